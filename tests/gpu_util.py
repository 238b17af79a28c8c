"""Helpers for GPU parity tests: numpy <-> device tensors, launch, oracle run."""

from __future__ import annotations

import ctypes
import re
import sys

import numpy as np

import oracle


def to_device(arr: np.ndarray, dtype: str, device):
    import torch

    if dtype == "bf16":
        t = torch.from_numpy(np.ascontiguousarray(arr).view(np.int16)).view(torch.bfloat16)
    else:
        t = torch.from_numpy(np.ascontiguousarray(arr))
    return t.to(device)


def to_host(t, dtype: str) -> np.ndarray:
    import torch

    t = t.detach().cpu()
    if dtype == "bf16":
        return t.view(torch.int16).numpy().view(np.uint16)
    return t.numpy()


def run_gpu(module, host_buffers, dtypes, device, func=None, case: str = "", kernels=None):
    """Copy buffers to the GPU, launch, synchronise, return host copies.  With
    `kernels`, the launch has to enqueue exactly these (kernels_of)."""
    import torch

    import xtile_amd as xt

    print(f"[gpu] {case}: {xt.plan(module, func)['kernel']}", flush=True)
    sys.stdout.flush()
    dev = [to_device(b, d, device) for b, d in zip(host_buffers, dtypes)]
    xt.launch(module, *dev, func=func)
    torch.cuda.synchronize()
    got = [to_host(t, d) for t, d in zip(dev, dtypes)]
    if kernels is not None:
        ran = kernels_of(module, dev, func)
        assert ran == kernels, ran
    return got


def kernels_of(module, buffers, func=None) -> list[str]:
    """The kernels a launch of `module` over these device buffers enqueues, as
    name<template arguments>, read from a graph that captures it."""
    import tempfile

    import torch

    import xtile_amd as xt

    xt.launch(module, *buffers, func=func)  # what a first launch loads stays out of the capture
    torch.cuda.synchronize()
    graph = torch.cuda.CUDAGraph(keep_graph=True)
    with torch.cuda.graph(graph):
        xt.launch(module, *buffers, func=func)
    hip = ctypes.CDLL(next(x.split()[-1] for x in open("/proc/self/maps") if "libamdhip64" in x))
    with tempfile.NamedTemporaryFile("r", suffix=".dot") as dot:
        assert hip.hipGraphDebugDotPrint(ctypes.c_void_p(graph.raw_cuda_graph()), dot.name.encode(), 1) == 0
        mangled = re.findall(r"(\w+)\\<\\<\\<", dot.read())
    names = []
    for name in mangled:  # a symbol of the library's, or a generated kernel's name
        m = re.search(r"_GLOBAL__N_1\d+([a-z]\w*?)(?:I((?:L[a-z]\d+E)+))?E", name)
        args = re.findall(r"L[a-z](\d+)E", m[2] or "") if m else []
        names.append((m[1] if m else name) + (f"<{', '.join(args)}>" if args else ""))
    return names


def run_oracle(module, host_buffers, nthreads: int):
    bufs = [np.array(b, copy=True) for b in host_buffers]
    oracle.run(str(module), bufs, nthreads)
    return bufs


def frob_rel(x: np.ndarray, ref: np.ndarray) -> float:
    x = np.asarray(x, dtype=np.float64)
    ref = np.asarray(ref, dtype=np.float64)
    return float(np.linalg.norm(x - ref) / max(np.linalg.norm(ref), 1e-300))
