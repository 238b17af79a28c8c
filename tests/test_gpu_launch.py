"""xt.launch: the native call takes the plain case; everything else reaches the
checked path, which launches it or raises the exception that names the fault."""

from __future__ import annotations

import pytest

import xtile_amd as xt
from xtile_amd import kernels as K

pytestmark = pytest.mark.gpu


def _buffers(cuda):
    import torch

    a, b = torch.rand(64, 128, device=cuda), torch.rand(64, 128, device=cuda)
    return a, b, torch.zeros(64, 128, device=cuda)


@pytest.mark.parametrize("how", ["plain", "func", "int", "object", "current", "subclass", "not built"])
def test_launches(cuda, monkeypatch, how):
    import torch

    m, (a, b, c) = K.add(64, 128), _buffers(cuda)
    side = torch.cuda.Stream()
    side.wait_stream(torch.cuda.current_stream())
    checked = []
    run = xt._launch_checked
    monkeypatch.setattr(xt, "_launch_checked", lambda *x: (checked.append(how), run(*x)))
    print(f"[gpu] launch {how}", flush=True)
    if how == "not built":  # what _load_launch returns then
        monkeypatch.setattr(xt, "_launch_native", lambda *_: False)
    if how == "func":
        xt.launch(m, a, b, c, func="add_kernel")
    elif how == "int":
        xt.launch(m, a, b, c, stream=side.cuda_stream)
    elif how == "object":
        xt.launch(m, a, b, c, stream=side)
    elif how == "current":
        with torch.cuda.stream(side):
            xt.launch(m, a, b, c)
    elif how == "subclass":
        class Wrapped(torch.Tensor):
            pass

        xt.launch(m, a.as_subclass(Wrapped), b, c)
    else:
        xt.launch(m, a, b, c)
    torch.cuda.synchronize()
    assert torch.equal(c, a + b)
    assert checked == ([how] if how in ("subclass", "not built") else [])


def test_refusals(cuda):
    import torch

    m, (a, b, c) = K.add(64, 128), _buffers(cuda)
    with pytest.raises(ValueError, match="takes 3 buffers, got 2"):
        xt.launch(m, a, b)
    with pytest.raises(TypeError, match="buffer 1 must be a torch.Tensor"):
        xt.launch(m, a, b.cpu().numpy(), c)
    with pytest.raises(ValueError, match="buffer 2 is not on a GPU"):
        xt.launch(m, a, b, c.cpu())
    with pytest.raises(TypeError, match="buffer 0 has dtype torch.float16; expected f32"):
        xt.launch(m, a.half(), b, c)
    with pytest.raises(ValueError, match=r"buffer 1 has shape \(128, 64\); expected \(64, 128\)"):
        xt.launch(m, a, b.reshape(128, 64), c)
    with pytest.raises(ValueError, match="buffer 0 must be contiguous"):
        xt.launch(m, torch.rand(128, 64, device=cuda).t(), b, c)
    with pytest.raises(NotImplementedError):
        xt.launch(K.add_rows(64, 128, 40), a, b, c)  # the last tile overruns
    with pytest.raises(TypeError, match="expected an xtile module object"):
        xt.launch(object(), a, b, c)
    with pytest.raises(RuntimeError):  # a batched tensor has no data of its own
        torch.func.vmap(lambda x: (xt.launch(m, x, b, c), x)[1])(torch.rand(2, 64, 128, device=cuda))
    torch.cuda.synchronize()
    assert not c.any()


def test_a_handle_is_known_by_its_type(cuda):
    """An object with an address for a module, and a capsule of the compiled
    binding while the ctypes one is in use, are refused by their type."""
    from xtile_amd import _compiled

    class Alike:
        _ptr = 16

    class Holder:
        _CAPIPtr = Alike()

    a, b, c = _buffers(cuda)
    for handle in (Alike(), Holder(), _compiled.load().parse(xt._wrap_module_asm(str(K.add(64, 128)))[0])):
        with pytest.raises(TypeError, match="expected an xtile module object"):
            xt.launch(handle, a, b, c)
    assert not c.any()


def test_a_pass_drops_the_plan(cuda):
    """The plan a launch used is not kept across a pass over its module."""
    import torch

    m, (a, b, c) = K.add(64, 128), _buffers(cuda)
    xt.launch(m, a, b, c)
    xt.xt_serialize(m)
    with pytest.raises((NotImplementedError, ValueError)):
        xt.launch(m, a, b, c)
    torch.cuda.synchronize()


def test_threads_on_one_module(cuda):
    """Threads that plan and launch one module at once, each on a stream of its
    own, through the native call (which holds no interpreter lock meanwhile)."""
    import threading

    import torch

    for _ in range(4):
        m = K.add(96, 640, 32, 64)  # planned by the first launch
        sets = [(torch.rand(96, 640, device=cuda), torch.rand(96, 640, device=cuda), torch.zeros(96, 640, device=cuda))
                for _ in range(8)]
        streams = [torch.cuda.Stream() for _ in sets]
        torch.cuda.synchronize()
        start, failed = threading.Barrier(len(sets)), []

        def work(bufs, stream):
            try:
                start.wait(timeout=30)
                with torch.cuda.stream(stream):
                    for _ in range(20):
                        xt.launch(m, *bufs)
                stream.synchronize()
            except Exception as exc:  # noqa: BLE001
                failed.append(exc)

        threads = [threading.Thread(target=work, args=x) for x in zip(sets, streams)]
        for t in threads:
            t.start()
        for t in threads:
            t.join(timeout=60)
        assert not failed and not any(t.is_alive() for t in threads)
        for a, b, c in sets:
            assert torch.equal(c, a + b)
