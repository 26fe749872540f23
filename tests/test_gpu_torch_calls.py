"""The C++ entry points on torch tensors (avelang_amd._torch_calls): a call they take gives what the Python wrapper gives
through ctypes, ``out`` comes back as the object that was passed, and what they do not take reaches the wrapper's checks."""
import ctypes.util
import threading
import time

import pytest
import torch

from avelang_amd import _lib, amdgpu_gemm_fp4 as api, moe
from tests import helpers as H

pytestmark = pytest.mark.gpu


class _Slow:
    def __getattr__(self, name):
        return lambda *args: None


def _calls(gpu, rows):
    mx = lambda r, k, seed: tuple(H.to_dev(x, gpu) for x in H.mx_operand(r, k, seed=seed))   # noqa: E731
    a, a_s = mx(rows, 1024, 1)
    w, w_s = mx(192, 1024, 2)
    e, e_s = (torch.stack(x).contiguous() for x in zip(mx(128, 1024, 3), mx(128, 1024, 4)))
    ro = torch.tensor([0, rows // 3, rows], dtype=torch.int32, device=gpu)
    x = torch.randn(rows, 1024, generator=torch.Generator().manual_seed(6)).to(gpu)
    g = (x.abs().max() / 2688).reshape(1)
    nv = api.quantize_nvfp4(x, g)
    logits = x[:, :8].contiguous()
    inv = torch.empty(rows, 2, dtype=torch.int32, device=gpu)
    _, _, weight = moe.moe_route_top2(logits, rows_of_token=inv)
    y = x.bfloat16().repeat(2, 1)
    idx = torch.arange(rows - 1, -1, -1, dtype=torch.int32, device=gpu)
    return {
        "gemm": lambda: api.gemm_mxfp4_transposed_b(a, a_s, w, w_s),
        "gemm variant": lambda: api.gemm_mxfp4_transposed_b(a, a_s, w, w_s, variant=_lib.GENERIC),
        "gemm fp4 dtypes": lambda: api.gemm_mxfp4_transposed_b(a.view(torch.float4_e2m1fn_x2), a_s.view(torch.float8_e8m0fnu), w, w_s),
        "nvfp4": lambda: api.gemm_nvfp4_transposed_b(*nv, g, *nv, g),
        "swiglu": lambda: api.gemm_mxfp4_swiglu_transposed_b(a, a_s, w, w_s),
        "swiglu quant": lambda: api.gemm_mxfp4_swiglu_quant_transposed_b(a, a_s, w, w_s),
        "swiglu quant padded": lambda: api.gemm_mxfp4_swiglu_quant_transposed_b(a, a_s, w, w_s, n_pad=128),
        "grouped": lambda: api.grouped_gemm_mxfp4_transposed_b(a, a_s, e, e_s, ro),
        "grouped swiglu": lambda: api.grouped_gemm_mxfp4_swiglu_transposed_b(a, a_s, e, e_s, ro),
        "grouped swiglu quant": lambda: api.grouped_gemm_mxfp4_swiglu_quant_transposed_b(a, a_s, e, e_s, ro),
        "quantize f32": lambda: api.quantize_mxfp4(x),
        "quantize bf16 padded": lambda: api.quantize_mxfp4(x.bfloat16(), k_pad=1536),
        "quantize nv": lambda: api.quantize_nvfp4(x.bfloat16(), g),
        "route": lambda: moe.moe_route_top2(logits),
        "combine": lambda: moe.moe_combine_top2(y, inv, weight, renormalize=True),
        "gather": lambda: moe.gather_rows_mxfp4(a, a_s, idx),
    }


@pytest.mark.parametrize("rows", [1, 130])
def test_same_results_as_through_the_wrapper(gpu, rows, monkeypatch):
    calls = _calls(gpu, rows)
    native = {k: f() for k, f in calls.items()}
    monkeypatch.setattr(api, "_native", _Slow())
    monkeypatch.setattr(moe, "_native", _Slow())
    for name, f in calls.items():
        want, got = f(), native[name]
        want, got = (x if isinstance(x, tuple) else (x,) for x in (want, got))
        assert type(got) is type(want) and len(got) == len(want), name
        for u, v in zip(got, want):
            assert u.dtype == v.dtype and u.device == v.device and torch.equal(u.view(torch.uint8), v.view(torch.uint8)), name


def test_out_is_returned_and_wrong_arguments_reach_the_checks(gpu):
    a, a_s, w, w_s = (H.to_dev(t, gpu) for t in (*H.mx_operand(16, 512, seed=1), *H.mx_operand(64, 512, seed=2)))
    out = torch.empty(16, 64, dtype=torch.bfloat16, device=gpu)
    assert api._native.gemm_mxfp4(a, a_s, w, w_s, out, 0, True) is out
    for bad in (out.float(), out[:, :32], out.cpu(), out.t().contiguous().t()):
        assert api._native.gemm_mxfp4(a, a_s, w, w_s, bad, 0, True) is None
        with pytest.raises(ValueError, match="out must"):
            api.gemm_mxfp4_transposed_b(a, a_s, w, w_s, bad)
    for bad in (a.int(), a[:, :8], a.t().contiguous().t(), None, 3, a.cpu()):
        assert api._native.gemm_mxfp4(bad, a_s, w, w_s, None, 0, True) is None
    with pytest.raises(ValueError, match="unknown kernel variant 99"):
        api.gemm_mxfp4_transposed_b(a, a_s, w, w_s, variant=99)
    with pytest.raises(TypeError, match="7 arguments expected, got 1"):
        api._native.gemm_mxfp4(a)


@pytest.mark.parametrize("n_pad", [None, 128])   # (padded results are allocated and cleared)
def test_other_threads_run_while_memory_is_allocated(gpu, n_pad):
    """A pool whose driver allocation is usleep: it takes as many microseconds as bytes are asked for (2 MB, a few tries) and hands out
    nothing.  Another Python thread counts on meanwhile; with the interpreter's lock held it would stand still."""
    a, a_s, w, w_s = (H.to_dev(t, gpu) for t in (*H.mx_operand(16, 512, seed=1), *H.mx_operand(64, 512, seed=2)))
    slow = torch.cuda.memory.CUDAPluggableAllocator(ctypes.util.find_library("c"), "usleep", "abs")
    pool = torch.cuda.MemPool(slow.allocator())
    stop, ticks = threading.Event(), [0]

    def count():
        while not stop.wait(0.01):
            ticks[0] += 1

    thread = threading.Thread(target=count)
    thread.start()
    try:
        start = time.monotonic()
        with torch.cuda.use_mem_pool(pool), pytest.raises(torch.OutOfMemoryError):
            ticks[0] = 0
            if api._native.gemm_mxfp4_swiglu_quant(a, a_s, w, w_s, None, None, n_pad) is not None:
                raise AssertionError("the pool had memory")
        counted, seconds = ticks[0], time.monotonic() - start
    finally:
        stop.set()
        thread.join()
    assert seconds > 1.0, seconds
    assert counted > 20 * seconds, (counted, seconds)   # 100 a second when nothing holds it up
