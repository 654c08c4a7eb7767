"""The drop-in boundary exercised the way the reference exercises it: libqtensor_hip.so loaded with a bare
ctypes handle, NO argtypes, pointers as c_void_p(tensor.data_ptr()), integers as c_int32, the null stream
(reference: qtensor/functional.py:17-60 binds the sixteen symbols, :68-84 get_ptr, :145-155, :193-211,
:251-282, :325-343 call them).  All sixteen are called on the device -- 4 and 8 bit, fp32 and bf16, plain
and with the exact diagonal, quantize and dequantize -- and compared bit for bit with the C oracle."""
import ctypes as ct
from pathlib import Path

import numpy as np
import pytest
import torch

import qtensor.functional as F
from oracle import quant_np as Q

pytestmark = pytest.mark.gpu
LIB = Path(__file__).resolve().parents[1] / "low-bit-shampoo_amd" / "qtensor" / "libqtensor_hip.so"


def get_ptr(t):
    return None if t is None else ct.c_void_p(t.data.data_ptr())


def bits_of(x):
    return np.ascontiguousarray(x, dtype=np.float32).view(np.uint32)


@pytest.mark.parametrize("order,blocksize", [(256, 64), (200, 128), (129, 64)])      # flat layout, ragged rows, odd order
@pytest.mark.parametrize("bits", [4, 8])
@pytest.mark.parametrize("dtype", ["fp32", "bf16"])
def test_sixteen_reference_symbols_bound_like_the_reference_binds_them(code_maps, order, blocksize, bits, dtype):
    assert torch.cuda.is_available()
    lib = ct.cdll.LoadLibrary(str(LIB))                    # what the reference's get_lib() returns
    code_np = code_maps[("linear-2", bits)]
    code = torch.from_numpy(code_np).cuda()
    g = torch.Generator().manual_seed(order * bits)
    A = torch.randn(order, order, generator=g)
    A[3, 3:40] = 0.0                                       # a zero stretch (a whole segment when blocksize is 64... or not)
    A[5, :blocksize] = 0.0                                 # an all-zero segment
    tdtype = torch.float32 if dtype == "fp32" else torch.bfloat16
    A_dev = A.cuda().to(tdtype).contiguous()
    A_host = A_dev.float().cpu().numpy()                   # what the kernel sees, exactly, as fp32
    nb = -(-order // blocksize)
    for diagreal in (False, True):
        mid = "_diagreal" if diagreal else ""
        absmax = torch.full((order * nb,), -1.0, device="cuda")
        diag = torch.full((order,), -1.0, device="cuda") if diagreal else None
        out = torch.zeros((order * order * bits + 7) // 8, dtype=torch.uint8, device="cuda")
        quan = getattr(lib, f"cquantize_blockwise{mid}_{bits}bit_{dtype}")
        args = [get_ptr(A_dev), get_ptr(code), ct.c_int32(order), get_ptr(absmax)] + ([get_ptr(diag)] if diagreal else [])
        quan(*args, get_ptr(out), ct.c_int32(blocksize))
        torch.cuda.synchronize()
        want = Q.quantize_c(A_host, code_np, order, blocksize, bits, diagreal)
        assert np.array_equal(out.cpu().numpy(), want[0]), (mid, "codes")
        assert np.array_equal(bits_of(absmax.cpu().numpy()), bits_of(want[1])), (mid, "absmax")
        if diagreal:
            assert np.array_equal(bits_of(diag.cpu().numpy()), bits_of(want[2])), (mid, "diag")
        back = torch.full((order, order), 7.0, dtype=tdtype, device="cuda")
        dequan = getattr(lib, f"cdequantize_blockwise{mid}_{bits}bit_{dtype}")
        args = [get_ptr(out), get_ptr(code), ct.c_int32(order), get_ptr(absmax)] + ([get_ptr(diag)] if diagreal else [])
        dequan(*args, get_ptr(back), ct.c_int32(blocksize))
        torch.cuda.synchronize()
        want_back = Q.dequantize_c(want[0], code_np, order, want[1], blocksize, bits, diag=want[2] if diagreal else None,
                                   to_bf16=dtype == "bf16")
        assert np.array_equal(bits_of(back.float().cpu().numpy()), bits_of(want_back)), (mid, "dequantized")


def test_pipe_switch_and_matrix_pipe_yardstick_through_the_bare_library():
    """The two entry points around the matrix pipes, called as a C program would: the process-wide switch
    (query, set, refuse) and the launch that is nothing but matrix instructions, whose rate must lie between a
    tenth of the published peak and the peak itself on either pipe."""
    lib = ct.cdll.LoadLibrary(str(LIB))
    lib.qtensor_hip_gemm_pipe.restype = ct.c_int
    lib.qtensor_hip_mfma_rate_flop.restype = ct.c_double
    lib.qtensor_hip_mfma_rate_flop.argtypes = [ct.c_int, ct.c_int, ct.c_int, ct.c_void_p, ct.c_void_p]
    lib.qtensor_hip_last_error.restype = ct.c_int
    before = lib.qtensor_hip_gemm_pipe(ct.c_int(-1))
    try:
        assert before in (0, 1)
        assert lib.qtensor_hip_gemm_pipe(ct.c_int(0)) == before and lib.qtensor_hip_gemm_pipe(ct.c_int(-1)) == 0
        assert lib.qtensor_hip_gemm_pipe(ct.c_int(1)) == 0 and lib.qtensor_hip_gemm_pipe(ct.c_int(-1)) == 1
        assert lib.qtensor_hip_gemm_pipe(ct.c_int(7)) == 1 and lib.qtensor_hip_last_error() != 0      # refused, unchanged
        assert lib.qtensor_hip_gemm_pipe(ct.c_int(-1)) == 1 and lib.qtensor_hip_last_error() == 0
    finally:
        lib.qtensor_hip_gemm_pipe(ct.c_int(before))
    sink = torch.zeros(1, device="cuda")
    stream = torch.cuda.current_stream().cuda_stream
    assert lib.qtensor_hip_mfma_rate_flop(2, 10, 1, sink.data_ptr(), stream) == 0.0 and lib.qtensor_hip_last_error() != 0
    assert lib.qtensor_hip_mfma_rate_flop(1, 0, 1, sink.data_ptr(), stream) == 0.0 and lib.qtensor_hip_last_error() != 0
    assert lib.qtensor_hip_mfma_rate_flop(1, 10, 1, None, stream) == 0.0 and lib.qtensor_hip_last_error() != 0
    for pipe, rounds, peak in ((1, 4000, 2500e12), (0, 1000, 157.3e12)):
        lib.qtensor_hip_mfma_rate_flop(pipe, rounds, 2, sink.data_ptr(), stream)              # warm-up
        e0, e1 = torch.cuda.Event(enable_timing=True), torch.cuda.Event(enable_timing=True)
        e0.record()
        flop = lib.qtensor_hip_mfma_rate_flop(pipe, rounds, 2, sink.data_ptr(), stream)
        e1.record()
        torch.cuda.synchronize()
        assert lib.qtensor_hip_last_error() == 0 and flop > 0
        rate = flop / (e0.elapsed_time(e1) * 1e-3)
        assert 0.1 * peak <= rate <= 1.02 * peak, (pipe, rate)
    assert float(sink[0]) == 0.0                                                              # the sink is never written


class _Subclass(torch.Tensor):
    pass


@pytest.mark.parametrize("bits,blocksize,order", [(4, 64, 1), (4, 64, 77), (8, 256, 256), (4, 2048, 130)])
@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("diag", [False, True])
def test_native_host_side_takes_the_good_calls_and_no_others(bits, blocksize, order, dtype, diag, monkeypatch):
    """The call with its host side in native code against the same call from Python, bit for bit: buffers made and buffers
    given, on a side stream; what is not plainly good is not taken and ends as it does from Python."""
    assert F._direct is not None
    taken = []
    native = F._direct

    class Spy:
        @staticmethod
        def quantize(*args):
            taken.append(native.quantize(*args))
            return taken[-1]

        @staticmethod
        def dequantize(*args):
            taken.append(native.dequantize(*args))
            return taken[-1]

    code = (F.create_linear_map(True, 4, 2) if bits == 4 else F.create_dynamic_map(True, 8, 1)).cuda()
    A = torch.randn(order, order, device="cuda").to(dtype)
    kw = dict(blocksize=blocksize, bits=bits)
    quantize, dequantize = ((F.quantize_blockwise_diagreal, F.dequantize_blockwise_diagreal) if diag else
                            (F.quantize_blockwise, F.dequantize_blockwise))

    def both(A, given=None, **more):
        made = quantize(A, code, order, **kw, **({} if given is None else given), **more)
        return made, dequantize(made[0], code, order, *made[1:], outdtype=dtype, **kw)

    monkeypatch.setattr(F, "_direct", None)
    want = both(A)
    monkeypatch.setattr(F, "_direct", Spy)
    got = both(A)
    given = dict(zip(("out", "absmax", "diag"), [torch.full_like(t, 7) for t in want[0]]))
    torch.cuda.synchronize()
    side = torch.cuda.Stream()
    with torch.cuda.stream(side):
        again = both(A, given)
    side.synchronize()
    assert len(taken) == 4 and all(t is not None for t in taken)
    assert all(a is b for a, b in zip(again[0], given.values()))
    for result in (got, again):
        assert all(torch.equal(a, b) and a.dtype == b.dtype and a.shape == b.shape for a, b in zip(result[0] + (result[1],), want[0] + (want[1],)))
    # not plainly good, but good: a subclass
    taken.clear()
    assert all(torch.equal(a, b) for a, b in zip(quantize(A.as_subclass(_Subclass), code, order, **kw), want[0]))
    # and not good
    wide = torch.randn(order, order + 1, device="cuda").to(dtype)
    for error, call in ((ValueError, lambda: quantize(wide, code, order, **kw)), (ValueError, lambda: quantize(A.double(), code, order, **kw)),
                        (ValueError, lambda: quantize(wide[:, 1:] if order > 1 else wide, code, order, **kw)),
                        (RuntimeError, lambda: quantize(A.cpu(), code, order, **kw)), (AssertionError, lambda: quantize(A, code, order, blocksize=65, bits=bits)),
                        (ValueError, lambda: quantize(A, code.cpu(), order, **kw)), (ValueError, lambda: quantize(A, code, order, out=A, **kw)),
                        (ValueError, lambda: dequantize(want[0][0], code, order, want[0][1][:0], *want[0][2:], **kw)),
                        (ValueError, lambda: dequantize(*([want[0][0], code, order] + list(want[0][1:])), outdtype=torch.float16, **kw))):
        with pytest.raises(error):
            call()
    assert len(taken) == 10 and all(t is None for t in taken)


def _inside(what, call):
    """What `call` returns, or the error it raises, with a transformation or a dispatch mode around it."""
    from torch.utils._python_dispatch import TorchDispatchMode
    seen = []

    def body(x):
        try:
            seen.append(call())
        except RuntimeError as error:
            seen.append(error)
        return (x * x).sum() if what == "grad" else x * x

    x = torch.ones(3, device="cuda")
    if what == "mode":
        class Mode(TorchDispatchMode):
            def __torch_dispatch__(self, func, types, args=(), kwargs=None):
                return func(*args, **(kwargs or {}))
        with Mode():
            body(x)
    elif what == "jvp":
        torch.func.jvp(body, (x,), (x,))
    elif what in ("vmap", "functionalize", "grad"):
        getattr(torch.func, what)(body)(x)
    else:
        torch.func.vjp(body, x)
    return seen[0]


@pytest.mark.parametrize("what", ["grad", "vjp", "jvp", "vmap", "functionalize", "mode"])
def test_calls_inside_a_transformation_or_mode_go_from_python(what, monkeypatch):
    """Plain tensors in, buffers to be made: what is made there may be a wrapper without memory.  The call ends as the one
    from Python does: the same error, the same tensors."""
    native, code = F._direct, F.create_linear_map(True, 4, 2).cuda()
    A = torch.randn(64, 64, device="cuda")
    codes, absmax = F.quantize_blockwise(A, code, 64, blocksize=64, bits=4)
    calls = (lambda: F.quantize_blockwise(A, code, 64, blocksize=64, bits=4),
             lambda: (F.dequantize_blockwise(codes, code, 64, absmax, blocksize=64, bits=4),))
    assert _inside(what, lambda: native.quantize(A, code, 64, None, None, None, 64, 4, False)) is None
    assert _inside(what, lambda: native.dequantize(codes, code, 64, absmax, None, torch.float32, None, 64, 4, False)) is None
    for call in calls:
        got = _inside(what, call)
        monkeypatch.setattr(F, "_direct", None)
        want = _inside(what, call)
        monkeypatch.setattr(F, "_direct", native)
        if isinstance(want, RuntimeError):
            assert isinstance(got, RuntimeError) and str(got) == str(want)
        else:
            assert all(torch.equal(a, b) for a, b in zip(got, want))
    assert what not in ("grad", "vjp", "jvp") or isinstance(want, RuntimeError)
