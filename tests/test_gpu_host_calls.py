"""The native host path of the small calls (csrc/host_calls.cpp) against the
Python path it stands for: the same bytes, and None (so the Python path) for
everything but the plain case."""
import ctypes

import pytest
import torch

from kb_nano_amd import Fp8Linear, FusedAddRMSNormFP8Quant, RMSNormFP8Quant, SiluMulQuantFp8, _ops

pytestmark = pytest.mark.gpu
BF16 = torch.bfloat16


def _both(monkeypatch, call):
    """call() through the native path, then through the Python path."""
    assert _ops._host is not None, "csrc/host_calls.cpp is not built"
    a = call()
    monkeypatch.setattr(_ops, "_host", None)
    b = call()
    monkeypatch.undo()
    return a, b


def _same(a, b):
    for x, y in zip(a, b, strict=True):
        assert x.dtype == y.dtype and x.shape == y.shape and x.stride() == y.stride()
        assert torch.equal(x.reshape(-1).view(torch.uint8), y.reshape(-1).view(torch.uint8))


@pytest.mark.parametrize("shape", [(1, 128), (61, 8192), (3, 7, 2048), (130, 200)])
@pytest.mark.parametrize("add", [False, True])
def test_norm_same_as_python_path(gpu_device, monkeypatch, shape, add):
    g = torch.Generator(device=gpu_device).manual_seed(sum(shape))
    x, r = (torch.randn(shape, device=gpu_device, generator=g).to(BF16) for _ in range(2))
    w = torch.randn(shape[-1], device=gpu_device, generator=g).to(BF16)

    def call():
        xx, rr = x.clone(), r.clone()
        if not add:
            return RMSNormFP8Quant()(xx, w)
        q, s, res = FusedAddRMSNormFP8Quant()(xx, rr, w)
        assert res is rr
        return q, s, rr, xx
    _same(*_both(monkeypatch, call))


@pytest.mark.parametrize("M,I,ue8m0", [(128, 128, True), (128, 2304, True), (256, 1024, False)])
def test_silu_same_as_python_path(gpu_device, monkeypatch, M, I, ue8m0):
    g = torch.Generator(device=gpu_device).manual_seed(I)
    x = torch.randn(M, 2 * I + 64, device=gpu_device, generator=g).to(BF16)[:, :2 * I]
    _same(*_both(monkeypatch, lambda: SiluMulQuantFp8()(x, use_ue8m0=ue8m0)))


@pytest.mark.parametrize("M", [1, 16, 40, 64, 65, 200, 300])
def test_linear_same_as_python_path(gpu_device, monkeypatch, M):
    """Decode buffers of 64 rows, prefill buffers of 256 and none beyond; the
    output is a view of the buffer the Python path writes; row strides."""
    from kb_nano_amd.fp8_linear import _Fp8PrefillBufs, _block_requant
    N, K = 2048, 2048
    g = torch.Generator(device=gpu_device).manual_seed(M)
    w, ws = _block_requant(torch.randn(N, K, device=gpu_device, generator=g) * 0.02, True)
    x = torch.randn(M, K + 128, device=gpu_device, generator=g).to(BF16)[:, :K]
    lin = Fp8Linear()
    lin._ensure_buffers(64, K, N, gpu_device)
    lin._pf = _Fp8PrefillBufs(256, K, N, gpu_device)
    bias = torch.randn(N, device=gpu_device, generator=g).to(BF16)

    def call():
        out = lin(x, w, ws)
        want = lin._o_buf if M <= 64 else lin._pf.o if M <= 256 else out
        assert out.shape == (M, N) and out.data_ptr() == want.data_ptr()
        return out.clone(), lin(x, w, ws, bias)
    call()   # the split workspace of this stream exists afterwards
    _same(*_both(monkeypatch, call))


def test_anything_but_the_plain_case_is_left_to_python(gpu_device):
    h = _ops._host
    x, w = torch.zeros(4, 256, device=gpu_device, dtype=BF16), torch.zeros(256, device=gpu_device, dtype=BF16)
    assert h.norm(x, w, 1e-6, None) is not None
    for bad in (x.cpu(), x.float(), x.t(), x[:0], x.view(torch.int16), [1.0], None):
        assert h.norm(bad, w, 1e-6, None) is None
    assert h.norm(x, w[:128], 1e-6, None) is None and h.norm(x, w, 1, None) is None
    assert h.norm(x, w, 1e-6, x[:2]) is None

    class Sub(torch.Tensor):
        pass
    assert h.norm(x.as_subclass(Sub), w, 1e-6, None) is None
    from torch.overrides import TorchFunctionMode
    from torch.utils._python_dispatch import TorchDispatchMode
    with TorchFunctionMode():
        assert h.norm(x, w, 1e-6, None) is None
    with TorchDispatchMode():
        assert h.norm(x, w, 1e-6, None) is None
    seen = []
    torch.func.vmap(lambda t: (seen.append(h.norm(x, w, 1e-6, None)), t)[1])(x)
    assert seen == [None]
    g = torch.cuda.CUDAGraph()
    with torch.cuda.graph(g):
        assert h.norm(x, w, 1e-6, None) is None
    assert h.norm(x, w, 1e-6, None) is not None
    y = torch.zeros(128, 512, device=gpu_device, dtype=BF16)
    assert h.silu(y, True, 1e-10) is not None
    assert h.silu(y[:100], True, 1e-10) is None and h.silu(y[:, :500], True, 1e-10) is None
    # shapes and types the Python path refuses still raise
    with pytest.raises((TypeError, ValueError)):
        RMSNormFP8Quant()(x, w[:128])
    with pytest.raises(AssertionError):
        SiluMulQuantFp8()(y[:100])


def _leave_an_error():
    """An error of an earlier runtime call on this thread, still unread: a
    device index that does not exist, refused by the runtime on the host."""
    with open("/proc/self/maps") as f:
        hip = next(line.split()[-1] for line in f if "libamdhip64" in line)
    assert ctypes.CDLL(hip).hipSetDevice(9999) != 0


@pytest.mark.parametrize("native", [True, False])
def test_a_pending_error_does_not_repeat_the_call(gpu_device, monkeypatch, native):
    """An error left pending is reported after the launch: the call raises, as
    the Python path does, and the operands were updated once, not twice."""
    from kb_nano_amd._lib import KbnError
    g = torch.Generator(device=gpu_device).manual_seed(3)
    x, r = (torch.randn(61, 2048, device=gpu_device, generator=g).to(BF16) for _ in range(2))
    w = torch.randn(2048, device=gpu_device, generator=g).to(BF16)
    x1, r1 = x.clone(), r.clone()
    FusedAddRMSNormFP8Quant()(x1, r1, w)
    torch.cuda.synchronize()
    if not native:
        monkeypatch.setattr(_ops, "_host", None)
    _leave_an_error()
    with pytest.raises(KbnError, match="launch failed"):
        FusedAddRMSNormFP8Quant()(x, r, w)
    torch.cuda.synchronize()
    assert torch.equal(r, r1) and torch.equal(x, x1)


def test_a_flag_without_a_truth_value(gpu_device):
    """``use_ue8m0`` may be any object; the error its truth value raises comes out as it is."""
    class Bad:
        def __bool__(self):
            raise ZeroDivisionError("no truth value")
    x = torch.ones(128, 512, device=gpu_device, dtype=BF16)
    with pytest.raises(ZeroDivisionError, match="no truth value"):
        SiluMulQuantFp8()(x, use_ue8m0=Bad())
    _same(SiluMulQuantFp8()(x, use_ue8m0=[]), SiluMulQuantFp8()(x, use_ue8m0=False))


def test_an_exception_inside_the_step_is_left_to_python(gpu_device):
    """Reading a tensor's address may throw in C++, and does so while the step
    holds no GIL: the step takes it again and the Python path reports the error."""
    x = torch.ones(61, 2048, device=gpu_device, dtype=BF16)
    w = torch.ones(2048, device=gpu_device, dtype=BF16)
    y = x.clone()
    torch._C._set_throw_on_mutable_data_ptr(y)
    assert _ops._host.norm(y, w, 1e-6, None) is None
    with pytest.raises(RuntimeError, match="data pointer"):
        RMSNormFP8Quant()(y, w)
    _same(RMSNormFP8Quant()(x, w), RMSNormFP8Quant()(x.clone(), w))
