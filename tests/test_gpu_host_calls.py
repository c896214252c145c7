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


def _linear(gpu_device, M, N=2048, K=2048, seed=0):
    from kb_nano_amd.fp8_linear import _block_requant
    g = torch.Generator(device=gpu_device).manual_seed(seed + M)
    w, ws = _block_requant(torch.randn(N, K, device=gpu_device, generator=g) * 0.02, True)
    x = torch.randn(M, K, device=gpu_device, generator=g).to(BF16)
    lin = Fp8Linear()
    lin._ensure_buffers(M, K, N, gpu_device)
    return lin, x, w, ws


# weights whose plan splits K, by the row count: summed in the split launch, and by a launch of its own
_SPLIT = {16: (2048, 2048), 100: (512, 7168)}


def _native(lin, x, w, ws):
    from kb_nano_amd.fp8_linear import is_e8m0_used
    return _ops._host.linear(x, w, ws, lin._a_buf, lin._s_buf, lin._o_buf, lin._pf, is_e8m0_used(), _ops._WS_BUFS)


@pytest.mark.parametrize("M", [16, 100])
def test_linear_on_side_streams_and_threads(gpu_device, M):
    """Each stream has its own split workspace; a side stream, and two threads
    on streams of their own at once, give the default stream's bits."""
    import threading
    N, K = _SPLIT[M]
    lin, x, w, ws = _linear(gpu_device, M, N, K)
    assert (_ops.lib().kbn_fp8_gemm_nt_workspace_bytes(M, N, K, 1) if M > 64 else
            _ops.lib().kbn_fp8_gemm_bf16a_workspace_bytes(M, N, K)) > 0
    ref = lin(x, w, ws).clone()
    torch.cuda.synchronize()
    got, errors = {}, []

    def work(name):
        try:
            mine = Fp8Linear()
            mine._ensure_buffers(M, K, N, gpu_device)
            stream = torch.cuda.Stream()
            with torch.cuda.stream(stream):
                first = mine(x, w, ws).clone()         # this stream's workspace is made by the Python path
                assert (0, stream.cuda_stream) in _ops._WS_BUFS
                for _ in range(20):
                    out = mine(x, w, ws)
                assert _native(mine, x, w, ws) is not None
                got[name] = [first, out.clone()]
            stream.synchronize()
        except BaseException as e:                     # an assertion of a thread fails the test below
            errors.append(e)
    work("side stream")
    threads = [threading.Thread(target=work, args=(i,)) for i in range(2)]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    assert not errors, errors
    assert len(got) == 3
    for outs in got.values():
        for out in outs:
            assert torch.equal(out, ref)


@pytest.mark.parametrize("M", [16, 100])
def test_linear_with_a_kept_workspace_that_is_too_small(gpu_device, M):
    lin, x, w, ws = _linear(gpu_device, M, *_SPLIT[M])
    ref = lin(x, w, ws).clone()
    key = (0, torch.cuda.current_stream().cuda_stream)
    full = _ops._WS_BUFS[key]
    _ops._WS_BUFS[key] = small = torch.empty(64, dtype=torch.uint8, device=gpu_device)
    lin._o_buf.fill_(float("nan"))
    assert _native(lin, x, w, ws) is None
    assert torch.equal(lin(x, w, ws), ref)             # the Python path makes a larger one
    assert _ops._WS_BUFS[key] is not small and _native(lin, x, w, ws) is not None
    _ops._WS_BUFS[key] = full


@pytest.mark.parametrize("M", [16, 100])
def test_linear_refusals_are_the_python_path_s(gpu_device, M):
    """What the entry points refuse, the step leaves to the Python path, which raises."""
    lin, x, w, ws = _linear(gpu_device, M)
    lin(x, w, ws)   # the split workspace of this stream exists afterwards
    assert _native(lin, x, w, ws) is not None
    flat = torch.zeros(M * 2048 + 8, device=gpu_device, dtype=BF16)
    cases = {
        "misaligned rows": (flat[1:1 + M * 2048].view(M, 2048), w, ws),
        "row stride": (torch.zeros(M, 2049, device=gpu_device, dtype=BF16)[:, :2048], w, ws),
        "too few scale rows": (x, w, ws[:8]),
        "scales not along K": (x, w, ws.t().contiguous().t()),
        "fp16 weight": (x, w.to(torch.float16), ws),
    }
    for name, args in cases.items():
        assert _native(lin, *args) is None, name
        with pytest.raises((RuntimeError, ValueError, TypeError)):
            lin(*args)
    assert torch.equal(lin(x, w, ws), lin(x.clone(), w, ws))


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
