"""The RMS norm and silu(gate) * up launches of a decoder layer against the torch ops they replace (needs a gfx950
GPU)."""
import pytest
import torch
import torch.nn.functional as F

import nanoquant_amd.decode as decode
from nanoquant_amd.decode import RMSNorm, silu_mul

pytestmark = pytest.mark.gpu
DTYPES = pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16], ids=["f16", "bf16"])


def _ulps(a, b, dtype):
    """The largest difference in units in the last place of the larger value's binade."""
    a, b = a.double(), b.double()
    bits = 10 if dtype == torch.float16 else 7
    unit = torch.exp2(torch.floor(torch.log2(torch.maximum(a.abs(), b.abs()).clamp_min(2.0 ** -14))) - bits)
    return ((a - b).abs() / unit).max().item()


@DTYPES
@pytest.mark.parametrize("shape", [(1, 8), (3, 2040), (5, 2048), (2, 7, 2056), (1, 4096), (300, 8192), (2, 16384)])
def test_rms_norm(shape, dtype):
    """The mean's summation order can move each of the two roundings to its neighbour: two units in the last place."""
    print("\n[case] rms norm", shape, dtype, flush=True)
    gen = torch.Generator(device="cuda").manual_seed(shape[-1])
    x = (torch.randn(shape, device="cuda", generator=gen) * 3).to(dtype)
    norm = RMSNorm(shape[-1], 1e-5, "cuda", dtype)
    norm.weight.data.copy_(torch.rand(shape[-1], device="cuda", generator=gen) + 0.5)
    assert decode._pointwise_kernel_takes(x, norm.weight)
    y = norm(x)
    want = norm.weight * F.rms_norm(x.float(), (shape[-1],), eps=1e-5).to(dtype)
    assert y.shape == want.shape and y.dtype == dtype and _ulps(y, want, dtype) <= 2.0
    x[0, ..., 3] = float("nan")
    assert norm(x)[0].isnan().any() and torch.equal(norm(x)[1:], y[1:])


@DTYPES
@pytest.mark.parametrize("shape", [(8,), (3, 264), (2, 5, 11008)])
def test_silu_mul(shape, dtype):
    """exp's last bit can move silu's rounding to its neighbour, and the product follows it: two units in the last
    place. Infinities and NaN as torch's."""
    print("\n[case] silu mul", shape, dtype, flush=True)
    gen = torch.Generator(device="cuda").manual_seed(shape[-1])
    gate, up = ((torch.randn(shape, device="cuda", generator=gen) * 4).to(dtype) for _ in range(2))
    assert decode._pointwise_kernel_takes(gate, up)
    assert _ulps(silu_mul(gate, up), F.silu(gate) * up, dtype) <= 2.0
    gate.view(-1)[:5] = torch.tensor([float("inf"), float("-inf"), float("nan"), -200.0, 60000.0], device="cuda")
    torch.testing.assert_close(silu_mul(gate, up).view(-1)[:5], (F.silu(gate) * up).view(-1)[:5], rtol=0, atol=0,
                               equal_nan=True)


def test_other_forms_keep_torch_ops():
    x = torch.randn(4, 64, device="cuda").half()
    norm = RMSNorm(64, 1e-5, "cuda", torch.float16)
    for form in (x.float(), x.t().contiguous().t(), torch.randn(4, 63, device="cuda").half(), x[:0],
                 torch.empty(260, device="cuda").half()[1:257].view(4, 64), x.clone().requires_grad_()):
        assert not decode._pointwise_kernel_takes(form, form)
    wide = RMSNorm(16392, 1e-5, "cuda", torch.float16)
    assert wide(torch.ones(2, 16392, device="cuda").half()).shape == (2, 16392)
    g = x.clone().requires_grad_()
    assert norm(g).requires_grad and silu_mul(g, x).requires_grad
    assert torch.equal(norm(x.t().contiguous().t()), norm.weight * F.rms_norm(x.float(), (64,), eps=1e-5).half())
    out = torch.func.vmap(lambda a: silu_mul(a, a))(x)
    assert torch.equal(out, F.silu(x) * x)
    assert silu_mul(x[:, :1], x).shape == (4, 64)  # torch's broadcasting


@DTYPES
@pytest.mark.parametrize("shape", [(3, 2040), (300, 8192), (2, 16384)])
def test_in_place(shape, dtype):
    """The C functions with their output in an input's place: bit for bit what they give elsewhere."""
    from nanoquant_amd import _lib
    print("\n[case] pointwise in place", shape, dtype, flush=True)
    lib, dt = _lib.load(), _lib.dtype_code(dtype)
    a, b = (torch.randn(shape, device="cuda").to(dtype) for _ in range(2))
    norm = RMSNorm(shape[-1], 1e-5, "cuda", dtype)
    want = norm(a)
    y = a.clone()
    _lib.check(lib.nq_rms_norm(dt, y.data_ptr(), norm.weight.data_ptr(), y.data_ptr(), shape[0], shape[1], 1e-5,
                               _lib.stream_of(y.device)), "rms_norm")
    assert torch.equal(y, want)
    want = silu_mul(a, b)
    for k in range(2):
        pair = [a.clone(), b.clone()]
        _lib.check(lib.nq_silu_mul(dt, pair[0].data_ptr(), pair[1].data_ptr(), pair[k].data_ptr(), a.numel(),
                                   _lib.stream_of(a.device)), "silu_mul")
        assert torch.equal(pair[k], want)


def test_small_calls_cost_no_more_than_torch_ops():
    """A call of one token, bound by its host path, against the two torch launches it replaces (it took 1.2 times their
    time); on a side stream too."""
    import time
    print("\n[case] pointwise, small calls", flush=True)
    x, u = (torch.randn(1, 1, 4096, device="cuda").half() for _ in range(2))

    def us(fn):
        best = float("inf")
        for _ in range(8):
            torch.cuda.synchronize()
            start = time.perf_counter()
            for _ in range(400):
                fn()
            torch.cuda.synchronize()
            best = min(best, (time.perf_counter() - start) / 400 * 1e6)
        return best

    with torch.no_grad():
        mine, theirs = us(lambda: silu_mul(x, u)), us(lambda: F.silu(x) * u)
    assert mine < 1.1 * theirs, (mine, theirs)
    want, stream = silu_mul(x, u), torch.cuda.Stream()
    stream.wait_stream(torch.cuda.current_stream())
    with torch.cuda.stream(stream):
        a = x
        for _ in range(20):
            a = a * 1
        got = silu_mul(a, u)
    torch.cuda.current_stream().wait_stream(stream)
    assert torch.equal(got, want)
