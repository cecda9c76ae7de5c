"""nq_dense_gemv of several batch rows on the matrix cores: its fragment counts, batch tiles and ragged
edges against float64 (needs a gfx950 GPU)."""
import numpy as np
import pytest
import torch

pytestmark = pytest.mark.gpu

CASES = [  # m, n, batch, ldy
    (15, 256, 3, 15),       # one fragment per wave, less than one row tile, the smallest batch
    (4113, 1024, 16, 4200),  # more row tiles than blocks, the last one of one row; output rows wider than m
    (1003, 2048, 17, 1003),  # two batch tiles, the second of one row
    (500, 3072, 33, 500),   # 12 fragments of 16, a second pass of one batch row
    (47, 1280, 4, 47),      # five fragments: the second stage of a wave holds one
    (77, 2816, 20, 80),     # eleven fragments, two batch tiles
    (333, 6144, 5, 333),    # an odd number of fragment groups
    (4100, 8192, 19, 4100),  # the widest rows; 16 batch rows a pass
]


def half_ulp(v, bits):
    _, e = np.frexp(np.abs(v))
    return np.ldexp(1.0, e - 1 - bits)


def call(w, x, g, y, batch, ldy):
    from nanoquant_amd import _lib
    (m, n), lib = w.shape, _lib.load()
    _lib.check(lib.nq_dense_gemv(_lib.dtype_code(w.dtype), w.data_ptr(), x.data_ptr(), _lib.ptr(g), 1e-5, y.data_ptr(),
                                 int(y.dtype == torch.float32), batch, n, m, ldy, _lib.stream_of(w.device)), "dense gemv")
    torch.cuda.synchronize()


@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16], ids=["f16", "bf16"])
@pytest.mark.parametrize("norm", [False, True], ids=["plain", "rmsnorm"])
@pytest.mark.parametrize("m,n,batch,ldy", CASES)
def test_dense_rows(m, n, batch, ldy, norm, dtype):
    """Each output within half a unit in the last place of the exact value, plus the fp32 sums' order: n <= 8192
    terms of about 0.15 each, 1e-5 of the largest output (measured below 2e-6). With the norm a rounded element
    of xn may fall on the other side of a tie (the mean's order): 5e-5."""
    print("\n[case] dense rows", dtype, (m, n, batch, ldy), norm, flush=True)
    gen = torch.Generator(device="cuda").manual_seed(m + n + batch)
    w = (torch.randn(m, n, device="cuda", generator=gen) * 0.05).to(dtype)
    x = (torch.randn(batch, n, device="cuda", generator=gen) * 3.0).to(dtype)
    g = (torch.rand(n, device="cuda", generator=gen) + 0.5).to(dtype) if norm else None
    y = torch.full((batch, ldy), 9.0, dtype=torch.float32 if norm else dtype, device="cuda")
    call(w, x, g, y, batch, ldy)
    xin = (g * torch.nn.functional.rms_norm(x.float(), (n,), eps=1e-5).to(dtype)) if norm else x
    ref = (xin.double().cpu() @ w.double().cpu().T).numpy()
    got = y[:, :m].double().cpu().numpy()
    bits = 11 if dtype == torch.float16 else 8
    allowed = np.maximum(half_ulp(ref, bits), half_ulp(got, bits))
    assert np.maximum(np.abs(got - ref) - allowed, 0.0).max() / np.abs(ref).max() <= (5e-5 if norm else 1e-5)
    if norm:
        assert torch.equal(y[:, :m].to(dtype).float(), y[:, :m])
    assert torch.equal(y[:, m:], torch.full_like(y[:, m:], 9.0))


def test_dense_rows_keep_infinities_and_nan_apart():
    """An infinite weight and a NaN input reach their own row and batch row only, rows past the batch nothing."""
    m, n, batch = 40, 512, 5
    w = torch.randn(m, n, device="cuda").half()
    x = torch.rand(batch, n, device="cuda").half() + 0.5
    clean = torch.empty(batch, m, dtype=torch.float16, device="cuda")
    call(w, x, None, clean, batch, m)
    w[7, 300] = float("inf")
    x[3, 41] = float("nan")
    y = torch.empty_like(clean)
    call(w, x, None, y, batch, m)
    assert y[3].isnan().all()
    keep = [b for b in range(batch) if b != 3]
    assert (y[keep, 7] == float("inf")).all()
    cols = [j for j in range(m) if j != 7]
    assert torch.equal(y[keep][:, cols], clean[keep][:, cols])
