"""Stage 2 of the decode GEMV with the rank split over a block's waves: its tiles' edges, singly against the float64
oracle, and the grouped epilogues against the single op (needs a gfx950 GPU)."""
import pytest
import torch

import oracle as O
from test_gpu_gemv_rows import BAR, _error, _oracle, _run
from test_gpu_group_batched import _entry, _group

pytestmark = pytest.mark.gpu

# (m, r, rows): one, two and four row tiles, four and eight waves, one, two and four column tiles; odd word counts,
# ragged ranks, outputs and last blocks of U that do not end on 16 bytes
SINGLES = [(8200, 3520, 8), (8191, 2219, 16), (4096, 4608, 9), (11003, 1100, 13), (10249, 2050, 12), (10250, 2050, 7),
           (27300, 3520, 2), (5003, 2300, 17), (4000, 4400, 30), (15999, 1000, 10)]
PAIRS = [(4096, 1632, 6), (11003, 1633, 3), (10249, 2050, 12), (27300, 3520, 2), (5003, 2300, 17), (10250, 2976, 32)]


@pytest.fixture(scope="module")
def lib():
    from nanoquant_amd import _lib
    return _lib.load()


@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16], ids=["f16", "bf16"])
@pytest.mark.parametrize("case", SINGLES, ids=lambda c: "x".join(map(str, c)))
def test_split_against_oracle(lib, case, dtype):
    m, r, rows = case
    print("\n[case] split", case, dtype, flush=True)
    c = O.random_case(m + rows, m, 256, r, rows, with_mid=True)
    y = _run(lib, c, dtype, offset=rows % 4)
    assert _error(y, _oracle(c, dtype), dtype) <= BAR  # the bar of the op, whichever kernels run
    assert torch.equal(y, _run(lib, c, dtype, offset=rows % 4)), "a second call over another workspace's bytes"


def _close(got, want, ulps, dtype, m):
    ulp = 2.0 ** (-10 if dtype == torch.float16 else -7)
    assert torch.equal(got[:, m:], torch.full_like(got[:, m:], 7.0))
    g, w = got[:, :m].float(), want.float()
    assert bool(((g - w).abs() <= ulps * ulp * torch.maximum(g.abs(), w.abs()) + 1e-6).all())


def _single(x, e):
    return torch.ops.binary_kernels.nanoquant_dyn_forward(x, e["s_in"], e["V"], e["s_mid"], e["U"], e["s_out"], 128, 128, 2, 2,
                                                          1, 1, 8, 8)


@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16], ids=["f16", "bf16"])
@pytest.mark.parametrize("case", PAIRS, ids=lambda c: "x".join(map(str, c)))
def test_split_pair_and_residual(lib, case, dtype):
    """The gated pair equals T(T(silu(gate)) * up) of the single ops, the residual T(resid + op): where the summation
    order differs it can move a rounding by one unit in the last place, and silu's and the product's add one each."""
    from nanoquant_amd import _lib
    m, r, rows = case
    print("\n[case] split pair", case, dtype, flush=True)
    x = torch.randn(rows, 256, device="cuda", generator=torch.Generator(device="cuda").manual_seed(m)).to(dtype)
    extra = rows % 3
    gate, up = (_entry(m + i, m, 256, r, dtype, extra, rows) for i in (0, 1))
    single = [_single(x, e) for e in (gate, up)]
    _group(lib, [gate, up], x, _lib.NQ_EPI_GATED, dtype)
    _close(gate["y"], torch.nn.functional.silu(single[0].float()).to(dtype) * single[1], 4, dtype, m)
    up["resid"] = up["y"] = torch.randn(rows, m + extra, device="cuda").to(dtype)  # in place
    up["y"][:, m:] = 7.0
    want = up["resid"][:, :m].float() + single[1].float()
    _group(lib, [up], x, _lib.NQ_EPI_RESIDUAL, dtype)
    ulp = 2.0 ** (-10 if dtype == torch.float16 else -7)
    assert bool(((up["y"][:, :m].float() - want).abs() <= ulp * (single[1].float().abs() + want.abs()) + 1e-6).all())


@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16], ids=["f16", "bf16"])
def test_split_group_of_unequal_items(lib, dtype):
    """Items too small for these kernels alone share the launch of the one that takes them: fewer rows, and ranks of one
    word (waves without a run) and of more words than its own."""
    from nanoquant_amd import _lib
    print("\n[case] split group", dtype, flush=True)
    x = torch.randn(16, 256, device="cuda").to(dtype)
    entries = [_entry(i, m, 256, r, dtype, 3, 16) for i, (m, r) in enumerate([(8192, 2240), (1025, 20), (500, 4600)])]
    single = [_single(x, e) for e in entries]
    _group(lib, entries, x, _lib.NQ_EPI_STORE, dtype)
    for e, want in zip(entries, single):
        _close(e["y"], want, 1, dtype, want.shape[1])
