"""A layer's Marlin words and scales in one launch (``nq_marlin_fused``) against the host packers (needs a gfx950 GPU)."""
import pytest
import torch

from nanoquant_amd.kernel import utils as ku

pytestmark = pytest.mark.gpu

# (n, r, m): one tile; a rank that is padded and fills its last words' tile partly; k and outputs past one block; a rank
# that needs no padding
SIZES = [(16, 32, 64), (272, 288, 64), (1040, 544, 192), (4112, 1120, 320), (512, 256, 1024)]


def _factors(n, r, m, seed=0):
    gen = torch.Generator().manual_seed(seed + n + r)
    sign = lambda *s: torch.randint(0, 2, s, dtype=torch.int8, generator=gen) * 2 - 1  # noqa: E731
    return sign(r, n), sign(m, r), [torch.randn(k, generator=gen).half() for k in (n, r, m)]


def _same(got, want):
    assert len(got) == len(want) == 6
    for a, b in zip(got, want):
        assert a.shape == b.shape and a.dtype == b.dtype and a.is_contiguous()
        assert torch.equal(a.cpu().view(torch.int16), b.view(torch.int16))


@pytest.mark.parametrize("sizes", SIZES, ids=lambda s: "x".join(map(str, s)))
def test_fused_packing(sizes, monkeypatch):
    print("\n[case] marlin fused", sizes, flush=True)
    V, U, scales = _factors(*sizes)
    want = ku.pack_binary_marlin_fused(V.T, U.T, *scales)
    on = [s.cuda() for s in scales]
    calls = []
    fused = ku._fused_on_gpu
    monkeypatch.setattr(ku, "_fused_on_gpu", lambda *a: calls.append(fused(*a)) or calls[-1])
    _same(ku.pack_binary_marlin_fused(V.cuda().T, U.cuda().T, *on), want)
    # factors laid out the other way, and as slices whose rows are further apart
    _same(ku.pack_binary_marlin_fused(V.cuda().T.contiguous(), U.cuda().T.contiguous(), *on), want)
    wide = torch.cat((V, V), 1).cuda()[:, :sizes[0]]
    _same(ku.pack_binary_marlin_fused(wide.T, U.cuda().T, *on), want)
    n, r, m = sizes
    for method in ("lsb_first", "half2"):
        Vp, Up = ku.pack_binary_gemv(V, method).cuda(), ku.pack_binary_gemv(U, method).cuda()
        if n % 32:  # bits past the last column are not the layer's
            Vp[:, -1] |= ku.pack_binary_gemv(torch.cat((torch.ones(1, n % 32), -torch.ones(1, 32 - n % 32)), 1).to(torch.int8),
                                             method).cuda()[0]
        _same(ku.pack_binary_marlin_fused_from_packed(Vp, (r, n), Up, (m, r), *on, method), want)
    assert len(calls) == 5 and all(c is not None for c in calls)


def test_fused_packing_other_calls(monkeypatch):
    """What the one launch does not take keeps the general route, errors included."""
    V, U, scales = _factors(272, 288, 64)
    want = ku.pack_binary_marlin_fused(V.T, U.T, *scales)
    V, U, scales = V.cuda(), U.cuda(), [s.cuda() for s in scales]
    shifted = torch.empty(V.numel() + 1, dtype=torch.int8, device="cuda")[1:].view_as(V)
    shifted.copy_(V)
    assert ku._fused_on_gpu(False, shifted, U, (272, 288, 64), 0, scales) is None
    wants16 = [t.clone() for t in (shifted, U)]
    _same(ku.pack_binary_marlin_fused(wants16[0].T, U.T, *scales), want)
    _same(ku.pack_binary_marlin_fused(V.float().T, U.float().T, *scales), want)  # other types of +-1
    with pytest.raises(RuntimeError, match="is invalid for input of size"):
        ku.pack_binary_marlin_fused(V[:270].T, U[:, :270].T, scales[0], scales[1][:270], scales[2])
    with pytest.raises(RuntimeError):
        ku.pack_binary_marlin_fused(V.T, U.T, scales[0], scales[1][:256], scales[2])
    with pytest.raises(TypeError, match="16-bit"):
        ku.pack_binary_marlin_fused(V.T, U.T, scales[0].float(), scales[1], scales[2])
    with pytest.raises(RuntimeError):
        ku.pack_binary_marlin_fused(V.T, U.T, scales[0].cpu(), scales[1], scales[2])
    with pytest.raises(ValueError, match="Unsupported method"):
        ku.pack_binary_marlin_fused_from_packed(ku.pack_binary_gemv(V), (288, 272), ku.pack_binary_gemv(U), (64, 288), *scales,
                                                "msb")
