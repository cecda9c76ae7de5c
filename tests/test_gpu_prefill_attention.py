"""Attention of a prompt on the KV cache (``nq_attention_prefill`` through ``rotary_attention``) against the torch
ops it replaces and float64 (needs a gfx950 GPU)."""
import math

import pytest
import torch

import nanoquant_amd.decode as decode
from nanoquant_amd.decode import LlamaShape, StaticKVCache, rotary_attention

pytestmark = pytest.mark.gpu

# (heads, kv_heads, batch, tokens, past): fewer rows than a wave's, one row past a block, one key past a tile,
# groups that do not divide a block, a chunk after a context, several blocks a head; keys shared by two groups of
# waves (few blocks of 768 tokens or more), with an odd number of tiles; more than one and two blocks a CU
CASES = [(4, 4, 1, 2, 0), (4, 4, 2, 33, 0), (8, 2, 2, 64, 1), (8, 1, 1, 129, 63), (6, 2, 3, 65, 64), (5, 1, 1, 300, 0),
         (2, 2, 1, 129, 511), (16, 2, 1, 700, 200), (2, 1, 1, 768, 0), (4, 2, 2, 800, 31), (1, 1, 1, 1025, 0), (16, 16, 2, 1030, 0),
         (16, 16, 4, 1030, 0)]


def _inputs(case, dtype, gap=37):
    heads, kv, batch, tokens, past = case
    gen = torch.Generator(device="cuda").manual_seed(tokens + past)
    draw = lambda *s: torch.randn(*s, device="cuda", generator=gen).to(dtype)  # noqa: E731
    shape = LlamaShape(hidden=heads * 128, layers=1, heads=heads, kv_heads=kv, ffn=256, vocab=64)
    cache = StaticKVCache(shape, batch, past + tokens + gap, "cuda", dtype)
    cache.k[0][:, :, :past].copy_(draw(batch, kv, past, 128))
    cache.v[0][:, :, :past].copy_(draw(batch, kv, past, 128))
    q, k, v = draw(batch, tokens, heads * 128), draw(batch, tokens, kv * 128), draw(batch, tokens, kv * 128)
    positions = torch.arange(past, past + tokens, device="cuda")
    inv = 1.0 / (10000.0 ** (torch.arange(0, 128, 2, device="cuda").float() / 128))
    angle = torch.cat((positions.float().view(-1, 1) * inv,) * 2, -1)
    return shape, q, k, v, angle.cos().to(dtype), angle.sin().to(dtype), positions, cache


def _exact(shape, q, k, v, cos, sin, positions, cache):
    rot = lambda t: torch.cat((-t[..., 64:], t[..., :64]), -1)  # noqa: E731
    split = lambda t: t.reshape(*t.shape[:2], -1, 128).transpose(1, 2).double()  # noqa: E731
    Q, K = (split(t) * cos.double() + rot(split(t)) * sin.double() for t in (q, k))
    kc, vc = cache.k[0].double(), cache.v[0].double()
    kc[:, :, positions], vc[:, :, positions] = K, split(v)
    hidden = torch.arange(kc.shape[2], device="cuda") > positions.view(-1, 1)
    group = shape.heads // shape.kv_heads
    s = Q.cpu() @ kc.repeat_interleave(group, 1).transpose(2, 3).contiguous().cpu() * 128 ** -0.5
    p = torch.softmax(s.masked_fill(hidden.cpu(), -math.inf), -1)
    return (p @ vc.repeat_interleave(group, 1).cpu()).transpose(1, 2).reshape(q.shape).cuda()


def _error(y, ref):
    return ((y.double() - ref).norm() / ref.norm()).item()


@pytest.fixture
def torch_ops(monkeypatch):
    def run(*args):
        with monkeypatch.context() as m:
            m.setattr(decode, "_prefill_kernel_takes", lambda *a: False)
            return rotary_attention(*args)
    return run


@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16], ids=["f16", "bf16"])
@pytest.mark.parametrize("case", CASES, ids=lambda c: "x".join(map(str, c)))
def test_prefill_attention(case, dtype, torch_ops):
    """The cache rows equal the torch path's bit for bit (the same roundings). The output rounds once less (its
    scores stay in float32), so its error against float64 is at most the torch path's, but for chance on few
    values: 1.1 times."""
    print("\n[case] prefill attention", case, dtype, flush=True)
    shape, q, k, v, cos, sin, pos, cache = args = _inputs(case, dtype)
    ref = _exact(*args)
    before = cache.k[0].clone(), cache.v[0].clone()
    assert decode._prefill_kernel_takes(shape, q, k, v, cos, sin, pos, cache.k[0], cache.v[0], cache.key_index)
    y = rotary_attention(shape, 0, q, k, v, cos, sin, pos, cache)
    after = cache.k[0].clone(), cache.v[0].clone()
    cache.k[0].copy_(before[0])
    cache.v[0].copy_(before[1])
    want = torch_ops(shape, 0, q, k, v, cos, sin, pos, cache)
    assert torch.equal(cache.k[0], after[0]) and torch.equal(cache.v[0], after[1])
    assert y.shape == want.shape and y.dtype == want.dtype and y.is_contiguous()
    assert _error(y, ref) <= 1.1 * _error(want, ref)


def test_prefill_attention_forms(torch_ops):
    """Forms the kernel takes beside a plain prompt: q, k and v as slices of one projection output, positions in any
    order, rows of the cache past the last position holding NaN."""
    shape, q, k, v, cos, sin, pos, cache = _inputs((8, 2, 1, 96, 20), torch.float16)
    qkv = torch.cat((q, k, v), -1)
    parts = qkv[..., :1024], qkv[..., 1024:1280], qkv[..., 1280:]
    order = torch.randperm(96, generator=torch.Generator().manual_seed(3)).cuda()
    args = (*(p[:, order] for p in (q, k, v)), cos[order], sin[order], pos[order])
    assert decode._prefill_kernel_takes(shape, *parts, cos, sin, pos, cache.k[0], cache.v[0], cache.key_index)
    y = rotary_attention(shape, 0, q, k, v, cos, sin, pos, cache)
    assert torch.equal(rotary_attention(shape, 0, *parts, cos, sin, pos, cache), y)
    # a row's sums depend on its block's tiles and mask only through its own keys
    assert torch.equal(rotary_attention(shape, 0, *args, cache), y[:, order])
    cache.k[0][:, :, 116:] = float("nan")
    cache.v[0][:, :, 116:] = float("nan")
    assert torch.equal(rotary_attention(shape, 0, q, k, v, cos, sin, pos, cache), y)


def test_prefill_attention_leaves_other_calls_to_torch(torch_ops):
    """Calls the kernel does not cover keep the torch ops: gradients, other strides and types, one token, a trace."""
    shape, q, k, v, cos, sin, pos, cache = _inputs((4, 4, 1, 40, 0), torch.float16)
    takes = lambda *a: decode._prefill_kernel_takes(shape, *a)  # noqa: E731
    tail = (cos, sin, pos, cache.k[0], cache.v[0], cache.key_index)
    assert takes(q, k, v, *tail)
    g = q.clone().requires_grad_()
    assert not takes(g, k, v, *tail)
    with torch.no_grad():
        assert takes(g, k, v, *tail)
    y = rotary_attention(shape, 0, g, k, v, cos, sin, pos, cache)
    assert y.requires_grad and torch.equal(y, torch_ops(shape, 0, q, k, v, cos, sin, pos, cache))
    assert not takes(q.float(), k.float(), v.float(), cos.float(), sin.float(), *tail[2:])
    assert not takes(q[:, :1], k[:, :1], v[:, :1], cos[:1], sin[:1], pos[:1], *tail[3:])
    assert not takes(q.transpose(1, 2).contiguous().transpose(1, 2), k, v, *tail)
    assert not takes(torch.empty(q.numel() + 4, dtype=q.dtype, device="cuda")[4:].view_as(q), k, v, *tail)
    assert not takes(q, k, v, cos, sin, pos.int(), *tail[3:])
    seen = []
    torch.func.vmap(lambda a: seen.append(takes(a, k, v, *tail)) or a)(q[None])
    with torch.autograd.forward_ad.dual_level():
        seen.append(takes(q, k, v, *tail))
    from torch._subclasses.fake_tensor import FakeTensorMode
    with FakeTensorMode(allow_non_fake_inputs=True):
        seen.append(takes(q, k, v, *tail))
    assert seen == [False, False, False]


@pytest.mark.parametrize("tokens", [70, 800])
@pytest.mark.parametrize("scale", [-0.09, 0.0, 3.0])
def test_prefill_attention_scales(scale, tokens):
    """Any factor of the scores, zero (the mean of the visible values) and negative ones too. P is rounded to float16
    (2^-11 of each term) and so is the output: the error stays below 2^-10 of the result's norm, but that a large
    factor makes the sum of rounded keys' errors count; the reference rounds them alike."""
    from nanoquant_amd import _lib
    shape, q, k, v, cos, sin, pos, cache = _inputs((2, 1, 1, tokens, 9), torch.float16)
    out = torch.empty_like(q)
    args = [t.data_ptr() for t in (cache.k[0], cache.v[0], cos, sin, pos, out)]
    _lib.check(_lib.load().nq_attention_prefill(
        _lib.NQ_F16, q.data_ptr(), 256, k.data_ptr(), 128, v.data_ptr(), 128, *args, 1, tokens, 2, 1, 128,
        cache.k[0].shape[2], scale, _lib.stream_of(q.device)), "prefill")
    split = q.view(1, tokens, 2, 128).transpose(1, 2)
    rot = (split * cos) + torch.cat((-split[..., 64:], split[..., :64]), -1) * sin  # rounded as the kernel rounds
    kc, vc = cache.k[0].double().cpu(), cache.v[0].double().cpu()
    s = rot.double().cpu() @ kc.repeat_interleave(2, 1).transpose(2, 3).contiguous() * scale
    hidden = torch.arange(kc.shape[2]) > pos.cpu().view(-1, 1)
    ref = torch.softmax(s.masked_fill(hidden, -math.inf), -1) @ vc.repeat_interleave(2, 1)
    assert _error(out.cpu(), ref.transpose(1, 2).reshape(1, tokens, 256)) <= 2 ** -10


def test_prefill_attention_argument_errors():
    from nanoquant_amd import _lib
    lib = _lib.load()

    def call(heads=4, kv=2, dim=128, stride=512, p=16):
        return lib.nq_attention_prefill(_lib.NQ_F16, p, stride, 16, 256, 16, 256, 16, 16, 16, 16, 16, 16, 1, 8, heads, kv,
                                        dim, 64, 0.1, None)

    assert call(dim=64) == _lib.NQ_ERR_UNSUPPORTED
    assert call(heads=3) == _lib.NQ_ERR_UNSUPPORTED
    assert call(stride=504) == _lib.NQ_ERR_SHAPE
    assert call(p=None) == _lib.NQ_ERR_INVALID_ARGUMENT
    assert call(p=24) == _lib.NQ_ERR_ALIGNMENT


# (heads, kv_heads, batch, tokens, past, gap): the shortest cache that is split, one tile a share and a short last one, a
# context of two tiles in a long cache (not shared), of six and seven tiles, a share that ends inside the tokens' own keys,
# groups, a second block of one row beside a full one, the last count of tokens, prompts
LONG_CASES = [(2, 2, 1, 2, 4094, 0), (2, 1, 2, 33, 5000, 99), (4, 4, 1, 2, 70, 5000), (4, 4, 1, 2, 382, 5000), (4, 4, 1, 2, 383, 5000),
              (4, 2, 1, 64, 4031, 1), (8, 1, 1, 5, 9001, 1), (43, 1, 1, 3, 5000, 0), (3, 3, 1, 64, 0, 5000), (6, 2, 1, 50, 350, 4000),
              (16, 16, 2, 2, 4500, 0)]


@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16], ids=["f16", "bf16"])
@pytest.mark.parametrize("case", LONG_CASES, ids=lambda c: "x".join(map(str, c)))
def test_prefill_attention_long_caches(case, dtype, torch_ops):
    """Keys shared over the grid: the same bars as above, the same value again and in a graph's replays."""
    from nanoquant_amd import _lib
    print("\n[case] prefill attention, long", case, dtype, flush=True)
    heads, kv, batch, tokens, past, gap = case
    shape, q, k, v, cos, sin, pos, cache = args = _inputs(case[:5], dtype, gap)
    assert _lib.load().nq_attention_prefill_workspace_bytes(batch, tokens, heads, kv, 128, past + tokens + gap) > 0
    ref = _exact(*args)
    run = lambda: rotary_attention(shape, 0, q, k, v, cos, sin, pos, cache)  # noqa: E731
    y = run()
    want = torch_ops(shape, 0, q, k, v, cos, sin, pos, cache)
    assert y.shape == want.shape and y.dtype == want.dtype and y.is_contiguous()
    assert _error(y, ref) <= 1.1 * _error(want, ref)
    assert torch.equal(run(), y)
    graph = torch.cuda.CUDAGraph()
    torch.cuda.synchronize()
    with torch.cuda.graph(graph):
        replayed = run()
    for _ in range(3):
        replayed.zero_()
        graph.replay()
        assert torch.equal(run(), y)
        torch.cuda.synchronize()
        assert torch.equal(replayed, y)


def test_prefill_attention_long_cache_edges():
    """With and without the shares: positions below 0 (NaN rows, no cache row), keys of NaN and infinity in one share, NaN
    past the last position, and a workspace that is too small."""
    from nanoquant_amd import _lib
    lib = _lib.load()
    shape, q, k, v, cos, sin, pos, cache = _inputs((4, 2, 1, 40, 4200), torch.float16, 60)
    L = cache.k[0].shape[2]
    need = lib.nq_attention_prefill_workspace_bytes(1, 40, 4, 2, 128, L)
    assert need > 0 and need % 16 == 0

    def call(nbytes):
        out = torch.empty_like(q)
        ws = torch.randint(0, 256, (max(nbytes, 16),), dtype=torch.uint8, device="cuda")
        _lib.check(lib.nq_attention_prefill_ws(
            _lib.NQ_F16, q.data_ptr(), 512, k.data_ptr(), 256, v.data_ptr(), 256, cache.k[0].data_ptr(), cache.v[0].data_ptr(),
            cos.data_ptr(), sin.data_ptr(), pos.data_ptr(), out.data_ptr(), 1, 40, 4, 2, 128, L, 0.088, ws.data_ptr(), nbytes,
            _lib.stream_of(q.device)), "prefill")
        return out

    def close(a, b):  # rounded once to float16, sums of another order: one unit of the row's largest value
        assert torch.equal(a.isnan(), b.isnan())
        torch.testing.assert_close(a, b, rtol=2e-3, atol=2e-4, equal_nan=True)

    cache.k[0][:, :, 4240:] = float("nan")
    cache.v[0][:, :, 4240:] = float("nan")
    plain = call(0)
    assert not plain.isnan().any() and torch.equal(call(need - 16), plain)
    close(call(need), plain)
    pos[3:5] = -1
    close(call(need), call(0))
    cache.k[0][0, 1, 700] = float("nan")
    close(call(need), call(0))
    cache.k[0][0, 1, 700] = 0
    cache.v[0][0, 0, 2000, 5] = float("inf")
    close(call(need), call(0))
    pos.fill_(-1)
    assert call(need).isnan().all()
    assert lib.nq_attention_prefill_workspace_bytes(1, 65, 4, 2, 128, L) == 0
    assert lib.nq_attention_prefill_workspace_bytes(1, 40, 4, 2, 128, 4095) == 0
