"""The launches around a decode step's layers (nq_decode_begin, nq_decode_end) against torch ops (needs a gfx950 GPU)."""
import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def lib():
    from nanoquant_amd import _lib
    return _lib.load()


@pytest.mark.parametrize("rows,n,ldx,offset", [(1, 32000, 32000, 0), (16, 4096, 4100, 0), (3, 1001, 1001, 0), (2, 8, 8, 1),
                                               (70, 36868, 36868, 0)])
def test_step_end(lib, rows, n, ldx, offset):
    """argmax (ties, a NaN, -inf), the token's place and the position, replayed in a graph to the end of the row and one
    step past it; ``offset``: logits off their 16-byte alignment."""
    from nanoquant_amd import _lib
    print("\n[case] step end", rows, n, ldx, offset, flush=True)
    L = 9
    g = torch.Generator(device="cuda").manual_seed(n)
    x = torch.randn(rows * ldx + offset, generator=g, device="cuda")[offset:].view(rows, ldx)
    x[:, n:] = 1e30
    x[0, n // 3] = x[0, n - 1] = x[0, :n].max() + 1.0
    if rows > 2:
        x[1, n // 2] = float("nan")
        x[2, :n] = float("-inf")
    tok, ids = torch.zeros(rows, dtype=torch.long, device="cuda"), torch.full((rows, L), -1, dtype=torch.long, device="cuda")
    pos, counter = torch.zeros(1, dtype=torch.long, device="cuda"), torch.zeros(1, dtype=torch.int32, device="cuda")

    def step():
        _lib.check(lib.nq_decode_end(x.data_ptr(), rows, n, ldx, tok.data_ptr(), ids.data_ptr(), L, pos.data_ptr(),
                                     counter.data_ptr(), _lib.stream_of(x.device)), "end")

    step()
    pos.fill_(4)
    ids.fill_(-1)
    torch.cuda.synchronize()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        step()
    want = torch.argmax(x[:, :n], dim=-1)
    for p in range(5, L + 1):
        graph.replay()
        torch.cuda.synchronize()
        assert torch.equal(tok, want) and int(pos) == p and int(counter) == 0
        if p < L:
            assert torch.equal(ids[:, p], want)
    assert bool((ids[:, :5] == -1).all())
    assert lib.nq_decode_end(x.data_ptr(), rows, n, n - 1, tok.data_ptr(), ids.data_ptr(), L, pos.data_ptr(),
                             counter.data_ptr(), None) == _lib.NQ_ERR_INVALID_ARGUMENT
    assert lib.nq_decode_end(x.data_ptr(), rows, n, ldx, tok.data_ptr(), ids.data_ptr(), L, pos.data_ptr(), None,
                             None) == _lib.NQ_ERR_INVALID_ARGUMENT


@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16], ids=["f16", "bf16"])
@pytest.mark.parametrize("batch,hidden,L,groups,rows,row", [(1, 4096, 100, 1, 4, 128), (3, 40, 33, 5, 7, 30),
                                                            (16, 8192, 65, 8, 0, 256), (2, 2056, 1, 1, 3, 1)])
def test_step_begin(lib, batch, hidden, L, groups, rows, row, dtype):
    from nanoquant_amd import _lib
    print("\n[case] step begin", batch, hidden, L, groups, rows, row, dtype, flush=True)
    vocab = 50
    embed, table = torch.randn(vocab, hidden, device="cuda").to(dtype), torch.randn(L, row, device="cuda").to(dtype)
    tok = torch.randint(0, vocab, (batch,), device="cuda")
    tok[-1] = vocab - 1
    for p in {0, L // 2, L - 1}:
        x = torch.full((batch + 1, hidden), 7.0, device="cuda", dtype=dtype)
        out = torch.full((row + 8,), 7.0, device="cuda", dtype=dtype)
        scores = torch.full((max(rows, 1) * L * groups + 8,), 7.0, device="cuda", dtype=dtype)
        pos = torch.tensor([p], device="cuda")

        def begin(with_embed, with_table, with_scores):
            _lib.check(lib.nq_decode_begin(
                _lib.dtype_code(dtype), embed.data_ptr() if with_embed else None, vocab, hidden, tok.data_ptr(), x.data_ptr(),
                batch, pos.data_ptr(), L, table.data_ptr() if with_table else None, row, out.data_ptr(),
                scores.data_ptr() if with_scores else None, rows, groups, _lib.stream_of(x.device)), "begin")
            torch.cuda.synchronize()

        begin(False, False, False)
        assert bool((x == 7).all() and (out == 7).all() and (scores == 7).all())
        begin(True, False, False)
        assert torch.equal(x[:batch], embed[tok]) and bool((x[batch] == 7).all() and (out == 7).all())
        begin(False, True, True)
        assert torch.equal(out[:row], table[p]) and bool((out[row:] == 7).all())
        want = torch.where(torch.arange(L, device="cuda") <= p, 0.0, float("-inf")).to(dtype)
        got = scores[:rows * L * groups].view(rows, L, groups)
        assert torch.equal(got, want.view(1, L, 1).expand_as(got)) and bool((scores[rows * L * groups:] == 7).all())
        x.fill_(0)
        begin(True, True, True)
        assert torch.equal(x[:batch], embed[tok])


@pytest.mark.parametrize("embed", [True, False], ids=["embed", "none"])
@pytest.mark.parametrize("table", [True, False], ids=["table", "none"])
def test_step_begin_reports(lib, embed, table):
    """Tokens and positions outside their ranges into pinned host words, the first and last good values not."""
    from nanoquant_amd import _lib
    print("\n[case] step begin reports", embed, table, flush=True)
    vocab, hidden, L, row, B = 50, 2056, 9, 16, 3
    weights, rows = torch.randn(vocab, hidden, device="cuda").half(), torch.randn(L, row, device="cuda").half()
    x, out = torch.zeros(B, hidden, device="cuda").half(), torch.zeros(row, device="cuda").half()
    fault = torch.zeros(2, dtype=torch.int32, pin_memory=True)
    for tokens, p, want in (([0, 49, 3], 0, (0, 0)), ([0, 49, 3], L - 2, (0, 0)), ([0, 50, 3], 1, (1, 0)),
                            ([0, 1, -1], 1, (1, 0)), ([0, 1, 2], L - 1, (0, 1)), ([0, 1, 2], -1, (0, 1)),
                            ([-5, 1, 2], 2 ** 40, (1, 1))):
        tok, pos = torch.tensor(tokens, device="cuda"), torch.tensor([p], device="cuda")
        fault.zero_()
        _lib.check(lib.nq_decode_begin_checked(
            _lib.NQ_F16, weights.data_ptr() if embed else None, vocab, hidden, tok.data_ptr(), x.data_ptr(), B,
            pos.data_ptr(), L, rows.data_ptr() if table else None, row, out.data_ptr(), None, 0, 1, fault.data_ptr(),
            _lib.stream_of(x.device)), "begin")
        torch.cuda.synchronize()
        assert fault.tolist() == [want[0] if embed else 0, want[1]], (tokens, p)
    assert lib.nq_decode_begin_checked(_lib.NQ_F16, None, vocab, hidden, None, None, B, pos.data_ptr(), L, None, 0, None,
                                       None, 0, 1, fault.data_ptr() + 1, None) == _lib.NQ_ERR_ALIGNMENT
