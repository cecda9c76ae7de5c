"""The decode GEMV of many batch rows (the kernels that share each decoded sign over 64 batch rows):
edges of its tiles, k ranges and k groups against the float64 oracle (needs a gfx950 GPU)."""
import numpy as np
import pytest
import torch

import oracle as O

pytestmark = pytest.mark.gpu

# An fp16 output is rounded by at most 2^-11 of itself; the intermediate (a bf16 pair, 2^-17) and the fp32
# sums over r and n of at most 2^13 terms stay below 1e-4 of the largest output. A bf16 output's own
# rounding is counted apart (half a unit in the last place).
BAR = 2.0 ** -11 + 1e-4

# (m, n, r, rows, s_mid): narrow inputs run from 129 rows, 256-511 words from 64, 512 words or more from 33, but for
# a small V (the k-split kernel, up to 96 rows) and where one round of the 16-row MFMA kernel does
CASES = [
    (300, 8192, 3200, 64, True),      # the first batch on 256 words; ragged outputs, k ranges
    (64, 16384, 2750, 33, True),      # the first batch on 512 words; a ragged rank
    (64, 16392, 1, 33, True),         # a rank of 1
    (1000, 12296, 130, 65, False),    # n % 64 == 8: the tail tile's first quarter; a second row tile of one row
    (129, 12344, 257, 100, True),     # n % 64 == 56; outputs that are not whole 16-byte stores
    (300, 8192, 70, 64, True),        # the sizes beside these that other kernels take
    (64, 16384, 1, 33, True),
    (1000, 8200, 130, 65, False),
    (129, 8248, 257, 100, True),
    (600, 4224, 1536, 129, True),     # 132 words, one round of the MFMA kernel
    (600, 4224, 2080, 129, True),     # and more than one
    (72, 16416, 96, 127, False),      # n % 64 == 32
    (4096, 11008, 1632, 96, True),    # several k ranges over k groups
    (520, 4096, 1632, 630, False),    # four k groups, no k range
    (11008, 4096, 1632, 300, True),   # 128-feature tiles; stage 2 on these kernels too
    (8200, 512, 4097, 700, False),    # the shortest rows, several tiles a CU; a large ragged rank, a ragged last tile
    (8100, 1024, 2000, 161, False),   # stage 2 in blocks of 32 rows, the last one of one row; a ragged last tile
    (2048, 1024, 2240, 2048, True),   # 256-feature tiles on every CU, one range
    (72, 33032, 130, 33, True),       # rows of more than 1024 words (n > 32768), n % 64 == 8
    (300, 40960, 300, 64, False),     # (the k-split kernel keeps this one)
    (300, 40960, 700, 64, False),     # several k ranges
    (64, 53248, 96, 100, True),
    (130, 33024, 65, 200, False),
    (132, 1472, 544, 513, True),      # many columns past the rank, zeroed by the blocks of five feature tiles
    (9804, 256, 384, 579, False),     # outputs of whole 8-byte stores
]


def _words(t, method="half2"):
    import nanoquant_amd as nq
    return nq.pack_binary_gemv(t, method=method)


@pytest.fixture(scope="module")
def lib():
    from nanoquant_amd import _lib
    return _lib.load()


def _run(lib, c, dtype, part=True, offset=0):
    """nq_gemv on a random-byte workspace, with or without room for the k ranges' sums; ``offset``: elements by
    which the output is moved off its 16-byte alignment."""
    from nanoquant_amd import _lib
    t = lambda a: torch.from_numpy(np.ascontiguousarray(a)).cuda()  # noqa: E731
    x, s_in, s_out = (t(c[k]).to(dtype) for k in ("x", "s_in", "s_out"))
    s_mid = None if c["s_mid"] is None else t(c["s_mid"]).to(dtype)
    V, U = _words(t(c["V"])), _words(t(c["U"]))
    (batch, n), (m, r) = c["x"].shape, c["U"].shape
    # the intermediate alone: rows of 32 columns never split
    nbytes = lib.nq_gemv_workspace_bytes(batch, n if part else 32, r, m)
    ws = torch.randint(0, 256, (nbytes,), dtype=torch.uint8, device="cuda")
    y = torch.empty(batch * m + 8, dtype=dtype, device="cuda")[offset:offset + batch * m].view(batch, m)
    _lib.check(lib.nq_gemv(_lib.dtype_code(dtype), x.data_ptr(), s_in.data_ptr(), V.data_ptr(), _lib.ptr(s_mid),
                           U.data_ptr(), s_out.data_ptr(), y.data_ptr(), batch, n, r, m, ws.data_ptr(), nbytes,
                           _lib.stream_of(x.device)), "nq_gemv")
    torch.cuda.synchronize()
    return y


def _oracle(c, dtype):
    """The fp64 result for the inputs as ``dtype`` holds them."""
    q = {k: None if c[k] is None else torch.from_numpy(c[k]).to(dtype).double().numpy() for k in ("x", "s_in", "s_mid", "s_out")}
    return O.nanoquant_forward_f64(q["x"], q["s_in"], c["V"], q["s_mid"], c["U"], q["s_out"])


def _error(y, y64, dtype):
    diff = np.abs(y.double().cpu().numpy() - y64)
    if dtype == torch.bfloat16:
        _, e = np.frexp(np.abs(y64))
        diff = np.maximum(diff - np.ldexp(1.0, e - 9), 0.0)
    return diff.max() / np.abs(y64).max()


@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16], ids=["f16", "bf16"])
@pytest.mark.parametrize("case", CASES, ids=lambda c: "x".join(str(int(v)) for v in c))
def test_rows_against_oracle(lib, case, dtype):
    m, n, r, rows, mid = case
    print("\n[case] gemv rows", case, dtype, flush=True)
    c = O.random_case(1000 + m + rows, m, n, r, rows, with_mid=mid)
    y64 = _oracle(c, dtype)
    y = _run(lib, c, dtype)
    assert _error(y, y64, dtype) <= BAR
    assert torch.equal(y, _run(lib, c, dtype)), "a second call over another workspace's bytes"


def _stage1_us(lib, rows, n, r):
    from nanoquant_amd import _lib
    x, s_in = torch.randn(rows, n, device="cuda").half(), torch.rand(n, device="cuda").half()
    V = torch.randint(-2 ** 31, 2 ** 31 - 1, (r, (n + 31) // 32), dtype=torch.int32, device="cuda")
    nbytes = lib.nq_gemv_workspace_bytes(rows, n, r, 64)
    ws = torch.zeros(nbytes, dtype=torch.uint8, device="cuda")
    times = []
    for _ in range(8):
        start, end = torch.cuda.Event(enable_timing=True), torch.cuda.Event(enable_timing=True)
        start.record()
        for _ in range(4):
            _lib.check(lib.nq_gemv_stage1(_lib.NQ_F16, x.data_ptr(), s_in.data_ptr(), V.data_ptr(), None, rows, n, r, 64,
                                          ws.data_ptr(), nbytes, _lib.stream_of(x.device)), "nq_gemv_stage1")
        end.record()
        torch.cuda.synchronize()
        times.append(start.elapsed_time(end) * 250)
    return min(times)


@pytest.mark.parametrize("rows", [48, 64, 100])
def test_rows_run_on_the_longest_inputs(lib, rows):
    """n > 32768: the kernels planned for (and given a workspace) run, not the general one, which passes over V for every
    eight batch rows and took 20 times the time of 32 rows where these take two to four times."""
    print("\n[case] gemv rows, time", rows, flush=True)
    few, many = _stage1_us(lib, 32, 53248, 1632), _stage1_us(lib, rows, 53248, 1632)
    assert many < 8 * few, f"{rows} rows take {many:.0f} us, 32 rows {few:.0f}"


def _graph_us(launch, count=16):
    """Microseconds of one launch among `count` in a graph, the least of five replays."""
    launch()
    torch.cuda.synchronize()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        for _ in range(count):
            launch()
    times = []
    for _ in range(6):
        start, end = torch.cuda.Event(enable_timing=True), torch.cuda.Event(enable_timing=True)
        start.record()
        graph.replay()
        end.record()
        torch.cuda.synchronize()
        times.append(start.elapsed_time(end) * 1000 / count)
    return min(times[1:])


def _stage_us(lib, stage, rows, n, r, m):
    from nanoquant_amd import _lib
    half = lambda *s: torch.rand(*s, device="cuda").half()  # noqa: E731
    words = lambda a, b: torch.randint(-2 ** 31, 2 ** 31 - 1, (a, (b + 31) // 32), dtype=torch.int32, device="cuda")  # noqa: E731
    x, s_in, s_out, V, U, y = half(rows, n), half(n), half(m), words(r, n), words(m, r), half(rows, m)
    nbytes = lib.nq_gemv_workspace_bytes(rows, n, r, m)
    ws = torch.zeros(nbytes, dtype=torch.uint8, device="cuda")
    if stage == 1:
        return _graph_us(lambda: _lib.check(lib.nq_gemv_stage1(
            _lib.NQ_F16, x.data_ptr(), s_in.data_ptr(), V.data_ptr(), None, rows, n, r, m, ws.data_ptr(), nbytes,
            torch.cuda.current_stream().cuda_stream), "stage 1"))
    return _graph_us(lambda: _lib.check(lib.nq_gemv_stage2(
        _lib.NQ_F16, U.data_ptr(), s_out.data_ptr(), y.data_ptr(), rows, n, r, m, ws.data_ptr(), nbytes,
        torch.cuda.current_stream().cuda_stream), "stage 2"))


def test_rows_time_does_not_jump_with_the_sizes_beside(lib):
    """Ranks with many columns to zero (r = 544; took twice the time of r = 512) and outputs that are not whole 16-byte
    stores (m = 9804; took 1.5 times the time of m = 9808) cost little more than their neighbours."""
    print("\n[case] gemv rows, neighbours", flush=True)
    a, b = (_stage_us(lib, 1, 513, 1472, r, 64) for r in (512, 544))
    assert b < 1.4 * a, (a, b)
    a, b = (_stage_us(lib, 2, 579, 256, 384, m) for m in (9808, 9804))
    assert b < 1.25 * a, (a, b)


def test_rows_leave_one_round_to_the_mfma_kernel(lib):
    """n = 4224 at 129 rows, one round of blocks of 64 features, takes about the time of 128 (it took 1.35 times that)."""
    print("\n[case] gemv rows, one round", flush=True)
    a, b = (_stage_us(lib, 1, rows, 4224, 1536, 64) for rows in (128, 129))
    assert b < 1.2 * a, (a, b)


@pytest.mark.parametrize("offset", [1, 4])
def test_rows_without_range_sums_and_unaligned_output(lib, offset):
    """No room for the k ranges' sums (one range runs), and outputs off their 16-byte alignment."""
    m, n, r, rows = 4096, 11008, 1632, 130
    print("\n[case] gemv rows, smallest workspace", offset, flush=True)
    assert lib.nq_gemv_workspace_bytes(rows, n, r, m) > lib.nq_gemv_workspace_bytes(rows, 32, r, m)
    c = O.random_case(77, m, n, r, rows, with_mid=True)
    assert _error(_run(lib, c, torch.float16, part=False, offset=offset), _oracle(c, torch.float16), torch.float16) <= BAR


def test_rows_take_inputs_off_their_alignment(lib):
    """x 2 bytes off a 16-byte boundary runs the general kernels, not these: the same result to the bar."""
    import nanoquant_amd  # noqa: F401
    m, n, r, rows = 300, 8192, 70, 130
    print("\n[case] gemv rows, unaligned x", flush=True)
    c = O.random_case(78, m, n, r, rows, with_mid=False)
    t = lambda a: torch.from_numpy(np.ascontiguousarray(a)).cuda()  # noqa: E731
    x = torch.empty(rows * n + 1, dtype=torch.float16, device="cuda")[1:].view(rows, n)
    x.copy_(t(c["x"]))
    y = torch.ops.binary_kernels.nanoquant_dyn_forward(x, t(c["s_in"]).half(), _words(t(c["V"])), None,
                                                       _words(t(c["U"])), t(c["s_out"]).half(), 128, 128, 2, 2, 1, 1, 8, 8)
    assert _error(y, _oracle(c, torch.float16), torch.float16) <= BAR
