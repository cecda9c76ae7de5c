"""The operators' C++ implementations against the general ones in Python (needs a gfx950 GPU)."""
import pytest
import torch

import nanoquant_amd  # noqa: F401
from nanoquant_amd import _lib
from nanoquant_amd.kernel import utils as ku

pytestmark = pytest.mark.gpu

TUNING = (128, 128, 2, 2, 1, 1, 8, 8)
NATIVE, GENERAL = torch.ops.binary_kernels, torch.ops.nanoquant_amd


@pytest.fixture(scope="module", autouse=True)
def library():
    assert _lib.ops is not None, "libnq_ops.so is not built"
    _lib.load()  # from here on the C++ operators have the library's functions


def _sign(*shape):
    return (torch.randint(0, 2, shape, device="cuda", dtype=torch.int8) * 2 - 1)


def _gemv(lead, n, r, m, dtype, mid):
    t = lambda k: torch.rand(k, device="cuda").to(dtype)  # noqa: E731
    return (torch.randn(*lead, n, device="cuda").to(dtype), t(n), ku.binary_packer(_sign(r, n), "half2"), t(r) if mid else None,
            ku.binary_packer(_sign(m, r), "half2"), t(m), *TUNING)


@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16], ids=["f16", "bf16"])
@pytest.mark.parametrize("lead,n,r,m,mid", [((), 33, 5, 7, True), ((1,), 256, 64, 100, False), ((2, 3), 1000, 96, 64, True),
                                            ((0, 4), 64, 32, 8, False), ((70,), 8192, 128, 256, True)])
def test_gemv_operator(lead, n, r, m, mid, dtype):
    args = _gemv(lead, n, r, m, dtype, mid)
    y, want = NATIVE.nanoquant_dyn_forward(*args), GENERAL.nanoquant_dyn_forward(*args)
    assert y.shape == want.shape == (*lead, m) and y.dtype == dtype and torch.equal(y, want)


@pytest.mark.parametrize("rows", [0, 1, 100, 300])
def test_gemm_operators(rows):
    n, r, m = 256, 200, 128
    V, U = _sign(r // 8 * 8, n), _sign(m, r // 8 * 8)
    scales = [torch.rand(k, device="cuda").half() for k in (n, V.shape[0], m)]
    V, U, scales[1] = V[:192], U[:, :192].contiguous(), scales[1][:192].contiguous()
    words_v, words_u, g, l, h, ws = ku.marlin_nanoquant_packer(V.T, U.T, *scales)
    x = torch.randn(rows, n, device="cuda").half()
    for args in ((x, words_v, words_u, g, l, h, ws), (x, words_v, words_u, g, None, None, ws)):
        assert torch.equal(NATIVE.marlin_nanoquant_forward(*args), GENERAL.marlin_nanoquant_forward(*args))
    for args in ((x, words_v, g, l, ws), (x, words_v, None, None, ws)):
        assert torch.equal(NATIVE.marlin_onebit_forward(*args), GENERAL.marlin_onebit_forward(*args))


def test_refusals_are_the_general_operators():
    """Every refused call raises what the Python checks raise."""
    good = list(_gemv((2,), 64, 32, 8, torch.float16, True))
    other = torch.ones(64, device="cuda")
    bad = {0: [good[0].float(), good[0].t().contiguous().t(), good[0].cpu()], 1: [other, other.half()[:32]],
           2: [good[2][:, :1].contiguous(), good[2].long()], 3: [good[3][:16], good[3].view(1, -1)],
           4: [good[4][:4], good[4].t()], 5: [good[5].view(1, -1), good[5].bfloat16()], 6: [100], 10: [4], 13: [3]}
    for i, values in bad.items():
        for v in values:
            args = good[:i] + [v] + good[i + 1:]
            with pytest.raises((RuntimeError, ValueError, NotImplementedError)) as want:
                GENERAL.nanoquant_dyn_forward(*args)
            with pytest.raises(type(want.value)) as got:
                NATIVE.nanoquant_dyn_forward(*args)
            if not isinstance(want.value, NotImplementedError):  # the dispatcher's own text names the operator
                assert str(got.value) == str(want.value)


def test_operator_on_a_side_stream_and_in_a_graph():
    args = _gemv((3,), 4096, 1120, 512, torch.float16, False)
    want = GENERAL.nanoquant_dyn_forward(*args)
    side = torch.cuda.Stream()
    side.wait_stream(torch.cuda.current_stream())
    with torch.cuda.stream(side):
        y = NATIVE.nanoquant_dyn_forward(*args)
    side.synchronize()
    assert torch.equal(y, want)
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        y = NATIVE.nanoquant_dyn_forward(*args)
    for _ in range(3):
        args[0].copy_(torch.randn_like(args[0]))
        graph.replay()
        torch.cuda.synchronize()
        assert torch.equal(y, GENERAL.nanoquant_dyn_forward(*args))
