"""Grouped stage 2 of many batch rows (a launch per item that shares each decoded sign over the batch):
the store, residual and gated epilogues against the single GEMV (needs a gfx950 GPU)."""
import numpy as np
import pytest
import torch

import oracle as O

pytestmark = pytest.mark.gpu

# (m, r, rows, y_stride past the row): whole and ragged row tiles, 8-byte and 2-byte stores, each launch shape
# (16 or 32 batch rows a block, 32- or 64-row tiles), and the smallest batch of a gated pair
CASES = [(10240, 64, 16, 0), (5001, 333, 40, 3), (9000, 100, 65, 8), (4102, 200, 90, 2), (20000, 1000, 8, 4),
         (4100, 1632, 24, 0), (16400, 4224, 2, 0), (8200, 1632, 32, 4), (4096, 64, 48, 0), (1199, 640, 40, 1),
         (1200, 640, 40, 0)]


def _group(lib, entries, x, epilogue, dtype):
    from nanoquant_amd import _lib
    arr = (_lib.GemvItem * len(entries))()
    for it, e in zip(arr, entries):
        it.v_bits, it.s_in, it.s_mid, it.u_bits, it.s_out = (e[k].data_ptr() for k in ("V", "s_in", "s_mid", "U", "s_out"))
        it.y, it.y_stride = e["y"].data_ptr(), e["y"].stride(0)
        it.resid = None if e.get("resid") is None else e["resid"].data_ptr()
        it.r, it.m = e["V"].shape[0], e["U"].shape[0]
    batch, n = x.shape
    need = lib.nq_gemv_group_workspace_bytes(len(entries), arr, batch)
    ws = torch.randint(0, 256, (need,), dtype=torch.uint8, device="cuda")
    st = torch.cuda.current_stream().cuda_stream
    _lib.check(lib.nq_gemv_group_stage1(_lib.dtype_code(dtype), len(entries), arr, x.data_ptr(), batch, n, -1.0,
                                        ws.data_ptr(), need, st), "stage 1")
    _lib.check(lib.nq_gemv_group_stage2(_lib.dtype_code(dtype), len(entries), arr, batch, epilogue, ws.data_ptr(), need, st),
               "stage 2")
    torch.cuda.synchronize()


def _entry(seed, m, n, r, dtype, stride, batch):
    import nanoquant_amd as nq
    c = O.random_case(seed, m, n, r, 1, with_mid=True)
    t = lambda a: torch.from_numpy(np.ascontiguousarray(a)).cuda()  # noqa: E731
    e = {"V": nq.pack_binary_gemv(t(c["V"]), method="half2"), "U": nq.pack_binary_gemv(t(c["U"]), method="half2")}
    # outputs of a few units, so that silu is neither linear nor zero
    scale = {"s_in": 0.06, "s_mid": 1.0, "s_out": 2.0 / np.sqrt(r)}
    e.update({k: (t(c[k]).float() * scale[k]).to(dtype) for k in scale})
    e["y"] = torch.full((batch, m + stride), 7.0, dtype=dtype, device="cuda")
    return e


@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16], ids=["f16", "bf16"])
@pytest.mark.parametrize("case", CASES, ids=lambda c: "x".join(map(str, c)))
def test_batched_epilogues(case, dtype):
    """Store and residual equal the single op (whose stage 2 is the same kernel) to a unit of its fp32 sum's order;
    the gated pair equals T(T(silu(gate)) * up) of the single ops' outputs. A difference of summation order can move
    a rounding by one unit in the last place, and silu's and the product's roundings add one each."""
    from nanoquant_amd import _lib
    lib = _lib.load()
    m, r, batch, extra = case
    n = 256
    print("\n[case] group batched", case, dtype, flush=True)
    gen = torch.Generator(device="cuda").manual_seed(m)
    x = torch.randn(batch, n, device="cuda", generator=gen).to(dtype)
    gate, up = (_entry(m + i, m, n, r, dtype, extra, batch) for i in (0, 1))
    single = [torch.ops.binary_kernels.nanoquant_dyn_forward(x, e["s_in"], e["V"], e["s_mid"], e["U"], e["s_out"], 128, 128,
                                                             2, 2, 1, 1, 8, 8) for e in (gate, up)]
    ulp = 2.0 ** (-10 if dtype == torch.float16 else -7)  # of a value's own binade, at most

    def close(got, want, ulps):
        assert torch.equal(got[:, m:], torch.full_like(got[:, m:], 7.0))
        g, w = got[:, :m].float(), want.float()
        assert bool(((g - w).abs() <= ulps * ulp * torch.maximum(g.abs(), w.abs()) + 1e-6).all())

    _group(lib, [gate, up], x, _lib.NQ_EPI_STORE, dtype)
    close(gate["y"], single[0], 1)
    close(up["y"], single[1], 1)
    gate["resid"] = torch.randn(batch, m + extra, device="cuda", generator=gen).to(dtype)
    gate["resid"][:, m:] = 7.0
    gate["y"].fill_(7.0)
    _group(lib, [gate], x, _lib.NQ_EPI_RESIDUAL, dtype)
    want = gate["resid"][:, :m] + single[0]
    g = gate["y"][:, :m].float()
    # the addend's own unit, then the sum's
    assert bool(((g - want.float()).abs() <= ulp * (single[0].float().abs() + want.float().abs()) + 1e-6).all())
    gate["y"].copy_(gate["resid"])
    gate["resid"] = gate["y"]  # in place
    _group(lib, [gate], x, _lib.NQ_EPI_RESIDUAL, dtype)
    assert torch.equal(gate["y"][:, :m].float(), g)
    gate["resid"] = None
    gate["y"].fill_(7.0)
    _group(lib, [gate, up], x, _lib.NQ_EPI_GATED, dtype)
    close(gate["y"], torch.nn.functional.silu(single[0].float()).to(dtype) * single[1], 4)


def test_small_items_share_a_launch():
    """Two stored items of a small rank take less than two launches of one (they took as much)."""
    from nanoquant_amd import _lib
    lib = _lib.load()
    m, r, batch, dtype = 3500, 224, 47, torch.float16
    print("\n[case] group batched, small items", flush=True)
    entries = [_entry(i, m, 64, r, dtype, 0, batch) for i in (1, 2)]
    arr = (_lib.GemvItem * 2)()
    for it, e in zip(arr, entries):
        it.v_bits, it.s_in, it.s_mid, it.u_bits, it.s_out = (e[k].data_ptr() for k in ("V", "s_in", "s_mid", "U", "s_out"))
        it.y, it.y_stride, it.r, it.m = e["y"].data_ptr(), m, r, m
    ws = torch.zeros(lib.nq_gemv_group_workspace_bytes(2, arr, batch), dtype=torch.uint8, device="cuda")

    def us(count):
        def launch():
            _lib.check(lib.nq_gemv_group_stage2(_lib.NQ_F16, count, arr, batch, _lib.NQ_EPI_STORE, ws.data_ptr(), ws.numel(),
                                                torch.cuda.current_stream().cuda_stream), "stage 2")
        launch()
        torch.cuda.synchronize()
        graph = torch.cuda.CUDAGraph()
        with torch.cuda.graph(graph):
            for _ in range(16):
                launch()
        times = []
        for _ in range(6):
            start, end = torch.cuda.Event(enable_timing=True), torch.cuda.Event(enable_timing=True)
            start.record()
            graph.replay()
            end.record()
            torch.cuda.synchronize()
            times.append(start.elapsed_time(end) * 1000 / 16)
        return min(times[1:])

    one, two = us(1), us(2)
    assert two < 1.7 * one, (one, two)
