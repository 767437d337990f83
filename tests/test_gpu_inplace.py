"""GPU parity of the in-place matmul (``csrc/qmv_inplace.hpp``: the MLX layout
through LDS) at the edges of its tiles: rows around 4 and 16, columns around
32 and 64, K with a last chunk that is not whole, rows whose scales are not
16-byte pieces, K longer than one scale segment; and its expert form over more
experts and items than one list holds.

Bar: bf16 outputs within rtol = atol = 1e-2 of the float64 oracle."""

import numpy as np
import pytest
import torch

from oracle import moe as OM
from oracle.bf16 import round_to_bf16
from oracle.qmv import make_affine4_weights, make_affine_weights, qmm_affine
from tests.gpu_util import assert_close, assert_swiglu_close, bf16_values, bits, from_bits, randn_bf16, u32

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("b,gs,n,k", [
    (4, 32, 1, 32), (4, 32, 33, 288),       # one group; a chunk and a piece of one
    (4, 64, 31, 1088), (4, 128, 65, 1664),  # 17 and 13 groups: scales element by element
    (4, 32, 40, 2880), (8, 32, 32, 2848),   # two scale segments: 90 groups, 89 (odd)
    (8, 64, 64, 64), (8, 64, 97, 5696),     # half a chunk; 89 groups
    (8, 128, 63, 12288), (8, 128, 8, 384),  # 96 groups: two segments; an odd number of groups
])
@pytest.mark.parametrize("m", [1, 4, 5, 16, 17, 37])
def test_tile_edges(gpu, b, gs, n, k, m):
    from mtplx_amd import _lib
    rng = np.random.default_rng(b * 7 + gs + n + k + m)
    w, s, bb = make_affine_weights(rng, n, k, gs, b)
    x = randn_bf16(rng, (m, k))
    y = torch.full((m + 1, n), float("nan"), dtype=torch.bfloat16, device="cuda")
    wd, sd, bd = u32(w), from_bits(s), from_bits(bb)
    _lib.call("mtp_qmv_affine", x.data_ptr(), wd.data_ptr(), sd.data_ptr(), bd.data_ptr(), y.data_ptr(), None, m, n, k,
              gs, b, torch.cuda.current_stream().cuda_stream)
    torch.cuda.synchronize()
    assert torch.isnan(y[m]).all()   # no row past the last is written
    assert_close(bf16_values(y[:m]), round_to_bf16(qmm_affine(bits(x), w, s, bb, gs, b)), what="in place")


@pytest.mark.parametrize("b,gs,k", [(4, 32, 288), (8, 64, 1024), (8, 128, 5120)])
@pytest.mark.parametrize("m", [1, 4, 5, 17])
def test_rows_at_any_alignment(gpu, b, gs, k, m):
    """x that starts 2 bytes into an allocation: the same outputs (the same
    products and sums: only the way x reaches LDS differs)."""
    from mtplx_amd import _lib
    rng = np.random.default_rng(6)
    n = 97
    w, s, bb = make_affine_weights(rng, n, k, gs, b)
    x, wd, sd, bd = randn_bf16(rng, (m, k)), u32(w), from_bits(s), from_bits(bb)
    xo = torch.cat([x.new_zeros(1), x.reshape(-1)])[1:].reshape(m, k)
    assert xo.data_ptr() % 16 == 2
    ys = []
    for x_ in (x, xo):
        y = torch.empty((m, n), dtype=torch.bfloat16, device="cuda")
        _lib.call("mtp_qmv_affine", x_.data_ptr(), wd.data_ptr(), sd.data_ptr(), bd.data_ptr(), y.data_ptr(), None, m,
                  n, k, gs, b, torch.cuda.current_stream().cuda_stream)
        ys.append(y)
    torch.cuda.synchronize()
    assert torch.equal(ys[0], ys[1])


def test_scales_at_any_alignment(gpu):
    """Scale arrays that start 2 bytes into an allocation: the same outputs."""
    from mtplx_amd import _lib
    rng = np.random.default_rng(5)
    m, n, k, gs = 4, 96, 1024, 64
    w, s, bb = make_affine_weights(rng, n, k, gs, 8)
    x, wd, sd, bd = randn_bf16(rng, (m, k)), u32(w), from_bits(s), from_bits(bb)
    so, bo = (torch.cat([t.new_zeros(1), t.reshape(-1)])[1:] for t in (sd, bd))
    assert so.data_ptr() % 16 == 2
    ys = []
    for s_, b_ in ((sd, bd), (so, bo)):
        y = torch.empty((m, n), dtype=torch.bfloat16, device="cuda")
        _lib.call("mtp_qmv_affine", x.data_ptr(), wd.data_ptr(), s_.data_ptr(), b_.data_ptr(), y.data_ptr(), None, m, n,
                  k, gs, 8, torch.cuda.current_stream().cuda_stream)
        ys.append(y)
    torch.cuda.synchronize()
    assert torch.equal(ys[0], ys[1])


@pytest.mark.parametrize("E,T,k,H,F,gs,skew", [
    (300, 100, 4, 256, 96, 64, 0.0),    # more experts than one list (128), one or two rows each
    (4, 70, 4, 512, 64, 128, 0.0),      # 70 rows each: five row tiles
    (160, 40, 8, 768, 4128, 64, 1.5),   # more items per workgroup than one list (32), both row classes
    (3, 9, 1, 1536, 40, 64, 0.0),       # columns past a tile; K in 6 chunks over 2 waves
    # tiles of 16 rows, scales in segments of 24 groups: 2 of them, the last one chunk of
    # one wave's (28 groups); 32; 3 (60); 2 of 12 chunks (32 groups of 128)
    (3, 40, 2, 1792, 40, 64, 0.0), (5, 60, 3, 2048, 48, 64, 0.8), (3, 40, 2, 3840, 33, 64, 0.0),
    (3, 40, 2, 4096, 40, 128, 0.0),
])
def test_experts(gpu, E, T, k, H, F, gs, skew):
    from mtplx_amd import _lib
    from mtplx_amd.moe_sorted_gather import expert_sort
    rng = np.random.default_rng(E + T)
    g0, u0 = (tuple(a.reshape(E, F, -1) for a in make_affine4_weights(rng, E * F, H, gs)) for _ in range(2))
    x = randn_bf16(rng, (T, H))
    p = 1.0 / np.arange(1, E + 1) ** skew
    idx = np.stack([rng.choice(E, size=k, replace=False, p=p / p.sum()) for _ in range(T)]).astype(np.int32)
    es = expert_sort(torch.from_numpy(idx).cuda(), E)
    row_map, sorted_ids, _, _ = OM.sort_rows(idx)
    st = torch.cuda.current_stream().cuda_stream
    R = T * k
    gd, ud = (u32(g0[0]), from_bits(g0[1]), from_bits(g0[2])), (u32(u0[0]), from_bits(u0[1]), from_bits(u0[2]))
    h = torch.full((R, F), float("nan"), dtype=torch.bfloat16, device="cuda")
    y = torch.full((R, F), float("nan"), dtype=torch.bfloat16, device="cuda")
    args = (x.data_ptr(), None, es.row_map.data_ptr(), es.expert_off.data_ptr(), es.active.data_ptr())
    _lib.call("mtp_gather_qmv_affine4", *args, *(t.data_ptr() for t in gd), *(t.data_ptr() for t in ud), h.data_ptr(),
              R, E, F, H, gs, 0, 3, F, None, 0, st)
    _lib.call("mtp_gather_qmv_affine4", *args, *(t.data_ptr() for t in gd), None, None, None, y.data_ptr(), R, E, F, H,
              gs, 0, 0, F, None, 0, st)
    torch.cuda.synchronize()
    gate = OM.gather_qmm_rows(bits(x), row_map, sorted_ids, *g0, gs)
    up = OM.gather_qmm_rows(bits(x), row_map, sorted_ids, *u0, gs)
    assert_close(bf16_values(y), round_to_bf16(gate), what="store")
    gb, ub = round_to_bf16(gate), round_to_bf16(up)
    want = round_to_bf16(round_to_bf16(gb / (1.0 + np.exp(-gb))) * ub)
    assert_swiglu_close(bf16_values(h), gb, ub, want, what="SwiGLU pair")


def _gather_nodes(call):
    """Kernels that ``call`` launches: the nodes of its captured graph."""
    import ctypes
    g = torch.cuda.CUDAGraph(keep_graph=True)
    with torch.cuda.graph(g):
        call()
    n = ctypes.c_size_t()
    hip = ctypes.CDLL(None)   # torch's HIP runtime is mapped
    assert hip.hipGraphGetNodes(ctypes.c_void_p(g.raw_cuda_graph()), None, ctypes.byref(n)) == 0
    return n.value


@pytest.mark.parametrize("emode", [0, 3])
def test_both_row_classes_in_one_launch(gpu, emode):
    """A gather whose experts have 1..4 rows and more is one kernel (small
    routed calls wait for launches), and a row's output has the same bits
    whichever class its expert falls in."""
    from mtplx_amd import _lib
    from mtplx_amd.moe_sorted_gather import expert_sort
    rng = np.random.default_rng(8)
    E, K, F = 5, 2048, 160
    gate, up = (tuple(a.reshape(E, F, -1) for a in make_affine4_weights(rng, E * F, K, 64)) for _ in range(2))
    gd, ud = ((u32(t[0]), from_bits(t[1]), from_bits(t[2])) for t in (gate, up))
    x = randn_bf16(rng, (24, K))

    def gather(ids):
        es = expert_sort(torch.from_numpy(ids).reshape(-1, 1).cuda(), E)
        y = torch.zeros((ids.size, F), dtype=torch.bfloat16, device="cuda")
        args = (x.data_ptr(), None, es.row_map.data_ptr(), es.expert_off.data_ptr(), es.active.data_ptr(),
                *(t.data_ptr() for t in gd), *(t.data_ptr() if emode else None for t in ud), y.data_ptr(), ids.size, E, F,
                K, 64, 0, emode, F, None, 0)
        run = lambda: _lib.call("mtp_gather_qmv_affine4", *args,   # noqa: E731
                                torch.cuda.current_stream().cuda_stream)
        return es, y, run

    ids = np.array([1] * 3 + [4] * 17 + [0] * 4, dtype=np.int32)   # both classes, two row tiles
    es, y, run = gather(ids)
    run()
    torch.cuda.synchronize()
    assert not torch.isnan(y.float()).any()
    flat = y[es.inv_order.long()].clone()
    es1, y1, run1 = gather(np.array([4], dtype=np.int32).repeat(3))   # x rows 0..2 of expert 4, in the small class
    es2, y2, run2 = gather(np.array([4], dtype=np.int32).repeat(20))  # and in the large one
    run1()
    run2()
    torch.cuda.synchronize()
    assert torch.equal(y1.view(torch.int16), y2[:3].view(torch.int16))
    assert torch.equal(y2[3:20].view(torch.int16), flat[3:20].view(torch.int16))
    assert _gather_nodes(run) == 1
