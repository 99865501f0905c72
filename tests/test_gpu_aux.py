"""GPU parity of the MXFP4 MoE orchestration ops (device counterparts of the reference's
moe_aux.cpp) and of the W4A4 mode of the layer, through the C ABI.

Bit-exact: quantised codes and scale bytes (token and sorted order), the routed combine.
W4A4 layer: against the oracle run on the same quantised activations
(`oracle.set_act_model(1)`), where only the order of the fp32 sums differs."""
from __future__ import annotations

import ctypes

import numpy as np
import pytest
import torch

import oracle
from vkernels_amd import synth
from vkernels_amd import vllm_experts as ve

import test_gpu_configs as cfgs
from gpu_util import (EXACT_SPLIT_MAX_ABS_TOL, EXACT_SPLIT_REL_L2_TOL, MAX_ABS_TOL, REL_L2_TOL, cpu_layer, dev,
                      edge_tokens, error_metrics, to_dev)

pytestmark = pytest.mark.gpu

_P, _I = ctypes.c_void_p, ctypes.c_int


def _edge_rows(M, hidden, seed):
    """Activations with everything the quantiser has cases for."""
    A = synth.make_activations(M, hidden, seed)
    f = synth.bf16_bits_to_f32(A)
    rng = np.random.default_rng(seed)
    A[0, :32] = 0                                                     # a zero group
    A[1, 40] = 0x7F80                                                 # inf: its group is zero
    A[2, 9] = 0x7FC1                                                  # NaN inside a finite group
    A[3, :] = rng.integers(0, 128, hidden).astype(np.uint16)          # bf16 subnormals
    A[4, :] = synth.f32_to_bf16_bits(f[4] * np.float32(2.0 ** 100))
    A[5, :] = synth.f32_to_bf16_bits(f[5] * np.float32(2.0 ** -100))
    A[6, :32] = synth.f32_to_bf16_bits(np.array([3, .125, .625, 1.25, 1.75, 2.5, -.125, -.124, -0.0, 0.0] + [0.1] * 22, np.float32))
    A[7, :64] = synth.f32_to_bf16_bits(np.r_[np.full(32, 1.5), np.full(32, 1.5078125)].astype(np.float32))  # m = 1.5 and above
    A[8, 0] = 0x7F00                                                  # 2^127 next to small values
    A[9, :32] = 0x8000                                                # negative zeros
    A[10, 3] = 0xFF80                                                 # -inf
    A[11, :32] = rng.integers(0, 65536, 32).astype(np.uint16)         # arbitrary bit patterns
    A[12:16] = rng.integers(0, 65536, (4, hidden)).astype(np.uint16)
    return A


def test_quant_bitwise(hip_lib):
    fn = hip_lib.vk_hip_mxfp4_moe_quant
    fn.restype = _I
    fn.argtypes = [_P, _P, _P, _I, _I, _I, _P]
    M, hidden = 48, 2880
    A = _edge_rows(M, hidden, 301)
    packed = torch.zeros((M, hidden // 2), dtype=torch.uint8, device=dev())
    scales = torch.zeros((M, hidden // 32), dtype=torch.uint8, device=dev())
    d_A = to_dev(A)
    assert fn(d_A.data_ptr(), packed.data_ptr(), scales.data_ptr(), M, hidden, 32, None) == 0
    torch.cuda.synchronize()
    rp, rs = oracle.mxfp4_moe_quant(A)
    gs, gp = scales.cpu().numpy(), packed.cpu().numpy()
    assert np.array_equal(gs, rs), f"scale bytes differ at (row, group) {np.argwhere(gs != rs)[:10].tolist()}"
    assert np.array_equal(gp, rp), f"codes differ at (row, byte) {np.argwhere(gp != rp)[:10].tolist()}"
    assert fn(None, None, None, 4, 64, 16, None) == ve.VK_ERROR_UNSUPPORTED


@pytest.mark.parametrize("hidden", [32, 64, 96, 544, 2048, 4096 + 32])
def test_quant_widths_and_magnitudes_bitwise(hip_lib, hidden):
    """Rows that share a wavefront, end inside a batch of loads or take several, at magnitudes
    around the ends of the packed routine's range of scale bytes (4 .. 143) and beyond, with
    every value near a rounding threshold."""
    fn = hip_lib.vk_hip_mxfp4_moe_quant
    fn.restype = _I
    fn.argtypes = [_P, _P, _P, _I, _I, _I, _P]
    M = 97
    rng = np.random.default_rng(hidden)
    near = np.array([.125, .625, 1.25, 1.75, 2.5, 3.0], np.float32)
    steps = rng.integers(-2, 3, (M, hidden))
    bits = synth.f32_to_bf16_bits(near[rng.integers(0, 6, (M, hidden))]).astype(np.int64) + steps
    exps = np.r_[np.arange(1 - 127, 8 - 127), np.arange(139 - 127, 148 - 127), rng.integers(-100, 100, M)][:M]
    vals = synth.bf16_bits_to_f32(bits.astype(np.uint16)).astype(np.float64) * 2.0 ** exps[:, None]
    vals *= rng.choice([-1.0, 1.0], (M, hidden))
    A = synth.f32_to_bf16_bits(vals.astype(np.float32))
    A[rng.random((M, hidden)) < 0.02] = 0x8001           # a negative subnormal among them
    A[11, hidden - 1] = 0x7FC0                           # a NaN, an infinity, a group of zeros
    A[12, 0] = 0xFF80
    A[13, :32] = 0x8000
    packed = torch.zeros((M, hidden // 2), dtype=torch.uint8, device=dev())
    scales = torch.zeros((M, hidden // 32), dtype=torch.uint8, device=dev())
    d_A = to_dev(A)
    assert fn(d_A.data_ptr(), packed.data_ptr(), scales.data_ptr(), M, hidden, 32, None) == 0
    torch.cuda.synchronize()
    rp, rs = oracle.mxfp4_moe_quant(A)
    assert np.array_equal(scales.cpu().numpy(), rs) and np.array_equal(packed.cpu().numpy(), rp)


@pytest.mark.parametrize("hidden,rows", [(2048, 3), (2080, 1), (2080, 4096), (2080, 4097), (4096, 65),
                                         (7168, 17), (8224, 2)])
def test_quant_a_workgroup_per_row_at_its_edges(hip_lib, hidden, rows):
    """Rows of one piece more than a wavefront takes in a batch, the most rows that have a
    workgroup each and one more, in token order and in sorted order with padding between."""
    q, sq = hip_lib.vk_hip_mxfp4_moe_quant, hip_lib.vk_hip_mxfp4_moe_sorted_quant
    q.restype = sq.restype = _I
    q.argtypes = [_P] * 3 + [_I] * 3 + [_P]
    sq.argtypes = [_P] * 4 + [_I] * 5 + [_P]
    rng = np.random.default_rng(hidden + rows)
    A = synth.f32_to_bf16_bits((rng.standard_normal((rows, hidden)) * 2.0 ** rng.integers(-120, 100, (rows, 1)))
                               .astype(np.float32))
    A[rng.integers(0, rows, 9), rng.integers(0, hidden, 9)] = 0x7FC0     # NaN, infinities, zero groups
    A[rng.integers(0, rows, 9), rng.integers(0, hidden, 9)] = 0xFF80
    A[rows - 1, hidden - 32:] = 0x8000
    packed = torch.full((rows + 1, hidden // 2), 7, dtype=torch.uint8, device=dev())
    scales = torch.full((rows + 1, hidden // 32), 7, dtype=torch.uint8, device=dev())
    d_A = to_dev(A)
    assert q(d_A.data_ptr(), packed.data_ptr(), scales.data_ptr(), rows, hidden, 32, None) == 0
    torch.cuda.synchronize()
    rp, rs = oracle.mxfp4_moe_quant(A)
    assert np.array_equal(packed.cpu().numpy(), np.r_[rp, np.full((1, hidden // 2), 7, np.uint8)])
    assert np.array_equal(scales.cpu().numpy(), np.r_[rs, np.full((1, hidden // 32), 7, np.uint8)])
    sids = rng.integers(0, 2 * rows, rows).astype(np.int32)              # top_k 1: half of them padding
    sids[rng.random(rows) < 0.1] = -5
    packed.fill_(7)
    scales.fill_(7)
    d_s = to_dev(sids)
    assert sq(d_A.data_ptr(), d_s.data_ptr(), packed.data_ptr(), scales.data_ptr(), rows, hidden, 32, 1, rows,
              None) == 0
    torch.cuda.synchronize()
    rp, rs = oracle.mxfp4_moe_sorted_quant(A, sids, 1)
    assert np.array_equal(packed.cpu().numpy(), np.r_[rp, np.full((1, hidden // 2), 7, np.uint8)])
    assert np.array_equal(scales.cpu().numpy(), np.r_[rs, np.full((1, hidden // 32), 7, np.uint8)])


@pytest.mark.parametrize("top_k", [1, 2, 3, 4, 6, 8])
def test_scatter_reduce_on_a_used_workspace(hip_lib, top_k):
    """The table of sorted positions holds what an earlier call left there: flat indices without
    a sorted row (a quarter of the experts is another rank's) add nothing, whatever their
    entries say."""
    sr = hip_lib.vk_hip_mxfp4_moe_scatter_reduce
    sr.restype = _I
    sr.argtypes = [_P, _P, _P, _P, _I, _I, _I, _I, _P, ctypes.c_size_t, _P]
    rng = np.random.default_rng(top_k)
    M, E, width = 53, 16, 132
    ids = np.stack([rng.permutation(E)[:top_k] for _ in range(M)]).astype(np.int32)
    emap = np.where(np.arange(E) % 4 == 1, -1, np.cumsum(np.arange(E) % 4 != 1) - 1).astype(np.int32)
    sids, _, em = oracle.moe_align_block_size_with_map(ids.ravel(), E, 16, emap)
    sids = sids[:em].copy()
    partial = rng.standard_normal((em, width)).astype(np.float32)
    tws = rng.random(em).astype(np.float32)
    base = rng.standard_normal((M, width)).astype(np.float32)
    ref = oracle.mxfp4_moe_scatter_reduce(partial, tws, sids, M, top_k, out=base.copy())
    d_p, d_w, d_s = to_dev(partial), to_dev(tws), to_dev(sids)
    for garbage in (np.full(M * top_k, -1), np.arange(M * top_k) % em, np.full(M * top_k, em),
                    rng.integers(-2 ** 31, 2 ** 31, M * top_k)):
        ws, out = to_dev(garbage.astype(np.int32)), to_dev(base.copy())
        assert sr(d_p.data_ptr(), d_w.data_ptr(), d_s.data_ptr(), out.data_ptr(), M, width, top_k, em,
                  ws.data_ptr(), ws.numel() * 4, None) == 0
        torch.cuda.synchronize()
        assert np.array_equal(out.cpu().numpy().view(np.uint32), ref.view(np.uint32))


@pytest.mark.parametrize("top_k", [1, 2, 3, 4, 5, 6, 7, 8, 9, 16])
def test_all_combines_on_a_used_workspace(hip_lib, top_k):
    """scatter_reduce, scatter_reduce_q and moe_combine (bias, a block without an expert) for every
    number of experts per token they are compiled for and for others, on workspaces that hold what
    an earlier call left there."""
    sr, srq, mc = (getattr(hip_lib, n) for n in ("vk_hip_mxfp4_moe_scatter_reduce",
                                                 "vk_hip_mxfp4_moe_scatter_reduce_q", "vk_hip_moe_combine"))
    sr.restype = srq.restype = mc.restype = _I
    sr.argtypes = [_P] * 4 + [_I] * 4 + [_P, ctypes.c_size_t, _P]
    srq.argtypes = [_P] * 5 + [_I] * 5 + [_P, ctypes.c_size_t, _P]
    mc.argtypes = [_P] * 6 + [_I] * 5 + [_P, ctypes.c_size_t, _P]
    rng = np.random.default_rng(100 + top_k)
    M, E, width = 53, 16, 192          # (the oracle's moe_combine takes whole tiles of 64 columns)
    ids = np.stack([rng.permutation(E)[:top_k] for _ in range(M)]).astype(np.int32)
    emap = np.where(np.arange(E) % 4 == 1, -1, np.cumsum(np.arange(E) % 4 != 1) - 1).astype(np.int32)
    sids, eids, em = oracle.moe_align_block_size_with_map(ids.ravel(), E, 16, emap)
    sids, eids = sids[:em].copy(), eids[:em // 16].copy()
    eids[len(eids) // 2] = -1
    partial = rng.standard_normal((em, width)).astype(np.float32)
    bias = rng.standard_normal((E, width)).astype(np.float32)
    fin = np.array(synth.FINITE_CODES, np.uint8)
    pq = fin[rng.integers(0, 12, (em, width // 2))] | (fin[rng.integers(0, 12, (em, width // 2))] << 4)
    ps = rng.integers(110, 140, (em, width // 32)).astype(np.uint8)
    ps[rng.random(ps.shape) < 0.1] = 0xFF
    tws = rng.random(em).astype(np.float32)
    base = rng.standard_normal((M, width)).astype(np.float32)
    refs = (oracle.mxfp4_moe_scatter_reduce(partial, tws, sids, M, top_k, out=base.copy()),
            oracle.mxfp4_moe_scatter_reduce_q(pq, ps, tws, sids, M, top_k, out=base.copy()),
            oracle.moe_combine(partial, bias, tws, sids, eids, M, width, top_k, em, out=base.copy()))
    d_p, d_b, d_pq, d_ps, d_w, d_s, d_e = (to_dev(a) for a in (partial, bias, pq, ps, tws, sids, eids))
    for garbage in (np.arange(M * top_k) % em, np.full(M * top_k, em),
                    np.repeat(np.arange(M) % em, top_k), rng.integers(-2 ** 31, 2 ** 31, M * top_k)):
        for i, ref in enumerate(refs):
            ws, out = to_dev(garbage.astype(np.int32)), to_dev(base.copy())
            scratch = (ws.data_ptr(), ws.numel() * 4, None)
            if i == 0:
                rc = sr(d_p.data_ptr(), d_w.data_ptr(), d_s.data_ptr(), out.data_ptr(), M, width, top_k, em, *scratch)
            elif i == 1:
                rc = srq(d_pq.data_ptr(), d_ps.data_ptr(), d_w.data_ptr(), d_s.data_ptr(), out.data_ptr(), M, width,
                         top_k, em, 32, *scratch)
            else:
                rc = mc(d_p.data_ptr(), d_b.data_ptr(), d_w.data_ptr(), d_s.data_ptr(), d_e.data_ptr(),
                        out.data_ptr(), M, width, top_k, em, 16, *scratch)
            assert rc == 0
            torch.cuda.synchronize()
            assert np.array_equal(out.cpu().numpy().view(np.uint32), ref.view(np.uint32)), i


@pytest.mark.parametrize("hidden", [32, 64, 96, 160, 256])
def test_sorted_quant_of_rows_that_share_a_wavefront(hip_lib, hidden):
    """2 to 16 rows to a wavefront: routed rows, padding and negative ids side by side, the last
    workgroup not full, groups that only the general routine takes beside others."""
    sq = hip_lib.vk_hip_mxfp4_moe_sorted_quant
    sq.restype = _I
    sq.argtypes = [_P, _P, _P, _P, _I, _I, _I, _I, _I, _P]
    rng = np.random.default_rng(hidden)
    M, top_k, em = 70, 3, 16 * 19 + 5
    A = _edge_rows(M, 64, 303)[:, :32] if hidden == 32 else _edge_rows(M, hidden, 303)
    sids = rng.integers(0, M * top_k, em).astype(np.int32)
    sids[rng.random(em) < 0.4] = M * top_k
    sids[rng.random(em) < 0.1] = -1
    packed = torch.full((em + 1, hidden // 2), 7, dtype=torch.uint8, device=dev())
    scales = torch.full((em + 1, hidden // 32), 7, dtype=torch.uint8, device=dev())
    d_A, d_s = to_dev(A), to_dev(sids)
    assert sq(d_A.data_ptr(), d_s.data_ptr(), packed.data_ptr(), scales.data_ptr(), M, hidden, 32, top_k, em,
              None) == 0
    torch.cuda.synchronize()
    rp, rs = oracle.mxfp4_moe_sorted_quant(A, sids, top_k)
    assert np.array_equal(packed.cpu().numpy(), np.r_[rp, np.full((1, hidden // 2), 7, np.uint8)])
    assert np.array_equal(scales.cpu().numpy(), np.r_[rs, np.full((1, hidden // 32), 7, np.uint8)])


def test_sorted_quant_and_scatter_reduce_bitwise(hip_lib):
    sq = hip_lib.vk_hip_mxfp4_moe_sorted_quant
    sq.restype = _I
    sq.argtypes = [_P, _P, _P, _P, _I, _I, _I, _I, _I, _P]
    sr = hip_lib.vk_hip_mxfp4_moe_scatter_reduce
    sr.restype = _I
    sr.argtypes = [_P, _P, _P, _P, _I, _I, _I, _I, _P, ctypes.c_size_t, _P]
    rng = np.random.default_rng(5)
    M, hidden, top_k, E = 70, 512, 4, 16
    A = _edge_rows(M, hidden, 302)
    ids = rng.integers(0, E, (M, top_k)).astype(np.int32)
    sids, _, em = oracle.moe_align_block_size(ids, 16, E)
    sids = sids[:em].copy()
    sids[5] = -3                                    # a negative id is padding too
    packed = torch.full((em, hidden // 2), 7, dtype=torch.uint8, device=dev())
    scales = torch.full((em, hidden // 32), 7, dtype=torch.uint8, device=dev())
    d_A, d_sids = to_dev(A), to_dev(sids)      # (kept alive until the synchronisation)
    assert sq(d_A.data_ptr(), d_sids.data_ptr(), packed.data_ptr(), scales.data_ptr(), M, hidden,
              32, top_k, em, None) == 0
    torch.cuda.synchronize()
    rp, rs = oracle.mxfp4_moe_sorted_quant(A, sids, top_k)
    assert np.array_equal(packed.cpu().numpy(), rp) and np.array_equal(scales.cpu().numpy(), rs)

    width = 2880
    partial = (rng.standard_normal((em, width)) * 100).astype(np.float32)
    tws = rng.random(em).astype(np.float32)
    base = rng.standard_normal((M, width)).astype(np.float32)      # the call accumulates
    out = to_dev(base.copy())
    ws = torch.zeros(M * top_k, dtype=torch.int32, device=dev())
    d_partial, d_tws = to_dev(partial), to_dev(tws)
    assert sr(d_partial.data_ptr(), d_tws.data_ptr(), d_sids.data_ptr(), out.data_ptr(), M,
              width, top_k, em, ws.data_ptr(), ws.numel() * 4, None) == 0
    torch.cuda.synchronize()
    ref = oracle.mxfp4_moe_scatter_reduce(partial, tws, sids, M, top_k, out=base.copy())
    assert np.array_equal(out.cpu().numpy().view(np.uint32), ref.view(np.uint32))
    assert sr(None, None, None, None, M, width, top_k, em, None, 0, None) == ve.VK_ERROR_INVALID_ARGUMENT


@pytest.mark.parametrize("hidden", [512, 2880, 76])
def test_sort_and_sort_scales_bitwise(hip_lib, hidden):
    """mxfp4_moe_sort / mxfp4_moe_sort_scales on the device: rows gathered into sorted
    order, padding rows (ids at or beyond M * top_k, negative ids) zeroed; byte for byte
    the oracle's.  hidden = 76: rows that are no multiple of 16 bytes (the byte-wise
    kernel), scale rows of 2 bytes."""
    st = hip_lib.vk_hip_mxfp4_moe_sort
    st.restype = _I
    st.argtypes = [_P, _P, _P, _I, _I, _I, _I, _P]
    ss = hip_lib.vk_hip_mxfp4_moe_sort_scales
    ss.restype = _I
    ss.argtypes = [_P, _P, _P, _I, _I, _I, _I, _P]
    rng = np.random.default_rng(hidden)
    M, top_k, E = 70, 4, 16
    A = rng.integers(0, 65536, (M, hidden)).astype(np.uint16)
    n_groups = max(hidden // 32, 1)
    scales = rng.integers(0, 256, (M, n_groups)).astype(np.uint8)
    ids = rng.integers(0, E, (M, top_k)).astype(np.int32)
    sids, _, em = oracle.moe_align_block_size(ids, 16, E)
    sids = sids[:em].copy()
    sids[3] = -1
    d_A, d_s, d_sids = to_dev(A), to_dev(scales), to_dev(sids)
    a_sorted = torch.full((em, hidden), 0x1234, dtype=torch.int16, device=dev())
    s_sorted = torch.full((em, n_groups), 9, dtype=torch.uint8, device=dev())
    assert st(d_A.data_ptr(), d_sids.data_ptr(), a_sorted.data_ptr(), M, hidden, top_k, em, None) == 0
    assert ss(d_s.data_ptr(), d_sids.data_ptr(), s_sorted.data_ptr(), M, n_groups, top_k, em, None) == 0
    torch.cuda.synchronize()
    assert np.array_equal(a_sorted.cpu().numpy().view(np.uint16), oracle.mxfp4_moe_sort(A, sids, top_k))
    assert np.array_equal(s_sorted.cpu().numpy(), oracle.mxfp4_moe_sort_scales(scales, sids, top_k))
    assert st(None, None, None, M, hidden, 0, em, None) == ve.VK_ERROR_INVALID_ARGUMENT
    assert ss(None, None, None, M, n_groups, top_k, em, None) == ve.VK_ERROR_INVALID_ARGUMENT
    assert st(None, None, None, M, hidden, top_k, 0, None) == 0              # nothing to do


def test_scatter_reduce_q_bitwise(hip_lib):
    """mxfp4_moe_scatter_reduce_q on the device: the routed combine of a quantised partial,
    dequantised inline; the same bits as the oracle (each product and each sum rounded on
    its own, rows in ascending order), with every code (inf and NaN included), scale bytes
    0, 1, 254 and 0xFF, and an `out` that already holds values."""
    fn = hip_lib.vk_hip_mxfp4_moe_scatter_reduce_q
    fn.restype = _I
    fn.argtypes = [_P, _P, _P, _P, _P, _I, _I, _I, _I, _I, _P, ctypes.c_size_t, _P]
    rng = np.random.default_rng(77)
    M, width, top_k, E = 70, 2880, 4, 16
    ids = rng.integers(0, E, (M, top_k)).astype(np.int32)
    sids, _, em = oracle.moe_align_block_size(ids, 16, E)
    sids = sids[:em].copy()
    sids[7] = -2
    pq = rng.integers(0, 256, (em, width // 2)).astype(np.uint8)
    fin = np.array(synth.FINITE_CODES, dtype=np.uint8)
    finite_rows = np.arange(em) % 4 != 0                               # three rows in four: finite codes only
    pq[finite_rows] = fin[pq[finite_rows] % 12 & 15] | (fin[(pq[finite_rows] >> 4) % 12] << 4)
    ps = rng.integers(110, 140, (em, width // 32)).astype(np.uint8)
    ps[:, 0] = 0
    ps[:, 1] = 1
    ps[:, 2] = 254
    ps[:, 3] = 255
    tws = rng.random(em).astype(np.float32)
    base = rng.standard_normal((M, width)).astype(np.float32)
    out = to_dev(base.copy())
    ws = torch.zeros(M * top_k, dtype=torch.int32, device=dev())
    d_pq, d_ps, d_tws, d_sids = to_dev(pq), to_dev(ps), to_dev(tws), to_dev(sids)
    assert fn(d_pq.data_ptr(), d_ps.data_ptr(), d_tws.data_ptr(), d_sids.data_ptr(), out.data_ptr(), M, width,
              top_k, em, 32, ws.data_ptr(), ws.numel() * 4, None) == 0, ve.last_error(hip_lib)
    torch.cuda.synchronize()
    ref = oracle.mxfp4_moe_scatter_reduce_q(pq, ps, tws, sids, M, top_k, out=base.copy())
    got = out.cpu().numpy()
    nan_g, nan_r = np.isnan(got), np.isnan(ref)
    assert np.array_equal(nan_g, nan_r) and nan_r.any() and not nan_r.all()
    assert np.array_equal(got.view(np.uint32)[~nan_r], ref.view(np.uint32)[~nan_r])
    assert fn(None, None, None, None, None, M, width, top_k, em, 32, None, 0, None) == ve.VK_ERROR_INVALID_ARGUMENT
    assert fn(None, None, None, None, None, M, width, top_k, em, 16, None, 0, None) == ve.VK_ERROR_UNSUPPORTED


def _check_w4a4(cfg, T, w, A_bits, logits, sample=128, wn=None):
    g = cfgs._run_gpu(cfg, w, A_bits, logits, None, True, prepack=True, w4a4=True)
    ids, tw = oracle.route_topk(logits, cfg.top_k, True)
    assert np.array_equal(g["ids"], ids)
    rows = np.arange(T) if sample is None or sample >= T else edge_tokens(g, T * cfg.top_k, cfg.top_k, sample, T)
    wn = w.numpy() if wn is None else wn
    oracle.set_act_model(1)
    try:
        cm = cpu_layer(A_bits[rows], wn, ids[rows], tw[rows], threads=16)
    finally:
        oracle.set_act_model(0)
    m_rel, m_l2, nf = error_metrics(g["out"][rows], cm["out"])
    c = cpu_layer(A_bits[rows], wn, ids[rows], tw[rows], threads=16)
    b_rel, b_l2, _ = error_metrics(g["out"][rows], c["out"])
    print(f"{cfg.name} T={T} W4A4 rows checked {rows.size}: vs oracle on the quantised activations "
          f"max_abs/rms={m_rel:.3e} rel_l2={m_l2:.3e}; vs the bf16-activation oracle rel_l2={b_l2:.3e}")
    # same operands on both sides: what differs is the order of the sums, and bf16 roundings
    # of act that fall the other way (each then moves its quantised value by a code step)
    assert nf and m_rel <= MAX_ABS_TOL and m_l2 <= REL_L2_TOL
    return g, wn


@pytest.mark.parametrize("T", [200, 513])
def test_w4a4_layer_config1(T):
    cfg = synth.CONFIGS["c1"]
    w = cfgs._weights(cfg, 1500)
    A, lg = cfgs._inputs(cfg, T, 6100 + T)
    _check_w4a4(cfg, T, w, A, lg)


def test_w4a4_layer_config3():
    cfg = synth.CONFIGS["c3"]
    w = cfgs._weights(cfg)
    A, lg = cfgs._inputs(cfg, 4096, 3000)
    _check_w4a4(cfg, 4096, w, A, lg, sample=96)


def test_w4a4_first_stage_matches_the_model_closely():
    """The first stage alone has no rounding between quantisation and output but the
    fp32 sums: act against the oracle's act on the quantised activations."""
    cfg = synth.CONFIGS["c1"]
    T = 200
    w = cfgs._weights(cfg, 1500)
    A, lg = cfgs._inputs(cfg, T, 6200)
    g = cfgs._run_gpu(cfg, w, A, lg, 16, True, prepack=True, w4a4=True)
    ids, tw = oracle.route_topk(lg, cfg.top_k, True)
    oracle.set_act_model(1)
    try:
        c = cpu_layer(A, w.numpy(), ids, tw, threads=16)
    finally:
        oracle.set_act_model(0)
    real = c["sorted_ids"] < T * cfg.top_k
    ga = synth.bf16_bits_to_f32(g["act"][:c["EM"]][real]).astype(np.float64)
    ca = synth.bf16_bits_to_f32(c["act"][real]).astype(np.float64)
    rms = float(np.sqrt(np.mean(ca ** 2)))
    excess = np.abs(ga - ca) - (1e-3 * rms + 2.0 ** -7 * np.abs(ca))
    assert float(excess.max()) <= 0.0
    assert float(np.linalg.norm(ga - ca) / np.linalg.norm(ca)) <= 2e-3


def test_w4a4_rows_outside_the_range_take_the_exact_path():
    cfg = synth.MoEConfig("t", 256, 512, 8, 2, (300,), "uniform")
    T, seed = 300, 6300
    w = synth.make_weights(cfg.E, cfg.H, cfg.I, seed, device=dev())
    r = synth.rand_u63(w.w13[0].numel(), seed, 32, dev()).reshape(w.w13[0].shape)
    w.w13[0][(r >> 10) % 4096 == 0] = 0x6E       # inf codes in one expert: flagged units
    A, lg = cfgs._inputs(cfg, T, seed)
    A = A.copy()
    A[2, :] = synth.f32_to_bf16_bits(synth.bf16_bits_to_f32(A[2, :]) * np.float32(2.0 ** 80))    # scale byte > 190
    A[3, :] = synth.f32_to_bf16_bits(synth.bf16_bits_to_f32(A[3, :]) * np.float32(2.0 ** -90))   # < 64
    A[4, :] = 0
    A[5, 7] = 0x7F80                              # an inf: its group quantises to zero
    g = cfgs._run_gpu(cfg, w, A, lg, None, True, prepack=True, w4a4=True)
    ids, tw = oracle.route_topk(lg, cfg.top_k, True)
    oracle.set_act_model(1)
    try:
        c = cpu_layer(A, w.numpy(), ids, tw, threads=16)
    finally:
        oracle.set_act_model(0)
    for t in range(T):
        max_rel, rel_l2, nf = error_metrics(g["out"][t], c["out"][t])
        assert nf and max_rel <= MAX_ABS_TOL and rel_l2 <= REL_L2_TOL, (t, max_rel, rel_l2)


@pytest.mark.parametrize("H,I", [(256, 64), (320, 128), (192, 192), (2304, 2176)])
def test_w4a4_stages_at_narrow_widths(H, I):
    """Second-stage rows that share a wavefront or have a workgroup each, widths that are no
    multiple of 128, and rows outside the range of the scaled products (their flag is per row)
    beside rows inside it, in the first stage, in the second or in both.  Each stage against the
    oracle on the same quantised operands, the second on the device's own act: the order of the
    fp32 sums is all that differs, and the bf16 rounding of act in the first stage."""
    cfg = synth.MoEConfig("t", H, I, 8, 2, (300,), "uniform")
    T, seed = 300, 6400 + I
    n_flat = T * cfg.top_k
    w = synth.make_weights(cfg.E, H, I, seed, device=dev())
    A, lg = cfgs._inputs(cfg, T, seed)
    # scale bytes beyond 64 .. 190: A's at 2^-66, act's at 2^-66, 2^-40 and 2^35
    power = np.array([0, 35, 0, -40, 0, -66, 20])[np.arange(T) % 7]
    A = synth.f32_to_bf16_bits((synth.bf16_bits_to_f32(A) * np.exp2(power)[:, None]).astype(np.float32))
    g = cfgs._run_gpu(cfg, w, A, lg, None, True, prepack=True, w4a4=True)
    ids, tw = oracle.route_topk(lg, cfg.top_k, True)
    wn = w.numpy()
    EM = g["max_EM"]
    eids16 = np.repeat(g["eids"], g["bs"] // 16).astype(np.int32)
    oracle.set_act_model(1)
    try:
        c = cpu_layer(A, wn, ids, tw, threads=16)
        partial = oracle.moe_down(g["act"], wn[2], wn[3], g["sids"], eids16, T, I, 0, I, H, cfg.top_k, EM)
    finally:
        oracle.set_act_model(0)
    ref = oracle.moe_combine(partial, None, oracle.gather_sorted_weights(tw, g["sids"]), g["sids"], eids16, T, H,
                             cfg.top_k, EM)
    g_act, c_act = np.zeros((n_flat, I)), np.zeros((n_flat, I))
    r = np.nonzero(g["sids"] < n_flat)[0]
    g_act[g["sids"][r]] = synth.bf16_bits_to_f32(g["act"][r])
    r = np.nonzero(c["sorted_ids"] < n_flat)[0]
    c_act[c["sorted_ids"][r]] = synth.bf16_bits_to_f32(c["act"][r])
    for p in np.unique(power):
        t = np.nonzero(power == p)[0]
        rows = (t[:, None] * cfg.top_k + np.arange(cfg.top_k)).ravel()
        ga, ca = g_act[rows], c_act[rows]
        assert np.all(np.isfinite(ga)) and np.all(np.isfinite(ca)), p
        excess = np.abs(ga - ca) - (1e-3 * np.sqrt(np.mean(ca ** 2)) + 2.0 ** -7 * np.abs(ca))
        assert float(excess.max()) <= 0.0, p
        got, exp = g["out"][t].astype(np.float64), ref[t].astype(np.float64)
        assert np.all(np.isfinite(got)) and np.all(np.isfinite(exp)), p
        scale = np.sqrt(np.mean(exp ** 2))
        if scale == 0.0:
            assert not got.any(), p
            continue
        worst, rel = np.abs(got - exp).max() / scale, np.linalg.norm(got - exp) / np.linalg.norm(exp)
        print(f"H={H} I={I} 2^{p}: max_abs/rms={worst:.3e} rel_l2={rel:.3e}")
        assert worst <= EXACT_SPLIT_MAX_ABS_TOL and rel <= EXACT_SPLIT_REL_L2_TOL, p
