"""The prefill kernels on the raw tensors: their loads, lane offsets and K loop's schedule walked on
the CPU (tests/prefill_raw_layout_check.cpp), and on the GPU against the same call on prepacked
weights with three terms in both stages, which multiplies and adds the same values in the same
order: the same bits, whatever the window, the epilogue or the path of a unit."""
from __future__ import annotations

import ctypes
import subprocess
import sys
from pathlib import Path

import pytest
import torch

ROOT = Path(__file__).resolve().parents[1]
sys.path.insert(0, str(ROOT))
from vkernels_amd import vllm_experts as ve  # noqa: E402


def _build(tmp_path, *defines):
    exe = tmp_path / "prefill_raw_layout_check"
    subprocess.run(["g++", "-O2", "-std=c++17", "-Wall", "-Werror", *defines, f"-I{ROOT / 'vkernels_amd' / 'csrc'}",
                    str(ROOT / "tests" / "prefill_raw_layout_check.cpp"), "-o", str(exe)], check=True)
    return exe


def test_offsets_and_schedule(tmp_path):
    exe = _build(tmp_path)
    for args in ("0 7168 2048 3", "1 2048 7168 3", "0 4096 1536 2", "1 1536 4096 2", "0 512 512 2", "1 512 512 2",
                 "1 512 704 2"):  # (the last unit of the last is ragged)
        res = subprocess.run([str(exe), *args.split()], capture_output=True, text=True)
        assert res.returncode == 0, f"{args}: {res.stderr.strip()}"


@pytest.mark.parametrize("wait", [0, 1])
def test_the_walk_notices_a_wait_that_counts_wrong(tmp_path, wait):
    exe = _build(tmp_path, f"-DVK_LAYOUT_BREAK_WAIT={wait}")
    assert subprocess.run([str(exe), "0", "7168", "2048", "3"], capture_output=True).returncode == 1


@pytest.fixture(scope="module")
def raw_rule(tmp_path_factory):
    """mx_raw_pays (moe_prefill_layout.hpp), compiled for the host: rows, EM, block, ispp, hidden -> taken?"""
    d = tmp_path_factory.mktemp("rule")
    (d / "rule.cpp").write_text('''#include "moe_prefill_layout.hpp"
extern "C" int pays(long long r, long long em, int b, int i, int h) { return vk::mx_raw_pays(r, em, b, i, h); }''')
    subprocess.run(["g++", "-O1", "-std=c++17", "-Wall", "-Werror", "-shared", "-fPIC",
                    f"-I{ROOT / 'vkernels_amd' / 'csrc'}", str(d / "rule.cpp"), "-o", str(d / "rule.so")], check=True)
    fn = ctypes.CDLL(str(d / "rule.so")).pays
    fn.argtypes = [ctypes.c_longlong, ctypes.c_longlong, ctypes.c_int, ctypes.c_int, ctypes.c_int]
    return fn


@pytest.mark.parametrize("H,I,E,k", [(7168, 2048, 256, 8), (4096, 1536, 64, 6), (1024, 512, 60, 4)])
@pytest.mark.parametrize("block,refused,taken", [
    # rows an expert: the raw form was measured behind at all the first, ahead at the second where
    # its rounds of workgroups are not nearly empty
    (16, (12, 24, 36, 64, 96), 192), (32, (12, 24, 36, 64, 96), 192), (64, (12, 24, 36, 48), 192),
    (128, (12, 24, 36, 48, 64), 192), (48, (12, 24, 36), 192), (80, (24, 36), 192), (96, (24, 36), 192), (112, (24, 36), 192),
])
def test_few_rows_a_segment_are_left_to_the_other_kernel(raw_rule, H, I, E, k, block, refused, taken):
    for rows in refused:
        T = rows * E // k
        assert not raw_rule(T * k, ve._align_em_bound(T, k, E, block), block, I, H), rows
        assert not raw_rule(T * k, (T * k + block - 1) // block * block + E * block, block, I, H), rows
    T = taken * E // k
    assert raw_rule(T * k, ve._align_em_bound(T, k, E, block), block, I, H)


@pytest.mark.parametrize("block", [16, 48, 64, 128, 256])
def test_the_rule_takes_any_sizes(raw_rule, block):
    """... of a valid call: EM below the rows (an expert map drops the others; refused), or far above."""
    for rows in (1, 513, 8192, 2 ** 31 - 1):
        for em in (block, rows // 2 // block * block + block, 2 ** 31 - 1):
            for width in (64, 512, 7168):
                assert raw_rule(rows, em, block, width, width) in ((0,) if em < rows else (0, 1))


def _weights(E, H, I, gen, special):
    def codes(*shape):
        c = torch.randint(0, 256, shape, dtype=torch.uint8, device="cuda", generator=gen)
        finite = c & ~((((c >> 1) & c) & 0x22) << 1)     # codes 6 and 7 of either sign become 2 and 3
        return finite
    def scales(*shape):
        return torch.randint(120, 131, shape, dtype=torch.uint8, device="cuda", generator=gen)
    w = [codes(E, 2 * I, H // 2), scales(E, 2 * I, H // 32), codes(E, H, I // 2), scales(E, H, I // 32)]
    if special:  # units that take the exact path: an infinity, a NaN, scale bytes at and past the range's ends
        w[0][0, 3, 5] = 0x06
        w[2][E - 1, H - 1, I // 2 - 1] = 0x70
        w[1][1, 2 * I - 1, H // 32 - 1] = 63
        w[1][1, 70, 0] = 64
        w[3][1, 200, 3] = 191
        w[3][2, 130, 1] = 190
    return w


# rows a block of 50 on, and rounds of workgroups that are not nearly empty (the call's own rule);
# H, I multiples of 512: the shortest loops (4 K steps), windows of 1 to 4 live row tiles
@pytest.mark.gpu
@pytest.mark.parametrize("H,I,E,k,T,epilogue,special", [
    (512, 512, 4, 2, 9999, "plain", False), (512, 512, 4, 2, 10111, "clamp", True),
    (1024, 512, 60, 4, 3000, "situ", False), (1024, 1536, 16, 2, 7001, "plain", True),
    (4096, 1536, 64, 6, 1100, "clamp", False),
])
def test_same_bits_as_on_prepacked_weights(H, I, E, k, T, epilogue, special):
    gen = torch.Generator(device="cuda").manual_seed(T)
    w = _weights(E, H, I, gen, special)
    kw = {}
    if epilogue != "plain":
        kw = dict(b13=torch.randn((E, 2 * I), device="cuda", generator=gen),
                  b2=torch.randn((E, H), device="cuda", generator=gen))
        kw.update(dict(swiglu_limit=7.0) if epilogue == "clamp" else dict(activation="situ", beta=3.0, linear_beta=20.0))
    A = torch.randn((T, H), device="cuda", generator=gen).to(torch.bfloat16)
    if special:
        A[5, 7], A[T - 1, H - 1] = float("inf"), 1e-38   # rows outside the range of the split
    logits = torch.randn((T, E), device="cuda", generator=gen)
    raw = ve.FusedExperts(*w, **kw)
    packed = ve.FusedExperts(*w, prepack=True, split_terms=3, **kw)
    ids, tw = raw.route(logits, k)
    assert raw.block_size_for(T, k) == 128
    a = raw.apply(A, ids, tw, output_dtype=torch.float32)
    b = packed.apply(A, ids, tw, output_dtype=torch.float32)
    assert torch.equal(torch.isnan(a), torch.isnan(b))
    assert torch.equal(torch.nan_to_num(a), torch.nan_to_num(b))
    # ... and it was the raw form that ran: the other kernel's two FP8 terms round differently
    other = _other_kernel(raw).apply(A, ids, tw, output_dtype=torch.float32)
    assert not torch.equal(torch.nan_to_num(a), torch.nan_to_num(other))


def _other_kernel(fe):
    """Has fe's calls run tile_wide_kernel: a workspace too short for the FP4-rate kernels' rows."""
    size = fe.ws_bytes_fn
    fe.ws_bytes_fn = lambda *a: size(*a) - 256
    return fe


# A rank's share of the experts: most rows are other ranks', which the rule cannot see in M * top_k
@pytest.mark.gpu
@pytest.mark.parametrize("entry", ["apply", "route_layer"])
def test_mapped_calls_are_left_to_the_other_kernel(entry):
    H, I, E, k, T, ranks = 1024, 512, 15, 4, 3000, 4
    gen = torch.Generator(device="cuda").manual_seed(3)
    w = _weights(E, H, I, gen, False)
    A = torch.randn((T, H), device="cuda", generator=gen).to(torch.bfloat16)
    logits = torch.randn((T, E * ranks), device="cuda", generator=gen)
    local = torch.full((E * ranks,), -1, dtype=torch.int32, device="cuda")
    local[::ranks] = torch.arange(E, dtype=torch.int32, device="cuda")
    def call(fe, A, logits):
        if entry == "route_layer":
            return fe.route_layer(A, logits, k)[0]
        ids, tw = fe.route(logits, k)
        return fe.apply(A, ids, tw, output_dtype=torch.float32)
    mapped = [call(f(ve.FusedExperts(*w, expert_map=local, local_num_experts=E)), A, logits)
              for f in (lambda fe: fe, _other_kernel)]
    assert torch.equal(*mapped)
    # (without a map the same sizes are the raw form's, which rounds differently)
    own = logits[:, :E].contiguous()
    plain = [call(f(ve.FusedExperts(*w)), A, own) for f in (lambda fe: fe, _other_kernel)]
    assert not torch.equal(*plain)
    torch.testing.assert_close(*plain, rtol=0, atol=2e-2 * float(plain[1].pow(2).mean().sqrt()))


# Several experts' rows in a window: the ring and each wavefront's scale bytes are used again from one
# segment to the next; blocks that are windows of their own (48, 112); rows that a map drops
@pytest.mark.gpu
@pytest.mark.parametrize("block,dropped", [(16, 0), (32, 0), (48, 0), (64, 0), (112, 0), (256, 0), (16, 7), (64, 7), (128, 7)])
def test_same_bits_in_other_blocks_and_under_a_map(block, dropped):
    H, I, E, k, T = 1024, 512, 60, 4, 3000 if block != 256 else 4500
    gen = torch.Generator(device="cuda").manual_seed(block)
    w = _weights(E, H, I, gen, True)
    kw = dict(b13=torch.randn((E, 2 * I), device="cuda", generator=gen), b2=torch.randn((E, H), device="cuda", generator=gen))
    if dropped:  # experts in another order, a few of them elsewhere
        perm = torch.randperm(E, device="cuda", generator=gen).to(torch.int32)
        kw["expert_map"] = torch.where(perm < E - dropped, perm, torch.full_like(perm, -1))
    A = torch.randn((T, H), device="cuda", generator=gen).to(torch.bfloat16)
    A[5, 7], A[T - 1, H - 1] = float("inf"), 1e-38
    logits = torch.randn((T, E), device="cuda", generator=gen)
    raw, packed = ve.FusedExperts(*w, **kw), ve.FusedExperts(*w, prepack=True, split_terms=3, **kw)
    ids, tw = raw.route(logits, k)
    a, b, other = (fe.apply(A, ids, tw, block_size=block, output_dtype=torch.float32).nan_to_num()
                   for fe in (raw, packed, _other_kernel(ve.FusedExperts(*w, **kw))))
    assert torch.equal(a, b)
    assert not torch.equal(a, other)


# The second stage alone; a last unit that is ragged (704 = 5 units of 128 and half of one), its bias too
@pytest.mark.gpu
@pytest.mark.parametrize("H,block", [(704, 128), (704, 64), (1024, 128)])
def test_same_bits_of_the_second_stage_alone(H, block):
    I, E, M = 512, 4, 11000
    gen = torch.Generator(device="cuda").manual_seed(H)
    w = _weights(E, H, I, gen, False)
    b2 = torch.randn((E, H), device="cuda", generator=gen)
    packed = ve.FusedExperts(*w, prepack=True)
    ids = torch.randint(0, E, (M, 1), device="cuda", generator=gen).to(torch.int32)
    tw = torch.rand((M, 1), device="cuda", generator=gen)
    sids, eids, _, em = packed.align(ids, block)
    act = torch.randn((em, I), device="cuda", generator=gen).to(torch.bfloat16)
    need = int(packed.ws_bytes_fn(M, H, I, 1, em))
    ws = torch.empty(need, dtype=torch.uint8, device="cuda")
    fn = packed.lib.vk_hip_moe_down_mxfp4_ex
    fn.restype, P, N = None, ctypes.c_void_p, ctypes.c_int
    fn.argtypes = [P] * 5 + [N] * 4 + [P, P, N, P, N, P, ctypes.c_size_t, ctypes.c_uint, P, N, P]

    def call(size, w2_packed):
        out = torch.full((M, H), float("nan"), device="cuda")
        packed.lib.vk_set_last_error(0, b"")
        fn(act.data_ptr(), w[2].data_ptr(), w[3].data_ptr(), tw.data_ptr(), out.data_ptr(), M, H, I, 1, sids.data_ptr(),
           eids.data_ptr(), em, b2.data_ptr(), block, ws.data_ptr(), size, ve.MOE_OVERWRITE_OUT | ve.MOE_SPLIT3,
           w2_packed, E, torch.cuda.current_stream().cuda_stream)
        torch.cuda.synchronize()
        assert packed.lib.vk_last_error_code() == 0, ve.last_error(packed.lib)
        return out
    raw = call(need, None)
    assert torch.isfinite(raw).all()
    assert torch.equal(raw, call(need, packed.w2_packed.data_ptr()))
    assert not torch.equal(raw, call(need - 256, None))    # (the kernel that takes it in a shorter workspace)
