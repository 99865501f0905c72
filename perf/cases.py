"""The work whose speed counts: the fused MXFP4 MoE layer as a serving program runs it.

Twelve listed cases and, through draw(), any other of the same ranges.  A case is

  path    "layer"  router, alignment and layer: FusedExperts.forward on weights prepacked at
                   load time (one copy of them), what a serving loop calls per MoE layer
          "apply"  FusedExperts.apply on the raw tensors, as they come from a checkpoint, with
                   the routing of the caller: the call of the reference's integration, a bf16
                   result included
          "split"  a tensor-parallel rank's share of the layer on its prepacked shard: the two
                   linear stages, the activation and the combine as separate calls, where the
                   all-reduces go between
          "aux"    the MXFP4 orchestration ops around somebody else's grouped GEMM: activations
                   quantised, once in token and once in sorted order, and the routed combine
  H, I, E, k       hidden and intermediate width, experts, experts per token
  T                tokens of the call
  skew             "uniform" router logits or "zipf": a few popular experts
  epilogue         "plain" SwiGLU, "clamp" (both biases and a clamp of 7) or "situ" (both
                   biases and the SiTU activation)
  w4a4             activations quantised to MXFP4 ("layer" only)
  tp               ranks that share K ("split" only, else 1)
"""
from __future__ import annotations

import ctypes
import math

import torch

from vkernels_amd import synth
from vkernels_amd import vllm_experts as ve

_P, _I, _F = ctypes.c_void_p, ctypes.c_int, ctypes.c_float


def _case(path, shape, T, *, skew="uniform", epilogue="plain", w4a4=False, tp=1, name=None):
    H, I, E, k = shape
    case = dict(path=path, H=H, I=I, E=E, k=k, T=T, skew=skew, epilogue=epilogue, w4a4=w4a4, tp=tp)
    return case if name is None else dict(case, name=name)


def _shape(config):
    cfg = synth.CONFIGS[config]
    return cfg.H, cfg.I, cfg.E, cfg.top_k


def listed():
    c1, c2, c3, c4 = (_shape(c) for c in ("c1", "c2", "c3", "c4"))
    return [
        # one user's next token: latency, launches and the host's work per call
        _case("layer", c1, 1, epilogue="clamp", name="decode_one"),
        # the decode batch of a busy server: the weights of every expert, once
        _case("layer", c1, 64, epilogue="clamp", name="decode_batch"),
        # the same from a caller that swapped the library in and keeps the raw tensors
        _case("apply", c1, 32, name="decode_raw"),
        # a large decode batch with popular experts: many passes for some, none for others
        _case("layer", c2, 512, skew="zipf", name="decode_skewed"),
        # decode and a piece of a prompt in one step, 24 rows an expert
        _case("layer", c4, 255, epilogue="situ", name="mixed_step"),
        # a ragged piece of a prompt (chunked prefill)
        _case("layer", c4, 1000, name="prefill_ragged"),
        # a large piece with popular experts, rows and columns that are no multiples of 128
        _case("layer", c2, 4096, skew="zipf", epilogue="clamp", name="prefill_skewed"),
        # the largest prefill: wide rows, many small experts, bound by the matrix cores
        _case("layer", c3, 16384, name="prefill_wide"),
        # a prefill from a caller that keeps the raw tensors
        _case("apply", c3, 4096, name="prefill_raw"),
        # a prefill with 4-bit activations
        _case("layer", c4, 8191, w4a4=True, name="prefill_w4a4"),
        # one of four tensor-parallel ranks, a piece of a prompt
        _case("split", c4, 2048, tp=4, name="rank_of_four"),
        # what goes around a 4-bit grouped GEMM of the caller's own
        _case("aux", c4, 4096, name="quant_and_combine"),
    ]


# Widths and expert counts beside the configurations': multiples of 64, as the layer asks for.
_WIDTHS = (256, 512, 704, 1024, 1536, 2048, 2880, 4096, 5120, 7168)
_LARGEST = 16384 * 8 * 7168 * 2048          # T k H I of the largest listed case
_LARGEST_WEIGHTS = 256 * 7168 * 2048        # E H I of it


def _log_int(rng, lo, hi):
    return min(hi, max(lo, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))))


def draw(rng):
    """Tokens spread over the logarithm of 1 .. 16384, on the configurations' shapes or on others."""
    path = rng.choice(("layer",) * 7 + ("apply",) * 3 + ("split",) + ("aux",))
    if rng.random() < 0.6:
        shape = _shape(rng.choice(("c0", "c1", "c2", "c3", "c4")))
    else:
        while True:
            H, I = rng.choice(_WIDTHS), rng.choice(_WIDTHS)
            E = rng.choice((8, 16, 32, 60, 64, 128, 256))
            if E * H * I <= _LARGEST_WEIGHTS // 2:
                break
        shape = (H, I, E, rng.choice((1, 2, 4, 6, 8)))
    H, I, E, k = shape
    most = min(16384 if path == "layer" else 4096, max(1, _LARGEST // (k * H * I) // 2))
    T = _log_int(rng, 1, most)
    tp = 1
    if path == "split":
        tp = max(t for t in (1, 2, rng.choice((2, 4))) if H % (64 * t) == 0 and I % (64 * t) == 0)
    return _case(path, shape, T, skew=rng.choice(("uniform", "uniform", "zipf")),
                 epilogue=rng.choice(("plain", "clamp", "situ")),
                 w4a4=path == "layer" and rng.random() < 0.15, tp=tp)


# ---- inputs ------------------------------------------------------------------------------------

def _popularity(E, seed):
    """log of a Zipf(s = 1.1) popularity over a permutation of the experts."""
    g = torch.Generator().manual_seed(seed)
    rank = torch.randperm(E, generator=g).double() + 1
    return torch.log(rank ** -1.1 / (rank ** -1.1).sum()).float()


def _codes(shape, gen, dev):
    """Packed E2M1 codes, the codes of inf and NaN (6 and 7 of either sign) replaced by finite
    ones, as a checkpoint's are."""
    n = math.prod(shape)
    out = torch.empty(n, dtype=torch.uint8, device=dev)
    words = out.view(torch.int64)           # (every width is a multiple of 64)
    step = 1 << 25
    for at in range(0, words.numel(), step):
        w = torch.randint(-2 ** 63, 2 ** 63 - 1, (min(step, words.numel() - at),), dtype=torch.int64,
                          device=dev, generator=gen)
        high = (w >> 1) & w & 0x2222222222222222     # bits 2 and 1 both set: 6 and 7
        w &= ~(high << 1)                            # ... become 2 and 3
        words[at:at + w.numel()] = w
    return out.view(shape)


def _scales(shape, gen, dev):
    """ue8m0 bytes, exponents -4 .. 2."""
    return torch.randint(123, 130, shape, dtype=torch.uint8, device=dev, generator=gen)


def _weights(E, H, I, gen, dev):
    return (_codes((E, 2 * I, H // 2), gen, dev), _scales((E, 2 * I, H // 32), gen, dev),
            _codes((E, H, I // 2), gen, dev), _scales((E, H, I // 32), gen, dev))


def _epilogue_args(case, gen, dev):
    if case["epilogue"] == "plain":
        return {}
    kw = dict(b13=0.5 * torch.randn((case["E"], 2 * case["I"]), device=dev, generator=gen),
              b2=0.5 * torch.randn((case["E"], case["H"]), device=dev, generator=gen))
    if case["epilogue"] == "clamp":
        return dict(kw, swiglu_limit=7.0)
    return dict(kw, activation="situ", beta=3.0, linear_beta=20.0)


def prepare(case, seed):
    dev = torch.device("cuda", torch.cuda.current_device())
    gen = torch.Generator(device=dev).manual_seed(seed)
    H, I, E, k, T = (case[n] for n in ("H", "I", "E", "k", "T"))
    state = dict(case=case, A=torch.randn((T, H), device=dev, generator=gen).to(torch.bfloat16))
    logits = torch.randn((T, E), device=dev, generator=gen)
    if case["skew"] == "zipf":
        logits += _popularity(E, seed).to(dev)
    if case["path"] == "aux":
        return _prepare_aux(state, logits, gen, dev)
    if case["path"] == "split":
        return _prepare_split(state, logits, gen, dev)
    packed = case["path"] == "layer"
    fe = ve.FusedExperts(*_weights(E, H, I, gen, dev), prepack=packed, keep_raw=not packed,
                         w4a4=case["w4a4"], **_epilogue_args(case, gen, dev))
    state["experts"] = fe
    if packed:
        state["logits"] = logits
    else:
        state["topk_ids"], state["topk_w"] = fe.route(logits, k)
    return state


def _ptr(t):
    return None if t is None else t.data_ptr()


def _bind(lib, name, argtypes):
    fn = getattr(lib, name)
    fn.restype, fn.argtypes = _I, argtypes
    return fn


def _aligned(logits, k, packed_experts, H, I):
    """Routing and alignment of the tokens on this device: (ids, weights, sorted ids, expert of
    each block, rows the arrays are sized for, block size)."""
    lib = ve.load_libvkernels_hip()
    T, E = logits.shape
    dev = logits.device
    bs = ve.default_block_size(T, k, lib, packed_experts=packed_experts, hidden=H, ispp=I)
    em = ve._align_em_bound(T, k, E, bs)
    ids = torch.empty((T, k), dtype=torch.int32, device=dev)
    w = torch.empty((T, k), dtype=torch.float32, device=dev)
    sids = torch.empty(em, dtype=torch.int32, device=dev)
    eids = torch.empty(em // bs, dtype=torch.int32, device=dev)
    out_em = torch.empty(1, dtype=torch.int32, device=dev)
    status = ve.resolve_route_align_fn(lib)(_ptr(logits), T, E, k, 1, None, bs, E, em, _ptr(ids), _ptr(w),
                                            _ptr(sids), _ptr(eids), _ptr(out_em), ve._stream(torch))
    assert status == 0, ve.last_error(lib)
    return ids, w, sids, eids, em, bs


def _prepare_aux(state, logits, gen, dev):
    case = state["case"]
    H, k = case["H"], case["k"]
    lib = ve.load_libvkernels_hip()
    _, w, sids, _, em, _ = _aligned(logits, k, 0, H, case["I"])
    partial = torch.randn((em, H), device=dev, generator=gen)   # what the grouped GEMM hands over
    state.update(
        topk_w=w, sorted_ids=sids, EM=em, partial=partial, A=state["A"],
        inverse=torch.empty(case["T"] * k, dtype=torch.int32, device=dev),
        quant=_bind(lib, "vk_hip_mxfp4_moe_quant", [_P] * 3 + [_I] * 3 + [_P]),
        sorted_quant=_bind(lib, "vk_hip_mxfp4_moe_sorted_quant", [_P] * 4 + [_I] * 5 + [_P]),
        reduce=_bind(lib, "vk_hip_mxfp4_moe_scatter_reduce", [_P] * 4 + [_I] * 4 + [_P, ctypes.c_size_t, _P]))
    return state


def _prepare_split(state, logits, gen, dev):
    case = state["case"]
    H, I, E, k, T, tp = (case[n] for n in ("H", "I", "E", "k", "T", "tp"))
    lib = ve.load_libvkernels_hip()
    size_fn, pack_fn, _ = ve.resolve_prepack_fns(lib)
    hk, ik = H // tp, I // tp
    packed = []
    for stage, (rows, K) in enumerate(((2 * I, hk), (H, ik))):
        w, s = _codes((E, rows, K // 2), gen, dev), _scales((E, rows, K // 32), gen, dev)
        n = size_fn(E, rows, K, stage)
        buf = torch.empty(n, dtype=torch.uint8, device=dev)
        status = pack_fn(_ptr(w), _ptr(s), E, rows, K, stage, _ptr(buf), n, ve._stream(torch))
        assert status == 0, ve.last_error(lib)
        packed.append(buf)
    ids, w, sids, eids, em, bs = _aligned(logits, k, E, H, I)
    # the routing weight of every sorted row (0 where none is routed)
    w_sorted = torch.cat([w.reshape(-1), w.new_zeros(1)])[sids.long().clamp(max=T * k)]
    ws_bytes = _bind(lib, "vk_hip_moe_preact_workspace_bytes", [_I] * 4)
    ws_bytes.restype = ctypes.c_size_t
    n = max(ws_bytes(0, T, em, hk), ws_bytes(1, T, em, ik), T * k * 4)
    stage_args = [_P] * 4 + [_I] + [_P] * 3 + [_I] * 8 + [_P, ctypes.c_size_t, _I, _P]
    state.update(
        packed=packed, sorted_ids=sids, expert_ids=eids, w_sorted=w_sorted, EM=em, bs=bs,
        epilogue=_epilogue_args(case, gen, dev),
        workspace=torch.empty(n, dtype=torch.uint8, device=dev),
        gate_up=torch.zeros((em, 2 * I), dtype=torch.float32, device=dev),
        act=torch.zeros((em, I), dtype=torch.bfloat16, device=dev),
        partial=torch.zeros((em, H), dtype=torch.float32, device=dev),
        gateup_fn=_bind(lib, "vk_hip_moe_gateup_preact_prepacked", stage_args),
        act_fn=_bind(lib, "vk_hip_moe_act_epilogue", [_P] * 5 + [_I] * 4 + [_F, _I, _F, _F, _I, _P]),
        down_fn=_bind(lib, "vk_hip_moe_down_preact_prepacked", stage_args),
        combine_fn=_bind(lib, "vk_hip_moe_combine", [_P] * 6 + [_I] * 5 + [_P, ctypes.c_size_t, _P]))
    return state


# ---- one pass -----------------------------------------------------------------------------------

def run(state):
    case = state["case"]
    if case["path"] == "layer":
        return state["experts"].forward(state["A"], state["logits"], case["k"])
    if case["path"] == "apply":
        return state["experts"].apply(state["A"], state["topk_ids"], state["topk_w"],
                                      output_dtype=torch.bfloat16)
    return (_run_split if case["path"] == "split" else _run_aux)(state)


def _run_split(s):
    """Without the all-reduces: the rank's own gate/up and down sums, and what the activation and
    the combine make of them."""
    case = s["case"]
    H, I, E, k, T, tp = (case[n] for n in ("H", "I", "E", "k", "T", "tp"))
    em, bs, epi, st = s["EM"], s["bs"], s["epilogue"], ve._stream(torch)
    sids, eids = _ptr(s["sorted_ids"]), _ptr(s["expert_ids"])
    ws, n = _ptr(s["workspace"]), s["workspace"].numel()
    out = torch.zeros((T, H), dtype=torch.float32, device=s["A"].device)
    status = s["gateup_fn"](_ptr(s["A"]), None, None, _ptr(s["packed"][0]), E, sids, eids, _ptr(s["gate_up"]),
                            T, H, I, k, em, 0, H // tp, bs, ws, n, 0, st)
    status |= s["act_fn"](_ptr(s["gate_up"]), _ptr(epi.get("b13")), _ptr(s["act"]), sids, eids, T, k, em, I,
                          epi.get("swiglu_limit", 0.0), int(epi.get("activation") == "situ"),
                          epi.get("beta", 4.0), epi.get("linear_beta", 25.0), bs, st)
    status |= s["down_fn"](_ptr(s["act"]), None, None, _ptr(s["packed"][1]), E, sids, eids, _ptr(s["partial"]),
                           T, I, H, k, em, 0, I // tp, bs, ws, n, 0, st)
    status |= s["combine_fn"](_ptr(s["partial"]), _ptr(epi.get("b2")), _ptr(s["w_sorted"]), sids, eids,
                              _ptr(out), T, H, k, em, bs, ws, n, st)
    if status:
        raise RuntimeError(ve.last_error(ve.load_libvkernels_hip()))
    return out, s["gate_up"], s["act"], s["partial"]


def _run_aux(s):
    case = s["case"]
    H, k, T, em = case["H"], case["k"], case["T"], s["EM"]
    dev, st = s["A"].device, ve._stream(torch)
    codes = torch.empty((T, H // 2), dtype=torch.uint8, device=dev)
    scales = torch.empty((T, H // 32), dtype=torch.uint8, device=dev)
    s_codes = torch.empty((em, H // 2), dtype=torch.uint8, device=dev)
    s_scales = torch.empty((em, H // 32), dtype=torch.uint8, device=dev)
    out = torch.zeros((T, H), dtype=torch.float32, device=dev)
    status = s["quant"](_ptr(s["A"]), _ptr(codes), _ptr(scales), T, H, 32, st)
    status |= s["sorted_quant"](_ptr(s["A"]), _ptr(s["sorted_ids"]), _ptr(s_codes), _ptr(s_scales),
                                T, H, 32, k, em, st)
    status |= s["reduce"](_ptr(s["partial"]), _ptr(s["topk_w"]), _ptr(s["sorted_ids"]), _ptr(out), T, H, k, em,
                          _ptr(s["inverse"]), T * k * 4, st)
    if status:
        raise RuntimeError(ve.last_error(ve.load_libvkernels_hip()))
    return codes, scales, s_codes, s_scales, out


# ---- what a pass cannot do without -----------------------------------------------------------------

def _active_experts(case):
    """Experts that at least one of the tokens is routed to."""
    E, k, T = case["E"], case["k"], case["T"]
    if case["skew"] == "uniform":
        return E * (1.0 - (1.0 - k / E) ** T)
    g = torch.Generator().manual_seed(1)
    logits = torch.randn((T, E), generator=g) + _popularity(E, 1)
    return float(torch.topk(logits, k, dim=1).indices.unique().numel())


def work(case):
    H, I, E, k, T, tp = (case[n] for n in ("H", "I", "E", "k", "T", "tp"))
    rows = T * k
    if case["path"] == "aux":
        quantised = H / 2 + H / 32
        em = ve._align_em_bound(T, k, E, ve.default_block_size(T, k))
        # activations in, codes out in both orders, the routed partial rows in, the result out
        return {"bytes": 2 * T * H + T * quantised + em * quantised + 4 * rows * H + 4 * T * H + 8 * rows,
                "flops": 2.0 * rows * H}
    active = _active_experts(case)
    weights = active * (17 / 32) * 3 * H * I / tp       # codes and scale bytes, each once
    flops = 6.0 * rows * H * I / tp
    if case["path"] == "split":
        # the linear parts leave as fp32 rows and come back (the all-reduces read them)
        between = rows * (2 * 4 * 2 * I + 2 * 2 * I + 2 * 4 * H)
        return {"bytes": weights + 2 * T * H / tp + between + 4 * T * H, "flops": flops}
    routing = 4 * T * E if case["path"] == "layer" else 8 * rows
    return {"bytes": weights + 2 * T * H + routing + (4 if case["path"] == "layer" else 2) * T * H,
            "flops": flops}


def tolerance(case):
    """Measured against the layer in 64-bit sums (48 tokens of every listed case and of drawn ones),
    times four: 1.8e-4 and at most 4.4e-3 for an element where the activations are multiplied
    exactly (decode sizes), 5.2e-4 and 4.8e-3 where they are two or three FP6 terms, 1.7e-3 and
    5e-3 where the result is rounded to bf16.  4-bit activations: 6e-8, but another order of
    the first stage's sums moves one activation in a million across a rounding threshold of the
    quantisation, a quarter of its value."""
    rows = case["T"] * case["k"]
    if case["path"] == "aux":
        return "exact"
    if case["path"] == "apply":
        return {"rel": 6e-3, "max": 2e-2}
    if case["path"] == "layer" and rows <= max(512, 28 * case["E"]):
        return {"rel": 7e-4, "max": 1.8e-2}
    if case["w4a4"]:
        return {"rel": 1e-3, "max": 5e-2}
    return {"rel": 2e-3, "max": 2e-2}
