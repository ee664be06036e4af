"""The calls that a user of this backend makes, as cases whose time is measured.

Sizes are those of the model that the backend serves (dim 4096, expert inner
size 2048, 256 experts of which a token takes 6, the attention projections of
bench.py's ATTN_FP8 and the 129280-row head) and of the repository's benchmark
configurations; token counts run from one decoded token to a 4096-token
prefill chunk. Kinds of case:

layer   apus_hip_moe_forward_dev: a whole MoE sublayer (router, expert choice
        by scores or by the hash table, routed experts, FP8 shared expert).
routed  apus_hip_moe_routed_dev: the routed experts alone, the routing given.
attn    apus_hip_linear_dev: the five FP8 projections of one attention layer.
linear  apus_hip_linear_dev: one FP8 or MXFP4 linear, resident (tiled) or
        row-major weights, whatever shape.
experts apus_hip_act_quant_dev + apus_hip_gemm_grouped_dev: expert matrices
        sharing a few activation rows.
plain   apus_hip_wlinear_dev: FP32 or BF16 weights (the LM head, the output
        projection's groups, the router gate).
hook    apus_hip_fp8_linear: the engine's hook, host pointers in and out.

Weights: E2M1 nibbles uniform over their 16 codes with E8M0 group scales that
bring the values to about 1/sqrt(K); E4M3 of N(0, 1) with log-uniform tile
scales. Activations are BF16-valued N(0, 1), as hidden states after a norm.
"""
import ctypes as C
import math
import os
import sys

import numpy as np
import torch

_ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
sys.path.insert(0, os.path.join(_ROOT, "apus-deepseek-v4-flash_amd"))
import apus_hip as H  # noqa: E402

DIM, INTER, EXPERTS, VOCAB = 4096, 2048, 256, 129280
LIMIT, ROUTE_SCALE = 10.0, 2.5
#: name, O, K and which input (0: hidden state, 1: query latent, 2: heads' output)
ATTN = (("wq_a", 1024, 4096, 0), ("wq_b", 32768, 1024, 1), ("wkv", 512, 4096, 0),
        ("wo_b", 4096, 8192, 2), ("idx_wq_b", 8192, 1024, 1))
ATTN_IN = (4096, 1024, 8192)
FP4, FP8 = 0, 1


def listed():
    return [
        # one decoded token through a MoE sublayer: the latency of chat decode
        {"name": "moe_layer_1", "kind": "layer", "tokens": 1, "topk": 6, "hash": False},
        # batched decode, 64 sequences, routed by seeded gating (benchmark config 2)
        {"name": "moe_routed_64", "kind": "routed", "tokens": 64, "topk": 6, "zipf": 0.0},
        # a 512-token prompt, expert popularity Zipf(1.1) (benchmark config 3)
        {"name": "moe_routed_512", "kind": "routed", "tokens": 512, "topk": 6, "zipf": 1.1},
        # a long prompt's prefill chunk through a hash-routed layer: the largest call
        {"name": "moe_layer_4096", "kind": "layer", "tokens": 4096, "topk": 6, "hash": True},
        # attention projections: one decoded token, a ragged prompt
        {"name": "attn_1", "kind": "attn", "tokens": 1},
        {"name": "attn_1000", "kind": "attn", "tokens": 1000},
        # batched decode: the attention output projection of 40 sequences
        {"name": "fp8_linear_40", "kind": "linear", "fmt": FP8, "tiled": True, "tokens": 40,
         "O": 4096, "K": 8192},
        # a square FP8 projection over a 512-token prompt (benchmark config 1)
        {"name": "fp8_linear_512", "kind": "linear", "fmt": FP8, "tiled": True, "tokens": 512,
         "O": 4096, "K": 4096},
        # the w1/w3 matrices of a token's six experts in one launch (benchmark config 0)
        {"name": "experts_12", "kind": "experts", "fmt": FP4, "entries": 12, "rows": 1,
         "O": 2048, "K": 4096},
        # the LM head for one token
        {"name": "head_1", "kind": "plain", "tokens": 1, "O": VOCAB, "K": DIM, "flags": 4},
        # one BF16 group of the attention output projection over a prompt
        {"name": "wo_a_512", "kind": "plain", "tokens": 512, "O": 1024, "K": 4096, "flags": 6},
        # a decode step's output projection from the CPU engine, through its hook
        {"name": "hook_wo_b_1", "kind": "hook", "tokens": 1, "O": 4096, "K": 8192},
    ]


def _log_int(rng, lo, hi):
    return min(hi, max(lo, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))))


def _no_result(fmt, m, K):
    """Resident FP8 weights with K = 1024 and 9..64 rows: when these cases were
    written the backend misread that shape's tile scales, so it has no result
    that a later one could be compared with."""
    return fmt == FP8 and K == 1024 and 9 <= m <= 64


def draw(rng):
    kind = rng.choice(("layer", "routed", "attn", "linear", "experts", "plain", "hook"))
    if kind == "layer":
        s = _log_int(rng, 1, 4096)
        # expert choice by scores up to decode batches; prompts by the hash
        # table, so that a near-tie of two scores is no difference
        return {"kind": kind, "tokens": s, "topk": rng.choice((6, 6, 8)) if s <= 2048 else 6,
                "hash": s > 128 or rng.random() < 0.3}
    if kind == "routed":
        s = _log_int(rng, 1, 4096)
        return {"kind": kind, "tokens": s, "topk": rng.choice((6, 6, 8)) if s <= 2048 else 6,
                "zipf": rng.choice((0.0, 0.6, 1.1))}
    if kind == "attn":
        s = _log_int(rng, 2, 4096)
        return {"kind": kind, "tokens": s + 56 if _no_result(FP8, s, 1024) else s}
    if kind == "linear":
        fmt = rng.choice((FP4, FP8))
        if rng.random() < 0.6:
            m, K = _log_int(rng, 1, 4096), rng.choice((1024, 2048, 4096, 8192))
            return {"kind": kind, "fmt": fmt, "tiled": True, "tokens": m, "O": 128 * _log_int(rng, 1, 64),
                    "K": 2048 if _no_result(fmt, m, K) else K}
        return {"kind": kind, "fmt": fmt, "tiled": False, "tokens": _log_int(rng, 1, 512),
                "O": _log_int(rng, 16, 4096), "K": 128 * _log_int(rng, 1, 64)}
    if kind == "experts":
        return {"kind": kind, "fmt": rng.choice((FP4, FP4, FP8)), "entries": _log_int(rng, 2, 48),
                "rows": _log_int(rng, 1, 8), "O": rng.choice((2048, 4096)), "K": rng.choice((2048, 4096))}
    if kind == "plain":
        if rng.random() < 0.3:
            return {"kind": kind, "tokens": 1, "O": _log_int(rng, 256, VOCAB), "K": rng.choice((2048, 4096)),
                    "flags": 4}
        return {"kind": kind, "tokens": _log_int(rng, 2, 2048), "O": rng.choice((64, 256, 1000, 1024)),
                "K": rng.choice((1000, 2048, 4096)), "flags": rng.choice((0, 0, 3, 6, 7))}
    m, (_, O, K, _) = _log_int(rng, 2, 512), rng.choice(ATTN)
    return {"kind": kind, "tokens": m + 56 if _no_result(FP8, m, K) else m, "O": O, "K": K}


# ------------------------------------------------------------------- inputs


def _gen(seed, what):
    return torch.Generator(device="cuda").manual_seed((seed * 1000003 + what) & 0x7FFFFFFF)


def _bytes(gen, lo, hi, *shape):
    return torch.randint(lo, hi, shape, dtype=torch.uint8, device="cuda", generator=gen)


def _acts(gen, *shape):
    """BF16-valued N(0, 1) rows held in fp32."""
    return torch.randn(*shape, device="cuda", generator=gen).bfloat16().float()


def _fp4_weight(gen, *shape_ok):
    """packed nibbles [.., O, K/2] and E8M0 bytes [.., O, K/32]; values about 1/sqrt(4096)"""
    *lead, O, K = shape_ok
    return _bytes(gen, 0, 256, *lead, O, K // 2), _bytes(gen, 117, 122, *lead, O, K // 32)


def _fp8_weight(gen, O, K):
    """E4M3 of N(0, 1) [O, K] and 128 x 128 tile scales, log-uniform in 2^-10 .. 2^-4"""
    w = torch.randn(O, K, device="cuda", generator=gen).to(torch.float8_e4m3fn).view(torch.uint8)
    return w, _bytes(gen, 117, 124, (O + 127) // 128, K // 128)


def _weight(fmt, gen, O, K):
    return _fp4_weight(gen, O, K) if fmt == FP4 else _fp8_weight(gen, O, K)


def _pack(fmt, w, ws):
    """the resident (tiled) form of one weight"""
    O, K = w.shape[0], w.shape[1] * (2 if fmt == FP4 else 1)
    tw, tws = torch.empty_like(w), ws if fmt == FP8 else torch.empty_like(ws)
    torch.cuda.synchronize()
    H._check(H.lib().apus_hip_pack_weights_dev(fmt, w.data_ptr(), ws.data_ptr(), tw.data_ptr(),
                                               tws.data_ptr(), O, K), "pack")
    H.synchronize()
    return tw, tws


class _Store:
    """One layer of experts in the backend's store, freed with the object."""

    def __init__(self, weights):
        L, err = H.lib(), C.create_string_buffer(256)
        self.ptr = L.apus_hip_store_create(1, EXPERTS, DIM, INTER, err, 256)
        if not self.ptr:
            raise H.ApusHipError("store_create: " + err.value.decode(errors="replace"))
        if not L.apus_hip_store_tiled(self.ptr):
            raise H.ApusHipError("the store is expected to hold its matrices tiled")
        torch.cuda.synchronize()
        p = (C.c_void_p * 6)()
        for e in range(EXPERTS):
            H._check(L.apus_hip_store_get(self.ptr, 0, e, p), "store_get")
            for i, (w, ws) in enumerate(weights):
                O, K = w.shape[1], w.shape[2] * 2
                H._check(L.apus_hip_pack_weights_dev(FP4, w[e].data_ptr(), ws[e].data_ptr(), p[2 * i],
                                                     p[2 * i + 1], O, K), "pack")
        H.synchronize()

    def __del__(self):
        try:
            H.synchronize()
            H.lib().apus_hip_store_free(self.ptr)
        except Exception:
            pass


def _experts(seed):
    """w1 [E, inter, dim], w2 [E, dim, inter], w3 [E, inter, dim]"""
    g = _gen(seed, 1)
    return [_fp4_weight(g, EXPERTS, O, K) for O, K in ((INTER, DIM), (DIM, INTER), (INTER, DIM))]


def _routing(case, seed):
    """distinct experts per token, drawn by popularity rank^-zipf; softmax weights"""
    rng = np.random.default_rng([seed, 7])
    s, k = case["tokens"], case["topk"]
    p = np.arange(1, EXPERTS + 1) ** -float(case["zipf"])
    logits = np.log(p[rng.permutation(EXPERTS)])[None, :] + rng.gumbel(size=(s, EXPERTS))
    idx = np.argsort(-logits, axis=1, kind="stable")[:, :k].astype(np.int32)
    w = np.exp(rng.standard_normal((s, k)))
    return idx, (w / w.sum(1, keepdims=True)).astype(np.float32)


def _layer_inputs(case, seed):
    g = _gen(seed, 2)
    x = _acts(g, case["tokens"], DIM)
    gate = torch.randn(EXPERTS, DIM, device="cuda", generator=g) / math.sqrt(DIM)
    bias = torch.randn(EXPERTS, device="cuda", generator=g) * 0.05
    shared = [_fp8_weight(g, O, K) for O, K in ((INTER, DIM), (DIM, INTER), (INTER, DIM))]
    rng = np.random.default_rng([seed, 9])
    # 4096 token ids in use, Zipf-popular as words are, each with its experts
    tid2eid = np.argsort(rng.random((4096, EXPERTS)), axis=1)[:, :case["topk"]].astype(np.int64)
    pop = np.arange(1, 4097) ** -1.0
    ids = rng.choice(4096, case["tokens"], p=pop / pop.sum()).astype(np.int64)
    return x, gate, bias, shared, torch.from_numpy(tid2eid).cuda(), torch.from_numpy(ids).cuda()


def _linear_inputs(case, seed):
    g = _gen(seed, 3)
    x = _acts(g, case["tokens"], case["K"])
    return x, _weight(case["fmt"], g, case["O"], case["K"])


def _attn_inputs(case, seed):
    g = _gen(seed, 4)
    return [_acts(g, case["tokens"], K) for K in ATTN_IN], [_fp8_weight(g, O, K) for _, O, K, _ in ATTN]


def _experts_inputs(case, seed):
    g = _gen(seed, 5)
    x = _acts(g, case["rows"], case["K"])
    return x, [_weight(case["fmt"], g, case["O"], case["K"]) for _ in range(case["entries"])]


def _plain_inputs(case, seed):
    g = _gen(seed, 6)
    w = torch.randn(case["O"], case["K"], device="cuda", generator=g) / math.sqrt(case["K"])
    x = torch.randn(case["tokens"], case["K"], device="cuda", generator=g)
    return x, w.bfloat16() if case["flags"] & 4 else w


def _out(*shape):
    return torch.zeros(*shape, device="cuda")


def _buf(nbytes):
    return torch.empty(max(256, int(nbytes)), dtype=torch.uint8, device="cuda")


def prepare(case, seed):
    H.enable()
    L, kind = H.lib(), case["kind"]
    st = {"kind": kind}
    if kind in ("layer", "routed"):
        s, k = case["tokens"], case["topk"]
        weights = _experts(seed)
        store = st["store"] = _Store(weights)
        del weights
        y = st["out"] = _out(s, DIM)
        if kind == "routed":
            idx, wgt = _routing(case, seed)
            st["x"] = _acts(_gen(seed, 2), s, DIM)
            st["idx"], st["wgt"] = torch.from_numpy(idx).cuda(), torch.from_numpy(wgt).cuda()
            st["ws"] = _buf(L.apus_hip_moe_workspace(store.ptr, s, k))
            st["args"] = (store.ptr, 0, st["x"].data_ptr(), st["idx"].data_ptr(), st["wgt"].data_ptr(), s, k,
                          LIMIT, y.data_ptr(), st["ws"].data_ptr())
            return st
        x, gate, bias, shared, tid2eid, ids = _layer_inputs(case, seed)
        shared = [_pack(FP8, w, ws) for w, ws in shared]
        ml = st["ml"] = H.ApusHipMoeLayer()
        ml.gate_w, ml.gate_bias = gate.data_ptr(), bias.data_ptr()
        ml.hash, ml.tid2eid = int(case["hash"]), tid2eid.data_ptr() if case["hash"] else None
        ml.route_scale, ml.limit, ml.shared_tiled = ROUTE_SCALE, LIMIT, 1
        ml.sw1, ml.sw1s, ml.sw2, ml.sw2s, ml.sw3, ml.sw3s = (t.data_ptr() for p in shared for t in p)
        st["keep"] = (x, gate, bias, shared, tid2eid, ids)
        st["ws"] = _buf(L.apus_hip_moe_forward_workspace(store.ptr, s, k))
        st["args"] = (store.ptr, 0, C.byref(ml), x.data_ptr(), ids.data_ptr() if case["hash"] else None, s, k,
                      y.data_ptr(), None, st["ws"].data_ptr())
        return st
    if kind == "attn":
        m = case["tokens"]
        xs, weights = _attn_inputs(case, seed)
        st["ws"] = _buf(max(L.apus_hip_linear_workspace(m, K) for K in ATTN_IN))
        st["keep"], st["out"], st["args"] = [xs], {}, []
        for (name, O, K, src), (w, ws) in zip(ATTN, weights):
            tw, tws = _pack(FP8, w, ws)
            y = st["out"][name] = _out(m, O)
            st["keep"] += [tw, tws]
            st["args"].append((FP8 | H.W_TILED, tw.data_ptr(), tws.data_ptr(), xs[src].data_ptr(), y.data_ptr(),
                               m, K, O, st["ws"].data_ptr()))
        return st
    if kind == "linear":
        x, (w, ws) = _linear_inputs(case, seed)
        fmt, m, O, K = case["fmt"], case["tokens"], case["O"], case["K"]
        if case["tiled"]:
            w, ws = _pack(fmt, w, ws)
        st["out"], st["ws"], st["keep"] = _out(m, O), _buf(L.apus_hip_linear_workspace(m, K)), (x, w, ws)
        st["args"] = [(fmt | (H.W_TILED if case["tiled"] else 0), w.data_ptr(), ws.data_ptr(), x.data_ptr(),
                       st["out"].data_ptr(), m, K, O, st["ws"].data_ptr())]
        return st
    if kind == "experts":
        x, weights = _experts_inputs(case, seed)
        n, m, O, K = case["entries"], case["rows"], case["O"], case["K"]
        packed = [_pack(case["fmt"], w, ws) for w, ws in weights]
        y = st["out"] = _out(n, m, O)
        codes, scales = _buf(m * K), _out(m, K // 128)
        ents = (H.ApusHipGemmEnt * n)()
        for i, (w, ws) in enumerate(packed):
            ents[i] = H.ApusHipGemmEnt(w.data_ptr(), ws.data_ptr(), y[i].data_ptr(), None, None, 0, 0, m, 0)
        table = torch.frombuffer(bytearray(bytes(ents)), dtype=torch.uint8).cuda()
        st["keep"] = (x, packed, codes, scales, table)
        st["quant"] = (x.data_ptr(), m, K, codes.data_ptr(), scales.data_ptr())
        st["args"] = (case["fmt"] | H.W_TILED, table.data_ptr(), n, codes.data_ptr(), scales.data_ptr(), O, K,
                      O, 0, m)
        return st
    if kind == "plain":
        x, w = _plain_inputs(case, seed)
        st["keep"], st["out"] = (x, w), _out(case["tokens"], case["O"])
        st["args"] = (w.data_ptr(), x.data_ptr(), st["out"].data_ptr(), case["tokens"], case["K"], case["O"],
                      case["flags"])
        return st
    # hook: everything in host memory; the first call makes the weight resident
    case = dict(case, fmt=FP8)
    x, (w, ws) = _linear_inputs(case, seed)
    x, w, ws = (t.cpu().numpy() for t in (x, w, ws))
    st["keep"], st["out"] = (x, w, ws), np.zeros((case["tokens"], case["O"]), np.float32)
    st["w"] = H.fp8_weight(w, ws)
    st["args"] = (C.byref(st["w"]), x.ctypes.data_as(H.f32p), st["out"].ctypes.data_as(H.f32p), case["tokens"],
                  case["K"], case["O"])
    run(st)
    return st


def run(st):
    L, kind, args = H.lib(), st["kind"], st["args"]
    if kind == "layer":
        rc = L.apus_hip_moe_forward_dev(*args)
    elif kind == "routed":
        rc = L.apus_hip_moe_routed_dev(*args)
    elif kind in ("attn", "linear"):
        rc = 0
        for a in args:
            rc |= L.apus_hip_linear_dev(*a)
    elif kind == "experts":
        rc = L.apus_hip_act_quant_dev(*st["quant"]) or L.apus_hip_gemm_grouped_dev(*args)
    elif kind == "plain":
        rc = L.apus_hip_wlinear_dev(*args)
    else:
        rc = L.apus_hip_fp8_linear(*args)
    H._check(rc, kind)
    return st["out"]


# --------------------------------------------------------------------- work


def _wbytes(fmt, O, K):
    return O * K // 2 + O * K // 32 if fmt == FP4 else O * K + (O + 127) // 128 * (K // 128)


def _linear_work(fmt, m, O, K):
    return _wbytes(fmt, O, K) + 4 * m * (O + K), 2 * m * O * K


def _moe_work(idx, s, k):
    """the weights of the experts that are met, once; x in and y out"""
    per = 2 * _wbytes(FP4, INTER, DIM) + _wbytes(FP4, DIM, INTER)
    return len(np.unique(idx)) * per + 8 * s * DIM, s * k * 6 * DIM * INTER


def work(case):
    kind = case["kind"]
    if kind == "routed":
        b, f = _moe_work(_routing(case, 0)[0], case["tokens"], case["topk"])
    elif kind == "layer":
        s, k = case["tokens"], case["topk"]
        rng = np.random.default_rng(0)
        if case["hash"]:
            pop = np.arange(1, 4097) ** -1.0
            met = len(np.unique(rng.choice(4096, s, p=pop / pop.sum())))
        else:
            met = s
        b, f = _moe_work(np.argsort(rng.random((met, EXPERTS)), axis=1)[:, :k], s, k)
        b += 3 * _wbytes(FP8, INTER, DIM) + 4 * EXPERTS * DIM
        f += 6 * s * DIM * INTER + 2 * s * EXPERTS * DIM
    elif kind == "attn":
        w = [_linear_work(FP8, case["tokens"], O, K) for _, O, K, _ in ATTN]
        b, f = sum(x for x, _ in w), sum(x for _, x in w)
    elif kind in ("linear", "hook"):
        b, f = _linear_work(case.get("fmt", FP8), case["tokens"], case["O"], case["K"])
    elif kind == "experts":
        n, m, O, K = case["entries"], case["rows"], case["O"], case["K"]
        b, f = n * _wbytes(case["fmt"], O, K) + 4 * m * K + 4 * n * m * O, 2 * n * m * O * K
    else:
        m, O, K = case["tokens"], case["O"], case["K"]
        b, f = O * K * (2 if case["flags"] & 4 else 4) + 4 * m * (O + K), 2 * m * O * K
    return {"bytes": float(b), "flops": float(f)}


def tolerance(case):
    kind = case["kind"]
    if kind in ("layer", "routed"):
        # 1e-3 to 2.2e-3 from exact(): BF16 sums, and h codes that round the other way
        return {"rel": 9e-3, "max": 0.1}
    if kind == "experts":
        # unrounded; the matrix cores' sums over a 128-group are 5e-6 (MXFP4) to 1.5e-5 (FP8) from exact()
        return {"rel": 6e-5, "max": 1e-3}
    if kind == "plain" and not case["flags"] & 2:
        return {"rel": 1e-5, "max": 1e-4}   # fp32 sums
    return {"rel": 7e-3, "max": 0.04}       # outputs rounded to BF16: 1.7e-3 from exact()


# -------------------------------------------------------------------- exact


def _bf16(v):
    return v.float().bfloat16().double()


def _quantised(x):
    """x rounded to BF16, then E4M3 per 128 columns under a power-of-two scale, as values"""
    m, K = x.shape
    v = x.float().bfloat16().float().view(m, K // 128, 128)
    r = v.abs().amax(2).clamp_min(1e-4) / 448.0
    mant, ex = torch.frexp(r)
    s = torch.ldexp(torch.ones_like(r), ex - (mant == 0.5).int()).unsqueeze(2)
    q = (v / s).clamp(-448, 448).to(torch.float8_e4m3fn).double() * s.double()
    return q.view(m, K)


def _value(fmt, w, ws):
    """the weight's values in 64 bits"""
    s = torch.pow(2.0, ws.double() - 127.0)
    if fmt == FP8:
        O, K = w.shape
        v = w.view(torch.float8_e4m3fn).double()
        return v * s.repeat_interleave(128, 0)[:O].repeat_interleave(128, 1)
    lut = torch.tensor([0, .5, 1, 1.5, 2, 3, 4, 6, -0., -.5, -1, -1.5, -2, -3, -4, -6], dtype=torch.float64,
                       device=w.device)
    v = torch.stack((lut[(w & 15).long()], lut[(w >> 4).long()]), -1).flatten(-2)
    return v * s.repeat_interleave(32, -1)


def _swiglu(g, u):
    g, u = _bf16(g).clamp_max(LIMIT), _bf16(u).clamp(-LIMIT, LIMIT)
    return _bf16(g * torch.sigmoid(g) * u)


def _ffn(xq, fmt, w1, w2, w3):
    h = _swiglu(xq @ _value(fmt, *w1).T, xq @ _value(fmt, *w3).T)
    return _bf16(_quantised(h) @ _value(fmt, *w2).T)


def _routed_exact(x, idx, wgt, seed):
    weights, xq = _experts(seed), _quantised(x)
    y = torch.zeros(x.shape[0], DIM, dtype=torch.float64, device="cuda")
    for e in range(EXPERTS):
        t, j = (idx == e).nonzero(as_tuple=True)
        if t.numel():
            eo = _ffn(xq[t], FP4, *[(w[e], ws[e]) for w, ws in weights])
            y.index_add_(0, t, wgt[t, j].double().unsqueeze(1) * eo)
    return y


def exact(case, seed):
    kind = case["kind"]
    if kind == "routed":
        idx, wgt = _routing(case, seed)
        return _routed_exact(_acts(_gen(seed, 2), case["tokens"], DIM), torch.from_numpy(idx).cuda(),
                             torch.from_numpy(wgt).cuda(), seed)
    if kind == "layer":
        x, gate, bias, shared, tid2eid, ids = _layer_inputs(case, seed)
        score = torch.nn.functional.softplus(x.double() @ gate.double().T).sqrt()
        idx = tid2eid[ids] if case["hash"] else (score + bias.double()).topk(case["topk"], 1).indices
        sp = score.gather(1, idx)
        y = _routed_exact(x, idx, sp / sp.sum(1, keepdim=True) * ROUTE_SCALE, seed)
        return y + _ffn(_quantised(x), FP8, *shared)
    if kind == "attn":
        xs, weights = _attn_inputs(case, seed)
        return {name: _quantised(xs[src]) @ _value(FP8, w, ws).T
                for (name, _, _, src), (w, ws) in zip(ATTN, weights)}
    if kind in ("linear", "hook"):
        case = dict(case, fmt=case.get("fmt", FP8))
        x, (w, ws) = _linear_inputs(case, seed)
        return _quantised(x) @ _value(case["fmt"], w, ws).T
    if kind == "experts":
        x, weights = _experts_inputs(case, seed)
        xq = _quantised(x)
        return torch.stack([xq @ _value(case["fmt"], w, ws).T for w, ws in weights])
    x, w = _plain_inputs(case, seed)
    x = _bf16(x) if case["flags"] & 1 else x.double()
    return x @ w.double().T
