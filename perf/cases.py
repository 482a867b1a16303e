"""The performance cases of this framework: the calls its users make, with the
inputs, one pass and the work of each.

Sizes are those of the Qwen3-0.6B-shaped model of ``artifact.QWEN3_0_6B`` and
of the benchmark's configurations: the fused int8 product of 64 rows, the MLP
block and the attention of 2048 tokens, the decode of 1 and 8 rows around 320
cache slots, the decode of 32 rows at 4096 slots; beside them short and ragged
sizes of the same calls. Every output is an integer that the integer
algorithm fixes to the last bit, so every case's tolerance is "exact".

Kinds (``case["kind"]``) and what they stand for:

* ``gemm_static``: int8 product and static requantisation in one call, a
  linear layer of at most 64 rows of a program that drives the C entry points.
* ``int_gemm``: ``backends.int_gemm``, the product that code written against
  the reference package calls with its [K, N] operand, ragged sizes included,
  2-D or batched.
* ``mlp``: the MLP half of a layer through the registered operators, from a
  few decode rows to a long prefill.
* ``attention``: the attention half of a layer through the registered
  operators: a whole prompt or a chunk after ``past`` slots, rows of different
  lengths.
* ``attn_decode``: the registered decode attention alone, one query per row.
* ``prefill``: the time to the first token, ``generate(max_new=1)``.
* ``generate``: a whole reply, prompt and all its tokens, graphed or eager.
* ``decode``: one graphed greedy step of a running batch.
"""

import functools
import math
import tempfile

import torch

from idempotent_llm_amd import artifact as art
from idempotent_llm_amd import backends, torch_ops  # noqa: F401  (torch_ops registers the ops)
from idempotent_llm_amd._lib import call
from idempotent_llm_amd.graphed import GraphedDecode
from idempotent_llm_amd.kvcache import PAGE, KVCache
from idempotent_llm_amd.model import IntQwen3

I64 = torch.int64
D = art.QWEN3_0_6B
H, I, HD = D["hidden"], D["intermediate"], D["head_dim"]
NQ, NKV, V, NL = D["n_q_heads"], D["n_kv_heads"], D["vocab"], D["n_layers"]
QKV = (NQ + 2 * NKV) * HD
LAYER_W = QKV * H + H * NQ * HD + 2 * I * H + H * I    # int8 weights of one layer
OPS = torch.ops.detllm_rocm


def listed():
    return [
        # the smallest call: one linear layer of 64 rows (latency and launch cost)
        dict(name="gemm_static_64", kind="gemm_static", M=64, K=1024, N=3072),
        # code of the reference package on ragged shapes (its operand is [K, N])
        dict(name="int_gemm_ragged", kind="int_gemm", batch=0, M=777, K=1000, N=1500),
        # the MLP of a batch of eight decode rows
        dict(name="mlp_8", kind="mlp", rows=8),
        # the MLP of a 2048-token prompt
        dict(name="mlp_2048", kind="mlp", rows=2048),
        # the attention of a 2048-token prompt
        dict(name="attention_2048", kind="attention", B=1, T=2048, past=0),
        # decode attention of eight rows at the end of a 512-token reply
        dict(name="attn_decode_8x576", kind="attn_decode", B=8, S=576),
        # time to first token of an ordinary short prompt
        dict(name="prefill_1x200", kind="prefill", B=1, T=200),
        # time to first token of a long prompt
        dict(name="prefill_1x2048", kind="prefill", B=1, T=2048),
        # eight chat replies: ragged prompts of up to 40 tokens, 32 new ones
        dict(name="generate_8x40", kind="generate", B=8, T=40, new=32, graph=True),
        # a single user's decode
        dict(name="decode_1x320", kind="decode", B=1, S=320),
        # a small serving batch's decode
        dict(name="decode_8x320", kind="decode", B=8, S=320),
        # a full serving batch's decode at a long context
        dict(name="decode_32x4000", kind="decode", B=32, S=4000),
    ]


def _log(rng, lo, hi):
    """A whole number of [lo, hi], even over its logarithm."""
    return min(hi, max(lo, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))))


def draw(rng):
    kind = rng.choice(["gemm_static", "int_gemm", "mlp", "attention", "attn_decode", "prefill",
                       "generate", "decode"])
    if kind == "gemm_static":
        return dict(kind=kind, M=_log(rng, 1, 64), K=16 * _log(rng, 16, 192),
                    N=_log(rng, 256, 6144))
    if kind == "int_gemm":
        if rng.random() < 0.3:    # per head, as the attention seams call it
            return dict(kind=kind, batch=rng.choice([4, 8, 16]), M=_log(rng, 1, 512),
                        K=HD, N=_log(rng, 16, 1024))
        return dict(kind=kind, batch=0, M=_log(rng, 1, 2048), K=_log(rng, 64, 3072),
                    N=_log(rng, 64, 4096))
    if kind == "mlp":
        return dict(kind=kind, rows=_log(rng, 1, 2048))
    if kind == "attention":
        B = _log(rng, 1, 8)
        T = _log(rng, 16, 2048 // B)
        return dict(kind=kind, B=B, T=T, past=rng.choice([0, 0, _log(rng, 16, 2048 - T + 16)]))
    if kind == "attn_decode":
        return dict(kind=kind, B=_log(rng, 1, 32), S=_log(rng, 64, 4096))
    if kind == "prefill":
        B = _log(rng, 1, 8)
        return dict(kind=kind, B=B, T=_log(rng, 16, 2048 // B))
    if kind == "generate":
        graph = rng.random() < 0.5
        return dict(kind=kind, B=_log(rng, 1, 8), T=_log(rng, 8, 128),
                    new=_log(rng, 4, 28 if graph else 10), graph=graph)
    return dict(kind=kind, B=_log(rng, 1, 32), S=_log(rng, 32, 4000))


# ------------------------------------------------------------------ preparation

@functools.lru_cache(maxsize=1)
def _model():
    """The program's one loaded model (random-init artifact, seed 3)."""
    with tempfile.TemporaryDirectory() as d:
        art.make_artifact(d, D, seed=3)
        return IntQwen3(d, backend="rocm")


def _gen(seed):
    return torch.Generator(device="cuda").manual_seed(int(seed) & 0x7FFFFFFFFFFFFFFF)


def _i8(g, *shape):
    return torch.randint(-127, 128, shape, dtype=torch.int8, device="cuda", generator=g)


def _ids(g, *shape):
    return torch.randint(100, 50000, shape, dtype=I64, device="cuda", generator=g)


def _ragged(g, B, T):
    """Validity [B, T] of right-padded rows: lengths in (T/2, T], the first T."""
    lens = torch.randint(T // 2 + 1, T + 1, (B,), device="cuda", generator=g)
    lens[0] = T
    return torch.arange(T, device="cuda")[None] < lens[:, None], lens


def _embed(m, L, ids, sm_m, sm_k):
    """The residual stream and the layer's int8 input for these tokens."""
    return OPS.embed_normq(ids.reshape(-1), m.embed_e8, m.embed_m, m.embed_k, sm_m, sm_k, m._err)


def _epilogue(m, L, x8, xm, xk, B, T, pos, kp, vp, table, base):
    P = backends.gemm_nt(x8, L.wqkv)
    return OPS.qkv_epilogue(P, B, T, NQ, NKV, xm, xk, pos, L.q_m, L.q_k, L.k_m, L.k_k, L.v_m,
                            L.v_k, L.q_norm_m, L.q_norm_k, L.k_norm_m, L.k_norm_k, L.qs_m,
                            L.qs_k, L.kq_m, L.kq_k, L.ks_m, L.ks_k, L.vq_m, L.vq_k, m.rope_cos,
                            m.rope_sin, kp, vp, table, base, m._err)


def _paged(B, slots):
    w = -(-slots // PAGE)
    kp = torch.zeros(B * w, NKV, PAGE, HD, dtype=torch.int8, device="cuda")
    vp = torch.zeros(B * w, NKV, HD, PAGE, dtype=torch.int8, device="cuda")
    table = torch.arange(B * w, dtype=torch.int32, device="cuda").view(B, w)
    return kp, vp, table, w


def _positions(B, lo, hi):
    return torch.arange(lo, hi, device="cuda").expand(B, hi - lo).contiguous()


def prepare(case, seed):
    g = _gen(seed)
    kind = case["kind"]
    if kind == "gemm_static":
        M, K, N = case["M"], case["K"], case["N"]
        return dict(case, A=_i8(g, M, K), W=_i8(g, N, K),
                    m=torch.randint(1 << 14, 1 << 15, (N,), dtype=I64, device="cuda",
                                    generator=g))
    if kind == "int_gemm":
        lead = (case["batch"],) if case["batch"] else ()
        return dict(case, a=_i8(g, *lead, case["M"], case["K"]),
                    b=_i8(g, *lead, case["K"], case["N"]))
    m = _model()
    L = m.layers[int(seed) % NL]
    if kind == "mlp":
        h, k_res, _, _, _ = _embed(m, L, _ids(g, case["rows"]), None, 0)
        return dict(case, L=L, h=h, k_res=k_res)
    if kind == "attention":
        B, T, past = case["B"], case["T"], case["past"]
        kp, vp, table, w = _paged(B, past + T)
        valid = torch.zeros(B, w * PAGE, dtype=torch.bool, device="cuda")
        if past:
            valid[:, :past] = _ragged(g, B, past)[0]
            _, _, x8, xm, xk = _embed(m, L, _ids(g, B, past), L.as_m, L.as_k)
            _epilogue(m, L, x8, xm, xk, B, past, _positions(B, 0, past), kp, vp, table, 0)
        valid[:, past:past + T] = _ragged(g, B, T)[0]
        _, _, x8, xm, xk = _embed(m, L, _ids(g, B, T), L.as_m, L.as_k)
        return dict(case, m=m, L=L, x8=x8, xm=xm, xk=xk, pos=_positions(B, past, past + T),
                    kp=kp, vp=vp, table=table, valid=valid)
    if kind == "attn_decode":
        B, S = case["B"], case["S"]
        kp, vp, table, w = _paged(B, S)
        valid = torch.zeros(B, w * PAGE, dtype=torch.bool, device="cuda")
        valid[:, :S - 1] = _ragged(g, B, S - 1)[0]
        valid[:, S - 1] = True
        _, _, x8, xm, xk = _embed(m, L, _ids(g, B, S), L.as_m, L.as_k)
        _epilogue(m, L, x8, xm, xk, B, S, _positions(B, 0, S), kp, vp, table, 0)
        _, _, x8, xm, xk = _embed(m, L, _ids(g, B, 1), L.as_m, L.as_k)
        q8, tpos = _epilogue(m, L, x8, xm, xk, B, 1, _positions(B, S - 1, S), kp, vp, table,
                             S - 1)
        return dict(case, m=m, q8=q8.view(B, NQ, HD), tpos=tpos.view(B, NQ), kp=kp, vp=vp,
                    table=table, valid=valid)
    if kind in ("prefill", "generate"):
        B, T = case["B"], case["T"]
        return dict(case, m=m, ids=_ids(g, B, T), valid=_ragged(g, B, T)[0])
    # a running batch: the prompt prefilled in chunks, the step's graph captured
    B, S = case["B"], case["S"]
    ids = _ids(g, B, S)
    valid, lens = _ragged(g, B, S)
    cache = KVCache().plan(m, B, S + 1)
    step = max(1, 1024 // B)
    for lo in range(0, S, step):
        hi = min(S, lo + step)
        logits, _, _, cache = m.forward(ids[:, lo:hi], _positions(B, lo, hi), cache,
                                        valid[:, lo:hi])
    cur = m.greedy_pick(logits[:, -1])
    gd = GraphedDecode(m, cache, lens)
    gd.step_greedy(cur)
    return dict(case, gd=gd, cur=cur)


# ------------------------------------------------------------------ one pass

def run(state):
    kind = state["kind"]
    if kind == "gemm_static":
        M, K, N = state["M"], state["K"], state["N"]
        y8 = torch.empty(M, N, dtype=torch.int8, device="cuda")
        call("detllm_igemv_requant_static", state["A"], state["W"], M, N, K, None, None,
             state["m"], 20, 1, 0, y8)
        return y8
    if kind == "int_gemm":
        return backends.int_gemm(state["a"], state["b"], "rocm")
    if kind == "mlp":
        # the residual is updated in place by the layer: this pass's own copy
        L, h, k_res = state["L"], state["h"].clone(), state["k_res"].clone()
        x8, xm, xk = OPS.norm_quant(h, L.ms_m, L.ms_k)
        P = backends.gemm_nt(x8, L.wgu)
        y8, ym, yk = OPS.swiglu_quant(P, xm, xk, L.gate_m, L.gate_k, L.up_m, L.up_k, L.ds_m,
                                      L.ds_k)
        P = backends.gemm_nt(y8, L.wd)
        x8, xm, xk = OPS.residual_normq(P, ym, yk, L.down_m, L.down_k, 20, h, k_res, L.as_m,
                                        L.as_k)
        return dict(h=h, k_res=k_res, x8=x8, xm=xm, xk=xk)
    if kind == "attention":
        m, L, B, T, past = (state[k] for k in ("m", "L", "B", "T", "past"))
        q8, tpos = _epilogue(m, L, state["x8"], state["xm"], state["xk"], B, T, state["pos"],
                             state["kp"], state["vp"], state["table"], past)
        ctx = OPS.attn_prefill(q8, tpos, state["kp"], state["vp"], state["table"],
                               state["valid"], past)
        a8, am, ak = OPS.merge_rowcol(ctx.view(B * T, NQ * HD), L.os_m, L.os_k,
                                      L.attn_out_col_m, L.attn_out_col_k)
        return dict(out=backends.gemm_nt(a8, L.wo), am=am, ak=ak, k=state["kp"], v=state["vp"])
    if kind == "attn_decode":
        return OPS.attn_decode(state["q8"], state["tpos"], state["kp"], state["vp"],
                               state["table"], state["valid"], state["S"], state["m"]._err)
    if kind in ("prefill", "generate"):
        new = state.get("new", 1)
        toks, logits = state["m"].generate(state["ids"], new, chunk_valid=state["valid"],
                                           use_graph=state.get("graph", False))
        return dict(tokens=toks, logits=logits)
    # back to the prompt's end, one greedy step from there
    gd = state["gd"]
    gd.length = gd.cache.length = state["S"]
    gd.steps = 0
    toks = gd.step_greedy(state["cur"])
    return dict(tokens=toks, logits=gd.out_pick[:, 0])


# ------------------------------------------------------------------ the work of a pass

def _scales():
    """Bytes of one layer's per-column scale vectors (int64)."""
    return 8 * (QKV + 2 * H + NQ * HD + 3 * I + 2 * H)


def work(case):
    kind = case["kind"]
    if kind == "gemm_static":
        M, K, N = case["M"], case["K"], case["N"]
        return dict(bytes=M * K + N * K + 8 * N + M * N, flops=2 * M * N * K)
    if kind == "int_gemm":
        M, K, N, b = case["M"], case["K"], case["N"], case["batch"] or 1
        return dict(bytes=b * (M * K + N * K + 4 * M * N), flops=2 * b * M * N * K)
    if kind == "mlp":
        R = case["rows"]
        return dict(bytes=3 * I * H + 8 * (3 * I + 3 * H) + R * (9 * H + 32),
                    flops=6 * R * I * H)
    if kind == "attention":
        B, T, past = case["B"], case["T"], case["past"]
        pairs = B * (T * past + T * (T + 1) // 2)
        return dict(bytes=QKV * H + H * NQ * HD + 8 * QKV + B * T * (5 * H + 32)
                    + 2 * B * (past + T) * NKV * HD,
                    flops=2 * B * T * (QKV + NQ * HD) * H + 4 * pairs * NQ * HD)
    if kind == "attn_decode":
        B, S = case["B"], case["S"]
        return dict(bytes=B * (2 * S * NKV * HD + S + NQ * (HD + 8 + 8 * HD)),
                    flops=4 * B * S * NQ * HD)
    B = case["B"]
    head = V * H + 8 * V
    if kind in ("prefill", "generate"):
        T, new = case["T"], case.get("new", 1)
        flops = B * (2 * T * NL * LAYER_W + NL * 2 * T * (T + 1) * NQ * HD + 2 * V * H)
        nbytes = NL * (LAYER_W + _scales()) + head + B * (4 * V + T * (H + 16))
        nbytes += B * T * NL * 2 * NKV * HD
        for s in range(1, new):
            step = _decode_work(B, T + s)
            flops += step["flops"]
            nbytes += step["bytes"]
        return dict(bytes=nbytes, flops=flops)
    return _decode_work(B, case["S"] + 1)


def _decode_work(B, S):
    kv = 2 * NKV * HD
    return dict(bytes=NL * (LAYER_W + _scales()) + V * H + 8 * V
                + B * (H + 16 + 4 * V + NL * kv * S),
                flops=B * (2 * (NL * LAYER_W + V * H) + NL * 4 * S * NQ * HD))


def tolerance(case):
    return "exact"     # integers, fixed to the last bit by the algorithm


def exact(case, seed):
    """The two products in 64-bit arithmetic (float64 sums of int8 products
    below 2^53 are exact). The other kinds are whole chains of the integer
    algorithm, which no plain 64-bit computation gives without restating it:
    their outputs are compared bit for bit instead."""
    if case["kind"] == "int_gemm":
        s = prepare(case, seed)
        return (s["a"].cpu().double() @ s["b"].cpu().double()).to(torch.int32)
    if case["kind"] == "gemm_static":
        s = prepare(case, seed)
        n = (s["A"].cpu().double() @ s["W"].cpu().double().T).to(I64) * s["m"].cpu()
        q = (n.abs() + (1 << 19)) >> 20    # round half away from zero by 2^20
        return torch.where(n < 0, -q, q).clamp(-128, 127).to(torch.int8)
    return None
