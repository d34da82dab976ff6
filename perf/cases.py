"""The work this library is used for, as cases to time and compare.

A case is one call (or one short run of calls) through the public entry points of
mynah_amd / libmynah_hip.so on inputs made from a seed:

  matvec    mynah_hip_matvec_dev: one projection of one token, weights and vectors in HBM
  dropin    ingot_matvec: the same through the host-pointer ABI, weights registered
  matmat    mynah_hip_matmat_dev / _matmat_mv_dev: a projection of many tokens, in the batched
            or the matvec order (with the residual), or on the int8 activation lane
  dequant   mynah_hip_dequant_dev: a whole matrix to f32
  forced    prefill of a prompt, then teacher-forced decode steps of a resident Qwen3
  generate  the greedy generation loop of a resident Qwen3, then one more step's logits

Weights are the shared generator's blocks (include/mynah_synth.h), activations N(0, 1); tokens
are uniform over the vocabulary.
"""
import math
import sys
from pathlib import Path

import numpy as np
import torch

sys.path.insert(0, str(Path(__file__).resolve().parent.parent / "mynah-slm_amd"))

import configs as CF  # noqa: E402
import mynah_amd as M  # noqa: E402

Q4_0, Q8_0, Q4_K, Q5_K, Q6_K = M.Q4_0, M.Q8_0, M.Q4_K, M.Q5_K, M.Q6_K
TYPES = {"q4_0": Q4_0, "q8_0": Q8_0, "q4_k": Q4_K, "q5_k": Q5_K, "q6_k": Q6_K}
GPU = "cuda"


def _matvec(qtype, rows, cols, order="exact"):
    return {"kind": "matvec", "type": qtype, "rows": rows, "cols": cols, "order": order}


def _matmat(qtype, rows, cols, tokens, lane="batched"):
    """lane: "batched" (the exact batched order), "matvec" (the matvec order plus a residual, as
    the prefill runs it) or "int8" (the int8 activation lane)."""
    return {"kind": "matmat", "type": qtype, "rows": rows, "cols": cols, "tokens": tokens,
            "lane": lane}


def _model(kind, shape, prompt, steps, attention="exact", layers=None, vocab=None):
    return {"kind": kind, "layers": layers or shape.n_layers, "d_model": shape.d_model,
            "d_ff": shape.d_ff, "heads": shape.n_heads, "kv_heads": shape.n_kv_heads,
            "vocab": vocab or shape.vocab, "prompt": prompt, "steps": steps,
            "attention": attention}


def listed():
    return [
        # One token's small projections: launches and latency count.
        {"name": "matvec_q4k_1024x3072", **_matvec("q4_k", 1024, 3072)},
        {"name": "matvec_q80_3072x1024", **_matvec("q8_0", 3072, 1024)},
        # A 4B feed-forward projection of one token.
        {"name": "matvec_q4k_9728x2560", **_matvec("q4_k", 9728, 2560)},
        # The 0.6B output head: the largest matrix of every decode step.
        {"name": "matvec_q6k_head", **_matvec("q6_k", 151936, 1024)},
        # The reference's own decoder linked against the library: host vectors in and out.
        {"name": "dropin_q6k_2048x1024", "kind": "dropin", "type": "q6_k", "rows": 2048,
         "cols": 1024},
        # Prompt projections: whole tiles, and a ragged batch in the prefill's order.
        {"name": "matmat_q4k_512tok", **_matmat("q4_k", 6144, 2048, 512)},
        {"name": "matmat_mv_q6k_201tok", **_matmat("q6_k", 2560, 9728, 201, "matvec")},
        # The int8 lane, whole tiles and a ragged batch of the other type that has it.
        {"name": "int8_q4k_512tok", **_matmat("q4_k", 6144, 2048, 512, "int8")},
        {"name": "int8_q5k_130tok", **_matmat("q5_k", 4096, 2560, 130, "int8")},
        # A matrix decoded to f32 (an embedding table or a projection for another consumer).
        {"name": "dequant_q6k_9728x2560", "kind": "dequant", "type": "q6_k", "rows": 9728,
         "cols": 2560},
        # A short chat turn of the 0.6B model: nearly all decode steps.
        {"name": "generate_06b", **_model("generate", CF.QWEN3_06B, 64, 48)},
        # Four layers of the 4B model with its head: a 2047-token prompt, then decode steps at
        # that context.
        {"name": "forced_4b_4layers", **_model("forced", CF.QWEN3_4B, 2047, 16, layers=4)},
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def _cols(rng, qtype, hi):
    step = 32 if qtype in ("q8_0", "q4_0") else 256
    return step * _log(rng, 1, hi // step)


def draw(rng):
    kind = rng.choice(("matvec", "matvec", "matmat", "matmat", "int8", "dequant", "dropin",
                       "forced"))
    qtype = rng.choice(("q4_k", "q4_k", "q6_k", "q6_k", "q8_0", "q5_k", "q4_0"))
    if kind == "matvec":
        cols = _cols(rng, qtype, 9728)
        order = rng.choice(("exact", "exact", "exact", "reordered"))
        return _matvec(qtype, min(_log(rng, 200, 151936), 150_000_000 // cols), cols, order)
    if kind == "dropin":
        cols = _cols(rng, qtype, 9728)
        return {"kind": kind, "type": qtype, "rows": min(_log(rng, 200, 9728), 25_000_000 // cols),
                "cols": cols}
    if kind == "dequant":
        cols = 256 * _log(rng, 2, 38)
        return {"kind": kind, "type": qtype,
                "rows": min(_log(rng, 200, 151936), 40_000_000 // cols), "cols": cols}
    if kind == "forced":
        shape = rng.choice((CF.QWEN3_TINY, CF.QWEN3_06B, CF.QWEN3_17B, CF.QWEN3_4B))
        return _model("forced", shape, _log(rng, 1, 1500), rng.randint(1, 24),
                      rng.choice(("exact", "exact", "split")), layers=rng.randint(1, 3),
                      vocab=rng.choice((4096, 32004)))
    cols = 256 * _log(rng, 2, 38)
    tokens = _log(rng, 2, 700)
    rows = min(_log(rng, 200, 9728), 9_000_000_000 // (cols * tokens))
    if kind == "int8":
        return _matmat(rng.choice(("q4_k", "q5_k")), rows, cols, tokens, "int8")
    return _matmat(qtype, rows, cols, tokens, rng.choice(("batched", "matvec")))


# ── inputs ───────────────────────────────────────────────────────────────────

def _seed(seed, k):
    return M.substream(seed, k)


def _weights(case, seed):
    return M.synth_blocks(TYPES[case["type"]], _seed(seed, 0), case["rows"], case["cols"])


def _normal(seed, k, *shape):
    n = math.prod(shape)
    return M.synth_normal(_seed(seed, k), n).reshape(shape)


def _shape(case):
    return CF.Qwen3Shape(case["layers"], case["d_model"], case["d_ff"], case["heads"],
                         case["kv_heads"], 128, case["vocab"])


def _tokens(case, seed):
    t = M.synth_uniform(_seed(seed, 3), case["prompt"] + case["steps"], case["vocab"])
    return t[:case["prompt"]], t[case["prompt"]:]


class Registered:
    """Host weights with their resident copy, as a program that maps a checkpoint holds them."""

    def __init__(self, w):
        self.w = w
        M.check(M.lib.mynah_hip_register(M.ptr(w), w.nbytes), "register")

    def __del__(self):
        M.lib.mynah_hip_unregister(M.ptr(self.w))


def prepare(case, seed):
    kind = case["kind"]
    if kind in ("forced", "generate"):
        dec = M.Qwen3Decoder(M.SynthQwen3(_shape(case), _seed(seed, 0)),
                             case["prompt"] + case["steps"] + 8)
        dec.set_attention(M.ATTN_SPLIT if case["attention"] == "split" else M.ATTN_EXACT)
        prompt, inputs = _tokens(case, seed)
        return {"case": case, "dec": dec, "prompt": prompt, "inputs": inputs}
    w = _weights(case, seed)
    if kind == "dropin":
        return {"case": case, "w": Registered(w), "x": _normal(seed, 1, case["cols"])}
    rows, cols, tokens = case["rows"], case["cols"], case.get("tokens", 1)
    s = {"case": case, "w": torch.from_numpy(w).to(GPU)}
    if kind == "dequant":
        s["y"] = torch.empty(rows, cols, device=GPU)
    else:
        s["x"] = torch.from_numpy(_normal(seed, 1, tokens, cols)).to(GPU)
        s["y"] = torch.empty(tokens, rows, device=GPU)
        if case.get("lane") == "matvec":
            s["res"] = torch.from_numpy(_normal(seed, 2, tokens, rows)).to(GPU)
    torch.cuda.synchronize()      # the library works on a stream of its own
    return s


def run(s):
    case = s["case"]
    kind = case["kind"]
    if kind == "generate":
        dec = s["dec"]
        dec.reset()
        ids, _, _ = dec.generate_tokens(s["prompt"], case["steps"], eos=(case["vocab"] - 1,))
        return {"ids": np.array(ids, np.int64), "logits": dec.forward(ids[-1])}
    if kind == "forced":
        dec = s["dec"]
        dec.reset()
        dec.prefill(s["prompt"])
        ids, logits = dec.forced(s["inputs"])
        return {"ids": np.array(ids, np.int64), "logits": logits}
    qtype, rows, cols = TYPES[case["type"]], case["rows"], case["cols"]
    if kind == "dropin":
        return M.matvec(qtype, s["w"].w, rows, cols, s["x"])
    w, y = s["w"].data_ptr(), s["y"].data_ptr()
    if kind == "dequant":
        M.dequant_dev(qtype, w, rows, cols, y)
    elif kind == "matvec":
        if case["order"] == "exact":
            M.matvec_dev(qtype, w, rows, cols, s["x"].data_ptr(), y)
        else:
            M.check(M.lib.mynah_hip_set_gemv_order(1), "set_gemv_order")
            M.matvec_dev(qtype, w, rows, cols, s["x"].data_ptr(), y)
            M.check(M.lib.mynah_hip_set_gemv_order(0), "set_gemv_order")
    elif case["lane"] == "batched":
        M.matmat_dev(qtype, w, rows, cols, s["x"].data_ptr(), y, case["tokens"])
    elif case["lane"] == "matvec":
        M.check(M.lib.mynah_hip_matmat_mv_dev(qtype, w, rows, cols, s["x"].data_ptr(), y,
                                              case["tokens"], s["res"].data_ptr(), None),
                "matmat_mv")
    else:
        M.set_int8(M.INT8_BATCHED)
        M.matmat_dev(qtype, w, rows, cols, s["x"].data_ptr(), y, case["tokens"])
        M.set_int8(M.INT8_OFF)
    return s["y"]


# ── what a pass cannot do without, and how far outputs may be apart ──────────

def work(case):
    kind = case["kind"]
    if kind in ("forced", "generate"):
        d, ff = case["d_model"], case["d_ff"]
        q, kv = 128 * case["heads"], 128 * case["kv_heads"]
        # The Q4_K_M mix: half of the v and down projections are Q6_K.
        q4 = d * (2 * q + kv) + 2 * ff * d + (d * kv + d * ff) / 2
        q6 = (d * kv + d * ff) / 2
        layer, params = q4 * 144 / 256 + q6 * 210 / 256, q4 + q6
        head = case["vocab"] * d
        n0, n = case["prompt"], case["steps"] + (1 if kind == "generate" else 0)
        passes = n + (1 if n0 > 1 else 0)
        pos = n0 + n
        attn = 4 * q * (pos * (pos + 1) / 2) * case["layers"]
        kv_read = 8 * kv * case["layers"] * (n * (n0 + n / 2) + n0)
        return {"bytes": passes * case["layers"] * layer + n * head * 210 / 256 + kv_read
                + 4 * case["vocab"],
                "flops": 2 * params * case["layers"] * pos + 2 * head * n + attn}
    rows, cols, tokens = case["rows"], case["cols"], case.get("tokens", 1)
    w = rows * M.row_bytes(TYPES[case["type"]], cols)
    if kind == "dequant":
        return {"bytes": w + 4 * rows * cols, "flops": 2 * rows * cols}
    res = 4 * tokens * rows if case.get("lane") == "matvec" else 0
    return {"bytes": w + 4 * tokens * (rows + cols) + res, "flops": 2 * rows * cols * tokens}


def tolerance(case):
    # Every default path promises the reference's own bits, whatever the launch. The reordered
    # GEMV and the split attention sum in an order of their own: against the exact order, over 60
    # and 20 drawn cases, 4.2e-7 (largest 3.3e-6) of the vector and 2.1e-6 (1.2e-5) of the logits;
    # four times that.
    if case.get("order") == "reordered":
        return {"rel": 2e-6, "max": 1.4e-5}
    if case.get("attention") == "split":
        return {"rel": 8e-6, "max": 5e-5}
    return "exact"


# ── the same results in 64 bits, from the block formats alone ────────────────

def _f16(b):
    return b.contiguous().view(torch.float16).double()


def _scale_min(s):
    """The eight 6-bit (scale, min) pairs of Q4_K / Q5_K from their 12 bytes."""
    s = s.int()
    a, b, c = s[..., 0:4], s[..., 4:8], s[..., 8:12]
    sc = torch.cat([a & 63, (c & 15) | ((a >> 6) << 4)], -1)
    mn = torch.cat([b & 63, (c >> 4) | ((b >> 6) << 4)], -1)
    return sc.double(), mn.double()


def _dequant64(qtype, raw, rows, cols):
    """The matrix [rows][cols] in 64 bits from its uint8 blocks on the GPU."""
    elems, size = M.BLOCK[qtype]
    b = raw.reshape(rows, cols // elems, size)
    if qtype == Q8_0:
        v = b[..., 2:].contiguous().view(torch.int8).double() * _f16(b[..., :2])
    elif qtype == Q4_0:
        q = torch.cat([b[..., 2:] & 15, b[..., 2:] >> 4], -1)
        v = (q.double() - 8) * _f16(b[..., :2])
    elif qtype in (Q4_K, Q5_K):
        sc, mn = _scale_min(b[..., 4:16])
        qs = b[..., size - 128:].reshape(rows, -1, 4, 1, 32)
        q = torch.cat([qs & 15, qs >> 4], 3).reshape(rows, -1, 8, 32).int()
        if qtype == Q5_K:
            j = torch.arange(8, device=raw.device, dtype=torch.int32).reshape(8, 1)
            q = q | (((b[..., 16:48].int().unsqueeze(-2) >> j) & 1) << 4)
        v = (q.double() * (sc * _f16(b[..., 0:2])).unsqueeze(-1)
             - (mn * _f16(b[..., 2:4])).unsqueeze(-1))
    else:
        ql = b[..., :128].reshape(rows, -1, 2, 1, 2, 32).int()
        ql = torch.cat([ql & 15, ql >> 4], 3).reshape(rows, -1, 2, 4, 32)
        k = 2 * torch.arange(4, device=raw.device, dtype=torch.int32).reshape(4, 1)
        qh = (b[..., 128:192].reshape(rows, -1, 2, 1, 32).int() >> k) & 3
        q = ((ql | (qh << 4)) - 32).double().reshape(rows, -1, 16, 16)
        sc = b[..., 192:208].contiguous().view(torch.int8).double()
        v = q * (sc * _f16(b[..., 208:210])).unsqueeze(-1)
    return v.reshape(rows, cols)


def _exact_model(case, seed):
    shape, f64 = _shape(case), torch.float64
    model = M.SynthQwen3(shape, _seed(seed, 0))
    prompt, inputs = _tokens(case, seed)
    ids = torch.from_numpy(np.concatenate([prompt, inputs]).astype(np.int64)).to(GPU)
    blob = torch.from_numpy(model.blob).to(GPU)
    tensors = {}
    for t in model.table[:model.count]:
        raw = blob[t.offset:t.offset + t.nbytes]
        tensors[t.name.decode()] = (t.type, raw, t.rows, t.cols)

    def get(name):
        qtype, raw, rows, cols = tensors[name]
        return raw.view(torch.float32).double() if qtype == 0 else _dequant64(qtype, raw, rows, cols)

    def norm(x, w):
        return x * torch.rsqrt(x.square().mean(-1, keepdim=True) + shape.rms_eps) * w

    n, hd, group = ids.numel(), 128, shape.n_heads // shape.n_kv_heads
    inv = shape.rope_theta ** (-torch.arange(0, hd, 2, device=GPU, dtype=f64) / hd)
    angle = torch.arange(n, device=GPU, dtype=f64).unsqueeze(1) * inv
    cos, sin = angle.cos().unsqueeze(1), angle.sin().unsqueeze(1)

    def rope(x):
        a, b = x[..., :hd // 2], x[..., hd // 2:]
        return torch.cat([a * cos - b * sin, b * cos + a * sin], -1)

    table = get("token_embd.weight")
    x = table[ids]
    mask = torch.ones(n, n, device=GPU, dtype=torch.bool).triu(1)
    for i in range(shape.n_layers):
        p = f"blk.{i}."
        h = norm(x, get(p + "attn_norm.weight"))
        q = (h @ get(p + "attn_q.weight").T).reshape(n, shape.n_heads, hd)
        k = (h @ get(p + "attn_k.weight").T).reshape(n, shape.n_kv_heads, hd)
        v = (h @ get(p + "attn_v.weight").T).reshape(n, shape.n_kv_heads, hd)
        q = rope(norm(q, get(p + "attn_q_norm.weight")))
        k = rope(norm(k, get(p + "attn_k_norm.weight")))
        out = torch.empty_like(q)
        for g in range(shape.n_heads):
            s = (q[:, g] @ k[:, g // group].T.contiguous()) / math.sqrt(hd)
            out[:, g] = s.masked_fill(mask, -math.inf).softmax(-1) @ v[:, g // group]
        x = x + out.reshape(n, -1) @ get(p + "attn_output.weight").T
        h = norm(x, get(p + "ffn_norm.weight"))
        g = h @ get(p + "ffn_gate.weight").T
        x = x + (g * g.sigmoid() * (h @ get(p + "ffn_up.weight").T)) @ get(p + "ffn_down.weight").T
    return {"ids": None, "logits": norm(x[-1], get("output_norm.weight")) @ table.T}


def exact(case, seed):
    kind = case["kind"]
    if kind == "generate":
        # Every input is the previous step's choice: one near-tie taken the other way changes
        # all that follows.
        return None
    if kind == "forced":
        return _exact_model(case, seed)
    rows, cols, tokens = case["rows"], case["cols"], case.get("tokens", 1)
    w = _dequant64(TYPES[case["type"]], torch.from_numpy(_weights(case, seed)).to(GPU), rows, cols)
    if kind == "dequant":
        return w
    x = torch.from_numpy(_normal(seed, 1, tokens, cols)).to(GPU)
    if case.get("lane") == "int8":
        # The lane's activations are whole numbers of 127ths of each 256 values' largest; which
        # whole numbers is the format's, in 32 bits.
        b = x.reshape(tokens, -1, 256)
        top = b.abs().amax(-1, keepdim=True)
        x = ((b * (127.0 / top)).round().double() * (top.double() / 127)).reshape(tokens, cols)
    y = x.double() @ w.T
    if case.get("lane") == "matvec":
        y = y + torch.from_numpy(_normal(seed, 2, tokens, rows)).to(GPU).double()
    return y[0] if kind == "dropin" else y
