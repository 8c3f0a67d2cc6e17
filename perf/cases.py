"""The work a host of this library has it do, as cases that can be timed.

A case is one linear layer, one FFN or attention block (a decode token or a
prompt), the ternary FFN, or a whole engine call. `numerics` is the weight
format and the order of the arithmetic with it: "q8" (packed Q8_0 tiles, Q8_0
activations), "ref" (row-major Q8 with fp32 scales, bf16 activations in the
reference's own order), "q4" / "q5" (the low-bit tensors). Shapes are those of
the two backbones the library is configured for: hidden 2048, FFN 8192, 32 q /
8 kv heads of 64, vocab 65536, 3 taps; and hidden 2048, FFN 7680, 16 / 4 heads
of 128, vocab 128000, 7 taps, sliding windows of 256.
"""
import math
import os
import sys

import numpy as np
import torch

sys.path.insert(0, os.path.join(os.path.dirname(os.path.abspath(__file__)), "..", "pulsar-asm_amd"))
import pulsar_amd as pq  # noqa: E402
from pulsar_amd.engine import Engine  # noqa: E402

DEV = "cuda"
EPS = 1e-5
CTX = 2048          # positions of a kept KV cache
BF16 = torch.bfloat16

# q heads, kv heads, rotated dims and RoPE base of an attention layer by head_dim
HEADS = {64: (32, 8), 128: (16, 4)}

# The two backbones at full width and fewer layers. "even" keeps the 2:1 mix of
# conv and attention layers, "sliding" the first five layers of its pattern
# (conv, conv, full attention, conv, sliding-window attention).
BACKBONES = {
    "even": dict(hidden=2048, ffn=8192, vocab=65536, nlayers=6, nh=32, nkv=8, hd=64, rot=32, ntaps=3, ctx=CTX,
                 eps=EPS, theta=1e6, attn_mask=0b110000, prefill_chunk=256),
    "sliding": dict(hidden=2048, ffn=7680, vocab=128000, nlayers=5, nh=16, nkv=4, hd=128, rot=64, ntaps=7, ctx=CTX,
                    eps=EPS, theta=1e6, attn_mask=0b10100, prefill_chunk=256, slide_mask=0b10000, slide_win=256,
                    slide_rot=128, slide_theta=1e4),
}


def listed():
    return [
        # the smallest call: one projection of one decode token (quantize, GEMV)
        dict(name="linear_q8_t1", kind="linear", numerics="q8", N=2048, K=2048, T=1),
        # the FFN of one decode token
        dict(name="mlp_decode_q8", kind="mlp", numerics="q8", H=2048, F=8192, T=1),
        dict(name="mlp_decode_q4", kind="mlp", numerics="q4", H=2048, F=8192, T=1),
        # the attention block of one decode token, far into a context
        dict(name="attn_decode_ref", kind="attn", numerics="ref", H=2048, hd=128, T=1, pos0=1500, win=0),
        # the FFN over a prompt: a whole chunk, the other backbone's width, a short ragged one
        dict(name="mlp_prefill_q8", kind="mlp", numerics="q8", H=2048, F=8192, T=256),
        dict(name="mlp_prefill_ref", kind="mlp", numerics="ref", H=2048, F=7680, T=256),
        dict(name="mlp_prefill_q5", kind="mlp", numerics="q5", H=2048, F=8192, T=77),
        # the attention block over a prompt, and over a chunk of a long one in a sliding-window layer
        dict(name="attn_prefill_q8", kind="attn", numerics="q8", H=2048, hd=64, T=512, pos0=0, win=0),
        dict(name="attn_prefill_ref", kind="attn", numerics="ref", H=2048, hd=128, T=203, pos0=300, win=256),
        # the ternary FFN's projections of one decode token
        dict(name="ternary_mlp", kind="ternary", H=4096, F=12288),
        # a whole answer: prompt, then greedy decoding, then the next logits
        dict(name="generate_q8", kind="engine", numerics="q8", backbone="even", prompt=300, steps=32),
        # a whole prompt in the reference's numerics, to its logits
        dict(name="prompt_ref", kind="engine", numerics="ref", backbone="sliding", prompt=256, steps=0),
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["linear", "linear", "mlp", "mlp", "mlp", "attn", "attn", "attn", "ternary", "engine"])
    if kind == "linear":
        num = rng.choice(["q8", "ref", "q4", "q5"])
        unit = 256 if num in ("q4", "q5") else 32
        K = unit * max(1, _log(rng, 256, 8192) // unit)
        N = _log(rng, 64, 65536)
        if num in ("q4", "q5"):
            N = 32 * (N // 32)
        T = rng.choice([1, _log(rng, 2, 512)])
        T = max(1, min(T, int(4e10 / (2.0 * N * K))))
        return dict(kind=kind, numerics=num, N=N, K=K, T=T)
    if kind == "mlp":
        num = rng.choice(["q8", "ref", "q4", "q5"])
        unit = 256 if num in ("q4", "q5") else 32
        T = rng.choice([1, _log(rng, 2, 512)])
        return dict(kind=kind, numerics=num, H=rng.choice([2048, 2048, 4096]),
                    F=unit * (_log(rng, 1024, 8192) // unit), T=T if num == "q8" else min(T, 256))
    if kind == "attn":
        num = rng.choice(["q8", "ref"])
        T = rng.choice([1, _log(rng, 2, 1024 if num == "q8" else 256)])
        return dict(kind=kind, numerics=num, H=2048, hd=rng.choice([64, 128]), T=T,
                    pos0=rng.choice([0, _log(rng, 1, CTX - T)]), win=rng.choice([0, 0, 256]))
    if kind == "ternary":
        return dict(kind=kind, H=256 * (_log(rng, 1024, 4096) // 256), F=256 * (_log(rng, 2560, 12288) // 256))
    return dict(kind=kind, numerics=rng.choice(["q8", "ref"]), backbone=rng.choice(["even", "sliding"]),
                prompt=_log(rng, 1, 256), steps=rng.choice([0, _log(rng, 1, 24)]))


# ----------------------------------------------------------------- inputs
def _gen(seed):
    g = torch.Generator(device=DEV)
    g.manual_seed(seed)
    return g


def _bf16(g, *shape, s=1.0):
    return (torch.randn(shape, device=DEV, generator=g) * s).to(BF16)


def _vec(g, n, a, b):
    return a + b * torch.randn(n, device=DEV, generator=g)


def _q8_rows(g, N, K):
    """Q8_0 weight rows of variance about 1/K: int8 codes, fp16 scales."""
    codes = torch.randint(-127, 128, (N, K), dtype=torch.int8, device=DEV, generator=g)
    scales = (torch.randn((N, K // 32), device=DEV, generator=g).abs() / (73.0 * math.sqrt(K))).half()
    return codes, scales


def _low_rows(g, N, K, bits):
    """Q4 / Q5 rows: one code per byte and (d' = 128 d, mn) fp16 per 32-group."""
    codes = torch.randint(0, 1 << bits, (N, K), dtype=torch.uint8, device=DEV, generator=g)
    d = torch.rand((N, K // 32), device=DEV, generator=g) * (4.0 / ((1 << bits) * math.sqrt(K)))
    return codes, torch.stack([128.0 * d, -d * ((1 << bits) / 2.0)], -1).half()


def _rows(g, num, N, K):
    return _low_rows(g, N, K, int(num[1])) if num in ("q4", "q5") else _q8_rows(g, N, K)


def _weight(num, rows, gate_up=False):
    """The handle a program keeps for these rows."""
    codes, scales = rows
    if num == "q8":
        return pq.Q8Weight(codes, scales, gate_up=gate_up)
    if num == "ref":
        return codes, scales.float()
    return pq.QlowWeight(codes, scales, int(num[1]))


def _workspace(ws_bytes):
    return torch.empty(max(16, ws_bytes), dtype=torch.uint8, device=DEV)


def _rope_table(hd, rot, theta):
    """[CTX][rot/2][cos, sin] fp32 of the fp32 angles pos * theta^(-2i/hd)."""
    i = np.arange(rot // 2, dtype=np.float32)
    invf = np.float32(1.0) / np.power(np.float32(theta), 2 * i / np.float32(hd), dtype=np.float32)
    a = (np.arange(CTX, dtype=np.float32)[:, None] * invf).astype(np.float64)
    return torch.from_numpy(np.stack([np.cos(a), np.sin(a)], -1).astype(np.float32)).to(DEV)


def _attn_shape(case):
    nh, nkv = HEADS[case["hd"]]
    rot, theta = (case["hd"], 1e4) if case["win"] else (case["hd"] // 2, 1e6)
    return nh, nkv, rot, theta


def _attn_inputs(case, seed):
    g = _gen(seed)
    H, hd, T = case["H"], case["hd"], case["T"]
    nh, nkv, rot, theta = _attn_shape(case)
    nin = (nh + 2 * nkv) * hd + nh          # q | k | v | gate rows
    dt = torch.float16 if case["numerics"] == "q8" else BF16
    cache = [(torch.randn((CTX, nkv * hd), device=DEV, generator=g) * s).to(dt) for s in (1.0, 1.0)]
    return dict(x=_bf16(g, T, H, s=4.0), h=_bf16(g, T, H), w0=_vec(g, H, 4.0, 0.4), w1=_vec(g, H, 1.0, 0.1),
                qn=_vec(g, hd, 1.0, 0.1), kn=_vec(g, hd, 1.0, 0.1), kc=cache[0], vc=cache[1],
                rows_in=_q8_rows(g, nin, H), rows_out=_q8_rows(g, H, nh * hd), cs=_rope_table(hd, rot, theta), nin=nin)


def _mlp_inputs(case, seed):
    g = _gen(seed)
    H, F, T, num = case["H"], case["F"], case["T"], case["numerics"]
    return dict(x=_bf16(g, T, H, s=4.0), h=_bf16(g, T, H), w0=_vec(g, H, 4.0, 0.4), w1=_vec(g, H, 1.0, 0.1),
                rows_gu=_rows(g, num, 2 * F, H), rows_down=_rows(g, num, H, F))


def _linear_inputs(case, seed):
    g = _gen(seed)
    return _bf16(g, case["T"], case["K"]), _rows(g, case["numerics"], case["N"], case["K"])


def _ternary_inputs(case, seed):
    g = _gen(seed)

    def tensor(N, K):
        c = torch.randint(0, 3, (N, K // 4, 4), dtype=torch.uint8, device=DEV, generator=g)
        codes = c[..., 0] | (c[..., 1] << 2) | (c[..., 2] << 4) | (c[..., 3] << 6)
        return codes, (torch.randn((N, K // 128), device=DEV, generator=g).abs() * (1.2 / math.sqrt(K))).half()

    H, F = case["H"], case["F"]
    return dict(x=torch.randn(H, device=DEV, generator=g), z=torch.randn(F, device=DEV, generator=g),
                gate=tensor(F, H), up=tensor(F, H), down=tensor(H, F))


def _engine_slots(cfg):
    """(layer, slot, N, K) of the Q8 tensors and (layer, slot, n, mean, spread) of the fp32 ones."""
    H, F, hd = cfg["hidden"], cfg["ffn"], cfg["hd"]
    q8, f32 = [(-1, 0, cfg["vocab"], H)], [(-1, 1, H, 1.0, 0.1)]
    for n in range(cfg["nlayers"]):
        attn = cfg["attn_mask"] >> n & 1
        q8 += [(n, 0, (cfg["nh"] + 2 * cfg["nkv"]) * hd + cfg["nh"] if attn else 3 * H, H),
               (n, 1, H, cfg["nh"] * hd if attn else H), (n, 2, 2 * F, H), (n, 3, H, F)]
        f32 += [(n, 4, H, 1.0, 0.1), (n, 5, H, 4.0, 0.4), (n, 6, H, 1.0, 0.1), (n, 7, H, 4.0, 0.4)]
        f32 += [(n, 8, hd, 1.0, 0.1), (n, 9, hd, 1.0, 0.1)] if attn else [(n, 10, H * cfg["ntaps"], 0.0, 0.5)]
    return q8, f32


def _engine_inputs(case, seed):
    cfg = BACKBONES[case["backbone"]]
    g = _gen(seed)
    q8, f32 = _engine_slots(cfg)
    prompt = torch.randint(0, cfg["vocab"], (case["prompt"],), device=DEV, generator=g)
    return cfg, {s[:2]: _q8_rows(g, *s[2:]) for s in q8}, {s[:2]: _vec(g, *s[2:]) for s in f32}, prompt


def prepare(case, seed):
    kind, num = case["kind"], case.get("numerics")
    if kind == "linear":
        x, rows = _linear_inputs(case, seed)
        s = dict(x=x[0] if case["T"] == 1 else x, w=_weight(num, rows))
        if num == "q8":
            s["ws"] = _workspace(pq.lib().pq_q8_gemm_workspace_bytes(case["N"], case["K"], case["T"]))
        elif num != "ref":
            s["ws"] = _workspace(pq.lib().pq_qlow_workspace_bytes(case["N"], case["K"], int(num[1])))
    elif kind == "mlp":
        s = _mlp_inputs(case, seed)
        s["gu"] = _weight(num, s.pop("rows_gu"), gate_up=True)
        s["down"] = _weight(num, s.pop("rows_down"))
        s["x_out"] = torch.empty_like(s["x"])
        H, F, T = case["H"], case["F"], case["T"]
        if num == "q8":
            s["ws"] = _workspace(max(pq.lib().pq_q8_gemm_workspace_bytes(2 * F, H, T),
                                     pq.lib().pq_q8_gemm_workspace_bytes(H, F, T)))
        elif num != "ref":
            s["ws"] = _workspace(pq.lib().pq_qlow_workspace_bytes(H, F, int(num[1])))
    elif kind == "attn":
        s = _attn_inputs(case, seed)
        s["w_in"] = _weight(num, s.pop("rows_in"))
        s["w_out"] = _weight(num, s.pop("rows_out"))
        nh, nkv, rot, _ = _attn_shape(case)
        H, hd, T = case["H"], case["hd"], case["T"]
        s["x_out"] = torch.empty_like(s["x"])
        s["scale"] = 1.0 / math.sqrt(hd)
        if T > 1:
            s["o"] = torch.empty((T, nh * hd), dtype=BF16, device=DEV)
            s["ws"] = _workspace(pq.lib().pq_attn_workspace_bytes(nh, hd, case["pos0"] + T, T))
            s["gws"] = _workspace(max(pq.lib().pq_q8_gemm_workspace_bytes(s["nin"], H, T),
                                      pq.lib().pq_q8_gemm_workspace_bytes(H, nh * hd, T)))
        else:
            s["o"] = torch.empty(nh * hd, dtype=BF16, device=DEV)
    elif kind == "ternary":
        s = _ternary_inputs(case, seed)
    else:
        cfg, q8, f32, prompt = _engine_inputs(case, seed)
        e = Engine(numerics=0 if num == "q8" else 1, **cfg)
        for (layer, slot), (codes, scales) in q8.items():
            e.set_q8(layer, slot, codes.cpu().numpy(), scales.cpu().numpy().view(np.uint16))
        for (layer, slot), v in f32.items():
            e.set_f32(layer, slot, v.cpu().numpy())
        e.mark_loaded()
        s = dict(engine=e, prompt=prompt.cpu().numpy().astype(np.int32))
    s["case"] = case
    return s


# ------------------------------------------------------------------ a pass
def _run_linear(c, s):
    num, T, x, w = c["numerics"], c["T"], s["x"], s["w"]
    if num == "ref":
        return pq.q8r_gemv(w[0], w[1], x)
    if num == "q8":
        qx, dx = pq.q8_quant(x)
        if T == 1:
            return pq.q8_gemv(w, qx, dx, out_dtype=pq.DT_BF16)
        return pq.q8_gemm(w, qx, dx, out_dtype=pq.DT_BF16, ws=s["ws"])
    return pq.qlow_gemv(w, x, ws=s["ws"]) if T == 1 else pq.qlow_gemm(w, x)


def _run_mlp_decode(c, s):
    """x += rms(h, w0); down(silu(gate) * up) of rms(x, w1), as a decode step fuses them."""
    num, gu, down = c["numerics"], s["gu"], s["down"]
    pro = dict(h=s["h"], x_in=s["x"], x_out=s["x_out"], w0=s["w0"], w1=s["w1"], eps=EPS)
    if num == "q8":
        qx, dx = pq.gemv_fused_swiglu(gu, pq.PRO_RESNORM, **pro)
        return s["x_out"], pq.q8_gemv(down, qx, dx, out_dtype=pq.DT_BF16)
    if num == "ref":
        a = pq.q8r_gemv_fused_swiglu(gu[0], gu[1], pq.PRO_RESNORM, **pro)
        return s["x_out"], pq.q8r_gemv(down[0], down[1], a)
    a = pq.qlow_gemv_fused_swiglu(gu, pq.PRO_RESNORM, **pro)
    return s["x_out"], pq.qlow_gemv(down, a, ws=s["ws"])


def _run_mlp_prefill(c, s):
    num, gu, down, T, F = c["numerics"], s["gu"], s["down"], c["T"], c["F"]
    if num == "q8":
        _, qx, dx = pq.rmsnorm(s["x"], s["w1"], eps=EPS, out=False, quant=True)
        a = pq.q8_gemm(gu, qx, dx, out_dtype=pq.DT_BF16, ws=s["ws"])
        _, qx, dx = pq.silu_mul(a, F, T, out=False, quant=True, interleaved=True)
        return pq.q8_gemm(down, qx, dx, out_dtype=pq.DT_BF16, ws=s["ws"])
    y, _, _ = pq.rmsnorm(s["x"], s["w1"], eps=EPS)
    a = pq.q8r_gemv(gu[0], gu[1], y) if num == "ref" else pq.qlow_gemm(gu, y)
    a, _, _ = pq.silu_mul(a, F, T)
    return pq.q8r_gemv(down[0], down[1], a) if num == "ref" else pq.qlow_gemm(down, a)


def _run_attn_decode(c, s):
    """x += rms(h, w0); o_proj(attention(rms(x, w1))) of one token, as a decode step fuses them."""
    nh, nkv, rot, _ = _attn_shape(c)
    hd, win, wout = c["hd"], s["w_in"], s["w_out"]
    pro = dict(h=s["h"], x_in=s["x"], x_out=s["x_out"], w0=s["w0"], w1=s["w1"], eps=EPS)
    if c["numerics"] == "q8":
        row = pq.gemv_fused(win, pq.PRO_RESNORM, **pro)
        qx, dx = pq.attn_layer_decode(row, s["qn"], s["kn"], s["cs"], s["kc"], s["vc"], c["pos0"], nh, nkv, hd, rot,
                                      s["scale"], eps=EPS, win=c["win"])
        return s["x_out"], s["kc"], s["vc"], pq.q8_gemv(wout, qx, dx, out_dtype=pq.DT_BF16)
    row = pq.q8r_gemv_fused(win[0], win[1], pq.PRO_RESNORM, **pro)
    pq.attn_decode_ref(row, s["qn"], s["kn"], s["cs"], s["kc"], s["vc"], c["pos0"], nh, nkv, hd, rot, s["scale"],
                       s["o"], gate=row[(nh + 2 * nkv) * hd:], eps=EPS, win=c["win"])
    return s["x_out"], s["kc"], s["vc"], pq.q8r_gemv(wout[0], wout[1], s["o"])


def _run_attn_prefill(c, s):
    nh, nkv, rot, _ = _attn_shape(c)
    hd, T, pos0, nin, win, wout = c["hd"], c["T"], c["pos0"], s["nin"], s["w_in"], s["w_out"]
    g0 = (nh + 2 * nkv) * hd
    if c["numerics"] == "q8":
        _, qx, dx = pq.rmsnorm(s["x"], s["w1"], eps=EPS, out=False, quant=True)
        rows = pq.q8_gemm(win, qx, dx, out_dtype=pq.DT_BF16, ws=s["gws"])
        pq.qk_prep(rows, nin, s["qn"], s["kn"], s["cs"], s["kc"], s["vc"], pos0, nh, nkv, hd, rot, T, eps=EPS)
        qx = torch.empty((T, nh * hd), dtype=torch.int8, device=DEV)
        dx = torch.empty((T, nh * hd // 32), dtype=torch.float32, device=DEV)
        pq.attn_decode(rows, nin, s["kc"], s["vc"], pos0, nh, nkv, hd, T, s["scale"], gate=rows[:, g0:],
                       gate_stride=nin, qx=qx, dx=dx, ws=s["ws"], win=c["win"])
        return s["kc"], s["vc"], pq.q8_gemm(wout, qx, dx, out_dtype=pq.DT_BF16, ws=s["gws"])
    y, _, _ = pq.rmsnorm(s["x"], s["w1"], eps=EPS)
    rows = pq.q8r_gemv(win[0], win[1], y)
    pq.qk_prep_ref(rows, nin, s["qn"], s["kn"], s["cs"], s["kc"], s["vc"], pos0, nh, nkv, hd, rot, T, eps=EPS)
    pq.attn_ref(rows, nin, s["kc"], s["vc"], pos0, nh, nkv, hd, T, s["scale"], s["o"], nh * hd, gate=rows[:, g0:],
                gate_stride=nin, win=c["win"])
    return s["kc"], s["vc"], pq.q8r_gemv(wout[0], wout[1], s["o"])


def _run_ternary(c, s):
    """gate and up read one activation; down reads the combined one (formed by the host's own code)."""
    g, u = pq.tq2_gemv_batch([s["gate"], s["up"]], pq.q8k_quant(s["x"]), c["H"])
    return g, u, pq.tq2_gemv(*s["down"], pq.q8k_quant(s["z"]), c["F"], c["H"])


def _run_engine(c, s):
    e = s["engine"]
    if c["steps"]:
        ids = e.greedy(s["prompt"], c["steps"] + 1)
        nxt, logits = e.feed(ids[-1:], want_logits=True)
        return ids, nxt, logits, e.hidden()
    e.reset()
    nxt, logits = e.feed(s["prompt"], want_logits=True)
    return nxt, logits, e.hidden()


def run(state):
    c = state["case"]
    if c["kind"] == "linear":
        return _run_linear(c, state)
    if c["kind"] == "mlp":
        return _run_mlp_decode(c, state) if c["T"] == 1 else _run_mlp_prefill(c, state)
    if c["kind"] == "attn":
        return _run_attn_decode(c, state) if c["T"] == 1 else _run_attn_prefill(c, state)
    return _run_ternary(c, state) if c["kind"] == "ternary" else _run_engine(c, state)


# ------------------------------------------------------------ what it needs
# bytes a weight takes: codes and the scales of a 32-block (or 128-group)
WEIGHT_BYTES = {"q8": 1 + 2 / 32, "ref": 1 + 4 / 32, "q4": 0.5 + 4 / 32, "q5": 0.625 + 4 / 32, "t2": 0.25 + 2 / 128}


def _keys(pos0, T, win):
    """Keys seen by T queries from pos0, and the cache rows they cover."""
    n = sum(min(p, win) if win else p for p in range(pos0 + 1, pos0 + T + 1))
    return n, min(pos0 + T, T + win) if win else pos0 + T


def work(case):
    kind = case["kind"]
    if kind == "linear":
        N, K, T = case["N"], case["K"], case["T"]
        return {"bytes": N * K * WEIGHT_BYTES[case["numerics"]] + 2 * T * (N + K), "flops": 2.0 * N * K * T}
    if kind == "mlp":
        H, F, T = case["H"], case["F"], case["T"]
        return {"bytes": 3 * H * F * WEIGHT_BYTES[case["numerics"]] + 8 * T * H, "flops": 6.0 * H * F * T}
    if kind == "attn":
        H, hd, T = case["H"], case["hd"], case["T"]
        nh, nkv = HEADS[hd]
        nin = (nh + 2 * nkv) * hd + nh
        keys, rows = _keys(case["pos0"], T, case["win"])
        weights = nin * H + H * nh * hd
        return {"bytes": weights * WEIGHT_BYTES[case["numerics"]] + 4 * rows * nkv * hd + 8 * T * H,
                "flops": 2.0 * T * weights + 4.0 * keys * nh * hd}
    if kind == "ternary":
        n = 3 * case["H"] * case["F"]
        return {"bytes": n * WEIGHT_BYTES["t2"] + 8 * (case["H"] + case["F"]) + 4 * case["F"], "flops": 2.0 * n}
    cfg = BACKBONES[case["backbone"]]
    q8, _ = _engine_slots(cfg)
    body, head = sum(N * K for n, _, N, K in q8 if n >= 0), cfg["vocab"] * cfg["hidden"]
    steps = case["steps"] + 1 if case["steps"] else 0     # the decode steps and the fed token
    keys, rows = _keys(0, case["prompt"] + steps, 0)
    n_attn = bin(cfg["attn_mask"]).count("1")
    w = WEIGHT_BYTES[case["numerics"]]
    return {"bytes": (1 + steps) * (body + head) * w + n_attn * 4.0 * cfg["nkv"] * cfg["hd"] * (rows + steps * rows),
            "flops": 2.0 * body * (case["prompt"] + steps) + 2.0 * head * (1 + steps)
                     + n_attn * 4.0 * keys * cfg["nh"] * cfg["hd"]}


def tolerance(case):
    """Every entry point states its order of operations and gives the same bits at any T, chunk or launch shape."""
    return "exact"


# -------------------------------------------------- the same in 64 bits
def _r16(v):
    return v.to(BF16).double()


def _rms(x, w):
    """The norm rounds to bf16 before the weight multiplies, and after it."""
    return _r16(_r16(x * torch.rsqrt((x * x).mean(-1, keepdim=True) + EPS)) * w.double())


def _act(num, x):
    """The GEMV's input as the numerics read it: Q8_0 blocks of 32, or x."""
    if num != "q8":
        return x
    b = x.float().reshape(*x.shape[:-1], -1, 32)
    d = b.abs().amax(-1, keepdim=True) / 127.0
    q = torch.round(b / torch.where(d > 0, d, torch.ones_like(d))).clamp(-127, 127)
    return (q.double() * d.double()).reshape(x.shape)


def _dense(num, rows):
    codes, scales = rows
    if num in ("q4", "q5"):
        s = scales.double()
        return codes.double() * (s[..., 0] / 128.0).repeat_interleave(32, 1) + s[..., 1].repeat_interleave(32, 1)
    return codes.double() * scales.double().repeat_interleave(32, 1)


def _mm(num, rows, x):
    """x [T][K] times the rows, a few thousand of them at a time."""
    codes, scales = rows
    a = _act(num, x)
    return torch.cat([a @ _dense(num, (codes[n:n + 8192], scales[n:n + 8192])).T for n in range(0, len(codes), 8192)], -1)


def _silu_mul(gu):
    g, u = gu.chunk(2, -1)
    return _r16(g * torch.sigmoid(g) * u)


def _attention(num, rows, qn, kn, cs, kc, vc, pos0, nh, nkv, hd, rot, win):
    """q | k | v | gate rows [T] -> gated attention output; kc / vc take the new rows."""
    T = rows.shape[0]

    def head(v, w):
        return _rms(v, w)

    def rope(v):
        c, s = (cs[pos0:pos0 + T, :, i].double()[:, None] for i in (0, 1))
        lo, hi = v[..., :rot // 2].clone(), v[..., hd // 2:hd // 2 + rot // 2].clone()
        v = v.clone()
        v[..., :rot // 2], v[..., hd // 2:hd // 2 + rot // 2] = _r16(lo * c - hi * s), _r16(hi * c + lo * s)
        return v

    q, k, v, gate = rows.split([nh * hd, nkv * hd, nkv * hd, nh], -1)
    q = rope(head(q.reshape(T, nh, hd), qn))
    k = rope(head(k.reshape(T, nkv, hd), kn))
    kc[pos0:pos0 + T] = k.reshape(T, -1).to(kc.dtype)
    vc[pos0:pos0 + T] = v.to(vc.dtype)
    n = pos0 + T
    K = kc[:n].double().reshape(n, nkv, hd).repeat_interleave(nh // nkv, 1)
    V = vc[:n].double().reshape(n, nkv, hd).repeat_interleave(nh // nkv, 1)
    at, key = torch.arange(pos0, n, device=DEV)[:, None], torch.arange(n, device=DEV)[None]
    seen = (key <= at) & ((key > at - win) if win else (key >= 0))
    out = torch.empty((T, nh, hd), dtype=torch.float64, device=DEV)
    for h in range(nh):
        p = (q[:, h] @ K[:, h].T / math.sqrt(hd)).masked_fill(~seen, -math.inf).softmax(-1)
        out[:, h] = _r16(p @ V[:, h])
    return _r16(out * torch.sigmoid(gate)[..., None]).reshape(T, nh * hd)


def _conv(bcx, taps, ntaps):
    B, C, x = bcx.chunk(3, -1)
    bx = torch.nn.functional.pad(_r16(B * x), (0, 0, ntaps - 1, 0))
    y = sum(taps[:, k] * bx[k:k + bcx.shape[0]] for k in range(ntaps))
    return _r16(C * _r16(y))


def _backbone(case, seed):
    cfg, q8, f32, prompt = _engine_inputs(case, seed)
    num, H, hd, nh, nkv = case["numerics"], cfg["hidden"], cfg["hd"], cfg["nh"], cfg["nkv"]
    codes, scales = q8[-1, 0]
    x = _r16(codes[prompt].double() * scales[prompt].double().repeat_interleave(32, 1))
    for n in range(cfg["nlayers"]):
        y = _rms(x, f32[n, 4])
        rows = _r16(_mm(num, q8[n, 0], y))
        if cfg["attn_mask"] >> n & 1:
            slide = cfg.get("slide_mask", 0) >> n & 1
            rot, theta, win = (cfg["slide_rot"], cfg["slide_theta"], cfg["slide_win"]) if slide else (
                cfg["rot"], cfg["theta"], 0)
            kc, vc = (torch.zeros((CTX, nkv * hd), dtype=torch.float16 if num == "q8" else BF16, device=DEV)
                      for _ in range(2))
            a = _attention(num, rows, f32[n, 8], f32[n, 9], _rope_table(hd, rot, theta), kc, vc, 0, nh, nkv, hd, rot,
                           win)
        else:
            a = _conv(rows, f32[n, 10].double().reshape(H, -1), cfg["ntaps"])
        x = _r16(x + _rms(_r16(_mm(num, q8[n, 1], a)), f32[n, 5]))
        a = _silu_mul(_r16(_mm(num, q8[n, 2], _rms(x, f32[n, 6]))))
        x = _r16(x + _rms(_r16(_mm(num, q8[n, 3], a)), f32[n, 7]))
    return _mm(num, q8[-1, 0], _rms(x[-1:], f32[-1, 1]))[0]


def _ternary_mm(tensor, x):
    codes, scales = tensor
    w = torch.stack([codes >> (2 * i) & 3 for i in range(4)], -1).reshape(codes.shape[0], -1).double() - 1.0
    b = x.reshape(-1, 256)
    top = b.gather(1, b.abs().argmax(1, keepdim=True))     # Q8_K: the largest |x| of a block takes code -127
    inv = -127.0 / top
    q = torch.round(inv * b).clamp(max=127)
    a = (q.double() / inv.double()).reshape(-1)
    return (w * scales.double().repeat_interleave(128, 1)) @ a


def exact(case, seed):
    kind, num = case["kind"], case.get("numerics")
    if kind == "linear":
        x, rows = _linear_inputs(case, seed)
        y = _mm(num, rows, x.double())
        return y[0] if case["T"] == 1 else y
    if kind == "mlp":
        s = _mlp_inputs(case, seed)
        x = s["x"].double()
        if case["T"] == 1:
            x = _r16(x + _rms(s["h"].double(), s["w0"]))
        gu = _mm(num, s["rows_gu"], _rms(x, s["w1"]))
        y = _mm(num, s["rows_down"], _silu_mul(_r16(gu)))
        return (x, y[0]) if case["T"] == 1 else y
    if kind == "attn":
        s = _attn_inputs(case, seed)
        nh, nkv, rot, _ = _attn_shape(case)
        x = s["x"].double()
        if case["T"] == 1:
            x = _r16(x + _rms(s["h"].double(), s["w0"]))
        rows = _r16(_mm(num, s["rows_in"], _rms(x, s["w1"])))
        a = _attention(num, rows, s["qn"], s["kn"], s["cs"], s["kc"], s["vc"], case["pos0"], nh, nkv, case["hd"], rot,
                       case["win"])
        y = _mm(num, s["rows_out"], a)
        kv = s["kc"].double(), s["vc"].double()
        return (x, *kv, y[0]) if case["T"] == 1 else (*kv, y)
    if kind == "ternary":
        s = _ternary_inputs(case, seed)
        return _ternary_mm(s["gate"], s["x"]), _ternary_mm(s["up"], s["x"]), _ternary_mm(s["down"], s["z"])
    if case["steps"]:
        return None      # the logits follow the ids, which a near tie may turn
    return None, _backbone(case, seed), None
