"""What a user of this framework has it do, as cases that can be timed and checked.

    q4k_*       the Q4_K decoder (decoder.HipDecoder): the next token of a conversation, and a prompt in front of it
    zepavik_*   the dense bf16 decoder with parallel layers, in bf16 and in true 32-bit
    gusolorn_*  the dense decoder with sequential layers: latent attention, matrix memory, routed experts
    matmul, ffn, attention   the ops a host strings together itself (doppler_amd.ops)

Sizes are the benchmark configurations of doppler_amd.synth and doppler_amd.design_bench (fewer layers where a pass shows the same
with them) and generic ones between.  Weights are random, scaled like trained ones (zero mean, products of unit size), drawn
from a pool per seed so that a large model is made quickly; weights and caches are the size of the real thing.
"""
import math

import numpy as np
import torch

F64 = torch.float64

# ------------------------------------------------------------------ the cases

WIDTHS = {      # heads, kv heads, head size, feed-forward: the three widths of design_bench
    1024: (16, 8, 64, 3072),
    2048: (16, 8, 128, 6144),
    4096: (32, 8, 128, 12288),
}
LATENT = {1024: (64, 32, 64, 256), 2048: (128, 64, 128, 512), 4096: (128, 64, 128, 512)}      # dim, rotated, value, rank
MEMORY = {1024: (4, 128, 256), 2048: (4, 256, 512), 4096: (8, 256, 512)}                     # heads, dim, value
EXPERTS, TOP, WINDOW = 16, 4, 1024


def listed():
    return [
        # the smallest call there is: one row through a small projection, where launch and latency are everything
        dict(name="matmul_1x2048x640", kind="matmul", M=1, N=2048, K=640, act="f32"),
        # a handful of rows (a few sequences, or drafted tokens to verify) through a large projection
        dict(name="matmul_8x4096x12288", kind="matmul", M=8, N=4096, K=12288, act="f32"),
        # a prompt's feed-forward block at a narrow model's width
        dict(name="ffn_512x1152x6912", kind="ffn", M=512, hidden=1152, inter=6912, activation="gelu"),
        # one token against a long conversation
        dict(name="attention_32768", kind="attention", heads=16, kv_heads=8, dim=128, keys=32768),
        # the headline: next token of a 9B-class model behind 2048 others
        dict(name="q4k_step_9b", kind="q4k_step", width=4096, layers=36, vocab=151936, ctx=2048),
        # the same for a small model and a short conversation, where launches count
        dict(name="q4k_step_small", kind="q4k_step", width=1024, layers=28, vocab=151936, ctx=517),
        # a long prompt through a large model (eight of its layers)
        dict(name="q4k_prefill_2048", kind="q4k_prefill", width=4096, layers=8, vocab=32000, tokens=2048),
        # dense weights: next token
        dict(name="zepavik_step_2048", kind="zepavik_step", width=2048, layers=6, tokens=1100, compute="bf16"),
        # dense weights: a long prompt at the largest width
        dict(name="zepavik_prefill_4096", kind="zepavik_prefill", width=4096, layers=3, tokens=2048, compute="bf16"),
        # the 32-bit compute type, for those who check a model against another implementation: a ragged prompt
        dict(name="zepavik_prefill_f32", kind="zepavik_prefill", width=1024, layers=6, tokens=301, compute="f32"),
        # sequential layers: a ragged prompt whose logits are wanted at a few places (scoring)
        dict(name="gusolorn_prefill_2048", kind="gusolorn_prefill", width=2048, layers=6, tokens=1531),
        # sequential layers: a short prompt, then token after token
        dict(name="gusolorn_steps_1024", kind="gusolorn_steps", width=1024, layers=6, tokens=40, steps=8),
    ]


def _log(rng, low, high):
    return int(round(math.exp(rng.uniform(math.log(low), math.log(high)))))


def draw(rng):
    kind = rng.choice(["matmul", "ffn", "attention", "q4k_step", "q4k_prefill", "zepavik_step", "zepavik_prefill", "gusolorn_prefill",
                       "gusolorn_steps"])
    if kind == "matmul":
        return dict(kind=kind, M=rng.randint(1, 15), N=_log(rng, 200, 12288), K=4 * _log(rng, 64, 3072), act=rng.choice(["f32", "f32", "f16"]))
    if kind == "ffn":
        return dict(kind=kind, M=_log(rng, 16, 2048), hidden=64 * rng.randint(8, 64), inter=64 * rng.randint(16, 192),
                    activation=rng.choice(["silu", "gelu"]))
    if kind == "attention":
        kv = rng.choice([1, 2, 4, 8])
        return dict(kind=kind, heads=kv * rng.choice([1, 2, 4, 7]), kv_heads=kv, dim=rng.choice([64, 128]), keys=_log(rng, 1, 32768))
    width = rng.choice(sorted(WIDTHS))
    if kind == "q4k_step":
        return dict(kind=kind, width=width, layers=rng.randint(2, 24), vocab=rng.choice([32000, 50257, 151936]), ctx=_log(rng, 16, 3500))
    if kind == "q4k_prefill":
        return dict(kind=kind, width=width, layers=rng.randint(2, 6), vocab=32000, tokens=_log(rng, 2, 2048))
    if kind == "zepavik_step":
        return dict(kind=kind, width=width, layers=rng.randint(2, 4), tokens=_log(rng, 16, 2048), compute=rng.choice(["bf16", "bf16", "f32"]))
    if kind == "zepavik_prefill":
        compute = rng.choice(["bf16", "bf16", "bf16", "f32"])
        return dict(kind=kind, width=width, layers=rng.randint(1, 3), tokens=_log(rng, 2, 2048 if compute == "bf16" else 600), compute=compute)
    if kind == "gusolorn_prefill":
        return dict(kind=kind, width=width, layers=3 if width == 4096 else rng.randint(3, 6), tokens=_log(rng, 2, 2048))
    return dict(kind=kind, width=width, layers=3 if width == 4096 else rng.randint(3, 6), tokens=_log(rng, 2, 600), steps=rng.randint(1, 12))


# ------------------------------------------------------------------ inputs

class _Pool:
    """Random numbers of a seed, dealt out in stretches that begin anywhere."""
    SIZE = (1 << 22) + 7

    def __init__(self, seed):
        self.g = np.random.Generator(np.random.PCG64(seed))
        self.normals = self.g.standard_normal(self.SIZE, dtype=np.float32)
        self.kept = {}

    def _stretch(self, a, n):
        at = int(self.g.integers(0, len(a)))
        return a[at:at + n] if at + n <= len(a) else np.resize(np.concatenate([a[at:], a[:at]]), (n,) + a.shape[1:])

    def _scaled(self, std, to, kind):
        key = (kind, round(float(std), 9))
        if key not in self.kept:
            self.kept[key] = to(self.normals * np.float32(std))
        return self.kept[key]

    def f32(self, shape, std=1.0, mean=0.0):
        return self._stretch(self.normals, int(np.prod(shape))).reshape(shape) * np.float32(std) + np.float32(mean)

    def f16(self, shape, std=1.0):
        """f16 bits."""
        return self._stretch(self._scaled(std, lambda a: a.astype(np.float16).view(np.uint16), "f16"), int(np.prod(shape))).reshape(shape)

    def bf16(self, shape, std=None):
        """bf16 bits; a matrix [out, in] by default so that its products are of unit size."""
        std = shape[-1] ** -0.5 if std is None else std
        return self._stretch(self._scaled(std, _bf16_bits, "bf16"), int(np.prod(shape))).reshape(shape)

    def rounded(self, shape, std, mean=0.0):
        """f32 values that bf16 holds."""
        return _from_bf16(_bf16_bits(self.f32(shape, std, mean)))

    def q4k(self, N, K):
        """Q4_K bytes of a matrix [N, K] with weights of zero mean and spread K^-1/2: mins equal scales and dmin = 7.5 d."""
        if "q4k" not in self.kept:
            n = 32771
            b = self.g.integers(0, 256, (n, 144), dtype=np.uint8)
            b[:, 8:12] = b[:, 4:8]
            b[:, 12:16] = (b[:, 12:16] & 0x0F) * 0x11
            self.kept["q4k"] = b, np.abs(self.normals[:n]) + np.float32(0.1)
        if ("q4k", K) not in self.kept:
            b, d = self.kept["q4k"]
            b = b.copy()
            d = (d * np.float32(K ** -0.5 / 188.0)).astype(np.float16)        # 188: spread of scale * (quant - 7.5) at these d
            b[:, 0:2] = d.view(np.uint8).reshape(-1, 2)
            b[:, 2:4] = (d.astype(np.float32) * np.float32(7.5)).astype(np.float16).view(np.uint8).reshape(-1, 2)
            self.kept["q4k", K] = b
        return np.ascontiguousarray(self._stretch(self.kept["q4k", K], N * (-(-K // 256)))).reshape(-1)

    def tokens(self, n, vocab):
        return self.g.integers(0, vocab, n).astype(np.uint32)


def _bf16_bits(x):
    return torch.from_numpy(np.ascontiguousarray(x, np.float32)).to(torch.bfloat16).view(torch.int16).numpy().view(np.uint16)


def _from_bf16(bits):
    return (bits.astype(np.uint32) << 16).view(np.float32)


def _rope(dim, positions, theta=1e6):
    a = np.arange(positions)[:, None] * theta ** (-2.0 * np.arange(dim // 2) / dim)
    return np.cos(a).astype(np.float32), np.sin(a).astype(np.float32)


def _q4k_model(case, seed, max_seq):
    p, W = _Pool(seed), case["width"]
    H, G, D, I = WIDTHS[W]
    cfg = dict(layers=case["layers"], hidden=W, inter=I, heads=H, kv_heads=G, head_dim=D, vocab=case["vocab"], eps=1e-6, qk_norm=1,
               max_seq=max_seq)
    # four different layers in turn: the decoder uploads each of them on its own
    made = [dict(wq=p.q4k(H * D, W), wk=p.q4k(G * D, W), wv=p.q4k(G * D, W), wo=p.q4k(W, H * D), wgate=p.q4k(I, W), wup=p.q4k(I, W),
                 wdown=p.q4k(W, I), input_norm=p.f32(W, 0.05, 1.0), post_attn_norm=p.f32(W, 0.05, 1.0), q_norm=p.f32(D, 0.05, 1.0),
                 k_norm=p.f32(D, 0.05, 1.0)) for _ in range(min(4, case["layers"]))]
    layers = [made[i % len(made)] for i in range(case["layers"])]
    cos, sin = _rope(D, max_seq)
    return cfg, layers, p.f16((case["vocab"], W), 0.5), p.f32(W, 0.05, 1.0), cos, sin, p


def _zepavik_model(case, seed, max_seq):
    p, W, V = _Pool(seed), case["width"], 32000
    H, G, D, ff = WIDTHS[W]
    mixer = dict(heads=H, kv_heads=G, dim=D, vdim=D, window=WINDOW, scale=D ** -0.5, log_bias=True, value_norm=True, gate=True)
    cfg = dict(hidden=W, vocab=V, eps=1e-5, logit_scale=1.0, max_positions=max_seq, bigram=dict(buckets=4096, mul_prev=31, mul_cur=7),
               layers=[dict(mixer=dict(mixer), mlp=dict(ff=ff, activation="relu2")) for _ in range(case["layers"])])
    layers = []
    for _ in range(case["layers"]):
        w = dict(norm=p.rounded(W, 0.05, 1.0), q=p.bf16((H * D, W)), k=p.bf16((G * D, W)), v=p.bf16((G * D, W)), q_bias=p.rounded(H * D, 0.2),
                 k_bias=p.rounded(G * D, 0.2), v_bias=p.rounded(G * D, 0.2), o=p.bf16((W, H * D)), gate=p.bf16((H, W)), up=p.bf16((ff, W)),
                 down=p.bf16((W, ff)))
        w["bias_r1"] = _from_bf16(_bf16_bits(p.g.uniform(0.02, 1.2, H)))
        w["bias_r2"] = _from_bf16(_bf16_bits(p.g.uniform(0.05, 0.6, H)))
        layers.append(w)
    weights = dict(embed=p.bf16((V, W), 1.0), bigram=p.bf16((4097, W), 1.0), pos=p.bf16((max_seq, W), 0.5), head=p.bf16((V, W)),
                   final_norm=p.rounded(W, 0.05, 1.0), layers=layers)
    return cfg, weights, p


def _gusolorn_model(case, seed):
    """Latent attention with a dense feed-forward, two of matrix memory with experts, and again on borrowed latent rows.  What experts are
    chosen by are columns of the embedding that no layer writes, apart by more than rounding, as a trained router's choices mostly are."""
    p, W, V = _Pool(seed), case["width"], 32000
    heads, ff = WIDTHS[W][0], WIDTHS[W][3]
    d, rot, e, rank = LATENT[W]
    H, md, me = MEMORY[W]
    eff, sff, E = ff // 2 // TOP, ff // 2, EXPERTS

    def out(shape):
        a = np.array(p.bf16(shape))
        a[..., :E, :] = 0
        return a
    layers, made = [], []
    for i in range(case["layers"]):
        lent = i - 3 if i % 6 == 3 else None
        w = dict(norm1=p.rounded(W, 0.05, 1.0), ls1=p.rounded(W, 0.1, 1.0), norm2=p.rounded(W, 0.05, 1.0), ls2=p.rounded(W, 0.1, 1.0))
        if i % 3 == 0:
            layers.append(dict(sequential=True, mixer=dict(type="latent_attention", heads=heads, dim=d, rot_dim=rot, vdim=e, kv_rank=rank,
                                                           window=WINDOW, scale=(d + rot) ** -0.5, rot_base=10000.0, kv_from=lent),
                               mlp=dict(type="dense", ff=ff, activation="gelu_erf")))
            w["mixer"] = dict(q=p.bf16((heads * (d + rot), W)), uk=p.bf16((heads * d, rank)), uv=p.bf16((heads * e, rank)), o=out((W, heads * e)))
            if lent is None:
                w["mixer"].update(dkv=p.bf16((rank + rot, W)), latent_norm=p.rounded(rank, 0.05, 1.0))
            w["mlp"] = dict(up=p.bf16((ff, W)), down=out((W, ff)))
        else:
            layers.append(dict(sequential=True, mixer=dict(type="mlstm", heads=H, dim=md, vdim=me, gate_cap=15.0),
                               mlp=dict(type="experts", experts=E, top=TOP, ff=eff, limit=7.0, shared=dict(ff=sff, limit=7.0))))
            w["mixer"] = dict(q=p.bf16((H * md, W)), k=p.bf16((H * md, W)), v=p.bf16((H * me, W)), g=p.bf16((H * me, W)), i=p.bf16((H, W)),
                              f=p.bf16((H, W)), o=out((W, H * me)), i_bias=p.rounded(H, 0.5, -2.0), f_bias=p.rounded(H, 0.5, 4.0),
                              head_norm=p.rounded(H * me, 0.05, 1.0))
            router = np.zeros((E, W), np.float32)
            router[np.arange(E), np.arange(E)] = 0.703125
            w["norm2"][:E] = 1.0
            w["mlp"] = dict(router=_bf16_bits(router), gate=p.bf16((E, eff, W)), up=p.bf16((E, eff, W)), down=out((E, W, eff)),
                            shared_gate=p.bf16((sff, W)), shared_up=p.bf16((sff, W)), shared_down=out((W, sff)), shared_sg=p.bf16((1, W)))
        made.append(w)
    embed = np.array(p.bf16((V, W), 1.0))
    embed[:, :E] = _bf16_bits(0.75 * (np.argsort(p.g.random((V, E), dtype=np.float32), axis=1) - (E - 1) / 2.0))
    cfg = dict(hidden=W, vocab=V, eps=1e-6, logit_scale=1.0, max_positions=0, bigram=None, layers=layers)
    return cfg, dict(embed=embed, head=p.bf16((V, W)), final_norm=p.rounded(W, 0.05, 1.0), layers=made), p


def _op_inputs(case, seed):
    """Host arrays of an op's inputs."""
    p = _Pool(seed)
    if case["kind"] == "matmul":
        M, N, K = case["M"], case["N"], case["K"]
        return dict(x=p.f32((M, K)) if case["act"] == "f32" else p.f16((M, K)), w=p.q4k(N, K))
    if case["kind"] == "ffn":
        M, W, I = case["M"], case["hidden"], case["inter"]
        return dict(x=p.f32((M, W)), norm=p.f32(W, 0.05, 1.0), gate=p.q4k(I, W), up=p.q4k(I, W), down=p.q4k(W, I))
    H, G, D, n = case["heads"], case["kv_heads"], case["dim"], case["keys"]
    return dict(q=p.f32((H, D)), k=p.f16((n, G, D)), v=p.f16((n, G, D)))


# ------------------------------------------------------------------ the framework's side

def _places(n):
    """Some places of a prompt whose logits are wanted."""
    return sorted({0, n // 3, n - 1})


def prepare(case, seed):
    from doppler_amd import decoder, dense_decoder, ops
    kind, s = case["kind"], dict(case=case)
    if kind in ("matmul", "ffn", "attention"):
        a = _op_inputs(case, seed)
        t = {k: ops.tensorFromNumpy(v) for k, v in a.items() if v.dtype != np.uint8}
        for k, v in a.items():
            if v.dtype == np.uint8:
                N, K = dict(w=("N", "K"), gate=("inter", "hidden"), up=("inter", "hidden"), down=("hidden", "inter"))[k]
                t[k] = ops.createWeightBuffer(ops.uploadData(ops.acquireBuffer(v.size), v), "q4k", "row", (case[N], case[K]))
        if kind == "matmul":
            s["out"] = ops.acquireBuffer(4 * case["M"] * case["N"])
        elif kind == "ffn":
            s["act"], s["out"] = ops.acquireBuffer(4 * case["M"] * case["inter"]), ops.acquireBuffer(4 * case["M"] * case["hidden"])
        else:
            s["out"] = ops.acquireBuffer(4 * ops.padToQ4KBlock(case["heads"] * case["dim"]))
            s["ws"] = ops.acquireBuffer(ops.attentionWorkspaceBytes(case["heads"], case["dim"], case["keys"]))
        s.update(t=t, ops=ops)
        return s
    if kind.startswith("q4k"):
        n = case["tokens"] if kind == "q4k_prefill" else case["ctx"]
        cfg, layers, embed, norm, cos, sin, p = _q4k_model(case, seed, n + (kind == "q4k_step"))
        s["dec"] = dec = decoder.HipDecoder(cfg, layers, embed, norm, cos, sin, cfg["max_seq"])
        s["tokens"] = p.tokens(n + 1, case["vocab"])
        row = cfg["kv_heads"] * cfg["head_dim"]
    elif kind.startswith("zepavik"):
        n = case["tokens"]
        cfg, weights, p = _zepavik_model(case, seed, n + (kind == "zepavik_step"))
        s["dec"] = dec = dense_decoder.DenseDecoder(cfg, weights, n + (kind == "zepavik_step"), compute=case["compute"])
        s["tokens"] = p.tokens(n + 1, cfg["vocab"])
        row = WIDTHS[case["width"]][1] * WIDTHS[case["width"]][2]
    else:
        n = case["tokens"] + case.get("steps", 0)
        cfg, weights, p = _gusolorn_model(case, seed)
        s["dec"] = dense_decoder.DenseDecoder(cfg, weights, n)
        s["tokens"] = [int(t) for t in p.tokens(n, cfg["vocab"])]
        return s
    if kind.endswith("step"):
        dec.prefill(s["tokens"][:n])
        s["updated"] = [d[c][n * row:] for d in dec.layers[:31] for c in ("cache_k", "cache_v")]     # the rows the step appends
    else:
        s["updated"] = [d[c] for d in dec.layers for c in ("cache_k", "cache_v")]
    return s


def run(s):
    case, kind = s["case"], s["case"]["kind"]
    if kind == "matmul":
        ops, t = s["ops"], s["t"]
        ops.runMatmul(t["x"], t["w"], case["M"], case["N"], case["K"], outputDtype="f32", outputBuffer=s["out"])
        return s["out"].view(torch.float32)
    if kind == "ffn":
        ops, t, M, W, I = s["ops"], s["t"], case["M"], case["hidden"], case["inter"]
        act = ops.runFusedNormedFFN(t["x"], t["norm"], 1e-6, t["gate"], t["up"], W, I, batchSize=M, activation=case["activation"],
                                    outputBuffer=s["act"])
        ops.runMatmul(act, t["down"], M, W, I, outputDtype="f32", outputBuffer=s["out"], residualTensor=t["x"])
        return s["out"].view(torch.float32)
    if kind == "attention":
        ops, t = s["ops"], s["t"]
        ops.runAttention(t["q"], t["k"], t["v"], None, case["heads"], case["dim"], seqLen=1, kvLen=case["keys"], numKVHeads=case["kv_heads"],
                         startPos=case["keys"] - 1, outputBuffer=s["out"], workspace=s["ws"])
        return s["out"].view(torch.float32)
    dec = s["dec"]
    if kind.endswith("step"):
        dec.step(int(s["tokens"][-1]), len(s["tokens"]) - 1, want_logits=True)
        return dict(logits=dec.logits, updated=s["updated"])
    if kind in ("q4k_prefill", "zepavik_prefill"):
        dec.prefill(s["tokens"][:-1], want_logits=True)
        return dict(logits=dec.logits, updated=s["updated"])
    dec.reset()
    if kind == "gusolorn_prefill":
        return dec.feed(s["tokens"], want=_places(len(s["tokens"])))
    n = case["tokens"]
    rows = [dec.feed(s["tokens"][:n], want=[n - 1])]
    for t in s["tokens"][n:]:
        rows.append(dec.feed([t], want=[0]))
    return rows


# ------------------------------------------------------------------ what a pass cannot do without

def _q4k_bytes(N, K):
    return 144.0 * N * -(-K // 256)


def _seen(n, window):
    """Pairs of query and key of a causal prompt."""
    return float(sum(min(t + 1, window) for t in range(n))) if window else n * (n + 1) / 2.0


def work(case):
    kind = case["kind"]
    if kind == "matmul":
        M, N, K = case["M"], case["N"], case["K"]
        return dict(bytes=_q4k_bytes(N, K) + M * K * (4 if case["act"] == "f32" else 2) + 4.0 * M * N, flops=2.0 * M * N * K)
    if kind == "ffn":
        M, W, I = case["M"], case["hidden"], case["inter"]
        return dict(bytes=2 * _q4k_bytes(I, W) + _q4k_bytes(W, I) + 8.0 * M * W, flops=6.0 * M * W * I)
    if kind == "attention":
        H, G, D, n = case["heads"], case["kv_heads"], case["dim"], case["keys"]
        return dict(bytes=4.0 * n * G * D + 8.0 * H * D, flops=4.0 * n * H * D)
    W, L = case["width"], case["layers"]
    H, G, D, ff = WIDTHS[W]
    if kind.startswith("q4k"):
        weights = float(W * (H + 2 * G) * D + W * H * D + 3 * W * ff)
        held = _q4k_bytes((H + 2 * G) * D, W) + _q4k_bytes(W, H * D) + 2 * _q4k_bytes(ff, W) + _q4k_bytes(W, ff)
        n, pairs = (1, case["ctx"] + 1.0) if kind == "q4k_step" else (case["tokens"], _seen(case["tokens"], 0))
        head = 1.0 * case["vocab"] * W
        rows = case["ctx"] if kind == "q4k_step" else 0
        return dict(bytes=L * (held + 4.0 * G * D * (rows + n)) + 2 * head + 2.0 * n * W + 4 * case["vocab"],
                    flops=2.0 * n * L * weights + 4.0 * L * H * D * pairs + 2 * head)
    V = 32000
    if kind.startswith("zepavik"):
        weights = float(W * (H + 2 * G) * D + W * H + W * H * D + 2 * W * ff)
        n = case["tokens"]
        elem = 2 if case["compute"] == "bf16" else 4
        if kind == "zepavik_step":
            keys = min(n + 1, WINDOW)
            return dict(bytes=L * (2 * weights + 2.0 * elem * G * D * keys) + 2.0 * V * W + 4 * V,
                        flops=L * (2 * weights + 4.0 * H * D * keys) + 2.0 * V * W)
        return dict(bytes=L * (2 * weights + 2.0 * elem * G * D * n) + 2.0 * V * W + 6.0 * n * W,
                    flops=L * (2.0 * n * weights + 4.0 * H * D * _seen(n, WINDOW)) + 2.0 * V * W)
    d, rot, e, rank = LATENT[W]
    mh, md, me = MEMORY[W]
    n, steps = case["tokens"], case.get("steps", 0)
    nbytes, flops = 0.0, 0.0
    for i in range(L):
        if i % 3 == 0:
            weights = float(W * (H * (d + rot) + (0 if i % 6 == 3 else rank + rot)) + H * rank * (d + e) + W * H * e + 2 * W * ff)
            stored = weights
            flops += 2.0 * H * (d + rot + e) * (_seen(n + steps, WINDOW))
        else:
            weights = float(W * mh * (2 * md + 3 * me + 2) + W * EXPERTS + 3 * W * ff)       # half of ff in the chosen experts, half in the shared one
            stored = weights + 3.0 * W * ff / 2 * (min(EXPERTS, TOP * n) / TOP - 1)
            flops += 4.0 * (n + steps) * mh * md * me
            nbytes += 8.0 * (steps + 1) * mh * md * me
        flops += 2.0 * (n + steps) * weights
        nbytes += 2 * stored + 2 * steps * weights
    places = steps + (len(_places(n)) if kind == "gusolorn_prefill" else 1)
    return dict(bytes=nbytes + 2.0 * V * W * (steps + 1) + 4.0 * places * V, flops=flops + 2.0 * V * W * places)


# ------------------------------------------------------------------ the same in 64 bits

def _dev(a):
    return torch.from_numpy(np.ascontiguousarray(a)).cuda()


def _q4k_f64(b, N, K):
    """[N, K] of Q4_K bytes."""
    b = _dev(np.ascontiguousarray(b).reshape(-1, 144))
    halves = b[:, 0:4].contiguous().view(torch.float16).to(F64)
    lo, hi, mix = b[:, 4:8].int(), b[:, 8:12].int(), b[:, 12:16].int()
    sc = torch.cat([lo & 63, (mix & 15) | (lo >> 6 << 4)], 1).to(F64) * halves[:, 0:1]
    mn = torch.cat([hi & 63, (mix >> 4) | (hi >> 6 << 4)], 1).to(F64) * halves[:, 1:2]
    q = b[:, 16:].reshape(-1, 4, 1, 32)
    q = torch.cat([q & 15, q >> 4], 2).reshape(-1, 8, 32).to(F64)
    return (q * sc[:, :, None] - mn[:, :, None]).reshape(N, -1)[:, :K]


def _bits(a, kind):
    return _dev(np.ascontiguousarray(a).view(np.int16)).view(torch.float16 if kind == "f16" else torch.bfloat16).to(F64)


def _norm(x, eps, w=None):
    y = x / torch.sqrt(x.square().mean(-1, keepdim=True) + eps)
    return y if w is None else y * w


def _head(h, table, kind, step=8192):
    """h @ table^T, a stretch of the table at a time."""
    return torch.cat([h @ _bits(table[i:i + step], kind).T for i in range(0, len(table), step)], -1)


def _softmax_attention(q, k, v, scale, window=0, r1=None, r2=None):
    """q [n, H, d], k [n, G, d], v [n, G, e] of one causal sequence -> [n, H, e]."""
    n, H, per = q.shape[0], q.shape[1], q.shape[1] // k.shape[1]
    dist = torch.arange(n, device=q.device)[:, None] - torch.arange(n, device=q.device)[None, :]
    hidden = (dist < 0) | (dist >= (window or n))
    out = []
    for h in range(H):
        s = scale * (q[:, h] @ k[:, h // per].T)
        if r1 is not None:
            s = s - r1[h] * torch.log1p(r2[h] * dist.clamp(min=0))
        out.append(torch.softmax(s.masked_fill(hidden, -math.inf), 1) @ v[:, h // per])
    return torch.stack(out, 1)


def _silu(z):
    return z * torch.sigmoid(z)


def _gelu_tanh(z):
    return 0.5 * z * (1 + torch.tanh(math.sqrt(2 / math.pi) * (z + 0.044715 * z ** 3)))


def _exact_q4k(case, seed):
    step = case["kind"] == "q4k_step"
    n = case["ctx"] + 1 if step else case["tokens"]
    cfg, layers, embed, final, cos, sin, p = _q4k_model(case, seed, n)
    tokens = p.tokens(n if step else n + 1, case["vocab"])[:n].astype(np.int64)
    W, I, H, G, D = cfg["hidden"], cfg["inter"], cfg["heads"], cfg["kv_heads"], cfg["head_dim"]
    cos, sin = _dev(cos[:n]).to(F64)[:, None], _dev(sin[:n]).to(F64)[:, None]

    def rot(x):
        a, b = x[..., :D // 2], x[..., D // 2:]
        return torch.cat([a * cos - b * sin, b * cos + a * sin], -1)
    x, updated = _bits(embed[tokens], "f16"), []
    for l in layers:
        f = lambda name: _dev(l[name]).to(F64)                                                  # noqa: B023, E731
        h = _norm(x, cfg["eps"], f("input_norm"))
        q = rot(_norm((h @ _q4k_f64(l["wq"], H * D, W).T).reshape(n, H, D), cfg["eps"], f("q_norm")))
        k = rot(_norm((h @ _q4k_f64(l["wk"], G * D, W).T).reshape(n, G, D), cfg["eps"], f("k_norm")))
        v = (h @ _q4k_f64(l["wv"], G * D, W).T).reshape(n, G, D)
        x = x + _softmax_attention(q, k, v, D ** -0.5).reshape(n, H * D) @ _q4k_f64(l["wo"], W, H * D).T
        h = _norm(x, cfg["eps"], f("post_attn_norm"))
        h = _silu(h @ _q4k_f64(l["wgate"], I, W).T) * (h @ _q4k_f64(l["wup"], I, W).T)
        x = x + h @ _q4k_f64(l["wdown"], W, I).T
        if len(updated) < 62 or not step:
            updated += [t[-1].reshape(-1) if step else t.reshape(-1) for t in (k, v)]
    return dict(logits=_head(_norm(x[-1], cfg["eps"], _dev(final).to(F64)), embed, "f16"), updated=updated)


def _exact_zepavik(case, seed):
    step = case["kind"] == "zepavik_step"
    n = case["tokens"] + step
    cfg, w, p = _zepavik_model(case, seed, n)
    tokens = p.tokens(n if step else n + 1, cfg["vocab"])[:n].astype(np.int64)
    b = cfg["bigram"]
    rows = np.concatenate([[b["buckets"]], (tokens[:-1] * b["mul_prev"] + tokens[1:] * b["mul_cur"]) % b["buckets"]])
    bf = lambda a: _bits(a, "bf16")                                                             # noqa: E731
    x, updated = bf(w["embed"][tokens]) + bf(w["bigram"][rows]) + bf(w["pos"][:n]), []
    for spec, l in zip(cfg["layers"], w["layers"]):
        m = spec["mixer"]
        H, G, D = m["heads"], m["kv_heads"], m["dim"]
        f = lambda name: _dev(l[name]).to(F64)                                                  # noqa: B023, E731
        h = _norm(x, cfg["eps"], f("norm"))
        q, k, v = ((h @ bf(l[t]).T + f(t + "_bias")).reshape(n, -1, D) for t in "qkv")
        v = _norm(v, cfg["eps"])
        o = _softmax_attention(q, k, v, m["scale"], m["window"], f("bias_r1"), f("bias_r2")) * torch.sigmoid(h @ bf(l["gate"]).T)[:, :, None]
        x = x + o.reshape(n, H * D) @ bf(l["o"]).T + (h @ bf(l["up"]).T).clamp(min=0).square() @ bf(l["down"]).T
        updated += [t[-1].reshape(-1) if step else t.reshape(-1) for t in (k, v)]
    return dict(logits=_head(_norm(x[-1], cfg["eps"], _dev(w["final_norm"]).to(F64)), w["head"], "bf16"), updated=updated)


def _memory(q, k, v, log_i, log_f):
    """Outputs [n, e] of one head: m_t = max(f_t + m_(t-1), i_t) from 0, S_t = e^(f_t + m_(t-1) - m_t) S_(t-1) + e^(i_t - m_t) k_t v_t^T."""
    n = len(q)
    F = torch.cumsum(log_f, 0)
    d = F[:, None] - F[None, :] + log_i[None, :]
    d = d.masked_fill(torch.ones(n, n, dtype=torch.bool, device=q.device).triu(1), -math.inf)
    m = torch.maximum(d.amax(1), F)
    a = torch.exp(d - m[:, None]) * (q @ k.T)
    return (a @ v) / (torch.maximum(a.sum(1).abs(), torch.exp(-m)) + 1e-6)[:, None]


def _clamped_glu(g, u, limit):
    g, u = g.clamp(max=limit), u.clamp(-limit, limit)
    return g * torch.sigmoid(1.702 * g) * (u + 1)


def _exact_gusolorn(case, seed):
    cfg, w, p = _gusolorn_model(case, seed)
    n = case["tokens"] + case.get("steps", 0)
    tokens = p.tokens(n, cfg["vocab"]).astype(np.int64)
    eps, bf, f64 = cfg["eps"], lambda a: _bits(a, "bf16"), lambda a: _dev(a).to(F64)

    def rot(x, base):
        dims = x.shape[-1]
        a = torch.arange(n, device="cuda", dtype=F64)[:, None] * base ** (-2.0 * torch.arange(dims // 2, device="cuda", dtype=F64) / dims)
        a = a.reshape((n,) + (1,) * (x.dim() - 2) + (dims // 2,))
        u, v = x[..., 0::2], x[..., 1::2]
        return torch.stack([u * torch.cos(a) - v * torch.sin(a), v * torch.cos(a) + u * torch.sin(a)], -1).reshape(x.shape)
    x, lent = bf(w["embed"][tokens]), {}
    for i, (spec, l) in enumerate(zip(cfg["layers"], w["layers"])):
        m, mlp, t = spec["mixer"], spec["mlp"], l["mixer"]
        H, d, e = m["heads"], m["dim"], m["vdim"]
        h = _norm(x, eps, f64(l["norm1"]))
        if m["type"] == "latent_attention":
            r = m["kv_rank"]
            if m["kv_from"] is None:
                y = h @ bf(t["dkv"]).T
                lent[i] = _norm(y[:, :r], eps, f64(t["latent_norm"])), rot(y[:, r:], m["rot_base"])
            c, k_rot = lent[i if m["kv_from"] is None else m["kv_from"]]
            q = (h @ bf(t["q"]).T).reshape(n, H, -1)
            q = torch.cat([q[:, :, :d], rot(q[:, :, d:], m["rot_base"])], 2)
            k = torch.cat([(c @ bf(t["uk"]).T).reshape(n, H, d), k_rot[:, None].expand(n, H, m["rot_dim"])], 2)
            y = _softmax_attention(q, k, (c @ bf(t["uv"]).T).reshape(n, H, e), m["scale"], m["window"]).reshape(n, H * e) @ bf(t["o"]).T
        else:
            q, k, v = (h @ bf(t["q"]).T).reshape(n, H, d) * d ** -0.5, (h @ bf(t["k"]).T).reshape(n, H, d), (h @ bf(t["v"]).T).reshape(n, H, e)
            cap = lambda z: m["gate_cap"] * torch.tanh(z / m["gate_cap"])                       # noqa: B023, E731
            log_i = cap(h @ bf(t["i"]).T + f64(t["i_bias"]))
            log_f = torch.nn.functional.logsigmoid(cap(h @ bf(t["f"]).T + f64(t["f_bias"])))
            o = torch.stack([_memory(q[:, a], k[:, a], v[:, a], log_i[:, a], log_f[:, a]) for a in range(H)], 1)
            y = (_norm(o, eps).reshape(n, H * e) * f64(t["head_norm"]) * torch.sigmoid(h @ bf(t["g"]).T)) @ bf(t["o"]).T
        x = x + f64(l["ls1"]) * y
        h, t = _norm(x, eps, f64(l["norm2"])), l["mlp"]
        if mlp["type"] == "dense":
            z = h @ bf(t["up"]).T
            y = (0.5 * z * (1 + torch.erf(z / math.sqrt(2)))) @ bf(t["down"]).T
        else:
            scores = torch.sigmoid(h @ bf(t["router"]).T)
            best, chosen = scores.topk(mlp["top"], 1)
            weight = torch.zeros_like(scores).scatter(1, chosen, best)
            y = torch.zeros_like(x)
            for a in range(mlp["experts"]):
                at = (weight[:, a] > 0).nonzero()[:, 0]
                ha = h[at] * weight[at, a:a + 1]
                y[at] += _clamped_glu(ha @ bf(t["gate"][a]).T, ha @ bf(t["up"][a]).T, mlp["limit"]) @ bf(t["down"][a]).T
            s = _clamped_glu(h @ bf(t["shared_gate"]).T, h @ bf(t["shared_up"]).T, mlp["shared"]["limit"]) @ bf(t["shared_down"]).T
            y = y + torch.sigmoid(h @ bf(t["shared_sg"]).T) * s
        x = x + f64(l["ls2"]) * y
    places = _places(n) if case["kind"] == "gusolorn_prefill" else list(range(case["tokens"] - 1, n))
    return _head(_norm(x[places], eps, f64(w["final_norm"])), w["head"], "bf16")


def exact(case, seed):
    kind = case["kind"]
    if kind in ("matmul", "ffn", "attention"):
        a = _op_inputs(case, seed)
    if kind == "matmul":
        x = _dev(a["x"]).to(F64) if case["act"] == "f32" else _bits(a["x"], "f16")
        return (x @ _q4k_f64(a["w"], case["N"], case["K"]).T).reshape(-1)
    if kind == "ffn":
        W, I = case["hidden"], case["inter"]
        x = _dev(a["x"]).to(F64)
        h = _norm(x, 1e-6, _dev(a["norm"]).to(F64))
        act = _silu if case["activation"] == "silu" else _gelu_tanh
        h = act(h @ _q4k_f64(a["gate"], I, W).T) * (h @ _q4k_f64(a["up"], I, W).T)
        return (x + h @ _q4k_f64(a["down"], W, I).T).reshape(-1)
    if kind == "attention":
        H, G, D = case["heads"], case["kv_heads"], case["dim"]
        q, k, v = _dev(a["q"]).to(F64), _bits(a["k"], "f16"), _bits(a["v"], "f16")
        o = torch.stack([torch.softmax(D ** -0.5 * (k[:, h // (H // G)] @ q[h]), 0) @ v[:, h // (H // G)] for h in range(H)])
        out = torch.zeros(-(-H * D // 256) * 256, dtype=F64, device="cuda")      # the op pads its output row to whole blocks
        out[:H * D] = o.reshape(-1)
        return out
    if kind.startswith("q4k"):
        return _exact_q4k(case, seed)
    if kind.startswith("zepavik"):
        return _exact_zepavik(case, seed)
    rows = _exact_gusolorn(case, seed)
    return rows if kind == "gusolorn_prefill" else [r[None] for r in rows]


def tolerance(case):
    """About four times the distance from exact() that the path showed over listed and drawn cases."""
    kind = case["kind"]
    if kind in ("matmul", "attention"):
        return dict(rel=1e-5)                   # 32-bit sums: 0.6e-6 to 2e-6
    if kind == "ffn":
        return dict(rel=2e-3)                   # f16 matrix-core operands: 5e-4
    if kind.startswith("q4k"):
        return dict(rel=8e-3)                   # the same, layer after layer (a step reads the cache a prompt left): 0.9e-3 to 2.3e-3
    if case.get("compute") == "f32":
        return dict(rel=1e-5)                   # 32-bit throughout: 1.6e-6
    if kind.startswith("zepavik"):
        return dict(rel=1.2e-2)                 # bf16 operands, layer after layer: 2.8e-3
    return dict(rel=2e-2)                       # twice as many products after one another, and gates: 5.8e-3
