"""The JavaScript host path: doppler_amd/js (op API with the reference's signatures) ->
Node-API addon -> libdopplerhip.so.  pytest writes seeded inputs and the oracle's expected
outputs to a scratch directory, one node process (tests/js/run_cases.mjs) runs every case,
and the results are compared here with the same bars as the Python-host tests."""
import json
import os
import shutil
import subprocess

import numpy as np
import pytest

import oracle
from doppler_amd import decoder, synth

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
NODE = shutil.which("node")
ADDON = os.path.join(ROOT, "doppler_amd", "js", "doppler_hip.node")


def rel_l2(a, b):
    a, b = np.asarray(a, np.float64).reshape(-1), np.asarray(b, np.float64).reshape(-1)
    return float(np.linalg.norm(a - b) / max(np.linalg.norm(b), 1e-30))


def test_addon_is_built_and_exports_the_op_api():
    """CPU-side: the addon loads in node and the JS entry module exposes every op name the
    reference's pipeline imports for this path."""
    if NODE is None:
        pytest.skip("node not installed")
    assert os.path.exists(ADDON), "run python -m doppler_amd.build"
    code = ("import('%s/doppler_amd/js/kernel-selector.js').then(m => console.log(JSON.stringify(Object.keys(m))))"
            % ROOT)
    out = subprocess.run([NODE, "-e", code], stdout=subprocess.PIPE, stderr=subprocess.PIPE, text=True, timeout=60)
    assert out.returncode == 0, out.stderr
    names = set(json.loads(out.stdout))
    for n in ("runMatmul", "recordMatmul", "runAttention", "recordAttention", "runRMSNorm", "recordRMSNorm", "runRMSNormQK", "recordRMSNormQK", "canUseRMSNormQK", "runSandwichRMSNormPair", "recordSandwichRMSNormPair",
              "runResidualNextRMSNormPair", "recordResidualNextRMSNormPair", "runRoPE", "runSplitQKV", "recordSplitQKV", "runBiasAdd", "recordBiasAdd", "runScale", "recordScale", "runRoPEQK", "recordRoPEQK", "canUseRoPEQK",
              "recordRoPE", "runKVCacheWriteF32ToF16", "recordKVCacheWriteF32ToF16", "runSplitQKVRMSNormRoPEQK",
              "recordSplitQKVRMSNormRoPEQK", "runSiLU", "recordSiLU", "runSiLURowSplit", "recordSiLURowSplit", "runGeLU",
              "recordGeLU", "runResidualAdd", "recordResidualAdd", "runGather", "recordGather", "runFusedFFN",
              "recordFusedFFN", "runDecodeAttentionFromQKV", "recordDecodeAttentionFromQKV", "runArgmax", "recordArgmax", "recordLmHeadArgmax", "recordLmHeadArgmaxF16",
              "createTensor", "createWeightBuffer", "acquireBuffer", "releaseBuffer", "uploadData", "readBuffer",
              "runMatmulRMSNormFused", "recordMatmulRMSNormFused", "shouldUseFusedMatmulRMSNorm",
              "selectMatmulRMSNormFusedVariant", "recordCheckFiniteness", "resolveFinitenessAbsThreshold",
              "shouldTriggerFinitenessValue", "parseFinitenessStatusWords", "createCommandRecorder", "CommandRecorder"):
        assert n in names, n


@pytest.mark.gpu
@pytest.mark.timeout(600)
def test_js_host_path_parity(tmp_path):
    if NODE is None:
        pytest.skip("node not installed")
    d = str(tmp_path)
    cases, checks = [], []

    def put(name, arr):
        np.ascontiguousarray(arr).tofile(os.path.join(d, name))
        return name

    def get(name, dtype):
        return np.fromfile(os.path.join(d, name), dtype)

    # dequant, bit exact
    W = synth.q4k_tensor(64, 768, 9000)
    cases.append(dict(name="dequant", op="dequant", W=put("dq.W", W), blocks=W.size // 144))
    checks.append(lambda: get("dequant.out.bin", np.float32).tobytes() == oracle.q4k_dequant_blocks(W).tobytes())

    # Q4_K matmul: config 0 GEMV, a config-1 shape at M=4 through recordMatmul, residual + f16 out
    def mm(name, M, N, K, seed, **kw):
        Wm = synth.q4k_tensor(N, K, seed)
        A = synth.normal_f32((M, K), seed + 1)
        if kw.get("a16"):
            A16 = A.astype(np.float16)
            A = A16.astype(np.float32)
        c = dict(name=name, op="matmul", wdtype="q4k", W=put(name + ".W", Wm),
                 A=put(name + ".A", A16.view(np.uint16) if kw.get("a16") else A), aDtype="f16" if kw.get("a16") else "f32",
                 M=M, N=N, K=K,
                 outputDtype=kw.get("outputDtype", "f32"), alpha=kw.get("alpha", 1.0), record=kw.get("record", False))
        if kw.get("normed"):
            nw = 1.0 + synth.normal_f32((K,), seed + 3, 0.1)
            c["normWeight"] = put(name + ".nw", nw)
            c["rmsNormEps"] = 1e-6
            want = oracle.q4k_matmul(oracle.rmsnorm(A, nw, 1e-6), Wm, M, N, K, c["alpha"])
        else:
            want = oracle.q4k_matmul(A, Wm, M, N, K, c["alpha"])
        if kw.get("residual"):
            R = synth.normal_f32((M, N), seed + 2)
            c["residual"] = put(name + ".R", R)
            want = want + R
        cases.append(c)
        dt = np.float16 if c["outputDtype"] == "f16" else np.float32
        checks.append(lambda: rel_l2(get(name + ".out.bin", dt).astype(np.float32), want) <= 1e-3)

    mm("mm_cfg0", 1, 2048, 640, 9100)
    mm("mm_cfg1", 4, 3072, 1024, 9110, record=True)
    mm("mm_res", 2, 512, 1024, 9120, alpha=0.5, residual=True)
    mm("mm_f16", 1, 512, 1024, 9130, outputDtype="f16", alpha=2.0 ** -8)
    mm("mm_normed", 1, 768, 1024, 9140, normed=True, residual=True)
    mm("mm_f16a", 4, 6144, 1536, 9150, a16=True, outputDtype="f16")        # the reference's f16a parity shape
    mm("mm_f16a_gemv", 1, 512, 1024, 9160, a16=True, residual=True, record=True)

    # dense matmul + RMSNorm over the output row, both weight layouts
    for nm, (fN, fK, tb, off, res, w16) in dict(mr_t=(1152, 1536, True, True, True, False),
                                                mr_n=(1000, 300, False, False, False, True)).items():
        g = synth.rng(9170 + fN)
        fx = g.standard_normal(fK).astype(np.float32)
        fW = (g.standard_normal((fN, fK)) * fK ** -0.5).astype(np.float32)
        fw = g.standard_normal(fN).astype(np.float32).astype(np.float16 if w16 else np.float32)
        fr = g.standard_normal(fN).astype(np.float32) if res else None
        stored = fW if tb else np.ascontiguousarray(fW.T)
        c = dict(name=nm, op="matmul_rmsnorm_fused", x=put(nm + ".x", fx), W=put(nm + ".W", stored),
                 normWeight=put(nm + ".nw", fw.view(np.uint16) if w16 else fw), N=fN, K=fK, eps=1e-6, transposeB=tb,
                 weightOffset=off, record=tb)
        if res:
            c["residual"] = put(nm + ".r", fr)
        cases.append(c)
        fwant = oracle.matmul_rmsnorm_fused(fx, stored, fw.astype(np.float32), fN, fK, 1e-6, transpose_b=tb,
                                            weight_offset=off, residual=fr)
        checks.append(lambda nm=nm, fwant=fwant: rel_l2(get(nm + ".out.bin", np.float32), fwant) <= 1e-5)

    # the all-f16 variant of the same op
    g = synth.rng(9175)
    hx = g.standard_normal(520).astype(np.float16)
    hW = (g.standard_normal((1032, 520)) * 520 ** -0.5).astype(np.float16)
    hw = g.standard_normal(1032).astype(np.float32)
    hr = g.standard_normal(1032).astype(np.float16)
    cases.append(dict(name="mr_h", op="matmul_rmsnorm_fused", dtype="f16", x=put("mr_h.x", hx.view(np.uint16)),
                      W=put("mr_h.W", hW.view(np.uint16)), normWeight=put("mr_h.nw", hw), residual=put("mr_h.r", hr.view(np.uint16)),
                      N=1032, K=520, eps=1e-6, transposeB=True, weightOffset=False, record=False))
    hwant = oracle.matmul_rmsnorm_fused(hx.astype(np.float32), hW.astype(np.float32), hw, 1032, 520, 1e-6,
                                        residual=hr.astype(np.float32))
    checks.append(lambda: rel_l2(get("mr_h.out.bin", np.float16).astype(np.float32), hwant) <= 5e-4)

    # finiteness guard: clean f32, then an f16 overflow that sets the status, then a later NaN that must not overwrite it
    fin_clean = synth.normal_f32(5000, 9180, 100.0)
    fin_over = synth.normal_f32(5000, 9181).astype(np.float16)
    fin_over[4999] = 65504
    fin_nan = fin_clean.copy()
    fin_nan[17] = np.nan
    fin = [dict(input=put("fin.a", fin_clean), dtype="f32", size=5000, layer=1, step=2),
           dict(input="fin.a", dtype="f32", size=5000, layer=1, step=3, threshold=50.0),
           dict(input=put("fin.b", fin_over.view(np.uint16)), dtype="f16", size=5000, layer=4, step=5),
           dict(input=put("fin.c", fin_nan), dtype="f32", size=5000, layer=6, step=7)]
    cases.append(dict(name="finiteness", op="check_finiteness", checks=fin[:1] + fin[2:]))
    cases.append(dict(name="finiteness_threshold", op="check_finiteness", checks=fin[1:2]))
    st = np.zeros(4, np.uint32)
    fin_want = []
    for arr, l, s_ in ((fin_clean, 1, 2), (fin_over, 4, 5), (fin_nan, 6, 7)):
        oracle.check_finiteness(arr, st, l, s_)
        fin_want += st.tolist()
    assert fin_want == [0, 0, 0, 0, 1, 4, 5, 0, 1, 4, 5, 0]
    checks.append(lambda: get("finiteness.out.bin", np.uint32).tolist() == fin_want)
    fin_thr = oracle.check_finiteness(fin_clean, np.zeros(4, np.uint32), 1, 3, 50.0).tolist()
    assert fin_thr[0] == 1
    checks.append(lambda: get("finiteness_threshold.out.bin", np.uint32).tolist() == fin_thr)

    # f16 weights
    E = synth.normal_f16_bits((3000, 512), 9200, 0.02)
    h = synth.normal_f32((1, 512), 9201)
    cases.append(dict(name="mm_f16w", op="matmul", wdtype="f16", W=put("e.W", E), A=put("e.A", h), M=1, N=3000, K=512,
                      outputDtype="f32", alpha=1.0, record=False))
    logits = oracle.f16w_matmul(h, E, 1, 3000, 512)
    checks.append(lambda: rel_l2(get("mm_f16w.out.bin", np.float32), logits) <= 1e-3)
    cases.append(dict(name="lm_head", op="lm_head", E="e.W", h="e.A", vocab=3000, hidden=512))
    checks.append(lambda: int(get("lm_head.out.bin", np.uint32)[0]) == oracle.argmax(logits[0]))
    # the final RMSNorm inside the LM head kernel (normWeight option)
    lnw = synth.normal_f32(512, 9202, 0.3)
    cases.append(dict(name="lm_head_normed", op="lm_head", E="e.W", h="e.A", vocab=3000, hidden=512,
                      normWeight=put("e.nw", lnw), rmsNormEps=1e-6))
    want_normed = oracle.f16w_matmul(oracle.rmsnorm(h, lnw, 1e-6).reshape(1, 512), E, 1, 3000, 512)
    checks.append(lambda: int(get("lm_head_normed.out.bin", np.uint32)[0]) == oracle.argmax(want_normed[0]))

    # fused FFN
    Wg, Wu = synth.q4k_tensor(1024, 768, 9300), synth.q4k_tensor(1024, 768, 9301)
    X = synth.normal_f32((2, 768), 9302, 0.02)
    cases.append(dict(name="ffn", op="fused_ffn", Wg=put("ffn.Wg", Wg), Wu=put("ffn.Wu", Wu), X=put("ffn.X", X), M=2,
                      hidden=768, inter=1024, activation="silu", alpha=1.0, swigluLimit=5.0))
    ffn_want = oracle.q4k_ffn_gate_up(X, Wg, Wu, 2, 768, 1024, activation="silu", swiglu_limit=5.0)
    checks.append(lambda: rel_l2(get("ffn.out.bin", np.float32), ffn_want) <= 1e-3)

    nwf = 1.0 + synth.normal_f32((768,), 9303, 0.1)
    Xn = synth.normal_f32((2, 768), 9304, 4.0)
    cases.append(dict(name="ffn_normed", op="fused_normed_ffn", Wg="ffn.Wg", Wu="ffn.Wu", X=put("ffnn.X", Xn),
                      normWeight=put("ffnn.nw", nwf), eps=1e-6, M=2, hidden=768, inter=1024, activation="gelu"))
    ffnn_want = oracle.q4k_ffn_gate_up(oracle.rmsnorm(Xn, nwf, 1e-6), Wg, Wu, 2, 768, 1024, activation="gelu")
    checks.append(lambda: rel_l2(get("ffn_normed.out.bin", np.float32), ffnn_want) <= 1e-3)

    # rmsnorm, rope, split qkv, kv write
    x = synth.normal_f32((3, 1152), 9400, 3.0)
    w = synth.normal_f32(1152, 9401, 0.1)
    r = synth.normal_f32((3, 1152), 9402)
    cases.append(dict(name="rms", op="rmsnorm", x=put("rms.x", x), w=put("rms.w", w), residual=put("rms.r", r), batch=3,
                      hidden=1152, eps=1e-6, weightOffset=True, outputScale=0.5))
    rms_want = oracle.rmsnorm(x, w, 1e-6, weight_offset=True, post_residual=r, output_scale=0.5)
    checks.append(lambda: rel_l2(get("rms.out.bin", np.float32), rms_want) <= 1e-5)

    qn = synth.normal_f32((2 * 16, 128), 9410, 2.0)
    kn = synth.normal_f32((2 * 8, 128), 9411, 0.5)
    qnw, knw = synth.normal_f32(128, 9412, 0.1), synth.normal_f32(128, 9413, 0.1)
    cases.append(dict(name="rmsqk", op="rmsnorm_qk", q=put("rmsqk.q", qn), k=put("rmsqk.k", kn), qw=put("rmsqk.qw", qnw),
                      kw=put("rmsqk.kw", knw), T=2, heads=16, kvHeads=8, headDim=128, eps=1e-6))
    rmsqk_q, rmsqk_k = oracle.rmsnorm(qn, qnw, 1e-6, weight_offset=True), oracle.rmsnorm(kn, knw, 1e-6, weight_offset=True)
    checks.append(lambda: rel_l2(get("rmsqk.q.out.bin", np.float32), rmsqk_q) <= 1e-5)
    checks.append(lambda: rel_l2(get("rmsqk.k.out.bin", np.float32), rmsqk_k) <= 1e-5)

    px, pr = synth.normal_f32((3, 1152), 9420, 3.0), synth.normal_f32((3, 1152), 9421)
    pwa, pwb = synth.normal_f32(1152, 9422, 0.1), synth.normal_f32(1152, 9423, 0.1)
    cases.append(dict(name="pair", op="rmsnorm_pair", x=put("pair.x", px), r=put("pair.r", pr), wa=put("pair.wa", pwa),
                      wb=put("pair.wb", pwb), batch=3, hidden=1152, eps=1e-6, outputScale=0.5))
    pair_post = oracle.rmsnorm(px, pwa, 1e-6, weight_offset=True, post_residual=pr)
    pair_pre = oracle.rmsnorm(pair_post.reshape(3, 1152), pwb, 1e-6, weight_offset=True)
    pair_res = ((px + pr) * np.float32(0.5)).astype(np.float32)
    pair_next = oracle.rmsnorm(pair_res, pwa, 1e-6, weight_offset=True)
    checks.append(lambda: rel_l2(get("pair.post.out.bin", np.float32), pair_post) <= 1e-5)
    checks.append(lambda: rel_l2(get("pair.pre.out.bin", np.float32), pair_pre) <= 1e-5)
    checks.append(lambda: np.array_equal(get("pair.res.out.bin", np.float32), pair_res.reshape(-1)))
    checks.append(lambda: rel_l2(get("pair.next.out.bin", np.float32), pair_next) <= 1e-5)

    cos, sin = synth.rope_tables(128, 64, 1e6)
    xr = synth.normal_f32((2, 16, 128), 9500)
    cases.append(dict(name="rope", op="rope", x=put("rope.x", xr), cos=put("cos", cos), sin=put("sin", sin), seq=2,
                      heads=16, headDim=128, startPos=40, interleaved=False))
    rope_want = oracle.rope_apply(xr, cos, sin, 2, 16, 128, 40)
    checks.append(lambda: rel_l2(get("rope.out.bin", np.float32), rope_want) <= 1e-6)
    # f16 activations (the reference's f16-activation plan, rope.js:44-63): the rotation of the f16 values,
    # computed in f32 and rounded to f16 once
    xr16 = xr.astype(np.float16)
    cases.append(dict(cases[-1], name="rope_f16", x=put("rope.x16", xr16.view(np.uint16)), dtype="f16"))
    rope16_want = oracle.rope_apply(xr16.astype(np.float32), cos, sin, 2, 16, 128, 40).astype(np.float16)
    checks.append(lambda: np.max(np.abs(get("rope_f16.out.bin", np.float16).astype(np.float32)
                                        - rope16_want.reshape(-1).astype(np.float32))
                                 / np.maximum(np.abs(rope16_want.reshape(-1).astype(np.float32)), 1e-3)) <= 2 ** -10)
    bx, bb = synth.normal_f32((3, 1024), 9510, 2.0), synth.normal_f32((2, 1024), 9511)
    cases.append(dict(name="biasscale", op="bias_scale", x=put("bs.x", bx), bias=put("bs.b", bb), tokens=3, dim=1024, scale=0.125))
    checks.append(lambda: np.array_equal(get("biasscale.bias.out.bin", np.float32).reshape(3, 1024), bx + bb[1]))
    checks.append(lambda: np.array_equal(get("biasscale.scale.out.bin", np.float32).reshape(3, 1024), (bx + bb[1]) * np.float32(0.125)))
    part = synth.normal_f32((6, 1536), 9512)
    part_want = np.concatenate([part[:1] * np.float32(0.3), np.zeros((5, 1536), np.float32)])
    cases.append(dict(name="scalepart", op="scale_part", x=put("scalepart.x", part), rows=6, dim=1536, scale=0.3))
    checks.append(lambda: np.array_equal(get("scalepart.out.bin", np.float32).reshape(6, 1536), part_want))
    sx = synth.normal_f32((3, 1024 + 256 + 256), 9520)
    cases.append(dict(name="splitplain", op="split_plain", x=put("sp.x", sx), tokens=3, q=1024, k=256, v=256))
    checks.append(lambda: np.array_equal(get("splitplain.q.out.bin", np.float32).reshape(3, 1024), sx[:, :1024]))
    checks.append(lambda: np.array_equal(get("splitplain.k.out.bin", np.float32).reshape(3, 256), sx[:, 1024:1280]))
    checks.append(lambda: np.array_equal(get("splitplain.v.out.bin", np.float32).reshape(3, 256), sx[:, 1280:]))
    kr = synth.normal_f32((2, 8, 128), 9501)
    cases.append(dict(name="ropeqk", op="rope_qk", q=put("ropeqk.q", xr), k=put("ropeqk.k", kr), cos=put("cos", cos),
                      sin=put("sin", sin), seq=2, heads=16, kvHeads=8, headDim=128, startPos=40))
    ropek_want = oracle.rope_apply(kr, cos, sin, 2, 8, 128, 40)
    checks.append(lambda: rel_l2(get("ropeqk.q.out.bin", np.float32), rope_want) <= 1e-6)
    checks.append(lambda: rel_l2(get("ropeqk.k.out.bin", np.float32), ropek_want) <= 1e-6)

    T, H, Hkv, D, start, max_seq = 2, 16, 8, 128, 37, 64
    qkv = synth.normal_f32((T, (H + 2 * Hkv) * D), 9600)
    qw, kw = 1 + synth.normal_f32(D, 9601, 0.1), 1 + synth.normal_f32(D, 9602, 0.1)
    cases.append(dict(name="split", op="split_qkv", qkv=put("split.qkv", qkv), qw=put("split.qw", qw), kw=put("split.kw", kw),
                      cos="cos", sin="sin", eps=1e-6, T=T, heads=H, kvHeads=Hkv, headDim=D, startPos=start, maxSeq=max_seq))
    wk, wv = np.zeros((max_seq, Hkv, D), np.uint16), np.zeros((max_seq, Hkv, D), np.uint16)
    want_q = oracle.qkv_norm_rope_kvwrite(qkv, qw, kw, cos, sin, T, H, Hkv, D, start, wk, wv, start * Hkv * D)
    checks.append(lambda: rel_l2(get("split.out.bin", np.float32), want_q) <= 1e-5)
    checks.append(lambda: np.array_equal(get("split.v.bin", np.uint16), wv.reshape(-1)))
    checks.append(lambda: rel_l2(get("split.k.bin", np.float16).astype(np.float32), wk.reshape(-1).view(np.float16).astype(np.float32)) <= 5e-4)

    # one decode step straight from the stacked projection: norm + RoPE + KV append inside the attention kernel
    fpos = start + T
    hk = synth.normal_f16_bits((max_seq, Hkv, D), 9610, D ** -0.5)
    hv = synth.normal_f16_bits((max_seq, Hkv, D), 9611, D ** -0.5)
    fq = synth.normal_f32((1, (H + 2 * Hkv) * D), 9612)
    cases.append(dict(name="fattn", op="attention_from_qkv", qkv=put("fattn.qkv", fq), qw="split.qw", kw="split.kw", cos="cos",
                      sin="sin", eps=1e-6, K=put("fattn.k", hk), V=put("fattn.v", hv), heads=H, kvHeads=Hkv, headDim=D,
                      startPos=fpos, maxSeq=max_seq))
    fk, fv = hk.copy().reshape(max_seq, Hkv, D), hv.copy().reshape(max_seq, Hkv, D)
    fqn = oracle.qkv_norm_rope_kvwrite(fq, qw, kw, cos, sin, 1, H, Hkv, D, fpos, fk.reshape(-1), fv.reshape(-1), fpos * Hkv * D)
    fwant = oracle.attention_decode_f16kv(fqn, fk, fv, H, Hkv, D, fpos + 1)
    checks.append(lambda: rel_l2(get("fattn.out.bin", np.float32), fwant) <= 2e-4)
    checks.append(lambda: np.array_equal(get("fattn.v.bin", np.uint16), fv.reshape(-1)))
    checks.append(lambda: rel_l2(get("fattn.k.bin", np.float16).astype(np.float32), fk.reshape(-1).view(np.float16).astype(np.float32)) <= 5e-4)

    kk, vv = synth.normal_f32(2048, 9700), synth.normal_f32(2048, 9701)
    cases.append(dict(name="kvw", op="kv_write", k=put("kvw.k", kk), v=put("kvw.v", vv), cacheElems=4096, srcOffset=64,
                      dstOffset=1024, count=1500))
    ek, ev = np.zeros(4096, np.uint16), np.zeros(4096, np.uint16)
    oracle.kv_write_f16(kk, vv, ek, ev, 64, 1024, 1500)
    checks.append(lambda: np.array_equal(get("kvw.out.bin", np.uint16), ek) and np.array_equal(get("kvw.v.bin", np.uint16), ev))

    # attention, config 3 at ctx 512
    ctx = 512
    c3, s3 = synth.rope_tables(128, ctx, 1e6)
    q = oracle.rope_apply(synth.normal_f32((1, 16, 128), 9800, 128 ** -0.5), c3, s3, 1, 16, 128, ctx - 1)
    q = q.astype(np.float16).astype(np.float32).reshape(16, 128)
    kb = oracle.rope_apply(synth.normal_f32((ctx, 8, 128), 9801, 128 ** -0.5), c3, s3, ctx, 8, 128, 0).astype(np.float16).view(np.uint16)
    vb = synth.normal_f16_bits((ctx, 8, 128), 9802, 128 ** -0.5)
    cases.append(dict(name="attn", op="attention", Q=put("attn.q", q), K=put("attn.k", kb), V=put("attn.v", vb), heads=16,
                      kvHeads=8, headDim=128, kvLen=ctx))
    attn_want = oracle.attention_decode_f16kv(q, kb, vb, 16, 8, 128, ctx)
    checks.append(lambda: rel_l2(get("attn.out.bin", np.float32), attn_want) <= 1e-3)
    # f16 Q (q above is f16-representable), f16 output
    cases.append(dict(cases[-1], name="attn_f16q", Q=put("attn.q16", q.astype(np.float16).view(np.uint16)), dtype="f16"))
    checks.append(lambda: rel_l2(get("attn_f16q.out.bin", np.float16).astype(np.float32), attn_want) <= 1e-3)
    # the same with the key count in a device buffer (kvLenBuffer): 300 of the 512 rows
    cases.append(dict(name="attn_len", op="attention_kvlen_buffer", Q="attn.q", K="attn.k", V="attn.v", heads=16, kvHeads=8,
                      headDim=128, kvLen=ctx, count=300))
    attn_len_want = oracle.attention_decode_f16kv(q, kb, vb, 16, 8, 128, 300)
    checks.append(lambda: rel_l2(get("attn_len.out.bin", np.float32), attn_len_want) <= 1e-3)

    # elementwise, gather, argmax
    a, b = synth.normal_f32(5000, 9900, 4.0), synth.normal_f32(5000, 9901)
    cases.append(dict(name="res", op="residual", a=put("ew.a", a), b=put("ew.b", b), n=5000, outputScale=0.25))
    checks.append(lambda: rel_l2(get("res.out.bin", np.float32), oracle.residual_add(a, b, 0.25)) <= 1e-7)
    for act in ("silu", "gelu"):
        cases.append(dict(name="gated_" + act, op="gated", gate="ew.a", up="ew.b", n=5000, activation=act))
        checks.append(lambda act=act: rel_l2(get("gated_%s.out.bin" % act, np.float32), oracle.act_gate(a, b, act)) <= 1e-5)
    xs = synth.normal_f32((4, 2 * 640), 9902, 3.0)
    cases.append(dict(name="rowsplit", op="silu_rowsplit", x=put("rs.x", xs), T=4, dim=640, activation="gelu"))
    checks.append(lambda: rel_l2(get("rowsplit.out.bin", np.float32), oracle.act_gate_rowsplit(xs, 4, 640, "gelu")) <= 1e-5)
    ids = np.array([5, 299, 300, 0], np.uint32)
    tab = synth.normal_f16_bits((300, 640), 9903, 0.02)
    cases.append(dict(name="gather", op="gather", ids=put("g.ids", ids), table=put("g.tab", tab), T=4, hidden=640, vocab=300))
    checks.append(lambda: np.array_equal(get("gather.out.bin", np.float32).reshape(4, 640), oracle.gather_f16(ids, tab, 640, 300)))
    # f16 rows out: the stored bits of the gathered rows (zeros for the id past the table)
    cases.append(dict(cases[-1], name="gather_f16", dtype="f16"))
    checks.append(lambda: np.array_equal(get("gather_f16.out.bin", np.float16).reshape(4, 640).astype(np.float32),
                                         oracle.gather_f16(ids, tab, 640, 300)))
    lg = synth.rng(9904).integers(-50, 50, 151936).astype(np.float32)
    pad = oracle.argmax(lg)
    cases.append(dict(name="argmax", op="argmax", logits=put("am.l", lg), vocab=151936, padTokenId=pad))
    checks.append(lambda: int(get("argmax.out.bin", np.uint32)[0]) == oracle.argmax(lg, pad_id=pad))

    # whole decode loop in JavaScript on a small model
    cfg = dict(layers=2, hidden=512, inter=1024, heads=8, kv_heads=4, head_dim=64, vocab=700, eps=1e-6, qk_norm=1,
               max_seq=24, theta=1e6)
    layers, embed, final_norm, mc, ms = decoder.random_model(cfg, seed=77, max_seq=24)
    jl = []
    for i, l in enumerate(layers):
        jl.append(dict(wqkv=put("L%d.qkv" % i, np.concatenate([l["wq"], l["wk"], l["wv"]])), wo=put("L%d.o" % i, l["wo"]),
                       wgate=put("L%d.g" % i, l["wgate"]), wup=put("L%d.u" % i, l["wup"]), wdown=put("L%d.d" % i, l["wdown"]),
                       inputNorm=put("L%d.in" % i, l["input_norm"]), postAttnNorm=put("L%d.pn" % i, l["post_attn_norm"]),
                       qNorm=put("L%d.qn" % i, l["q_norm"]), kNorm=put("L%d.kn" % i, l["k_norm"])))
    prompt = [int(t) for t in synth.rng(78).integers(0, 700, 6)]
    cases.append(dict(name="decoder", op="decoder", layers=jl, embed=put("m.embed", embed), finalNorm=put("m.fn", final_norm),
                      cos=put("m.cos", mc), sin=put("m.sin", ms), prompt=prompt, steps=10,
                      config=dict(layers=2, hidden=512, inter=1024, heads=8, kvHeads=4, headDim=64, vocab=700, eps=1e-6, maxSeq=24)))
    cases.append(dict(cases[-1], name="decoder_separate_qkv_kernel",
                      config=dict(cases[-1]["config"], fuseQkvAttention=False)))
    # the same steps with the decode step captured into a HIP graph at position 3 and replayed from
    # there on, and one step under a profiling recorder (per-label HIP-event timings)
    cases.append(dict(cases[-2], name="decoder_graph_replay", graphFrom=3, profileAt=4))
    # the finiteness guard on: same tokens while nothing crosses the bound; this random-weight model's
    # residual stream is far outside the f16 range (about 1e9 after layer 0), so with the default
    # bound of 65500 the first step throws and names layer 0
    cases.append(dict(cases[-3], name="decoder_guarded",
                      config=dict(cases[-3]["config"], finitenessGuard=True, finitenessAbsThreshold=1e30)))
    cases.append(dict(cases[-4], name="decoder_guarded_graph", graphFrom=2,
                      config=dict(cases[-4]["config"], finitenessGuard=True, finitenessAbsThreshold=1e30)))
    cases.append(dict(cases[-5], name="decoder_guard_trips", expectFinitenessAt=0,
                      config=dict(cases[-5]["config"], finitenessGuard=True)))
    ol = []
    for l in layers:
        dd = dict(l)
        dd["cache_k"] = np.zeros((24, 4, 64), np.uint16)
        dd["cache_v"] = np.zeros((24, 4, 64), np.uint16)
        ol.append(dd)
    cpu = oracle.DecoderOracle(cfg, ol, embed, final_norm, mc, ms)
    want_tokens, tok = [], None
    for pos in range(len(prompt) + 10):
        tok = cpu.step(prompt[pos] if pos < len(prompt) else tok, pos)
        want_tokens.append(tok)
    checks.append(lambda: [int(t) for t in get("decoder.out.bin", np.uint32)] == want_tokens)
    checks.append(lambda: [int(t) for t in get("decoder_separate_qkv_kernel.out.bin", np.uint32)] == want_tokens)
    checks.append(lambda: [int(t) for t in get("decoder_graph_replay.out.bin", np.uint32)] == want_tokens)
    checks.append(lambda: [int(t) for t in get("decoder_guarded.out.bin", np.uint32)] == want_tokens)
    checks.append(lambda: [int(t) for t in get("decoder_guarded_graph.out.bin", np.uint32)] == want_tokens)
    checks.append(lambda: get("decoder_guard_trips.out.bin", np.uint32).size == 0)

    # ---- the chained layer launch from the JS decoder: a model wide enough for it (the small one above
    #      keeps one launch per op), weights centred so that the logits depend on what the stack is fed;
    #      eager and from the captured graph, and the same model with the chain switched off
    ccfg = dict(layers=2, hidden=2048, inter=4096, heads=16, kv_heads=4, head_dim=128, vocab=700, eps=1e-6, qk_norm=1,
                max_seq=24, theta=1e6)
    clayers, cembed, cfinal, cmc, cms = decoder.random_model(ccfg, seed=91, max_seq=24)
    for l in clayers:
        for n in ("wq", "wk", "wv", "wo", "wgate", "wup", "wdown"):
            l[n] = synth.q4k_centred(l[n], 5)
    cjl = []
    for i, l in enumerate(clayers):
        cjl.append(dict(wqkv=put("C%d.qkv" % i, np.concatenate([l["wq"], l["wk"], l["wv"]])), wo=put("C%d.o" % i, l["wo"]),
                        wgate=put("C%d.g" % i, l["wgate"]), wup=put("C%d.u" % i, l["wup"]), wdown=put("C%d.d" % i, l["wdown"]),
                        inputNorm=put("C%d.in" % i, l["input_norm"]), postAttnNorm=put("C%d.pn" % i, l["post_attn_norm"]),
                        qNorm=put("C%d.qn" % i, l["q_norm"]), kNorm=put("C%d.kn" % i, l["k_norm"])))
    cprompt = [int(t) for t in synth.rng(92).integers(0, 700, 5)]
    cases.append(dict(name="decoder_chained", op="decoder", layers=cjl, embed=put("c.embed", cembed), finalNorm=put("c.fn", cfinal),
                      cos=put("c.cos", cmc), sin=put("c.sin", cms), prompt=cprompt, steps=9, graphFrom=7, expectChained=True,
                      config=dict(layers=2, hidden=2048, inter=4096, heads=16, kvHeads=4, headDim=128, vocab=700, eps=1e-6, maxSeq=24)))
    cases.append(dict(cases[-1], name="decoder_chain_off", expectChained=False,
                      config=dict(cases[-1]["config"], chainGemvs=False)))
    # the generation loop with staged token readback (decodeGreedy) from position 6 on, chained and not
    for src, name in ((cases[-2], "decoder_chained_greedy"), (cases[-1], "decoder_chain_off_greedy")):
        cases.append(dict({k: v for k, v in src.items() if k != "graphFrom"}, name=name, greedyFrom=6))
    col = []
    for l in clayers:
        dd = dict(l)
        dd["cache_k"] = np.zeros((24, 4, 128), np.uint16)
        dd["cache_v"] = np.zeros((24, 4, 128), np.uint16)
        col.append(dd)
    ccpu = oracle.DecoderOracle(ccfg, col, cembed, cfinal, cmc, cms)
    cwant, ctok = [], None
    for pos in range(len(cprompt) + 9):
        ctok = ccpu.step(cprompt[pos] if pos < len(cprompt) else ctok, pos)
        cwant.append(ctok)
    assert len(set(cwant)) > 2, cwant
    checks.append(lambda: [int(t) for t in get("decoder_chained.out.bin", np.uint32)] == cwant)
    checks.append(lambda: [int(t) for t in get("decoder_chain_off.out.bin", np.uint32)] == cwant)
    checks.append(lambda: [int(t) for t in get("decoder_chained_greedy.out.bin", np.uint32)] == cwant)
    checks.append(lambda: [int(t) for t in get("decoder_chain_off_greedy.out.bin", np.uint32)] == cwant)

    # ---- top-k temperature sampling through the JS op (seeded draw as in the reference)
    slog = (synth.rng(79).standard_normal(4000) * 3).astype(np.float32)
    cases.append(dict(name="sample", op="sample", logits=put("s.logits", slog), vocab=4000, temperature=0.9, topK=40, seed=42))
    want_sample = oracle.sample_topk(slog, 0.9, 40, oracle.seeded_random(42))
    checks.append(lambda: int(get("sample.out.bin", np.uint32)[0]) == want_sample)

    # ---- the same model again, this time written as an RDRR artifact (small shards, so tensors
    #      span shard boundaries) and read back by the JavaScript loader
    from doppler_amd import rdrr
    art_dir = os.path.join(d, "artifact")
    rdrr.write_artifact(art_dir, cfg, layers, embed, final_norm, shard_bytes=300_000)
    art_obj = rdrr.Artifact(art_dir)
    c2, l2, e2, fn2 = rdrr.load_model_arrays(art_obj)        # norms rounded to f16 by the artifact
    ol2 = []
    for l in l2:
        dd = dict(l)
        dd["cache_k"] = np.zeros((24, 4, 64), np.uint16)
        dd["cache_v"] = np.zeros((24, 4, 64), np.uint16)
        ol2.append(dd)
    cpu2 = oracle.DecoderOracle(cfg, ol2, e2, fn2, mc, ms)
    want2, tok = [], None
    for pos in range(len(prompt) + 10):
        tok = cpu2.step(prompt[pos] if pos < len(prompt) else tok, pos)
        want2.append(tok)
    cases.append(dict(name="rdrr_decoder", op="rdrr_decoder", dir=art_dir, maxSeq=24, prompt=prompt, steps=10))
    checks.append(lambda: [int(t) for t in get("rdrr_decoder.out.bin", np.uint32)] == want2)

    # ---- generate(): prompt through the prefill path, then the decode loop, greedy and with seeded
    #      top-k sampling; the Python host runs the same kernels on the same artifact
    from doppler_amd import rdrr as _rdrr
    pyd = _rdrr.load_decoder(art_dir, 24)
    want_greedy = pyd.generate(prompt, 8)
    pyd2 = _rdrr.load_decoder(art_dir, 24)
    samp = dict(temperature=0.9, topK=20, seed=5)
    want_sampled = pyd2.generate(prompt, 8, sampling=samp)
    assert want_greedy[0] == want2[len(prompt) - 1]            # prefill path agrees with the checker's token
    cases.append(dict(name="gen_greedy", op="generate", dir=art_dir, maxSeq=24, prompt=prompt, maxTokens=8))
    cases.append(dict(name="gen_sampled", op="generate", dir=art_dir, maxSeq=24, prompt=prompt, maxTokens=8, sampling=samp))
    checks.append(lambda: [int(t) for t in get("gen_greedy.out.bin", np.uint32)] == want_greedy)
    checks.append(lambda: [int(t) for t in get("gen_sampled.out.bin", np.uint32)] == want_sampled)

    json.dump(dict(cases=cases), open(os.path.join(d, "manifest.json"), "w"))
    p = subprocess.run([NODE, os.path.join(ROOT, "tests", "js", "run_cases.mjs"), d], stdout=subprocess.PIPE,
                       stderr=subprocess.STDOUT, text=True, timeout=500)
    assert p.returncode == 0, p.stdout
    res = json.load(open(os.path.join(d, "results.json")))
    assert res["cases"] == [c["name"] for c in cases]
    for i, chk in enumerate(checks):
        assert chk(), "check %d failed" % i
    # the profiled step: every op of the step carries a label with a positive time (2 layers x 5 ops
    # + gather + LM head with the final norm inside)
    prof = res["profile"]
    assert res["profileOps"] == 12, res["profileOps"]
    assert set(prof) == {"gather", "matmul:qkv_proj", "attention:from_qkv", "matmul:o_proj", "fused_normed_ffn",
                         "matmul:down_proj", "lm_head_argmax"}, prof
    assert all(0.0 < ms < 50.0 for ms in prof.values()), prof
    bad = [e for e in res["errors"] if not e["ok"]]
    assert not bad and len(res["errors"]) >= 21, bad
