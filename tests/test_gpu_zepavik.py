"""Zepavik on the GPU: every mechanism alone against the plain restatement, then whole models through the framework's own
loading, step, cache, prefill and generation.

Tolerances: 32-bit paths must agree with the float64 restatement to ~1e-5; bf16 paths to what rounding operands to bf16
(products) and f16 (cached keys and values, queries) explains."""
import ctypes
import math
import json
import os
import subprocess
import time
import sys

import numpy as np
import pytest
import torch

from doppler_amd import capi, decoder, dense_decoder, generate, models
from oracle import plain_zepavik as plain
from tests import zepavik_models as zm

pytestmark = pytest.mark.gpu
ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
F32_ROW, BF16_ROW = 3e-5, 0.03       # largest error of a row of logits (see zm.row_errors)


@pytest.fixture(scope="module")
def L():
    torch.cuda.init()
    return capi.init(torch.cuda.current_device())


def dev(a, dtype=torch.float32):
    return torch.from_numpy(np.ascontiguousarray(a)).to(dtype).cuda()


def host(t):
    torch.cuda.synchronize()
    capi.check(capi.load().dh_sync())
    return t.float().cpu().numpy().astype(np.float64)


def rel(a, b):
    return float(np.linalg.norm(a - b) / max(np.linalg.norm(b), 1e-30))


def rng(seed):
    return np.random.Generator(np.random.PCG64(seed))


# ------------------------------------------------------------------ embedding, norms

@pytest.mark.parametrize("hidden,buckets,mp,mc", [(136, 61, 31, 13), (70, 1, 5, 9), (4104, 501, 2000003, 1999993), (2051, 77, 3, 2)])
def test_embedding_sum(L, hidden, buckets, mp, mc):
    """Portions of a sequence; products of ids and multipliers far above 32 bits."""
    V, P, n = 3001, 90, 40
    g = rng(1)
    E, B, T = (zm.bf16(g.standard_normal((r, hidden))) for r in (V, buckets + 1, P))
    toks = [int(t) for t in g.integers(0, V, n)]
    toks[3] = V - 1
    want = E[toks] + B[plain.bigram_rows(toks, buckets, mp, mc)] + T[np.arange(n)]
    dE, dB, dT = (dev(a, torch.bfloat16) for a in (E, B, T))
    ld = hidden + 24
    out = torch.full((n, ld), 7.0, device="cuda")
    ids = dev(np.array([0] + toks, np.int32), torch.int32)      # one unused word in front
    for a, b in ((0, 1), (1, 3), (3, 4), (4, 17), (17, n)):
        capi.check(L.dh_embed_sum(ids.data_ptr(), 1 + a, ids.data_ptr() + 4 * a, dE.data_ptr(), V, dB.data_ptr(), buckets, mp, mc,
                                  dT.data_ptr(), P, out.data_ptr() + 4 * ld * a, ld, b - a, hidden, a, None))
    got = host(out)
    assert np.abs(got[:, :hidden] - want).max() < 1e-5 and (got[:, hidden:] == 7.0).all()
    # the position from a key count on the device
    kv = dev(np.array([30], np.int32), torch.int32)
    row = torch.zeros(ld, device="cuda")
    capi.check(L.dh_embed_sum(ids.data_ptr(), 30, ids.data_ptr() + 4 * 29, dE.data_ptr(), V, dB.data_ptr(), buckets, mp, mc,
                              dT.data_ptr(), P, row.data_ptr(), ld, 1, hidden, 0, kv.data_ptr()))
    assert np.abs(host(row)[:hidden] - want[29]).max() < 1e-5
    assert L.dh_embed_sum(ids.data_ptr(), 0, None, dE.data_ptr(), V, dB.data_ptr(), buckets, mp, mc, dT.data_ptr(), P, out.data_ptr(),
                          ld, 1, hidden, 5, None) != 0
    assert L.dh_embed_sum(ids.data_ptr(), 0, ids.data_ptr(), dE.data_ptr(), V, dB.data_ptr(), buckets, mp, mc, dT.data_ptr(), P,
                          out.data_ptr(), ld, 1, hidden, P, None) != 0


@pytest.mark.parametrize("hidden,ld", [(136, 192), (70, 128), (4096, 4096), (9000, 9024)])
@pytest.mark.parametrize("eps", [1e-5, 0.3])
def test_row_norms(L, hidden, ld, eps):
    g = rng(2)
    x = g.standard_normal((5, ld)).astype(np.float32)
    x[1] *= 1e-3                                   # eps inside the root decides this row
    w = np.zeros(ld, np.float32)
    w[:hidden] = 1 + 0.3 * g.standard_normal(hidden)
    rows = np.array([4, 1, 1, 0], np.int32)
    dx, dw, dr = dev(x), dev(w), dev(rows, torch.int32)
    want = plain.rms_norm(x[rows][:, :hidden].astype(np.float64), eps, w[:hidden].astype(np.float64))
    out = torch.full((4, ld), 3.0, device="cuda")
    capi.check(L.dh_rmsnorm_rows(dx.data_ptr(), ld, dr.data_ptr(), dw.data_ptr(), out.data_ptr(), capi.F32, ld, 4, hidden, eps))
    got = host(out)
    assert rel(got[:, :hidden], want) < 1e-6 and not got[:, hidden:].any()
    out16 = torch.full((5, ld), 3.0, dtype=torch.bfloat16, device="cuda")
    capi.check(L.dh_rmsnorm_rows(dx.data_ptr(), ld, None, dw.data_ptr(), out16.data_ptr(), capi.BF16, ld, 5, hidden, eps))
    got = host(out16)
    want = plain.rms_norm(x[:, :hidden].astype(np.float64), eps, w[:hidden].astype(np.float64))
    assert np.abs(got[:, :hidden] - want).max() <= np.abs(want).max() * 2.0 ** -8 and not got[:, hidden:].any()


# ------------------------------------------------------------------ dense products

def act_of(name, z):
    return {"relu2": np.square(np.maximum(z, 0)), "silu": z / (1 + np.exp(-z)), None: z,
            "gelu_tanh": 0.5 * z * (1 + np.tanh(np.sqrt(2 / np.pi) * (z + 0.044715 * z ** 3)))}[name]


# both tiles, whole and in k slices, edges in both directions
@pytest.mark.parametrize("M,N,K,first", [(1, 5, 64, 5), (2, 130, 128, 40), (65, 200, 192, 72), (130, 2100, 320, 2100), (300, 1500, 256, 0),
                                         (1030, 4100, 128, 1000), (2048, 8200, 64, 8000),
                                         (3, 100, 4096, 60), (200, 1000, 8256, 904), (96, 70, 33088, 70)])
@pytest.mark.parametrize("operand", ["bf16", "f32"])
def test_dense_matmul(L, M, N, K, first, operand):
    g = torch.Generator().manual_seed(M + N)
    A = torch.randn(M, K, generator=g).to(torch.bfloat16 if operand == "bf16" else torch.float32)
    W = (torch.randn(N, K, generator=g) / K ** 0.5).to(torch.bfloat16)
    bias, res = torch.randn(max(first, 1), generator=g), torch.randn(M, max(first, 1) + 8, generator=g)
    acc = 0.75 * (A.double() @ W.double().T).numpy()
    dA, dW, db = A.cuda(), W.cuda(), bias.cuda()
    code = capi.BF16 if operand == "bf16" else capi.F32
    for name, act in (("relu2", capi.ACT_RELU2), ("silu", capi.ACT_SILU), ("gelu_tanh", capi.ACT_GELU)):
        C = res.cuda()
        ldc2 = N - first + 4
        C2 = torch.full((M, max(ldc2, 1)), 9.0, dtype=torch.bfloat16 if operand == "bf16" else torch.float32, device="cuda")
        capi.check(L.dh_dense_matmul(dA.data_ptr(), code, K, dW.data_ptr(), K, M, N, K, 0.75, db.data_ptr(), C.data_ptr(), C.data_ptr(),
                                     first + 8, first, C2.data_ptr(), code, ldc2, act))
        got, got2 = host(C), host(C2)
        if first:
            want = acc[:, :first] + bias.double().numpy()[:first] + res.double().numpy()[:, :first]
            assert np.abs(got[:, :first] - want).max() < 2e-5
            assert np.array_equal(got[:, first:], res.double().numpy()[:, first:])
        if first < N:
            want = act_of(name, acc[:, first:])
            tol = (2.0 ** -8 if operand == "bf16" else 1e-5) * max(1.0, np.abs(want).max())
            assert np.abs(got2[:, :N - first] - want).max() < tol
            assert (got2[:, N - first:] == 9.0).all()


# the larger tiles of the 16-bit products: k steps of either parity, edges in both directions, both outputs in one tile
@pytest.mark.parametrize("M,N,K,first", [(2060, 6150, 1536, 6150), (2060, 6150, 1600, 3001), (1540, 4090, 2048, 33), (1537, 4097, 2112, 4000)])
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
def test_dense_matmul_large_tiles(L, M, N, K, first, dtype):
    g = torch.Generator(device="cuda").manual_seed(M + N + K)
    A = torch.randn(M, K, generator=g, device="cuda").to(dtype)
    W = (torch.randn(N, K, generator=g, device="cuda") / K ** 0.5).to(dtype)
    scale, res = torch.randn(N, generator=g, device="cuda"), torch.randn(M, first, generator=g, device="cuda")
    C, C2 = res.clone(), torch.full((M, N - first + 2), 9.0, dtype=dtype, device="cuda")
    code = capi.BF16 if dtype == torch.bfloat16 else capi.F16
    torch.cuda.synchronize()
    capi.check(L.dh_dense_matmul_scaled(A.data_ptr(), code, K, W.data_ptr(), K, M, N, K, 1.5, None, scale.data_ptr(), C.data_ptr(), C.data_ptr(),
                                        first, first, C2.data_ptr(), code, N - first + 2, capi.ACT_RELU2))
    capi.check(L.dh_sync())
    acc = 1.5 * (A.double() @ W.double().T)
    # unit products: sums of up to 2112 terms in 32 bits stay within 2^-24 * sqrt(K) * a few of them
    assert (C.double() - (acc[:, :first] * scale[:first].double() + res.double())).abs().max() < 5e-5
    if first < N:
        want = acc[:, first:].clamp(min=0).square()
        assert ((C2[:, :N - first].double() - want).abs() <= 2.0 ** (-8 if dtype == torch.bfloat16 else -10) * want + 1e-4).all()
        assert (C2[:, N - first:] == 9.0).all()


# every tile of the 16-bit products, whole and in k slices (with a short last one), k steps of either parity, ragged in both directions; the
# tile and the slices are those of 256 compute units
TILES = [(129, 130, 192, (64, 64, 1)), (2, 33, 1664, (64, 64, 3)), (195, 9798, 640, (128, 128, 1)), (148, 11027, 704, (128, 128, 1)),
         (67, 4706, 4096, (128, 128, 6)), (1274, 65, 11776, (128, 128, 16)), (1412, 2912, 896, (256, 128, 1)), (1540, 4090, 2112, (256, 128, 1)),
         (1165, 1684, 9664, (256, 128, 3)), (2720, 4759, 1152, (256, 256, 1)), (2060, 6150, 1600, (256, 256, 1)), (129, 11422, 14144, (256, 256, 5))]
# with a second output through the exact gelu, whose epilogue counts
ERF_TILES = [(129, 130, 192, (64, 64, 1)), (2, 33, 1664, (64, 64, 3)), (330, 5525, 768, (128, 128, 1)), (67, 4706, 4096, (128, 128, 6)),
             (1224, 4121, 2176, (256, 128, 1)), (1165, 1684, 9664, (256, 128, 3)), (2441, 5063, 1216, (256, 256, 1)), (129, 11422, 14144, (256, 256, 5))]
# gate and up products of a shared expert (32 gate rows, 32 up rows, ..)
GLU_TILES = [(300, 256, 704, (64, 128, 1)), (1234, 1664, 704, (128, 128, 1)), (1928, 2176, 640, (256, 128, 1)), (2224, 5632, 1344, (256, 256, 1))]


def tile_of(L, M, N, K, code, glu=False, num_cus=0, erf=False):
    out = (ctypes.c_int64 * 3)()
    capi.check(L.dh_dense_matmul_layout(M, N, K, code, 2 if erf else int(glu), num_cus, out))
    return tuple(out)


@pytest.mark.parametrize("M,N,K,tile", TILES)
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
def test_dense_matmul_every_tile(L, M, N, K, tile, dtype):
    assert tile_of(L, M, N, K, capi.BF16 if dtype == torch.bfloat16 else capi.F16) == tile
    check_forms(L, M, N, K, dtype, ((N, capi.ACT_NONE, None), (N // 3, capi.ACT_NONE, lambda z: z),
                                    (N // 3, capi.ACT_RELU2, lambda z: z.clamp(min=0).square())))


@pytest.mark.parametrize("M,N,K,tile", ERF_TILES)
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
def test_dense_matmul_gelu_on_every_tile(L, M, N, K, tile, dtype):
    assert tile_of(L, M, N, K, capi.BF16 if dtype == torch.bfloat16 else capi.F16, erf=True) == tile
    check_forms(L, M, N, K, dtype, ((N // 3, capi.ACT_GELU_ERF, lambda z: 0.5 * z * (1 + torch.erf(z * 0.5 ** 0.5))),))


@pytest.mark.parametrize("M,N,K,tile", TILES + [(1, 70, 64, (64, 64, 1)), (9, 100, 128, (64, 64, 1)), (33, 64, 64, (64, 64, 1))])
def test_dense_matmul_with_a_residual_in_place_on_every_tile(L, M, N, K, tile):
    """(acc + bias) * scale + what the output held, alone and in front of a second output.  5e-5 of the sums as in check_forms, times scales of
    up to 4; squared, twice a sum of up to 5."""
    assert tile_of(L, M, N, K, capi.BF16) == tile
    g = torch.Generator(device="cuda").manual_seed(M + N + K)
    A = torch.randn(M, K, generator=g, device="cuda").to(torch.bfloat16)
    W = (torch.randn(N, K, generator=g, device="cuda") / K ** 0.5).to(torch.bfloat16)
    bias, scale = (torch.randn(N, generator=g, device="cuda") for _ in range(2))
    acc = A.double() @ W.double().T
    for first in (N, N // 3):
        C, C2 = torch.randn(M, first + 3, generator=g, device="cuda"), torch.full((M, N - first + 2), 9.0, device="cuda")
        want = (acc[:, :first] + bias[:first].double()) * scale[:first].double() + C[:, :first].double()
        beside = C[:, first:].clone()
        torch.cuda.synchronize()
        capi.check(L.dh_dense_matmul_scaled(A.data_ptr(), capi.BF16, K, W.data_ptr(), K, M, N, K, 1.0, bias.data_ptr(), scale.data_ptr(), C.data_ptr(),
                                            C.data_ptr(), first + 3, first, C2.data_ptr(), capi.F32, N - first + 2, capi.ACT_RELU2))
        capi.check(L.dh_sync())
        assert (C[:, :first].double() - want).abs().max() < 2e-4 and torch.equal(C[:, first:], beside)
        if first < N:
            assert (C2[:, :N - first].double() - acc[:, first:].clamp(min=0).square()).abs().max() < 5e-4 and (C2[:, N - first:] == 9.0).all()


def check_forms(L, M, N, K, dtype, forms):
    code = capi.BF16 if dtype == torch.bfloat16 else capi.F16
    g = torch.Generator(device="cuda").manual_seed(M + N + K)
    A = torch.randn(M, K, generator=g, device="cuda").to(dtype)
    W = (torch.randn(N, K, generator=g, device="cuda") / K ** 0.5).to(dtype)
    acc = A.double() @ W.double().T
    for first, act, fn in forms:
        C, C2 = torch.full((M, first + 3), 9.0, device="cuda"), torch.full((M, N - first + 2), 9.0, dtype=dtype, device="cuda")
        torch.cuda.synchronize()
        capi.check(L.dh_dense_matmul(A.data_ptr(), code, K, W.data_ptr(), K, M, N, K, 1.0, None, None, C.data_ptr(), first + 3, first,
                                     C2.data_ptr(), code, N - first + 2, act))
        capi.check(L.dh_sync())
        # unit products: sums of up to 14144 exact terms in 32 bits; a second output is rounded once more
        assert (C[:, :first].double() - acc[:, :first]).abs().max() < 5e-5 and (C[:, first:] == 9.0).all()
        if first < N:
            want = fn(acc[:, first:])
            assert ((C2[:, :N - first].double() - want).abs() <= 2.0 ** (-8 if code == capi.BF16 else -10) * want.abs() + 2e-4).all()
            assert (C2[:, N - first:] == 9.0).all()


@pytest.mark.parametrize("T,N,K,tile", GLU_TILES)
def test_shared_expert_on_every_tile(L, T, N, K, tile):
    """The routed expert's weights are zero, so that what is added to the rows is the shared expert's result alone.  Its activations are
    rounded to bf16 in front of the down product (2^-9 of each, added up over ff of them in a product of random signs)."""
    assert tile_of(L, T, N, K, capi.BF16, glu=True) == tile
    ff, hidden, limit = N // 2, 128, 1.5
    g = torch.Generator(device="cuda").manual_seed(T)
    h = torch.randn(T, K, generator=g, device="cuda").to(torch.bfloat16)
    w = lambda rows, k: (torch.randn(rows, k, generator=g, device="cuda") / k ** 0.5).to(torch.bfloat16)
    up, down, router, norm = w(N, K), w(K, ff)[:hidden].contiguous(), w(2, K), torch.ones(K, device="cuda")
    none = torch.zeros(max(128, K), max(64, K), dtype=torch.bfloat16, device="cuda")
    spec = capi.Experts(hidden, K, 1, 1, 64, ff, 1e-5, 7.0, limit, norm.data_ptr(), None, router.data_ptr(), none.data_ptr(), none.data_ptr(), up.data_ptr(),
                        down.data_ptr())
    ws = torch.empty(L.dh_experts_prefill_workspace_bytes(ctypes.byref(spec), capi.BF16, T), dtype=torch.uint8, device="cuda")
    x = torch.zeros(T, hidden, device="cuda")
    torch.cuda.synchronize()
    capi.check(L.dh_experts_prefill(ctypes.byref(spec), h.data_ptr(), capi.BF16, x.data_ptr(), hidden, ws.data_ptr(), T))
    capi.check(L.dh_sync())
    z = (h.double() @ up.double().T).view(T, ff // 32, 2, 32)
    gate, lin = (z[:, :, i].reshape(T, ff) for i in (0, 1))
    gate = gate.clamp(max=limit)
    act = gate * torch.sigmoid(1.702 * gate) * (lin.clamp(-limit, limit) + 1) * torch.sigmoid(h.double() @ router[1].double())[:, None]
    want = act @ down.double().T
    assert ((x.double() - want).norm(dim=1) <= 2.0 ** -8 * want.norm(dim=1)).all()
    assert ((x.double() - want).norm(dim=0) <= 2.0 ** -8 * want.norm(dim=0)).all()


# the smallest tile: k steps of every remainder by its four buffers, one row and column over and under its edges
@pytest.mark.parametrize("M,N,K", [(64, 64, 64), (65, 63, 128), (33, 129, 192), (63, 65, 256), (3, 97, 320), (130, 31, 448)])
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
def test_dense_matmul_small_tiles(L, M, N, K, dtype):
    g = torch.Generator(device="cuda").manual_seed(M + N + K)
    A = torch.randn(M, K, generator=g, device="cuda").to(dtype)
    W = (torch.randn(N, K, generator=g, device="cuda") / K ** 0.5).to(dtype)
    C = torch.full((M, N + 3), 9.0, device="cuda")
    code = capi.BF16 if dtype == torch.bfloat16 else capi.F16
    torch.cuda.synchronize()
    capi.check(L.dh_dense_matmul(A.data_ptr(), code, K, W.data_ptr(), K, M, N, K, 1.0, None, None, C.data_ptr(), N + 3, N, None, 0, 0, capi.ACT_NONE))
    capi.check(L.dh_sync())
    # unit products: sums of up to 448 exact terms in 32 bits
    assert (C[:, :N].double() - A.double() @ W.double().T).abs().max() < 2e-5 and (C[:, N:] == 9.0).all()


# 32-bit products in k slices: one tile, a ragged last slice, a narrow product, as many slices as there are
@pytest.mark.parametrize("M,N,K", [(1, 3, 128), (17, 70, 4160), (65, 130, 1088), (301, 1024, 4096), (40, 129, 16448)])
def test_dense_matmul_f32_slices(L, M, N, K):
    g = torch.Generator(device="cuda").manual_seed(M + N + K)
    A = torch.randn(M, K, generator=g, device="cuda")
    W = (torch.randn(N, K, generator=g, device="cuda") / K ** 0.5).to(torch.bfloat16)
    bias, C = torch.randn(N, generator=g, device="cuda"), torch.full((M, N + 4), 9.0, device="cuda")
    torch.cuda.synchronize()
    capi.check(L.dh_dense_matmul(A.data_ptr(), capi.F32, K, W.data_ptr(), K, M, N, K, -0.5, bias.data_ptr(), None, C.data_ptr(), N + 4, N, None, 0,
                                 0, capi.ACT_NONE))
    capi.check(L.dh_sync())
    want = -0.5 * (A.double() @ W.double().T) + bias.double()
    # unit products: sums of up to 16448 terms in 32 bits
    assert (C[:, :N].double() - want).abs().max() < 5e-5 and (C[:, N:] == 9.0).all()


# the tiles of the 32-bit products, whole and in k slices, ragged in both directions; one of a single step, which goes through registers
F32_TILES = [(33, 65, 64, (64, 64, 1)), (2, 33, 128, (32, 64, 1)), (33, 70, 960, (32, 64, 1)), (17, 70, 4160, (32, 64, 13)), (200, 4000, 192, (64, 64, 1)),
             (400, 3001, 2112, (64, 64, 1)), (301, 1024, 4096, (64, 64, 3)), (590, 10255, 2112, (128, 128, 1)), (600, 2050, 8256, (128, 128, 3))]


@pytest.mark.parametrize("M,N,K,tile", F32_TILES)
def test_dense_matmul_f32_tiles(L, M, N, K, tile):
    """Both outputs, in place, rows further apart than they are long.  Of K terms a sum is rounded fewer than K / 8 times, by 2^-25 of its size
    on average: within 2^-24 sqrt(K) / 4 of the exact one (2-norm), and 2^-22 for what the epilogue adds."""
    assert tile_of(L, M, N, K, capi.F32, num_cus=256) == tile
    g = torch.Generator(device="cuda").manual_seed(M + N + K)
    A = torch.randn(M, K + 8, generator=g, device="cuda")
    W = (torch.randn(N, K + 16, generator=g, device="cuda") / K ** 0.5).to(torch.bfloat16)
    first = N // 2
    bias, scale, res = (torch.randn(*s, generator=g, device="cuda") for s in ((first,), (first,), (M, first + 3)))
    C, C2 = res.clone(), torch.full((M, N - first + 2), 9.0, device="cuda")
    torch.cuda.synchronize()
    capi.check(L.dh_dense_matmul_scaled(A.data_ptr(), capi.F32, K + 8, W.data_ptr(), K + 16, M, N, K, 0.5, bias.data_ptr(), scale.data_ptr(), C.data_ptr(),
                                        C.data_ptr(), first + 3, first, C2.data_ptr(), capi.F32, N - first + 2, capi.ACT_RELU2))
    capi.check(L.dh_sync())
    acc = 0.5 * (A[:, :K].double() @ W[:, :K].double().T)
    want, near = (acc[:, :first] + bias.double()) * scale.double() + res[:, :first].double(), 2.0 ** -24 * K ** 0.5 / 4 + 2.0 ** -22
    assert (C[:, :first].double() - want).norm() < near * want.norm() and torch.equal(C[:, first:], res[:, first:])
    want = acc[:, first:].clamp(min=0).square()
    assert (C2[:, :N - first].double() - want).norm() < 2 * near * want.norm() and (C2[:, N - first:] == 9.0).all()


@pytest.mark.parametrize("M,N,K", [(9, 70, 128), (300, 1030, 1024), (301, 1024, 4096), (600, 10255, 2112)])
def test_dense_matmul_f32_extreme_values(L, M, N, K):
    """Infinities, no numbers and overflow stay where they belong; rows and products near the smallest numbers keep their bits."""
    g = torch.Generator(device="cuda").manual_seed(K)
    A = torch.randn(M, K, generator=g, device="cuda")
    W = (torch.randn(N, K, generator=g, device="cuda") / K ** 0.5).to(torch.bfloat16)
    A[0, 3], A[1, K - 1] = math.inf, -math.inf
    A[2, 7] = torch.tensor([0x7f800001], dtype=torch.int32, device="cuda").view(torch.float32)[0]        # a NaN whose upper half is an infinity
    W[3, 9], A[3, 9] = math.inf, 0.5           # the lower parts of 0.5 are zero
    W[N - 1, 0] = -math.inf
    A[4] *= 2.0 ** -122
    A[0, 4:], W[5, 4:] = 0, 0
    A[3, 11], W[6, 11] = 3.4e38, 1.0
    got, want = torch.zeros(M, N, device="cuda"), A.double() @ W.double().T
    torch.cuda.synchronize()
    capi.check(L.dh_dense_matmul(A.data_ptr(), capi.F32, K, W.data_ptr(), K, M, N, K, 1.0, None, None, got.data_ptr(), N, N, None, 0, 0, capi.ACT_NONE))
    capi.check(L.dh_sync())
    finite = want.float().isfinite()
    assert torch.equal(got.isnan(), want.isnan()) and torch.equal(got[want.isinf()].double(), want[want.isinf()])
    # row 4's products are rounded at 2^-149 each
    assert (got[4].double() - want[4])[finite[4]].abs().max() < 1e-6 * 2.0 ** -122 * 6 + K * 2.0 ** -150
    rows = [m for m in range(M) if m not in (3, 4)]
    assert (got.double() - want)[rows][finite[rows]].abs().max() < 5e-5


@pytest.mark.parametrize("M,N,K", [(9, 70, 128), (300, 1030, 1024), (301, 1024, 4096), (600, 10255, 2112)])
def test_dense_matmul_f32_far_from_one(L, M, N, K):
    """Activations with bits below bf16's smallest number, down to f32's, against small, ordinary and huge weights.  f32 sums: half a unit of the
    last place of K / 8 partial sums at worst, which are no larger than the terms together, and 2^-150 for each product and sum below f32's normal numbers."""
    g = torch.Generator(device="cuda").manual_seed(K + 1)
    A = torch.randn(M, K, generator=g, device="cuda")
    W = torch.randn(N, K, generator=g, device="cuda")
    for rows, power in ((slice(0, 2), -136), (slice(2, 4), -124), (slice(4, 6), -110), (slice(6, 7), -100)):
        A[rows] *= 2.0 ** (power // 2)
        A[rows] *= 2.0 ** (power - power // 2)
    for columns, power in ((slice(0, 9), 100), (slice(9, 20), 50), (slice(20, 30), 30), (slice(30, 40), -60)):
        W[columns] *= 2.0 ** power
    A[7, 1:] = 0
    A[7, 0] = 2.0 ** -140
    W = W.to(torch.bfloat16)
    got, a, w = torch.zeros(M, N, device="cuda"), A.double(), W.double()
    torch.cuda.synchronize()
    capi.check(L.dh_dense_matmul(A.data_ptr(), capi.F32, K, W.data_ptr(), K, M, N, K, 1.0, None, None, got.data_ptr(), N, N, None, 0, 0, capi.ACT_NONE))
    capi.check(L.dh_sync())
    bound = K / 8 * 2.0 ** -25 * (a.abs() @ w.abs().T) + 2 * K * 2.0 ** -150
    assert bool(((got.double() - a @ w.T).abs() <= bound).all())
    # the rows beside them are what they are without them
    A[:8] = A[8]
    beside = torch.zeros(M, N, device="cuda")
    torch.cuda.synchronize()
    capi.check(L.dh_dense_matmul(A.data_ptr(), capi.F32, K, W.data_ptr(), K, M, N, K, 1.0, None, None, beside.data_ptr(), N, N, None, 0, 0, capi.ACT_NONE))
    capi.check(L.dh_sync())
    assert torch.equal(got[8:], beside[8:])


@pytest.mark.parametrize("M,N,K", [(9, 70, 128), (301, 1024, 4096), (600, 10255, 2112)])
def test_dense_matmul_f32_parts_below_normal_numbers(L, M, N, K):
    """What parts that bf16 holds only below its normal numbers leave of two activations, where the rest of them cancels; and weights there."""
    A, W = torch.zeros(M, K, device="cuda"), torch.full((N, K), 2.0 ** 60, device="cuda").to(torch.bfloat16)
    A[:, 5], A[:, K - 1] = 2.0 ** -104 * (1 + 2.0 ** -22), -2.0 ** -104
    A[3], W[7] = 0, 2.0 ** -130
    A[3, 9], A[3, 11] = 2.0 ** 67 * (1 + 2.0 ** -16), -2.0 ** 67
    got = torch.zeros(M, N, device="cuda")
    torch.cuda.synchronize()
    capi.check(L.dh_dense_matmul(A.data_ptr(), capi.F32, K, W.data_ptr(), K, M, N, K, 1.0, None, None, got.data_ptr(), N, N, None, 0, 0, capi.ACT_NONE))
    capi.check(L.dh_sync())
    want = A.double() @ W.double().T
    want[:, 7] = torch.where(torch.arange(M, device="cuda") == 3, want[:, 7], torch.zeros(()).double().cuda())       # 2^-256
    assert torch.equal(got.double(), want)


def test_dense_matmul_f32_rows_that_are_no_numbers_cost_little(L):
    """Sums that the split operands do not give are made again a tile at a time: with one such row of 600 the call takes 2.5 times as long, with all of
    them what 32-bit instructions take besides, 4.4 times."""
    M, N, K = 600, 18464, 4096
    g = torch.Generator(device="cuda").manual_seed(11)
    A = torch.randn(M, K, generator=g, device="cuda")
    W = (torch.randn(N, K, generator=g, device="cuda") / K ** 0.5).to(torch.bfloat16)
    C = torch.zeros(M, N, device="cuda")
    torch.cuda.synchronize()

    def fastest():
        times = []
        for rep in range(6):
            t0 = time.perf_counter()
            capi.check(L.dh_dense_matmul(A.data_ptr(), capi.F32, K, W.data_ptr(), K, M, N, K, 1.0, None, None, C.data_ptr(), N, N, None, 0, 0, capi.ACT_NONE))
            capi.check(L.dh_sync())
            times.append(time.perf_counter() - t0)
        return min(times[1:])

    plain, sums = fastest(), C.clone()
    A[200, 17] = math.nan
    torch.cuda.synchronize()
    one = fastest()
    rows = [m for m in range(M) if m != 200]
    assert C[200].isnan().all() and torch.equal(C[rows], sums[rows])
    A[:, 5] = math.inf
    torch.cuda.synchronize()
    every = fastest()
    print("600 x 18464 x 4096: %.0f us, with a row that is no number %.0f, with infinite rows %.0f" % (plain * 1e6, one * 1e6, every * 1e6))
    assert one < 4 * plain and every < 8 * plain


def test_dense_matmul_f32_rows_2_gb_apart(L):
    M, N, K, ld = 2, 70, 192, 2 ** 29
    g = torch.Generator(device="cuda").manual_seed(7)
    A, W, C = torch.randn(M, K, generator=g, device="cuda"), torch.randn(N, K, generator=g, device="cuda").to(torch.bfloat16), torch.zeros(M, N, device="cuda")
    wide = torch.zeros(ld + K, device="cuda")
    wide[:K], wide[ld:] = A
    torch.cuda.synchronize()
    capi.check(L.dh_dense_matmul(wide.data_ptr(), capi.F32, ld, W.data_ptr(), K, M, N, K, 1.0, None, None, C.data_ptr(), N, N, None, 0, 0, capi.ACT_NONE))
    capi.check(L.dh_sync())
    # 192 terms of size up to 4 x 4 in 32 bits
    assert (C.double() - A.double() @ W.double().T).abs().max() < 192 * 16 * 2.0 ** -23


@pytest.mark.parametrize("M,N,K,operand", [(70000, 16, 4096, "f32"), (66000, 17, 12288, "bf16"), (66000, 20, 12288, "f16")])
def test_tall_narrow_products_in_slices(L, M, N, K, operand):
    """More rows than a grid's second dimension holds, and few enough columns that k is cut into slices."""
    dtype, code = dict(f32=(torch.float32, capi.F32), bf16=(torch.bfloat16, capi.BF16), f16=(torch.float16, capi.F16))[operand]
    g = torch.Generator(device="cuda").manual_seed(N)
    A = torch.randn(M, K, generator=g, device="cuda").to(dtype)
    W = (torch.randn(N, K, generator=g, device="cuda") / K ** 0.5).to(torch.bfloat16 if operand == "f32" else dtype)
    C = torch.full((M, N + 3), 9.0, device="cuda")
    torch.cuda.synchronize()
    capi.check(L.dh_dense_matmul(A.data_ptr(), code, K, W.data_ptr(), K, M, N, K, 1.0, None, None, C.data_ptr(), N + 3, N, None, 0, 0, capi.ACT_NONE))
    capi.check(L.dh_sync())
    want = torch.cat([A[i:i + 8192].double() @ W.double().T for i in range(0, M, 8192)])
    # unit products: sums of up to 12288 terms in 32 bits
    assert (C[:, :N].double() - want).abs().max() < 5e-5 and (C[:, N:] == 9.0).all()


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("far", ["activations", "weights"])
def test_dense_matmul_rows_4_gb_apart(L, far, dtype):
    """Two rows as far apart as a 32-bit stride allows."""
    M, N, K, ld = (2, 70, 64, 2 ** 31 - 64) if far == "activations" else (70, 2, 64, 2 ** 31 - 64)
    g = torch.Generator(device="cuda").manual_seed(7)
    A, W = torch.randn(M, K, generator=g, device="cuda").to(dtype), torch.randn(N, K, generator=g, device="cuda").to(dtype)
    wide = torch.zeros(ld + K, dtype=dtype, device="cuda")
    wide[:K], wide[ld:] = (A if far == "activations" else W)
    C, code = torch.zeros(M, N, device="cuda"), capi.BF16 if dtype == torch.bfloat16 else capi.F16
    torch.cuda.synchronize()
    capi.check(L.dh_dense_matmul(wide.data_ptr() if M == 2 else A.data_ptr(), code, ld if M == 2 else K, wide.data_ptr() if N == 2 else W.data_ptr(),
                                 ld if N == 2 else K, M, N, K, 1.0, None, None, C.data_ptr(), N, N, None, 0, 0, capi.ACT_NONE))
    capi.check(L.dh_sync())
    # 64 terms of size up to 4 x 4 in 32 bits
    assert (C.double() - A.double() @ W.double().T).abs().max() < 64 * 16 * 2.0 ** -23


def test_f32_products_are_not_reduced_precision(L):
    """Activations that differ from a constant in their last bits only: bf16- or TF32-like operands would lose them."""
    M, N, K = 40, 70, 256
    # Sums pass through magnitudes of 1 to 3, where each of the 256 additions rounds by up to 2^-24 or 2^-23: against sums of about
    # sqrt(256) 2^-20 that is 0.038 on average over draws and 0.059 in the worst of 300 (sequential f32 sums on the CPU; 1 of 27 is above
    # the bound), so the draw is fixed.  Operands of 16 bits or TF32 give 1.
    A = (1.0 + torch.randn(M, K, dtype=torch.float64, generator=torch.Generator().manual_seed(256)) * 2.0 ** -20).float()
    W = torch.ones(N, K, dtype=torch.bfloat16)
    W[:, ::2] = -1.0
    dA, dW, C = A.cuda(), W.cuda(), torch.zeros(M, N, device="cuda")
    capi.check(L.dh_dense_matmul(dA.data_ptr(), capi.F32, K, dW.data_ptr(), K, M, N, K, 1.0, None, None, C.data_ptr(), N, N, None, 0, 0,
                                 capi.ACT_NONE))
    want = (A.double() @ W.double().T).numpy()
    assert rel(host(C), want) < 0.05 and np.abs(want).max() < 1e-4


@pytest.mark.parametrize("N,K,hidden,first", [(1, 64, 40, 1), (77, 192, 136, 77), (1003, 1024, 1000, 300), (33000, 512, 512, 20000), (130, 8256, 8200, 64),
                                              (700, 16448, 16400, 700), (65, 32768, 32768, 0)])
def test_dense_gemv(L, N, K, hidden, first):
    g = torch.Generator().manual_seed(N + K)
    x = torch.zeros(K)
    x[:hidden] = torch.randn(hidden, generator=g)
    w = torch.zeros(K)
    w[:hidden] = 1 + 0.3 * torch.randn(hidden, generator=g)
    W = (torch.randn(N, K, generator=g) / K ** 0.5).to(torch.bfloat16)
    bias, res = torch.randn(N, generator=g), torch.randn(N, generator=g)
    dx, dw, dW, db = x.cuda(), w.cuda(), W.cuda(), bias.cuda()
    for normed in (True, False):
        xn = plain.rms_norm(x[:hidden].double().numpy(), 1e-2, w[:hidden].double().numpy()) if normed else x[:hidden].double().numpy()
        acc = 1.25 * (W[:, :hidden].double().numpy() @ xn)
        C, C2 = res.cuda(), torch.full((N - first + 1,), 5.0, device="cuda")
        capi.check(L.dh_dense_gemv(dx.data_ptr(), dw.data_ptr() if normed else None, hidden, 1e-2, dW.data_ptr(), K, N, K, 1.25,
                                   db.data_ptr(), C.data_ptr(), C.data_ptr(), first, C2.data_ptr(), capi.ACT_RELU2))
        want = acc[:first] + bias.double().numpy()[:first] + res.double().numpy()[:first]
        got, got2 = host(C), host(C2)
        if first:
            assert np.abs(got[:first] - want).max() < 1e-5
        assert np.array_equal(got[first:], res.double().numpy()[first:])
        if first < N:
            assert np.abs(got2[:-1] - act_of("relu2", acc[first:])).max() < 2e-5
        assert got2[-1] == 5.0


@pytest.mark.parametrize("K", [960, 1024, 1088, 2048, 2112, 3072, 3136, 4160, 8192])
@pytest.mark.parametrize("N", [5, 2047, 2048, 2049, 4101, 5136])
def test_dense_gemv_widths(L, N, K):
    """Either side of where the stage's length and the workgroup's width change; a product of K terms of size 1 / sqrt(K) in f32 in at
    most K / 64 + 6 roundings a lane and sum: 2^-24 (K / 64 + 6) <= 8e-6 of terms below 6."""
    g = torch.Generator(device="cuda").manual_seed(N + K)
    x, w = torch.randn(K, generator=g, device="cuda"), torch.rand(K, generator=g, device="cuda") + 0.5
    W = (torch.randn(N, K, generator=g, device="cuda") / K ** 0.5).to(torch.bfloat16)
    C = torch.full((N + 1,), 5.0, device="cuda")
    torch.cuda.synchronize()
    for normed in (True, False):
        capi.check(L.dh_dense_gemv(x.data_ptr(), w.data_ptr() if normed else None, K, 1e-5, W.data_ptr(), K, N, K, 1.0, None, None,
                                   C.data_ptr(), N, None, capi.ACT_NONE))
        capi.check(L.dh_sync())
        xn = x.double()
        if normed:
            xn = xn / torch.sqrt(xn.square().mean() + 1e-5) * w.double()
        assert (C[:N].double() - W.double() @ xn).abs().max() < 2e-5 and C[N] == 5.0
    # heads of 64 in front of the product
    H = K // 64
    y, gate = torch.zeros(N, device="cuda"), torch.randn(K, generator=g, device="cuda")
    torch.cuda.synchronize()
    capi.check(L.dh_dense_gemv_heads(x.data_ptr(), gate.data_ptr(), w.data_ptr(), H, 64, 64, 1e-5, W.data_ptr(), K, N, K, None, None, y.data_ptr()))
    capi.check(L.dh_sync())
    heads = x.double().reshape(H, 64)
    heads = (heads / torch.sqrt(heads.square().mean(1, keepdim=True) + 1e-5)).reshape(-1) * w.double() * torch.sigmoid(gate.double())
    assert (y.double() - W.double() @ heads).abs().max() < 2e-5


@pytest.mark.parametrize("vocab,K,hidden", [(301, 192, 136), (70001, 512, 500), (900, 9024, 9000)])
def test_dense_head_argmax(L, vocab, K, hidden):
    g = torch.Generator().manual_seed(vocab)
    x, w = torch.zeros(K), torch.zeros(K)
    x[:hidden], w[:hidden] = torch.randn(hidden, generator=g), torch.rand(hidden, generator=g) + 0.5
    W = (torch.randn(vocab, K, generator=g) / K ** 0.5).to(torch.bfloat16)
    want = 0.3 * (W[:, :hidden].double().numpy() @ plain.rms_norm(x[:hidden].double().numpy(), 1e-5, w[:hidden].double().numpy()))
    best = int(want.argmax())
    W[min(best + 40, vocab - 1)] = W[best]             # a tie: the lower index wins
    logits, tok = torch.zeros(vocab, device="cuda"), torch.zeros(4, dtype=torch.int32, device="cuda")
    ws = torch.zeros(int(L.dh_lmhead_argmax_workspace_bytes(vocab)), dtype=torch.uint8, device="cuda")
    dx, dw, dW = x.cuda(), w.cuda(), W.cuda()
    capi.check(L.dh_dense_lmhead_argmax(dx.data_ptr(), dw.data_ptr(), hidden, 1e-5, dW.data_ptr(), K, vocab, K, 0.3, ws.data_ptr(),
                                        tok.data_ptr(), 2, logits.data_ptr()))
    got = host(logits)
    keep = np.arange(vocab) != min(best + 40, vocab - 1)
    assert np.abs(got - want)[keep].max() < 1e-5 and tok.cpu().tolist() == [0, 0, best, 0]


# ------------------------------------------------------------------ attention

class Attn:
    """One attention layer fed through the C ABI: projection rows in, gated outputs out."""

    def __init__(self, L, H, G, d, e, window, cache="f16", scale=None, seed=0, n=200, gain=1.0, bias=True, gate=True, norm=True, value_std=1.0):
        self.L, self.H, self.G, self.d, self.e, self.window = L, H, G, d, e, window
        self.D, self.VD = (d + 7) // 8 * 8, (e + 7) // 8 * 8
        self.scale, self.eps, self.n = scale or d ** -0.5, 2e-3, n
        g = rng(seed)
        self.q, self.k, self.v = (g.standard_normal((n, h, s)).astype(np.float32) for h, s in ((H, d), (G, d), (G, e)))
        self.q *= gain
        self.v *= value_std
        self.gate = g.standard_normal((n, H)).astype(np.float32)
        self.r1, self.r2 = (g.uniform(a, b, H).astype(np.float32) for a, b in ((0.02, 1.5), (0.05, 0.9)))
        self.bias, self.gated, self.norm = bias, gate, norm
        self.ko = H * self.D
        self.vo = self.ko + G * self.D
        self.go = self.vo + G * self.VD
        self.ld = (self.go + H + 7) // 8 * 8
        self.cache_t = torch.float16 if cache == "f16" else torch.float32
        self.kc = torch.full((n, G, self.D), 60.0, dtype=self.cache_t, device="cuda")     # rows of an earlier sequence
        self.vc = torch.full((n, G, self.VD), -60.0, dtype=self.cache_t, device="cuda")
        self.dr1, self.dr2 = dev(self.r1), dev(self.r2)
        self.spec = capi.AttnSpec(H, G, self.D, self.VD, e, window, capi.F16 if cache == "f16" else capi.F32, int(norm), self.ko, self.vo,
                                  self.go if gate else -1, self.ld, self.scale, self.eps, self.dr1.data_ptr() if bias else None,
                                  self.dr2.data_ptr() if bias else None)
        self.ws = torch.zeros(int(L.dh_attn_spec_workspace_bytes(H, self.VD, n)), dtype=torch.uint8, device="cuda")

    def rows(self):
        r = np.zeros((self.n, self.ld), np.float32)
        for a, at, heads, size in ((self.q, 0, self.H, self.D), (self.k, self.ko, self.G, self.D), (self.v, self.vo, self.G, self.VD)):
            block = np.zeros((self.n, heads, size), np.float32)
            block[:, :, :a.shape[2]] = a
            r[:, at:at + heads * size] = block.reshape(self.n, -1)
        r[:, self.go:self.go + self.H] = self.gate
        return dev(r)

    def want(self):
        z = np.zeros(self.H)
        f = lambda a: a.astype(np.float64)
        v = plain.rms_norm(f(self.v), self.eps) if self.norm else f(self.v)
        o = plain.attention(f(self.q), f(self.k), v, self.scale, f(self.r1) if self.bias else z, f(self.r2) if self.bias else z,
                            self.window or 10 ** 9)
        return o * (plain.sigmoid(f(self.gate))[:, :, None] if self.gated else 1.0)

    def run(self, portions, out="f32"):
        """portions: sizes; 1 goes through the decode op, more through KV write + prefill."""
        L, rows, at = self.L, self.rows(), 0
        o = torch.zeros((self.n, self.H * self.VD), dtype=torch.float32 if out == "f32" else torch.bfloat16, device="cuda")
        one = torch.zeros(self.H * self.VD, device="cuda")
        spec = ctypes.byref(self.spec)
        for t in portions:
            src = rows.data_ptr() + 4 * self.ld * at
            if t == 1:
                capi.check(L.dh_attn_spec_decode(spec, src, self.kc.data_ptr(), self.vc.data_ptr(), one.data_ptr(), at, None, 0, self.ws.data_ptr()))
                capi.check(L.dh_sync())
                o[at] = one.to(o.dtype)
                torch.cuda.synchronize()
            else:
                capi.check(L.dh_attn_spec_kv_write(spec, src, self.kc.data_ptr(), self.vc.data_ptr(), t, at))
                capi.check(L.dh_attn_spec_prefill(spec, src, self.kc.data_ptr(), self.vc.data_ptr(),
                                                  o.data_ptr() + o.element_size() * self.H * self.VD * at,
                                                  capi.F32 if out == "f32" else capi.BF16, self.H * self.VD, t, at))
            at += t
        return host(o)[:at].reshape(at, self.H, self.VD)


SHAPES = [(4, 4, 64, 64), (6, 2, 24, 40), (8, 2, 128, 128), (5, 1, 64, 104), (3, 3, 96, 20), (12, 1, 16, 8), (9, 1, 136, 24), (2, 1, 40, 264),
          (10, 2, 300, 500), (1, 1, 8, 8)]


@pytest.mark.parametrize("cache", ["f16", "f32"])
@pytest.mark.parametrize("H,G,d,e", SHAPES)
def test_attention_shapes_prefill_decode_and_portions(L, H, G, d, e, cache):
    n, window = 150, 70
    tol = 3e-3 if cache == "f16" else 3e-6
    for k, portions in enumerate(([n], [1] * n, [2, 3, 1, 1, 61, 2, 7, 1, 64, 5, 3])):
        a = Attn(L, H, G, d, e, window, cache, n=n, seed=H + d)
        got, want = a.run(portions), a.want()
        assert not got[:, :, e:].any()
        err = [rel(got[t, :, :e], want[t]) for t in range(n)]
        assert max(err) < tol, (k, int(np.argmax(err)), max(err))


@pytest.mark.parametrize("cache", ["f16", "f32"])
@pytest.mark.parametrize("window", [1, 2, 7, 63, 64, 65, 128, 129, 0])
def test_attention_window_edges(L, window, cache):
    """In every head one key stands out; the queries that just see it and just do not are far apart."""
    n, H, G, d, e = 300, 4, 2, 64, 48
    planted = 100
    tol = 4e-3 if cache == "f16" else 1e-5
    for portions in ([n], [1] * n, [64] * 4 + [44], [99, 2, 1, 60, 1, 1, 66, 70]):
        a = Attn(L, H, G, d, e, window, cache, n=n, seed=5, gain=0.1)
        a.q[:, :, 0] = 24.0
        a.k[:, :, 0] = 0.0
        a.k[planted, :, 0] = 9.0
        a.v[planted] = 5.0 * np.sign(a.v[planted])
        got, want = a.run(portions)[:, :, :e], a.want()
        err = np.abs(got - want).max(axis=(1, 2)) / np.abs(want).max(axis=(1, 2))
        assert err.max() < tol, (int(err.argmax()), err.max())
        if window:
            inside, outside = planted + window - 1, planted + window
            edge = n - 1 if inside >= n else inside
            probe = np.einsum("he,ge->hg", want[edge] / np.linalg.norm(want[edge], axis=1, keepdims=True),
                              np.sign(a.v[planted]) / np.sqrt(e))
            assert probe.max(axis=1).min() > 0.9                # the planted key decides the last query that sees it
            if outside < n:
                assert np.abs(want[outside] - want[edge]).max() > 0.1


@pytest.mark.parametrize("start,T", [(0, 15), (0, 16), (3, 17), (30, 33), (255, 2), (1, 257), (40, 130)])
@pytest.mark.parametrize("H,G,d,e,window", [(4, 2, 64, 64, 0), (3, 1, 72, 40, 33), (2, 2, 128, 128, 0), (2, 1, 24, 104, 100)])
def test_attention_f32_tiles(L, H, G, d, e, window, start, T):
    """Tiles of 16 queries and 32 keys dealt to eight waves, remainders of both, either output type; the tolerance is the shapes test's."""
    a = Attn(L, H, G, d, e, window, "f32", n=start + T, seed=T)
    want = a.want()[start:]
    portions = [start, T] if start else [T]
    got = a.run(portions)[start:, :, :e]
    assert max(rel(got[t], want[t]) for t in range(T)) < 3e-6
    assert max(rel(x, y) for x, y in zip(a.run(portions, "bf16")[start:, :, :e], want)) < 2.0 ** -8


@pytest.mark.parametrize("start,T", [(0, 31), (3, 17), (30, 33), (1, 257), (40, 130), (700, 40)])
@pytest.mark.parametrize("H,G,d,e,window", [(16, 2, 64, 64, 0), (5, 1, 72, 40, 33), (8, 1, 128, 128, 0), (7, 1, 24, 104, 100)])
def test_attention_f32_tiles_of_many_heads(L, H, G, d, e, window, start, T):
    """The same where the tiles serve the call whatever its length: five and more heads to a key-value head."""
    a = Attn(L, H, G, d, e, window, "f32", n=start + T, seed=T)
    assert L.dh_attn_spec_prefill_plan(ctypes.byref(a.spec), 0, T, start, 256) == 1
    test_attention_f32_tiles(L, H, G, d, e, window, start, T)


@pytest.mark.parametrize("bad", [float("inf"), float("-inf"), float("nan")])
@pytest.mark.parametrize("H,G,d,e,window,at", [(8, 1, 64, 64, 0, 37), (5, 1, 128, 104, 40, 50), (16, 2, 64, 128, 33, 95), (7, 1, 120, 24, 20, 64),
                                                   (8, 1, 64, 64, 70, 0), (16, 2, 64, 64, 0, 149)])
def test_a_non_finite_value_in_a_tile_stays_with_the_queries_that_see_it(L, H, G, d, e, window, at, bad):
    a = Attn(L, H, G, d, e, window, "f32", n=150, seed=at)
    assert L.dh_attn_spec_prefill_plan(ctypes.byref(a.spec), 0, 150, 0, 256) == 1
    test_a_non_finite_value_stays_with_the_queries_that_see_it(L, H, G, d, e, window, at, bad)


@pytest.mark.parametrize("bad", [float("inf"), float("-inf"), float("nan")])
@pytest.mark.parametrize("H,G,d,e,window,at", [(2, 2, 64, 64, 0, 37), (2, 1, 128, 104, 40, 50), (1, 1, 64, 128, 33, 95), (2, 1, 120, 24, 1, 64),
                                                   (1, 1, 64, 64, 70, 0), (1, 1, 64, 64, 0, 149)])
def test_a_non_finite_value_stays_with_the_queries_that_see_it(L, H, G, d, e, window, at, bad):
    """f32 caches: every query in front of the value's token, or past its window, has the same bits as without it; those that see it do
    not, in that element alone."""
    n = 150
    a = Attn(L, H, G, d, e, window, "f32", n=n, seed=at)
    clean = a.run([n])
    rows, out = a.rows(), torch.zeros(n, H * a.VD, device="cuda")
    a.vc.view(-1, a.vc.numel() // a.vc.shape[0])[at, 3] = bad                # one element of the first key-value head's value
    torch.cuda.synchronize()
    capi.check(L.dh_attn_spec_prefill(ctypes.byref(a.spec), rows.data_ptr(), a.kc.data_ptr(), a.vc.data_ptr(), out.data_ptr(), capi.F32, H * a.VD, n, 0))
    got = host(out).reshape(n, H, a.VD)
    sees = np.zeros(n, bool)
    sees[at:at + window if window else n] = True
    hit = np.zeros(got.shape, bool)
    hit[sees, :H // G, 3] = True                                            # the query heads of that key-value head
    assert not np.isfinite(got[hit]).any() and np.array_equal(got[~hit], clean[~hit])


@pytest.mark.parametrize("bias,gate,norm", [(False, True, True), (True, False, True), (True, True, False), (False, False, False)])
def test_attention_mechanisms_one_at_a_time(L, bias, gate, norm):
    for cache, tol in (("f16", 3e-3), ("f32", 3e-6)):
        for portions in ([90], [30] + [1] * 60):
            a = Attn(L, 6, 3, 32, 56, 40, cache, n=90, seed=9, bias=bias, gate=gate, norm=norm, scale=0.31)
            assert rel(a.run(portions)[:, :, :56], a.want()) < tol


def test_value_norm_with_small_values_keeps_eps_inside_the_root(L):
    for cache, tol in (("f16", 3e-3), ("f32", 1e-5)):
        a = Attn(L, 4, 2, 64, 20, 50, cache, n=80, seed=10, value_std=0.03)      # mean square 9e-4 against eps 2e-3
        assert rel(a.run([40] + [1] * 40)[:, :, :20], a.want()) < tol


def test_first_tokens_and_large_distances(L):
    """A window longer than the sequence over many key tiles and splits: the far keys' bias, and the first positions."""
    n = 1500
    for cache, tol in (("f16", 4e-3), ("f32", 3e-5)):
        a = Attn(L, 8, 2, 64, 64, 2000, cache, n=n, seed=11, gain=0.1)
        a.q[:, :, 3] = 30.0
        a.k[:, :, 3] = 0.0
        a.k[2, :, 3] = 6.0
        a.r1[0], a.r2[0] = 0.0, 0.0
        a.dr1.copy_(torch.from_numpy(a.r1))
        a.dr2.copy_(torch.from_numpy(a.r2))
        want = a.want()
        got = a.run([5, 1, 1, 1, 1492])
        assert max(rel(got[t], want[t]) for t in range(n)) < tol
        tail = a.run([1490] + [1] * 10)
        assert max(rel(tail[t], want[t]) for t in range(1490, n)) < tol


@pytest.mark.parametrize("window", [0, 40])
def test_decode_with_the_key_count_on_the_device(L, window):
    n = 200
    a, b = (Attn(L, 6, 2, 24, 40, window, "f16", n=n, seed=12) for _ in range(2))
    want = a.run([100] + [1] * 100)
    rows, one = b.rows(), torch.zeros(6 * 40, device="cuda")
    b.run([100])
    kv = torch.zeros(1, dtype=torch.int32, device="cuda")
    for p in range(100, n):
        kv.fill_(p + 1)
        torch.cuda.synchronize()
        capi.check(L.dh_attn_spec_decode(ctypes.byref(b.spec), rows.data_ptr() + 4 * b.ld * p, b.kc.data_ptr(), b.vc.data_ptr(),
                                         one.data_ptr(), 0, kv.data_ptr(), n, b.ws.data_ptr()))
        assert rel(host(one).reshape(6, 40), want[p]) < 1e-5, p
    assert torch.equal(a.kc, b.kc) and torch.equal(a.vc, b.vc)


@pytest.mark.parametrize("cache", ["f16", "f32"])
@pytest.mark.parametrize("H,G,d,e,window,n,rows,ff,merged", [(4, 2, 64, 48, 0, 700, 2050, 72, True), (2, 2, 24, 40, 129, 400, 30, 0, True), (16, 8, 128, 128, 1024, 1200, 2048, 64, True),
                                                             (40, 40, 64, 24, 300, 400, 1030, 704, False), (16, 16, 64, 24, 300, 400, 1030, 704, True), (18, 6, 64, 24, 300, 400, 1030, 704, False),
                                                             (32, 32, 64, 24, 300, 400, 2050, 704, True), (33, 33, 64, 24, 300, 400, 2050, 704, False), (6, 2, 24, 40, 300, 400, 100, 8, False), (4, 2, 64, 64, 64, 300, 100, 0, False),
                                                             (32, 16, 128, 128, 1024, 1100, 4096, 0, False), (3, 3, 40, 264, 0, 300, 64, 0, False)])
def test_splits_left_to_the_product_behind(L, H, G, d, e, window, n, rows, ff, merged, cache):
    """A step's attention and the product that reads it, the key splits merged by the product or by a launch of their own, and with the key count on the
    device: one to eight splits of 128 keys, heads of up to 16 lanes one and two at a time, part of a wave's heads and all four of them in products of four and of eight waves, other activations
    beside the heads'; more heads at once, few keys, many bytes of splits and long heads are merged as ever.  The same 32-bit sums in another order: 24
    roundings of the terms' sizes."""
    a, b, c = (Attn(L, H, G, d, e, window, cache, n=n, seed=31) for _ in range(3))
    wide, K = H * a.VD, (H * a.VD + ff + 63) // 64 * 64
    g = torch.Generator(device="cuda").manual_seed(n)
    W, x = (torch.randn(rows, K, generator=g, device="cuda") / K ** 0.5).to(torch.bfloat16), torch.randn(rows, generator=g, device="cuda")
    inputs = [torch.randn(K, generator=g, device="cuda")]
    inputs += [inputs[0].clone(), inputs[0].clone()]
    src, took, kv = a.rows(), [], torch.zeros(1, dtype=torch.int32, device="cuda")
    for t in (a, b, c):
        capi.check(L.dh_attn_spec_kv_write(ctypes.byref(t.spec), src.data_ptr(), t.kc.data_ptr(), t.vc.data_ptr(), n, 0))
    for p in sorted({0, 1, 63, 64, 127, 128, 129, 255, 256, n // 2, n - 1}):
        outs = []
        for t, mixed, on_device in ((a, inputs[0], None), (b, inputs[1], False), (c, inputs[2], True)):
            step = (ctypes.byref(t.spec), src.data_ptr() + 4 * t.ld * p, t.kc.data_ptr(), t.vc.data_ptr(), mixed.data_ptr())
            left, y = ctypes.c_int(-1), x.clone()
            kv.fill_(p + 1)
            torch.cuda.synchronize()
            where = (0, kv.data_ptr(), n) if on_device else (p, None, n)
            if on_device is None:
                capi.check(L.dh_attn_spec_decode(*step, *where, t.ws.data_ptr()))
            else:
                capi.check(L.dh_attn_spec_decode_for(*step, *where, t.ws.data_ptr(), rows, ctypes.byref(left)))
                took.append(left.value)
            if left.value > 0:
                mixed[:wide] = float("nan")                    # what lies there is not read
                torch.cuda.synchronize()
                capi.check(L.dh_dense_gemv_attn(step[0], step[1], t.ws.data_ptr(), left.value, where[1], n, mixed.data_ptr(), W.data_ptr(), K, rows, K,
                                                y.data_ptr(), y.data_ptr()))
            else:
                capi.check(L.dh_dense_gemv(mixed.data_ptr(), None, 0, 0.0, W.data_ptr(), K, rows, K, 1.0, None, y.data_ptr(), y.data_ptr(), rows, None, capi.ACT_NONE))
            capi.check(L.dh_sync())
            outs.append(y.double())
        size = x.abs().double() + W.abs().double() @ inputs[0].abs().double()
        for y in outs[1:]:
            assert ((y - outs[0]).abs() <= 24 * 2.0 ** -24 * size).all(), p
    assert (max(took) > 0) == merged
    assert torch.equal(a.kc, b.kc) and torch.equal(a.vc, b.vc) and torch.equal(a.kc, c.kc)


@pytest.mark.parametrize("H,G,d,e,n,merged", [(2, 2, 64, 64, 8400, False), (3, 3, 64, 64, 8400, False), (4, 2, 32, 32, 9000, False), (1, 1, 64, 128, 8320, False),
                                              (1, 1, 64, 64, 8192, True), (2, 1, 32, 32, 8150, True)])
def test_few_heads_over_many_keys(L, H, G, d, e, n, merged):
    """Splits of few small heads are few bytes at any number of them; the product behind merges up to 64 of a head.  The product against 64 bits over the
    layer's outputs: 32-bit sums of n keys and of K columns, no chain of which is longer than one in 32 of the terms, each a rounding of the sizes."""
    a = Attn(L, H, G, d, e, 0, "f32", n=n, seed=61, bias=False, gate=False)
    rows, K = 64, (H * a.VD + 63) // 64 * 64
    g = torch.Generator(device="cuda").manual_seed(n)
    W, src = (torch.randn(rows, K, generator=g, device="cuda") / K ** 0.5).to(torch.bfloat16), a.rows()
    kv, spec = torch.zeros(1, dtype=torch.int32, device="cuda"), ctypes.byref(a.spec)
    capi.check(L.dh_attn_spec_kv_write(spec, src.data_ptr(), a.kc.data_ptr(), a.vc.data_ptr(), n, 0))
    q = dev(a.q).double()
    for p in sorted({8127, 8128, 8191, 8192, n - 1} & set(range(n))):
        k, v = a.kc[:p + 1].double(), a.vc[:p + 1].double()
        o = torch.zeros(H, a.VD, dtype=torch.float64, device="cuda")
        for h in range(H):
            o[h] = torch.softmax(k[:, h * G // H, :d] @ q[p, h] * a.scale, 0) @ v[:, h * G // H]
        want = W[:, :H * a.VD].double() @ o.reshape(-1)
        size = W[:, :H * a.VD].double().abs() @ v.abs().amax(0).repeat_interleave(H // G, 0).reshape(-1)
        for on_device in (False, True):
            left, mixed, y = ctypes.c_int(-1), torch.zeros(K, device="cuda"), torch.zeros(rows, device="cuda")
            kv.fill_(p + 1)
            torch.cuda.synchronize()
            row, where = src.data_ptr() + 4 * a.ld * p, (0, kv.data_ptr(), n) if on_device else (p, None, n)
            capi.check(L.dh_attn_spec_decode_for(spec, row, a.kc.data_ptr(), a.vc.data_ptr(), mixed.data_ptr(), *where, a.ws.data_ptr(), rows, ctypes.byref(left)))
            assert (left.value > 0) == merged and left.value <= 64
            if merged:
                capi.check(L.dh_dense_gemv_attn(spec, row, a.ws.data_ptr(), left.value, where[1], n, mixed.data_ptr(), W.data_ptr(), K, rows, K, None, y.data_ptr()))
            else:
                capi.check(L.dh_dense_gemv(mixed.data_ptr(), None, 0, 0.0, W.data_ptr(), K, rows, K, 1.0, None, None, y.data_ptr(), rows, None, capi.ACT_NONE))
            capi.check(L.dh_sync())
            assert ((y.double() - want).abs() <= (n / 32 + K / 32) * 2.0 ** -24 * size).all(), (p, on_device)


def test_splits_in_front_of_a_product_of_other_rows(L):
    """More heads than a product's waves make factors of at once: the bits of a product of eight waves that has the same rows and more."""
    a, K = Attn(L, 32, 32, 64, 24, 300, n=400, seed=31), 32 * 24
    g = torch.Generator(device="cuda").manual_seed(3)
    W, src, x = (torch.randn(2050, K, generator=g, device="cuda") / K ** 0.5).to(torch.bfloat16), a.rows(), torch.zeros(K, device="cuda")
    left, row, spec = ctypes.c_int(), src.data_ptr() + 4 * a.ld * 399, ctypes.byref(a.spec)
    torch.cuda.synchronize()
    capi.check(L.dh_attn_spec_kv_write(spec, src.data_ptr(), a.kc.data_ptr(), a.vc.data_ptr(), 400, 0))
    capi.check(L.dh_attn_spec_decode_for(spec, row, a.kc.data_ptr(), a.vc.data_ptr(), x.data_ptr(), 399, None, 400, a.ws.data_ptr(), 2050, ctypes.byref(left)))
    outs = []
    for rows in (2050, 100):
        outs.append(torch.zeros(rows, device="cuda"))
        torch.cuda.synchronize()
        capi.check(L.dh_dense_gemv_attn(spec, row, a.ws.data_ptr(), left.value, None, 400, x.data_ptr(), W.data_ptr(), K, rows, K, None, outs[-1].data_ptr()))
        capi.check(L.dh_sync())
    assert left.value > 1 and outs[0].abs().sum() > 0 and torch.equal(outs[0][:100], outs[1])


@pytest.mark.parametrize("what", ["key", "value", "query", "new key"])
def test_what_is_no_number_is_none_behind_a_product_either(L, what):
    """A lost element of a key, a value or the step's row: the product's outputs are lost in front of a product as they are behind a merge of their own, in one
    split of 128 keys, in several, and where 64 keys are one."""
    n, H, G, d = 300, 4, 2, 64
    W = torch.ones(70, H * d, dtype=torch.bfloat16, device="cuda")
    for p in (5, 62, 63, 64, 100, 127, 128, 200, 299):
        ys = []
        for rows in (0, 70):
            a = Attn(L, H, G, d, d, 0, n=n, seed=3, bias=False)
            src = a.rows()
            capi.check(L.dh_attn_spec_kv_write(ctypes.byref(a.spec), src.data_ptr(), a.kc.data_ptr(), a.vc.data_ptr(), n, 0))
            capi.check(L.dh_sync())
            if what == "key": a.kc[p // 2, 1, 7] = float("nan")
            if what == "value": a.vc[p // 2, 1, 7] = float("nan")
            if what == "query": src[p, 2 * d + 3] = float("nan")
            if what == "new key": src[p, a.ko + d + 3] = float("nan")
            x, y, left = torch.zeros(H * d, device="cuda"), torch.zeros(70, device="cuda"), ctypes.c_int(0)
            torch.cuda.synchronize()
            step = (ctypes.byref(a.spec), src.data_ptr() + 4 * a.ld * p, a.kc.data_ptr(), a.vc.data_ptr(), x.data_ptr(), p, None, n, a.ws.data_ptr())
            if rows:
                capi.check(L.dh_attn_spec_decode_for(*step, rows, ctypes.byref(left)))
            else:
                capi.check(L.dh_attn_spec_decode(*step))
            if left.value:
                capi.check(L.dh_dense_gemv_attn(*step[:2], a.ws.data_ptr(), left.value, None, n, x.data_ptr(), W.data_ptr(), H * d, 70, H * d, None, y.data_ptr()))
            else:
                capi.check(L.dh_dense_gemv(x.data_ptr(), None, 0, 0.0, W.data_ptr(), H * d, 70, H * d, 1.0, None, None, y.data_ptr(), 70, None, capi.ACT_NONE))
            capi.check(L.dh_sync())
            ys.append(y)
        assert torch.equal(ys[0].isnan(), ys[1].isnan()), p


def test_splits_of_another_count_are_refused(L):
    """The device's key count says how many splits a product reads: they have to be those of the most keys it can be."""
    a = Attn(L, 4, 2, 64, 48, 0, n=700, seed=9)
    src, W, x, y, left = a.rows(), torch.zeros(64, 192, dtype=torch.bfloat16, device="cuda"), torch.zeros(192, device="cuda"), torch.zeros(64, device="cuda"), ctypes.c_int()
    count = torch.full((1,), 700, dtype=torch.int32, device="cuda")
    capi.check(L.dh_attn_spec_kv_write(ctypes.byref(a.spec), src.data_ptr(), a.kc.data_ptr(), a.vc.data_ptr(), 700, 0))
    torch.cuda.synchronize()
    capi.check(L.dh_attn_spec_decode_for(ctypes.byref(a.spec), src.data_ptr() + 4 * a.ld * 699, a.kc.data_ptr(), a.vc.data_ptr(), x.data_ptr(), 0, count.data_ptr(), 700,
                                         a.ws.data_ptr(), 64, ctypes.byref(left)))
    merge = lambda splits, most: L.dh_dense_gemv_attn(ctypes.byref(a.spec), src.data_ptr() + 4 * a.ld * 699, a.ws.data_ptr(), splits, count.data_ptr(), most, x.data_ptr(),
                                                    W.data_ptr(), 192, 64, 192, None, y.data_ptr())
    for splits, most in ((left.value - 1, 700), (left.value + 1, 700), (left.value, 1100), (0, 700)):
        assert merge(splits, most) != 0 and "splits" in L.dh_last_error().decode()
    assert merge(left.value, 700) == 0 and L.dh_sync() == 0


def test_a_workspace_on_any_float(L):
    """Splits in a workspace that begins on a multiple of four bytes: the bits of one on a multiple of sixteen, and with a product behind a launch merges them."""
    outs = []
    for off in (0, 4, 8, 12):
        a = Attn(L, 4, 2, 64, 48, 0, n=700, seed=9)
        src, ws = a.rows(), torch.zeros(a.ws.numel() + 16, dtype=torch.uint8, device="cuda")
        capi.check(L.dh_attn_spec_kv_write(ctypes.byref(a.spec), src.data_ptr(), a.kc.data_ptr(), a.vc.data_ptr(), 700, 0))
        for p in (130, 699):
            step, left = (ctypes.byref(a.spec), src.data_ptr() + 4 * a.ld * p, a.kc.data_ptr(), a.vc.data_ptr()), ctypes.c_int(-1)
            for rows in (0, 64):
                out = torch.zeros(4 * 48, device="cuda")
                torch.cuda.synchronize()
                if rows and off:
                    capi.check(L.dh_attn_spec_decode_for(*step, out.data_ptr(), p, None, 700, ws.data_ptr() + off, rows, ctypes.byref(left)))
                    assert left.value == 0
                else:
                    capi.check(L.dh_attn_spec_decode(*step, out.data_ptr(), p, None, 700, ws.data_ptr() + off))
                capi.check(L.dh_sync())
                outs.append((p, out))
    assert all(torch.equal(o, next(x for q, x in outs if q == p)) for p, o in outs)


def test_shared_key_rows_four_gigabytes_apart(L):
    """Row strides whose bytes no longer fit 32 bits: the bits of rows beside one another."""
    H, D, S, VD, T, far = 2, 8, 8, 8, 2, 1 << 30
    g = torch.Generator(device="cuda").manual_seed(5)
    ld = H * (D + S) + 16
    qkv, kc, vc, ks = (torch.randn(T, n, generator=g, device="cuda") for n in (ld, D, VD, S))
    spec = capi.AttnSpec(H, 1, D, VD, VD, 0, capi.F32, 0, H * (D + S), H * (D + S) + 8, -1, ld, D ** -0.5, 1e-5, None, None)
    apart, outs = torch.empty(far + S, device="cuda"), []
    apart[:S], apart[far:] = ks[0], ks[1]
    for rows, stride in ((ks, S), (apart, far)):
        o = torch.zeros(T, H * VD, device="cuda")
        torch.cuda.synchronize()
        capi.check(L.dh_attn_spec_prefill_shared(ctypes.byref(spec), qkv.data_ptr(), kc.data_ptr(), rows.data_ptr(), S, stride, vc.data_ptr(), o.data_ptr(),
                                                 capi.F32, H * VD, T, 0))
        capi.check(L.dh_sync())
        outs.append(o)
    assert outs[0].abs().sum() > 0 and torch.equal(*outs)


def test_prefill_output_in_bf16(L):
    a = Attn(L, 6, 2, 24, 40, 30, "f16", n=70, seed=13)
    f = a.run([70])
    b = Attn(L, 6, 2, 24, 40, 30, "f16", n=70, seed=13)
    assert np.array_equal(b.run([70], out="bf16"), zm.bf16(f))


def test_bad_specs_are_refused(L):
    a = Attn(L, 4, 2, 64, 64, 10, n=20)
    rows = a.rows()
    for field, value, message in (("H", 5, "multiple"), ("D", 12, "multiples of 8"), ("VD", 520, "up to 512"), ("window", -1, "window"),
                                  ("cache_dtype", capi.BF16, "caches"), ("ld_qkv", 64, "does not hold"), ("value_dim", 65, "value_dim"),
                                  ("d_bias_r2", None, "both")):
        spec = capi.AttnSpec.from_buffer_copy(a.spec)
        setattr(spec, field, value)
        assert L.dh_attn_spec_kv_write(ctypes.byref(spec), rows.data_ptr(), a.kc.data_ptr(), a.vc.data_ptr(), 2, 0) != 0
        assert message in L.dh_last_error().decode(), (field, L.dh_last_error())
    assert L.dh_dense_matmul(rows.data_ptr(), 7, 64, rows.data_ptr(), 64, 1, 8, 64, 1.0, None, None, rows.data_ptr(), 8, 8, None, 0, 0, -1) != 0
    assert L.dh_dense_gemv(rows.data_ptr(), None, 0, 0.0, rows.data_ptr(), 100, 8, 100, 1.0, None, None, rows.data_ptr(), 8, None, -1) != 0


# ------------------------------------------------------------------ whole models

@pytest.fixture(scope="module")
def folders(tmp_path_factory):
    base = tmp_path_factory.mktemp("zepavik")
    out = {}
    for name, cfg, seed in (("mixed", zm.MIXED, 21), ("wide-heads", zm.WIDE_HEADS, 22), ("even", zm.EVEN, 23), ("odd", zm.ODD, 24)):
        t = zm.tensors(cfg, seed)
        out[name] = (zm.write(base / name, cfg, t), cfg, t)
    return out


def feed_all(dec, tokens, portions):
    dec.reset()
    out, at = [], 0
    for n in portions:
        part = tokens[at:at + n]
        out.append(dec.feed(part, list(range(len(part)))))
        at += n
    assert at >= len(tokens)
    return np.concatenate(out)


@pytest.mark.parametrize("dtype,tol", [("float32", F32_ROW), ("bfloat16", BF16_ROW)])
@pytest.mark.parametrize("name", ["mixed", "wide-heads", "even", "odd"])
def test_logits_whole_decoded_and_in_portions(folders, name, dtype, tol):
    folder, cfg, t = folders[name]
    toks = zm.prompt(cfg, 180, 31)
    want = plain.forward(cfg, t, toks)
    dec = models.load(folder, 200, dtype)
    for portions in ([180], [1] * 180, [2] * 90, [3, 1, 62, 2, 1, 1, 64, 33, 13], [65, 115]):
        err = zm.row_errors(feed_all(dec, toks, portions), want)
        assert err.max() < tol, (portions[:4], int(err.argmax()), err.max())
    # one prompt in chunks of the batched path's own
    dec.reset()
    assert zm.row_errors(dec.prefill(toks, chunk=50, want=[0, 49, 50, 179]), want[[0, 49, 50, 179]]).max() < tol


def test_layers_of_the_residual_stream(folders, tmp_path):
    """Models cut after every layer: the stream itself, read from the step's residual row."""
    _, cfg, t = folders["mixed"]
    toks = zm.prompt(cfg, 40, 32)
    _, streams = plain.forward(cfg, t, toks, want_layers=True)
    for n in range(1, len(cfg["layers"]) + 1):
        dec = models.load(zm.write(tmp_path / str(n), dict(cfg, layers=cfg["layers"][:n]), t), 64, "float32")
        dec.prefill(toks[:-1])
        dec.step(toks[-1], 39)
        assert rel(host(dec.x)[:cfg["width"]], streams[n - 1, -1]) < 1e-5, n


@pytest.mark.parametrize("dtype,tol", [("float32", F32_ROW), ("bfloat16", BF16_ROW)])
def test_unequal_sequences_one_after_another_reuse_the_cache(folders, dtype, tol):
    """Long, short, long again: rows an earlier sequence left behind must not be seen, nor its last token."""
    folder, cfg, t = folders["mixed"]
    dec = models.load(folder, 160, dtype)
    for i, n in enumerate((150, 1, 2, 70, 9, 160)):
        toks = zm.prompt(cfg, n, 40 + i)
        want = plain.forward(cfg, t, toks)
        cut = n // 2
        assert zm.row_errors(feed_all(dec, toks, [cut, n - cut] if cut else [n]), want).max() < tol, n


def test_long_decoding_passes_every_window(folders):
    folder, cfg, t = folders["mixed"]
    toks = zm.prompt(cfg, 390, 51)
    want = plain.forward(cfg, t, toks)
    dec = models.load(folder, 400, "float32")
    got = feed_all(dec, toks, [20] + [1] * 370)
    assert zm.row_errors(got, want).max() < F32_ROW
    with pytest.raises(ValueError, match="max_seq"):
        feed_all(dec, toks + [1] * 11, [390, 11])


def test_the_caches_hold_what_the_equations_say(folders):
    folder, cfg, t = folders["wide-heads"]
    toks = zm.prompt(cfg, 30, 52)
    dec = models.load(folder, 40, "float32")
    feed_all(dec, toks, [20] + [1] * 10)
    m, eps = cfg["layers"][0]["mixer"], cfg["norm"]["eps"]
    h = plain.rms_norm(plain.embed(cfg, t, toks), eps, t["l0.norm1"])
    k, v = dec.read_kv(0, 30)
    want_k = (h @ t["l0.mix.k"].T + t["l0.mix.k.b"]).reshape(30, m["kv_heads"], m["dim"])
    want_v = plain.rms_norm((h @ t["l0.mix.v"].T + t["l0.mix.v.b"]).reshape(30, m["kv_heads"], m["vdim"]), eps)
    assert rel(k[:, :, :m["dim"]], want_k) < 1e-5 and rel(v[:, :, :m["vdim"]], want_v) < 1e-5


def test_widths_beyond_the_single_row_kernel(tmp_path):
    """Rows longer than the decode GEMV holds take the matrix-core path for single tokens too."""
    cfg = zm.config(33000, 40, [zm.layer(2, 1, 8, 8, 3, ff=24)], max_positions=12, buckets=5)
    t = zm.tensors(cfg, 61)
    toks = zm.prompt(cfg, 10, 62)
    want = plain.forward(cfg, t, toks)
    dec = models.load(zm.write(tmp_path, cfg, t), 12, "float32")
    assert zm.row_errors(feed_all(dec, toks, [4, 1, 1, 2, 1, 1]), want).max() < 1e-4
    dec.prefill(toks[:6])
    assert dec.step(toks[6], 6) == int(want[6].argmax())


# ------------------------------------------------------------------ generation

def test_greedy_generation_every_way(folders):
    """The framework's own loops: generate, blocking steps, staged readback, batched submits, the captured step."""
    folder, cfg, t = folders["even"]
    prompt = zm.prompt(cfg, 30, 71)
    n = 40
    want = plain.greedy(cfg, t, prompt, n)
    dec = models.load(folder, 120, "float32")
    assert isinstance(dec, decoder.DecoderBase)
    assert dec.generate(prompt, n) == want
    assert dec.generate(prompt, n, chunk=7) == want
    first = dec.prefill(prompt)
    assert [first] + dec.decode_greedy(first, 30, n - 1) == want
    dec.release_readback()
    first = dec.prefill(prompt)
    assert [first] + dec.decode_batch(first, 30, 20) + dec.decode_batch(want[20], 50, n - 21) == want
    # token by token from nothing, then the captured step replayed with eager work between replays
    out = [dec.step(tok, p) for p, tok in enumerate(prompt)][-1:]
    graph = [dec.step_graph(out[0], 30)]
    for i in range(1, n - 1):
        if i % 7 == 0:
            assert dec.step(graph[-1], 30 + i) == want[i + 1]
        graph.append(dec.step_graph(graph[-1], 30 + i))
    assert out + graph == want
    # a replay for another sequence, from its first position on
    other = zm.prompt(cfg, 9, 72)
    for p, tok in enumerate(other):
        g = dec.step_graph(tok, p)
    assert g == plain.greedy(cfg, t, other, 1)[0]
    dec.release_graph()
    with pytest.raises(ValueError, match="does not fit"):
        dec.generate(prompt, 120)


def test_generation_in_the_served_precision_and_sampling(folders):
    folder, cfg, t = folders["mixed"]
    prompt = zm.prompt(cfg, 25, 73)
    dec = models.load(folder, 80)
    assert dec.compute == "bf16"
    a = dec.generate(prompt, 30)
    seq = prompt + a
    logits = plain.forward(cfg, t, seq)
    # every greedy token is the plain model's best or within the precision's reach of it
    for i, tok in enumerate(a):
        row = logits[len(prompt) + i - 1]
        assert row.max() - row[tok] < 0.1 * row.std()
    s = dict(temperature=0.9, topK=12, seed=5)
    b = dec.generate(prompt, 30, sampling=s)
    assert b == dec.generate(prompt, 30, sampling=s) and b != dec.generate(prompt, 30, sampling=dict(s, seed=6))
    logits = plain.forward(cfg, t, prompt + b)
    for i, tok in enumerate(b):
        row = logits[len(prompt) + i - 1]
        assert (row > row[tok] + 0.1 * row.std()).sum() < 12


def test_finiteness_guard(folders, tmp_path):
    _, cfg, t = folders["even"]
    dec = models.load(zm.write(tmp_path / "a", cfg, t), 40, finiteness_guard=True)
    tok = dec.prefill(zm.prompt(cfg, 5, 74))
    dec.step(tok, 5)
    bad = dict(t)
    bad["l1.mlp.down"] = zm.bf16(t["l1.mlp.down"] * 1e8)
    dec = models.load(zm.write(tmp_path / "b", cfg, bad), 40, finiteness_guard=True)
    tok = dec.prefill(zm.prompt(cfg, 5, 74))
    with pytest.raises(decoder.FinitenessError, match="layer 1"):
        dec.step(tok, 5)


def test_command_line_generates(folders, capsys):
    folder, cfg, t = folders["even"]
    prompt = zm.prompt(cfg, 12, 75)
    assert generate.main(["--model", folder, "--dtype", "float32", "--prompt", ",".join(map(str, prompt)), "--max-tokens", "15"]) == 0
    out = json.loads(capsys.readouterr().out.strip().splitlines()[-1])
    assert out["prompt"] == prompt and out["tokens"] == plain.greedy(cfg, t, prompt, 15)


@pytest.mark.parametrize("dtype,tol", [("float32", F32_ROW), ("bfloat16", BF16_ROW)])
def test_trace_replay(folders, tmp_path, dtype, tol):
    folder, cfg, t = folders["mixed"]
    a, b = zm.prompt(cfg, 90, 81), zm.prompt(cfg, 33, 82)
    steps = [("a", a[:50], [0, 49], []), ("a", a[50:52], [], []), ("a", a[52:53], [0], []), ("a", a[53:], [36, 3], ["a"]), ("b", b[:1], [0], []),
             ("b", b[1:], [31], ["b"])]
    lines = [json.dumps({"step": i, "entries": [{"id": r, "tokens": toks, "want": w}], "end": end}) for i, (r, toks, w, end) in enumerate(steps)]
    r = subprocess.run([os.path.join(ROOT, "bin", "trace_run"), "--model", folder, "--dtype", dtype, "--out", str(tmp_path), "--max-tokens", "90"],
                       input="\n".join(lines) + "\n", capture_output=True, text=True, timeout=100)
    assert r.returncode == 0, r.stderr[-2000:]
    assert [l for l in r.stdout.splitlines() if l.startswith("done")] == ["done %d" % i for i in range(6)]
    assert not os.path.exists(str(tmp_path / "1.f32"))
    la, lb = plain.forward(cfg, t, a), plain.forward(cfg, t, b)
    for step, want in ((0, la[[0, 49]]), (2, la[[52]]), (3, la[[89, 56]]), (4, lb[[0]]), (5, lb[[32]])):
        got = np.fromfile(str(tmp_path / ("%d.f32" % step)), "<f4").reshape(-1, cfg["vocab"])
        assert zm.row_errors(got, want).max() < tol, step


def test_the_quantised_decoder_feeds_the_same_way():
    """feed() belongs to every decoder: portions and single steps of the Q4_K model give the logits of its steps."""
    cfg = dict(layers=2, hidden=256, inter=512, heads=4, kv_heads=2, head_dim=64, vocab=300, eps=1e-6, qk_norm=1, max_seq=40, theta=1e6)
    layers, embed, final_norm, cos, sin = decoder.random_model(cfg, seed=11, max_seq=40)
    dec = decoder.HipDecoder(cfg, layers, embed, final_norm, cos, sin, 40)
    toks = [int(v) for v in rng(3).integers(0, 300, 30)]
    want = []
    for p, tok in enumerate(toks):
        dec.step(tok, p, want_logits=True)
        want.append(dec.read_logits())
    got = feed_all(dec, toks, [17, 1, 1, 11])
    assert zm.row_errors(got, np.array(want, np.float64)).max() < 2e-2


def test_random_weights_make_a_model():
    cfg = dict(hidden=128, vocab=90, eps=1e-5, logit_scale=1.0, max_positions=64, bigram=dict(buckets=7, mul_prev=3, mul_cur=5),
               layers=[dict(mixer=dict(heads=4, kv_heads=2, dim=32, vdim=32, window=16, scale=0.2, log_bias=True, value_norm=True, gate=True),
                            mlp=dict(ff=96, activation="relu2"))] * 2)
    w = dense_decoder.random_weights(cfg, seed=4)
    a = dense_decoder.DenseDecoder(cfg, w, 64, compute="f32").generate([1, 2, 3], 20)
    b = dense_decoder.DenseDecoder(cfg, w, 64, compute="f32").generate([1, 2, 3], 20, chunk=2)
    assert a == b and len(a) == 20
    with pytest.raises(ValueError, match="positions"):
        dense_decoder.DenseDecoder(cfg, w, 65)
