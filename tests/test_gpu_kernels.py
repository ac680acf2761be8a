"""Parity of the gfx950 kernels with the CPU oracle, called through the C ABI
(include/gehtp_kernels.h) on device buffers. Inputs are the seeded BASELINE shapes."""
from __future__ import annotations

import ctypes as C
import math

import numpy as np
import pytest

from helpers import (assert_close, from_dev, normal_f16, ptr, stream_ptr, to_dev, w4g_weights)

pytestmark = pytest.mark.gpu


def _sync():
    import torch
    torch.cuda.synchronize()


def _w4g(lib, dev, x, wq, ws, M, N, K, which="auto"):
    import torch
    xd, qd, sd = to_dev(x, dev), to_dev(wq, dev), to_dev(ws, dev)
    yd = torch.empty((M, N), dtype=torch.float16, device=dev)
    fn = {"auto": lib.gehtp_w4g_matmul, "gemv": lib.gehtp_w4g_gemv, "gemm": lib.gehtp_w4g_gemm}[which]
    rc = fn(ptr(xd), K, ptr(qd), ptr(sd), ptr(yd), N, M, N, K, stream_ptr())
    assert rc == 0, rc
    _sync()
    return from_dev(yd)


# ---------------------------------------------------------------- W4A16 ------
def test_w4g_dequant_bit_exact(lib, oracle, torch_dev):
    import torch
    rng = np.random.default_rng(7)
    N, K = 384, 1024
    q, wq, ws = w4g_weights(rng, N, K)
    # include extreme scales: subnormal products, large values
    ws[0, :] = np.float16(6e-5)
    ws[1, :] = np.float16(1000.0)
    ws[2, :] = np.float16(-0.0137)
    wd = torch.empty((N, K), dtype=torch.float16, device=torch_dev)
    assert lib.gehtp_w4g_dequant(ptr(to_dev(wq, torch_dev)), ptr(to_dev(ws, torch_dev)), ptr(wd), N, K,
                                 stream_ptr()) == 0
    _sync()
    got = from_dev(wd).view(np.uint16)
    ref = oracle.w4g_dequant(wq, ws, K).view(np.uint16)
    assert np.array_equal(got, ref)


@pytest.mark.parametrize("M", [1, 2, 3, 4])
def test_w4g_gemv_config1(lib, oracle, torch_dev, M):
    """Config 1: x [M,1024] ~N(0,1), W int4 [3072,1024] g64, scales U[0.005,0.02]."""
    rng = np.random.default_rng(100 + M)
    N, K = 3072, 1024
    _, wq, ws = w4g_weights(rng, N, K)
    x = normal_f16(rng, M, K)
    got = _w4g(lib, torch_dev, x, wq, ws, M, N, K, "gemv")
    ref = oracle.matmul_w4g(x, wq, ws, threads=8)
    assert_close(got, ref, what=f"gemv M={M}")


@pytest.mark.parametrize("N,K", [(2560, 2560), (4096, 2560), (9728, 2560), (2560, 9728), (1000, 192), (7, 64)])
def test_w4g_gemv_shapes(lib, oracle, torch_dev, N, K):
    rng = np.random.default_rng(N * 7 + K)
    _, wq, ws = w4g_weights(rng, N, K)
    x = normal_f16(rng, 1, K)
    got = _w4g(lib, torch_dev, x, wq, ws, 1, N, K, "gemv")
    ref = oracle.matmul_w4g(x, wq, ws, threads=8)
    assert_close(got, ref, what=f"gemv {N}x{K}")


@pytest.mark.parametrize("M", [1, 2, 4])
@pytest.mark.parametrize("N", [2000, 4000, 6144, 8000, 9728, 19456, 24000, 30000])
def test_w4g_gemv_pass_forms(lib, oracle, torch_dev, M, N):
    """K = 2560 (80 threads per row, 4 rows per pass, ~512 workgroups on 256 CUs): at M = 1
    N = 2000 / 4000 / 6144 / 8000 run 1 / 2 / 3 / 4 passes per thread in the straight-line
    form, N = 9728 / 19456 / 24000 the unrolled 8 / 10 / 12-pass batch schedules, N = 30000
    (15 passes, rounded to 16) the batch loop; M = 2 and 4 cap the passes by the partial-sum
    space (12 and 6, the latter run as 4). Each against the oracle, every shape with a last
    workgroup moved back to end at row N where N is not a multiple of its rows."""
    rng = np.random.default_rng(N + M)
    K = 2560
    _, wq, ws = w4g_weights(rng, N, K)
    x = normal_f16(rng, M, K)
    got = _w4g(lib, torch_dev, x, wq, ws, M, N, K, "gemv")
    ref = oracle.matmul_w4g(x, wq, ws, threads=8)
    assert_close(got, ref, what=f"gemv M={M} {N}x{K}")


@pytest.mark.parametrize("N,K", [(7, 192), (9, 64), (301, 576)])
def test_w4g_gemv_scales_off_word(lib, oracle, torch_dev, N, K):
    """A scale array starting 2 bytes past a 4-byte boundary with an odd number of scales
    (each scale is loaded as its own 16-bit value) gives the oracle's result."""
    import torch
    rng = np.random.default_rng(N * K)
    _, wq, ws = w4g_weights(rng, N, K)
    assert (N * (K // 64)) % 2 == 1
    x = normal_f16(rng, 1, K)
    buf = torch.zeros(ws.size + 2, dtype=torch.float16, device=torch_dev)
    buf[1:1 + ws.size] = torch.from_numpy(ws.reshape(-1)).to(torch_dev)
    sd = buf[1:]
    assert sd.data_ptr() % 4 == 2
    xd, qd = to_dev(x, torch_dev), to_dev(wq, torch_dev)
    yd = torch.empty((1, N), dtype=torch.float16, device=torch_dev)
    assert lib.gehtp_w4g_gemv(ptr(xd), K, ptr(qd), sd.data_ptr(), ptr(yd), N, 1, N, K, stream_ptr()) == 0
    _sync()
    assert_close(from_dev(yd), oracle.matmul_w4g(x, wq, ws, threads=8), what=f"gemv {N}x{K} scales at +2 bytes")


def test_w4g_gemm_config2(lib, oracle, torch_dev):
    """Config 2: RMSNorm(eps 1e-6, gamma U(0.8,1.2)) then W4A16 GEMM [512,1024] x [3072,1024]^T."""
    import torch
    rng = np.random.default_rng(2)
    M, N, K = 512, 3072, 1024
    x = normal_f16(rng, M, K)
    gamma = rng.uniform(0.8, 1.2, K).astype(np.float16)
    _, wq, ws = w4g_weights(rng, N, K)
    xd, gd = to_dev(x, torch_dev), to_dev(gamma, torch_dev)
    hd = torch.empty((M, K), dtype=torch.float16, device=torch_dev)
    assert lib.gehtp_rmsnorm2(ptr(xd), ptr(gd), None, ptr(hd), M, K, stream_ptr()) == 0
    _sync()
    h_ref = oracle.rmsnorm2(x, gamma)
    h_got = from_dev(hd)
    ulps = np.abs(h_got.view(np.int16).astype(np.int32) - h_ref.view(np.int16).astype(np.int32))
    assert ulps.max() <= 1, f"rmsnorm differs by {ulps.max()} ulp"
    got = _w4g(lib, torch_dev, h_ref, wq, ws, M, N, K, "gemm")
    ref = oracle.matmul_w4g(h_ref, wq, ws, threads=8)
    assert_close(got, ref, what="gemm config2")


@pytest.mark.parametrize("M,N,K", [(5, 384, 128), (200, 130, 192), (129, 257, 64), (2048, 256, 2560)])
def test_w4g_gemm_ragged(lib, oracle, torch_dev, M, N, K):
    rng = np.random.default_rng(M + N + K)
    _, wq, ws = w4g_weights(rng, N, K)
    x = normal_f16(rng, M, K)
    got = _w4g(lib, torch_dev, x, wq, ws, M, N, K, "gemm")
    ref = oracle.matmul_w4g(x, wq, ws, threads=8)
    assert_close(got, ref, what=f"gemm {M}x{N}x{K}")


@pytest.mark.parametrize("mode", [0, 1], ids=["plain", "swiglu"])
def test_w4g_gemm_wide_tile_ragged(lib, oracle, torch_dev, mode):
    """A grid large enough for the 128x256 tile, with a partial last row tile (M = 2000)
    and a last column tile partly past N (N = 16382): every row band equals, bit for bit,
    the same rows computed by a small call (which takes the 128x128 tile; both kernels
    share the K order and MFMA sequence), and a sample of rows matches the oracle."""
    import torch
    rng = np.random.default_rng(91 + mode)
    M, N, K = 2000, 16382, 256
    _, wq, ws = w4g_weights(rng, N, K)
    x = normal_f16(rng, M, K)
    n_out = N // 2 if mode else N
    xd, qd, sd = to_dev(x, torch_dev), to_dev(wq, torch_dev), to_dev(ws, torch_dev)
    y = torch.empty((M, n_out), dtype=torch.float16, device=torch_dev)
    assert lib.gehtp_w4g_fused(ptr(xd), K, ptr(qd), ptr(sd), ptr(y), n_out, M, N, K, None, None, n_out, mode,
                               stream_ptr()) == 0
    for r0, r1 in ((0, 128), (896, 1024), (1920, 2000)):
        ys = torch.empty((r1 - r0, n_out), dtype=torch.float16, device=torch_dev)
        assert lib.gehtp_w4g_fused(ptr(xd) + r0 * K * 2, K, ptr(qd), ptr(sd), ptr(ys), n_out, r1 - r0, N, K, None,
                                   None, n_out, mode, stream_ptr()) == 0
        _sync()
        assert np.array_equal(from_dev(y)[r0:r1].view(np.uint16), from_dev(ys).view(np.uint16)), (r0, r1)
    rows = np.r_[0:8, 1990:2000]
    acc = oracle.matmul_w4g(np.ascontiguousarray(x[rows]), wq, ws, threads=8)
    ref = oracle.binary(oracle.unary(acc[:, 0::2].copy(), 12), acc[:, 1::2].copy(), 2) if mode else acc
    assert_close(from_dev(y)[rows], ref, what=f"wide tile mode={mode}")


def test_w4g_gemv_equals_gemm_small_m(lib, torch_dev):
    """The two implementations agree to two fp16 ulps (4e-3 absolute near zero): both round
    each dequantized weight to fp16 (the reference's fp16(q*s)) and accumulate in fp32,
    in different orders, and each result is rounded to fp16 once."""
    rng = np.random.default_rng(11)
    N, K = 1536, 2560
    _, wq, ws = w4g_weights(rng, N, K)
    x = normal_f16(rng, 4, K)
    a = _w4g(lib, torch_dev, x, wq, ws, 4, N, K, "gemv")
    b = _w4g(lib, torch_dev, x, wq, ws, 4, N, K, "gemm")
    assert_close(a, b, min_cos=0.99999, what="gemv vs gemm")
    ulp = np.spacing(np.maximum(np.abs(a), np.abs(b)).astype(np.float16)).astype(np.float32)
    assert (np.abs(a - b) <= np.maximum(2 * ulp, 4e-3)).all(), "gemv and gemm differ by more than 2 ulps"


# ---------------------------------------------------------------- rows -------
@pytest.mark.parametrize("rows,rw", [(512, 1024), (1, 2560), (4096, 128), (3, 100), (5, 8192), (2, 9728),
                                     (7, 1536), (9, 24)])
def test_rmsnorm2(lib, oracle, torch_dev, rows, rw):
    import torch
    rng = np.random.default_rng(rows + rw)
    x = normal_f16(rng, rows, rw)
    x[0, :] = 0   # zero row
    gamma = rng.uniform(0.8, 1.2, rw).astype(np.float16)
    beta = (rng.standard_normal(rw) * 0.1).astype(np.float16)
    for b in (None, beta):
        y = torch.empty((rows, rw), dtype=torch.float16, device=torch_dev)
        assert lib.gehtp_rmsnorm2(ptr(to_dev(x, torch_dev)), ptr(to_dev(gamma, torch_dev)),
                                  ptr(to_dev(b, torch_dev)) if b is not None else None, ptr(y),
                                  rows, rw, stream_ptr()) == 0
        _sync()
        ref = oracle.rmsnorm2(x, gamma, b)
        got = from_dev(y)
        d = np.abs(got.view(np.int16).astype(np.int32) - ref.view(np.int16).astype(np.int32))
        assert d.max() <= 1, f"rmsnorm max ulp diff {d.max()}"
        assert (d == 0).mean() > 0.999


@pytest.mark.parametrize("rows,n", [(64, 1024), (16, 100), (3, 4096)])
def test_softmax(lib, oracle, torch_dev, rows, n):
    import torch
    rng = np.random.default_rng(n)
    x = (rng.standard_normal((rows, n)) * 3).astype(np.float16)
    y = torch.empty((rows, n), dtype=torch.float16, device=torch_dev)
    assert lib.gehtp_softmax(ptr(to_dev(x, torch_dev)), ptr(y), rows, n, stream_ptr()) == 0
    _sync()
    ref = oracle.softmax(x, rows, n)
    assert_close(from_dev(y), ref, max_abs=1e-3, what="softmax")


def test_argmax_first_max(lib, oracle, torch_dev):
    import torch
    rng = np.random.default_rng(5)
    n = 151936
    x = normal_f16(rng, n)
    x[[1000, 77777, 150000]] = np.float16(9.0)   # ties: first index wins
    x[5] = np.float16(-np.inf)
    out = torch.zeros(1, dtype=torch.int32, device=torch_dev)
    assert lib.gehtp_argmax(ptr(to_dev(x, torch_dev)), n, ptr(out), stream_ptr()) == 0
    _sync()
    assert int(out.item()) == oracle.argmax(x) == 1000
    allneg = np.full(300, -np.inf, np.float16)
    assert lib.gehtp_argmax(ptr(to_dev(allneg, torch_dev)), 300, ptr(out), stream_ptr()) == 0
    _sync()
    assert int(out.item()) == oracle.argmax(allneg) == 0
    # ragged length (tail past the 8-wide loads) and a 2-byte-aligned start
    tail = normal_f16(rng, 1004)
    tail[1002] = np.float16(20.0)
    xd = to_dev(tail, torch_dev)
    for off, n2 in ((0, 1003), (1, 1003)):
        assert lib.gehtp_argmax(ptr(xd) + 2 * off, n2, ptr(out), stream_ptr()) == 0
        _sync()
        assert int(out.item()) == oracle.argmax(tail[off:off + n2]) == 1002 - off
    # several load batches per thread (20 x 1024 16-byte chunks each); ties across batches
    big = normal_f16(rng, 400003)
    big[[170001, 390000, 400002]] = np.float16(11.0)
    assert lib.gehtp_argmax(ptr(to_dev(big, torch_dev)), big.size, ptr(out), stream_ptr()) == 0
    _sync()
    assert int(out.item()) == oracle.argmax(big) == 170001


def test_rope_bit_exact(lib, oracle, torch_dev):
    import torch
    rng = np.random.default_rng(9)
    n_tok, H, hd = 37, 4, 128
    x = normal_f16(rng, n_tok, H * hd)
    for pos0 in (0, 1000):
        y = torch.empty_like(to_dev(x, torch_dev))
        assert lib.gehtp_rope(ptr(to_dev(x, torch_dev)), ptr(y), n_tok, H, hd, pos0, 1e6, H * hd,
                              stream_ptr()) == 0
        _sync()
        ref = oracle.rope(x, H, hd, pos0, 1e6)
        got = from_dev(y)
        assert np.array_equal(got.view(np.uint16), ref.view(np.uint16))


def test_matmul_f16_flags(lib, oracle, torch_dev):
    """OP_MATMUL_F16 layouts: plain, t0, t1, batched, SPLIT window; GEMV and GEMM sizes."""
    import torch
    rng = np.random.default_rng(21)
    for (M, K, N) in [(1, 256, 300), (3, 64, 130), (40, 96, 72), (128, 128, 128)]:
        for flags in (0, 1, 2, 3):
            a = normal_f16(rng, M * K)
            w = normal_f16(rng, K * N)
            y = torch.zeros(M * N, dtype=torch.float16, device=torch_dev)
            assert lib.gehtp_matmul_f16(ptr(to_dev(a, torch_dev)), ptr(to_dev(w, torch_dev)), ptr(y),
                                        M, K, N, 0, N, flags, stream_ptr()) == 0
            _sync()
            ref = oracle.matmul_f16(a, w, M, K, N, flags=flags)
            assert_close(from_dev(y), ref, max_abs=3e-2, what=f"mm {M}x{K}x{N} f{flags}")
    # batched (Bn=4), t1 (q . k^T form)
    Bn, M, K, N = 4, 33, 128, 70
    a = normal_f16(rng, Bn * M * K)
    w = normal_f16(rng, Bn * N * K)
    flags = (Bn << 16) | 4 | 2
    y = torch.zeros(Bn * M * N, dtype=torch.float16, device=torch_dev)
    assert lib.gehtp_matmul_f16(ptr(to_dev(a, torch_dev)), ptr(to_dev(w, torch_dev)), ptr(y), M, K, N, 0, N,
                                flags, stream_ptr()) == 0
    _sync()
    assert_close(from_dev(y), oracle.matmul_f16(a, w, M, K, N, flags=flags), max_abs=3e-2, what="batched")
    # SPLIT window: columns [64, 128) of N_full = 192 only
    M, K, Nf = 8, 64, 192
    a = normal_f16(rng, M * K)
    w = normal_f16(rng, Nf * K)
    y = torch.zeros(M * Nf, dtype=torch.float16, device=torch_dev)
    assert lib.gehtp_matmul_f16(ptr(to_dev(a, torch_dev)), ptr(to_dev(w, torch_dev)), ptr(y), M, K, Nf, 64, 64,
                                2, stream_ptr()) == 0
    _sync()
    got = from_dev(y).reshape(M, Nf)
    ref = oracle.matmul_f16(a, w, M, K, Nf, 64, 64, 2).reshape(M, Nf)
    assert np.all(got[:, :64] == 0) and np.all(got[:, 128:] == 0)
    assert_close(got[:, 64:128], ref[:, 64:128], max_abs=3e-2, what="split")


@pytest.mark.parametrize("K,N,n0", [(2560, 4099, 0), (1024, 3000, 0), (4096, 777, 0), (512, 96, 32)])
def test_matmul_f16_gemv_m1_prefetch_form(lib, oracle, torch_dev, K, N, n0):
    """M = 1, w stored [N, K], K a multiple of 512 (the lm_head): the GEMV form that
    requests all of a wave's weight rows before computing. Its output equals row 0 of the
    M = 2 form (the same per-lane order and wave reduction) bit for bit, and the oracle
    within fp16 tolerance; with a SPLIT window only columns [n0, n0 + N) are written."""
    import torch
    rng = np.random.default_rng(K + N)
    Nf = n0 + N + (16 if n0 else 0)
    a = normal_f16(rng, K)
    w = normal_f16(rng, Nf * K) * np.float16(0.25)
    y1 = torch.zeros(Nf, dtype=torch.float16, device=torch_dev)
    y2 = torch.zeros(2 * Nf, dtype=torch.float16, device=torch_dev)
    ad, wd = to_dev(a, torch_dev), to_dev(np.concatenate([a, a]), torch_dev)
    wdev = to_dev(w, torch_dev)
    assert lib.gehtp_matmul_f16(ptr(ad), ptr(wdev), ptr(y1), 1, K, Nf, n0, N, 2, stream_ptr()) == 0
    assert lib.gehtp_matmul_f16(ptr(wd), ptr(wdev), ptr(y2), 2, K, Nf, n0, N, 2, stream_ptr()) == 0
    _sync()
    got, two = from_dev(y1), from_dev(y2).reshape(2, Nf)
    assert np.array_equal(got.view(np.uint16), two[0].view(np.uint16))
    assert np.all(got[:n0] == 0) and np.all(got[n0 + N:] == 0)
    ref = oracle.matmul_f16(a, w, 1, K, Nf, n0, N, 2)
    assert_close(got[n0:n0 + N], ref[n0:n0 + N], max_abs=3e-2, what=f"gemv m1 {K}x{N}")


# ---------------------------------------------------------------- attention --
SCALE = float(np.float16(1.0 / math.sqrt(128)))


@pytest.mark.parametrize("S,H,KVH,causal", [(1024, 16, 8, True), (200, 4, 2, True), (130, 8, 8, False),
                                            (1, 2, 1, True)])
def test_attn_prefill(lib, oracle, torch_dev, S, H, KVH, causal):
    """Config 3 prefill: Q/K/V ~N(0,1), 16 Q / 8 KV heads, hd 128, scale 1/sqrt(128)."""
    import torch
    rng = np.random.default_rng(S + H)
    hd = 128
    q, k, v = normal_f16(rng, S, H, hd), normal_f16(rng, S, KVH, hd), normal_f16(rng, S, KVH, hd)
    out = torch.empty((S, H, hd), dtype=torch.float16, device=torch_dev)
    assert lib.gehtp_attn_prefill(ptr(to_dev(q, torch_dev)), ptr(to_dev(k, torch_dev)), ptr(to_dev(v, torch_dev)),
                                  ptr(out), S, H, KVH, hd, SCALE, int(causal), stream_ptr()) == 0
    _sync()
    ref = oracle.attn_prefill(q, k, v, SCALE, causal)
    got = from_dev(out)
    assert_close(got, ref, what=f"attn S={S}")
    if causal:   # query 0 sees only key 0: the output is V[0] exactly
        rep = H // KVH
        for h in range(H):
            assert np.array_equal(got[0, h], v[0, h // rep])


@pytest.mark.parametrize("ramp", [0.0, 4.0])
def test_attn_prefill_wide_ragged(lib, oracle, torch_dev, ramp):
    """The 128-query tiles (32 heads x 8 tiles cover the 256 CUs) at S = 1000: the last key
    stage holds 40 keys, read as zero rows past S by the kernel's buffer loads and masked.
    With ramp > 0 the keys are scaled by 1 + ramp * j / S, so later stages hold larger
    scores: at ramp 4 the lazily kept reference max of about one row half in fourteen
    moves after its first stage (the scores of a later stage exceed it by more than 8 in
    log2 units), so O is rescaled mid-row there."""
    import torch
    rng = np.random.default_rng(77 + int(ramp * 10))
    S, H, KVH, hd = 1000, 32, 8, 128
    q, k, v = normal_f16(rng, S, H, hd), normal_f16(rng, S, KVH, hd), normal_f16(rng, S, KVH, hd)
    if ramp:
        k = (k.astype(np.float32) * (1.0 + ramp * np.arange(S, dtype=np.float32) / S)[:, None, None]).astype(np.float16)
    out = torch.empty((S, H, hd), dtype=torch.float16, device=torch_dev)
    assert lib.gehtp_attn_prefill(ptr(to_dev(q, torch_dev)), ptr(to_dev(k, torch_dev)), ptr(to_dev(v, torch_dev)),
                                  ptr(out), S, H, KVH, hd, SCALE, 1, stream_ptr()) == 0
    _sync()
    assert_close(from_dev(out), oracle.attn_prefill(q, k, v, SCALE, True, threads=8),
                 what=f"attn S={S} ramp={ramp}")


@pytest.mark.parametrize("causal", [False, True])
def test_attn_prefill_tile_sizes(lib, oracle, torch_dev, causal):
    """The prefill runs 128-, 64- or 32-query tiles by their modelled cost (past 512 tokens
    also with four key parts). On 256 CUs at S = 512, 64 heads take the 128-query tiles, their first 32 heads (over the
    first 4 KV heads, the same grouping) the 64-query ones and their first 16 the
    32-query ones. Every query sums the same key stages in the same order each time
    (with the mask too: a tile's two halves split its stages where the enclosing larger
    tile's do, the larger tile's extra stage being wholly masked for the queries before
    it), so the outputs are bit-identical; they match the oracle."""
    import torch
    rng = np.random.default_rng(11 + causal)
    S, hd = 512, 128
    q, k, v = normal_f16(rng, S, 64, hd), normal_f16(rng, S, 8, hd), normal_f16(rng, S, 8, hd)
    outs = {}
    for H, KVH in ((64, 8), (32, 4), (16, 2)):
        qs, ks, vs = (np.ascontiguousarray(t[:, :n]) for t, n in ((q, H), (k, KVH), (v, KVH)))
        out = torch.empty((S, H, hd), dtype=torch.float16, device=torch_dev)
        assert lib.gehtp_attn_prefill(ptr(to_dev(qs, torch_dev)), ptr(to_dev(ks, torch_dev)),
                                      ptr(to_dev(vs, torch_dev)), ptr(out), S, H, KVH, hd, SCALE, int(causal),
                                      stream_ptr()) == 0
        _sync()
        outs[H] = from_dev(out)
    big, mid, small = outs[64][:, :16], outs[32][:, :16], outs[16]
    assert np.array_equal(big.view(np.uint16), small.view(np.uint16))
    assert np.array_equal(mid.view(np.uint16), small.view(np.uint16))
    ref = oracle.attn_prefill(np.ascontiguousarray(q[:, :16]), np.ascontiguousarray(k[:, :2]),
                              np.ascontiguousarray(v[:, :2]), SCALE, causal)
    assert_close(small, ref, what=f"32-query tiles causal={causal}")
    assert_close(big, ref, what=f"128-query tiles causal={causal}")


@pytest.mark.parametrize("S,H,causal", [(513, 8, True), (600, 16, True), (577, 8, False), (700, 16, False), (641, 48, True),
                                        (769, 32, False), (700, 16, True), (1001, 16, True), (768, 24, True)])
def test_attn_prefill_four_parts(lib, oracle, torch_dev, S, H, causal):
    """Past 512 tokens, grids of up to one workgroup per CU split a tile's key stages over
    four parts (32-query tiles at 8 heads; 64-query ones at 16 heads and 700 or 1001 tokens,
    causal with a partial last key stage and query tile; 9 stages of 513..576 tokens leave the
    last part empty, and one key in the last stage at 513, 577); larger grids (48 heads, 24
    at 768 tokens, 32 without a mask) and 600 tokens of 16 heads take two parts. Keys grow
    along S, so that late stages move the reference max and the parts' maxima differ."""
    import torch
    rng = np.random.default_rng(S)
    KVH, hd = 8, 128
    q, k, v = normal_f16(rng, S, H, hd), normal_f16(rng, S, KVH, hd), normal_f16(rng, S, KVH, hd)
    k = (k.astype(np.float32) * (1.0 + 3.0 * np.arange(S, dtype=np.float32) / S)[:, None, None]).astype(np.float16)
    out = torch.full((S + 1, H, hd), 7.0, dtype=torch.float16, device=torch_dev)
    assert lib.gehtp_attn_prefill(ptr(to_dev(q, torch_dev)), ptr(to_dev(k, torch_dev)), ptr(to_dev(v, torch_dev)),
                                  ptr(out), S, H, KVH, hd, SCALE, int(causal), stream_ptr()) == 0
    _sync()
    got = from_dev(out)
    assert_close(got[:S], oracle.attn_prefill(q, k, v, SCALE, causal, threads=8), what=f"attn S={S} H={H}")
    assert (got[S] == 7.0).all()   # nothing written past the last query


@pytest.mark.parametrize("n_kv,H,KVH", [(4096, 16, 8), (77, 32, 8), (1, 16, 8)])
def test_attn_decode(lib, oracle, torch_dev, n_kv, H, KVH):
    """Config 3 decode: batch 1 over a KV cache of n_kv tokens in the reference ring layout."""
    import torch
    rng = np.random.default_rng(n_kv + H)
    hd = 128
    kv_elems = KVH * hd
    state_bytes = 4096 * kv_elems * 4
    ring = oracle.KVRing(state_bytes, kv_elems)
    ks, vs = normal_f16(rng, n_kv, kv_elems), normal_f16(rng, n_kv, kv_elems)
    for t in range(n_kv):
        ring.append(ks[t], vs[t])
    q = normal_f16(rng, H, hd)
    ring_d = torch.zeros(state_bytes, dtype=torch.uint8, device=torch_dev)
    assert lib.gehtp_kv_append(ptr(ring_d), state_bytes, ptr(to_dev(ks, torch_dev)), ptr(to_dev(vs, torch_dev)),
                               kv_elems, n_kv, 0, stream_ptr()) == 0
    _sync()
    assert np.array_equal(ring_d.cpu().numpy(), ring.buf), "device ring differs from the reference ring"
    wf = lib.gehtp_attn_decode_work_floats(n_kv, H, hd)
    work = torch.zeros(wf, dtype=torch.float32, device=torch_dev)
    out = torch.empty((H, hd), dtype=torch.float16, device=torch_dev)
    assert lib.gehtp_attn_decode(ptr(to_dev(q, torch_dev)), ptr(ring_d), state_bytes, ptr(out), n_kv, H, KVH, hd,
                                 SCALE, ptr(work), wf, stream_ptr()) == 0
    _sync()
    ref = ring.attn_decode(q, n_kv, H, KVH, hd, SCALE)
    assert_close(from_dev(out), ref, what=f"decode n_kv={n_kv}")


@pytest.mark.parametrize("n_kv,H", [(4096 + 1, 16), (4096 + 64 * 9, 8), (8192, 32), (8192 + 64 * 7 + 5, 16), (12300, 16)])
def test_attn_decode_merge_rounds(lib, oracle, torch_dev, n_kv, H):
    """The merge takes a head's chunks of 64 keys in rounds of 64 (8 thread groups x 8
    records): contexts that end one key, nine chunks or 7 chunks and 5 keys into a round, or
    on its edge. Keys grow along the context, so that later rounds move the maximum."""
    import torch
    rng = np.random.default_rng(n_kv)
    KVH, hd = 8, 128
    kv_elems = KVH * hd
    state_bytes = n_kv * kv_elems * 4
    ring = oracle.KVRing(state_bytes, kv_elems)
    ks, vs = normal_f16(rng, n_kv, kv_elems), normal_f16(rng, n_kv, kv_elems)
    ks = (ks.astype(np.float32) * (1.0 + np.arange(n_kv, dtype=np.float32) / n_kv)[:, None]).astype(np.float16)
    for t in range(n_kv):
        ring.append(ks[t], vs[t])
    q = normal_f16(rng, H, hd)
    ring_d = torch.zeros(state_bytes, dtype=torch.uint8, device=torch_dev)
    assert lib.gehtp_kv_append(ptr(ring_d), state_bytes, ptr(to_dev(ks, torch_dev)), ptr(to_dev(vs, torch_dev)),
                               kv_elems, n_kv, 0, stream_ptr()) == 0
    wf = lib.gehtp_attn_decode_work_floats(n_kv, H, hd)
    work = torch.zeros(wf, dtype=torch.float32, device=torch_dev)
    out = torch.empty((H, hd), dtype=torch.float16, device=torch_dev)
    assert lib.gehtp_attn_decode(ptr(to_dev(q, torch_dev)), ptr(ring_d), state_bytes, ptr(out), n_kv, H, KVH, hd,
                                 SCALE, ptr(work), wf, stream_ptr()) == 0
    _sync()
    assert_close(from_dev(out), ring.attn_decode(q, n_kv, H, KVH, hd, SCALE), what=f"decode n_kv={n_kv}")


def test_decode_matches_prefill_last_row(lib, torch_dev):
    """Decode of token t over keys [0, t] equals row t of the causal prefill (reference's
    decode==prefill gate, scripts/judge_logits.py: cos >= 0.9999)."""
    import torch
    rng = np.random.default_rng(3)
    S, H, KVH, hd = 300, 16, 8, 128
    q, k, v = normal_f16(rng, S, H, hd), normal_f16(rng, S, KVH, hd), normal_f16(rng, S, KVH, hd)
    out = torch.empty((S, H, hd), dtype=torch.float16, device=torch_dev)
    assert lib.gehtp_attn_prefill(ptr(to_dev(q, torch_dev)), ptr(to_dev(k, torch_dev)), ptr(to_dev(v, torch_dev)),
                                  ptr(out), S, H, KVH, hd, SCALE, 1, stream_ptr()) == 0
    state_bytes = 512 * KVH * hd * 4
    ring_d = torch.zeros(state_bytes, dtype=torch.uint8, device=torch_dev)
    assert lib.gehtp_kv_append(ptr(ring_d), state_bytes, ptr(to_dev(k.reshape(S, -1), torch_dev)),
                               ptr(to_dev(v.reshape(S, -1), torch_dev)), KVH * hd, S, 0, stream_ptr()) == 0
    wf = lib.gehtp_attn_decode_work_floats(S, H, hd)
    work = torch.zeros(wf, dtype=torch.float32, device=torch_dev)
    dec = torch.empty((H, hd), dtype=torch.float16, device=torch_dev)
    qd = to_dev(q, torch_dev)
    assert lib.gehtp_attn_decode(ptr(qd[S - 1]), ptr(ring_d), state_bytes, ptr(dec), S, H, KVH, hd, SCALE,
                                 ptr(work), wf, stream_ptr()) == 0
    _sync()
    assert_close(from_dev(dec), from_dev(out)[S - 1], max_abs=4e-3, min_cos=0.99999, what="decode vs prefill")


# ---------------------------------------------------------------- fused ops --
@pytest.mark.parametrize("mode,use_norm,use_res", [(0, True, False), (0, False, True), (1, True, False),
                                                    (1, False, True)])
def test_w4g_fused_gemv(lib, oracle, torch_dev, mode, use_norm, use_res):
    """OP_W4G_FUSED_F16 GEMV = RMSNORM2 -> MATMUL_W4G (-> silu*up) (-> ADD), same roundings."""
    import torch
    rng = np.random.default_rng(31 + mode * 2 + use_norm)
    N, K = (2 * 1536 if mode else 2048), 2560
    _, wq, ws = w4g_weights(rng, N, K)
    x = normal_f16(rng, 1, K)
    gamma = rng.uniform(0.8, 1.2, K).astype(np.float16)
    n_out = N // 2 if mode else N
    res = normal_f16(rng, 1, n_out)
    y = torch.empty((1, n_out), dtype=torch.float16, device=torch_dev)
    rc = lib.gehtp_w4g_fused(ptr(to_dev(x, torch_dev)), K, ptr(to_dev(wq, torch_dev)), ptr(to_dev(ws, torch_dev)),
                             ptr(y), n_out, 1, N, K, ptr(to_dev(gamma, torch_dev)) if use_norm else None,
                             ptr(to_dev(res, torch_dev)) if use_res else None, n_out, mode, stream_ptr())
    assert rc == 0
    _sync()
    h = oracle.rmsnorm2(x, gamma, np.zeros(K, np.float16)) if use_norm else x
    acc = oracle.matmul_w4g(h, wq, ws, threads=8)
    ref = oracle.binary(oracle.unary(acc[:, 0::2], 12), acc[:, 1::2].copy(), 2) if mode else acc
    if use_res:
        ref = oracle.binary(ref, res, 0)
    assert_close(from_dev(y), ref, what=f"w4g_fused mode={mode} norm={use_norm} res={use_res}")


@pytest.mark.parametrize("K", [1024, 2048, 2560, 3072, 4096])
@pytest.mark.parametrize("N,mode,use_norm,use_res", [(6144, 0, True, False), (2562, 0, False, True),
                                                      (19456, 1, True, False), (1002, 1, True, True),
                                                      (14, 0, False, False), (26, 1, True, True)])
def test_w4g_gemv_row_in_wave(lib, oracle, torch_dev, K, N, mode, use_norm, use_res):
    """The M = 1 GEMV whose rows sit inside one wave: 16 lanes per row with 2 / 4 / 5 slices
    each (K = 1024 / 2048 / 2560) and 32 lanes with 3 / 4 (K = 3072 / 4096); RMSNorm,
    SwiGLU (the gate/up partner through a row swap) and residual epilogues; N = 2562 and
    1002 leave a last workgroup moved back to end at row N, N = 14 / 26 fit only small
    workgroups. Against the oracle's RMSNORM2 -> MATMUL_W4G (-> silu * up) (-> ADD). The
    activations are scaled (x by 1/4, gamma U[0.2, 0.3], both by sqrt(2560 / K) above K =
    2560) so that outputs stay below 16,
    where the 2e-2 bound is above the fp16 spacing that the summation order can move."""
    import torch
    rng = np.random.default_rng(K + 3 * N + mode)
    _, wq, ws = w4g_weights(rng, N, K)
    f = min(1.0, float(np.sqrt(2560.0 / K)))
    x = (normal_f16(rng, 1, K) * np.float16(0.25 * f)).astype(np.float16)
    gamma = (rng.uniform(0.2, 0.3, K) * f).astype(np.float16)
    n_out = N // 2 if mode else N
    res = normal_f16(rng, 1, n_out)
    y = torch.empty((1, n_out), dtype=torch.float16, device=torch_dev)
    rc = lib.gehtp_w4g_fused(ptr(to_dev(x, torch_dev)), K, ptr(to_dev(wq, torch_dev)), ptr(to_dev(ws, torch_dev)),
                             ptr(y), n_out, 1, N, K, ptr(to_dev(gamma, torch_dev)) if use_norm else None,
                             ptr(to_dev(res, torch_dev)) if use_res else None, n_out, mode, stream_ptr())
    assert rc == 0
    _sync()
    h = oracle.rmsnorm2(x, gamma, np.zeros(K, np.float16)) if use_norm else x
    acc = oracle.matmul_w4g(h, wq, ws, threads=8)
    ref = oracle.binary(oracle.unary(np.ascontiguousarray(acc[:, 0::2]), 12), np.ascontiguousarray(acc[:, 1::2]),
                        2) if mode else acc
    if use_res:
        ref = oracle.binary(ref, res, 0)
    assert np.abs(ref.astype(np.float32)).max() < 16.0
    assert_close(from_dev(y), ref, what=f"row-in-wave gemv K={K} N={N} mode={mode} norm={use_norm} res={use_res}")


@pytest.mark.parametrize("M,N,use_res", [(1, 40, True), (1, 100, False), (2, 702, True), (1, 30000, False)])
def test_w4g_fused_gemv_swiglu_odd_rows(lib, oracle, torch_dev, M, N, use_res):
    """SwiGLU GEMV at K = 704 (22 threads per row, 23 rows per pass of a 512-thread
    workgroup): a gate/up pair must not straddle workgroups, so the launcher makes each
    workgroup's row count even (two passes instead of one when 46 <= N: N = 100, 702; 22
    rows per pass when N < 46: N = 40; one pass fewer when the pass count is odd: N =
    30000, three passes -> two), and no workgroup may span more than N rows (the last one
    is moved back to end at row N). Against the oracle's MATMUL_W4G -> silu * up (-> ADD)."""
    import torch
    rng = np.random.default_rng(7 * N + M)
    K = 704
    _, wq, ws = w4g_weights(rng, N, K)
    x = normal_f16(rng, M, K)
    gamma = rng.uniform(0.8, 1.2, K).astype(np.float16)
    n_out = N // 2
    res = normal_f16(rng, M, n_out)
    y = torch.empty((M, n_out), dtype=torch.float16, device=torch_dev)
    rc = lib.gehtp_w4g_fused(ptr(to_dev(x, torch_dev)), K, ptr(to_dev(wq, torch_dev)), ptr(to_dev(ws, torch_dev)),
                             ptr(y), n_out, M, N, K, ptr(to_dev(gamma, torch_dev)),
                             ptr(to_dev(res, torch_dev)) if use_res else None, n_out, 1, stream_ptr())
    assert rc == 0
    _sync()
    acc = oracle.matmul_w4g(oracle.rmsnorm2(x, gamma, np.zeros(K, np.float16)), wq, ws, threads=8)
    ref = oracle.binary(oracle.unary(np.ascontiguousarray(acc[:, 0::2]), 12), np.ascontiguousarray(acc[:, 1::2]), 2)
    if use_res:
        ref = oracle.binary(ref, res, 0)
    assert_close(from_dev(y), ref, what=f"swiglu gemv K=704 M={M} N={N}")


def test_w4g_fused_gemm_epilogues(lib, oracle, torch_dev):
    """The GEMM path (M > 4) applies the same SwiGLU and residual epilogues."""
    import torch
    rng = np.random.default_rng(41)
    M, N, K = 96, 2 * 320, 512
    _, wq, ws = w4g_weights(rng, N, K)
    x = normal_f16(rng, M, K)
    res = normal_f16(rng, M, N // 2)
    y = torch.empty((M, N // 2), dtype=torch.float16, device=torch_dev)
    assert lib.gehtp_w4g_fused(ptr(to_dev(x, torch_dev)), K, ptr(to_dev(wq, torch_dev)), ptr(to_dev(ws, torch_dev)),
                               ptr(y), N // 2, M, N, K, None, ptr(to_dev(res, torch_dev)), N // 2, 1,
                               stream_ptr()) == 0
    _sync()
    acc = oracle.matmul_w4g(x, wq, ws, threads=8)
    ref = oracle.binary(oracle.binary(oracle.unary(acc[:, 0::2].copy(), 12), acc[:, 1::2].copy(), 2), res, 0)
    assert_close(from_dev(y), ref, what="gemm swiglu+res")


@pytest.mark.parametrize("K", [4160, 2624])
@pytest.mark.parametrize("mode,use_res,M,N", [(0, False, 384, 1280), (0, True, 200, 1280), (1, False, 384, 1280),
                                              (1, True, 131, 1280), (0, True, 77, 1276), (1, True, 45, 1284),
                                              (0, True, 640, 2560)])
def test_w4g_gemm_split_k(lib, oracle, torch_dev, mode, use_res, M, N, K):
    """Narrow N, long K: with a workspace the GEMM splits K (fp32 sums of each part, added
    in part order in a second pass through the same epilogue: 8 columns per thread when N
    and the output rows allow 16-byte access, else column pairs). K = 4160 (65 K steps)
    splits in three unequal parts: on the 128 x 256 tile for M = 640, N = 2560 (150
    workgroups of it, over half of 256 CUs), on the 128 x 128 kernel's shorter tiles for
    the smaller grids; K = 2624 (41 steps) in two on the 128 x 128 kernel. Checked against
    the oracle (the first 128 rows for M = 640) and against the one-pass GEMM (only the
    fp32 sum order differs: almost everywhere identical)."""
    import torch
    rng = np.random.default_rng(60 + 2 * mode + use_res + N + K)
    n_out = N // 2 if mode else N
    need = lib.gehtp_w4g_split_bytes(M, N, K)
    assert need == (3 if K // 64 >= 48 else 2) * M * N * 4
    assert lib.gehtp_w4g_split_bytes(2, N, K) == 0            # GEMV sizes never split
    assert lib.gehtp_w4g_split_bytes(M, 1 << 16, K) == 0       # enough tiles already
    _, wq, ws = w4g_weights(rng, N, K)
    # x / 4 keeps the 4160-term sums near unit size (as in the shorter-K tests), so a
    # rounding flip of a SwiGLU gate is not multiplied by a large up value
    x = normal_f16(rng, M, K) * np.float16(0.25)
    res = normal_f16(rng, M, n_out)
    xd, wqd, wsd = to_dev(x, torch_dev), to_dev(wq, torch_dev), to_dev(ws, torch_dev)
    rd = ptr(to_dev(res, torch_dev)) if use_res else None
    work = torch.empty(need // 4, dtype=torch.float32, device=torch_dev)
    y1 = torch.empty((M, n_out), dtype=torch.float16, device=torch_dev)
    y2 = torch.empty((M, n_out), dtype=torch.float16, device=torch_dev)
    assert lib.gehtp_w4g_fused_ws(ptr(xd), K, ptr(wqd), ptr(wsd), ptr(y1), n_out, M, N, K, None, rd, n_out, mode,
                                  ptr(work), need, stream_ptr()) == 0
    assert lib.gehtp_w4g_fused_ws(ptr(xd), K, ptr(wqd), ptr(wsd), ptr(y2), n_out, M, N, K, None, rd, n_out, mode,
                                  None, 0, stream_ptr()) == 0
    _sync()
    R = M if M <= 384 else 128
    acc = oracle.matmul_w4g(np.ascontiguousarray(x[:R]), wq, ws, threads=8)
    ref = oracle.binary(oracle.unary(acc[:, 0::2].copy(), 12), acc[:, 1::2].copy(), 2) if mode else acc
    if use_res:
        ref = oracle.binary(ref, np.ascontiguousarray(res[:R]), 0)
    a, b = from_dev(y1), from_dev(y2)
    assert_close(a[:R], ref, what=f"split-K gemm mode={mode} res={use_res}")
    # fp32 reordering over K = 4160 terms moves a sum by ~1e-5, which flips the fp16
    # rounding of a few outputs (and, where the residual cancels the product, shows as
    # that product's ulp on a small result): both stay within the parity bar.
    assert_close(b[:R], ref, what=f"one-pass gemm mode={mode} res={use_res}")
    assert np.abs(a.astype(np.float32) - b.astype(np.float32)).max() <= 2e-2
    assert (a == b).mean() > 0.99


@pytest.mark.parametrize("mode,use_res", [(0, False), (1, True)])
def test_w4g_gemm_tile_heights(lib, oracle, torch_dev, mode, use_res):
    """An unsplit GEMM whose grid of 128 x 128 tiles leaves CUs idle runs 64- or 32-row
    tiles (on 256 CUs, N = 3072, K = 1024: M = 2048 keeps 128 rows, M = 512, the single
    prefill GEMM shape of the benchmark's second config, takes 64, M = 40 takes 32 with a
    partial tile). Each output's K order and MFMA sequence do not depend on the tile
    height: the rows the three calls share are bit-identical, and M = 512 matches the
    oracle."""
    import torch
    rng = np.random.default_rng(70 + mode + use_res)
    N, K = 3072, 1024
    n_out = N // 2 if mode else N
    _, wq, ws = w4g_weights(rng, N, K)
    x = normal_f16(rng, 2048, K)
    res = normal_f16(rng, 2048, n_out)
    xd, wqd, wsd, resd = (to_dev(v, torch_dev) for v in (x, wq, ws, res))
    outs = {}
    for M in (2048, 512, 40):
        assert lib.gehtp_w4g_split_bytes(M, N, K) == 0
        y = torch.empty((M, n_out), dtype=torch.float16, device=torch_dev)
        assert lib.gehtp_w4g_fused_ws(ptr(xd), K, ptr(wqd), ptr(wsd), ptr(y), n_out, M, N, K, None,
                                      ptr(resd) if use_res else None, n_out, mode, None, 0, stream_ptr()) == 0
        _sync()
        outs[M] = from_dev(y)
    assert np.array_equal(outs[512].view(np.uint16), outs[2048][:512].view(np.uint16))
    assert np.array_equal(outs[40].view(np.uint16), outs[2048][:40].view(np.uint16))
    acc = oracle.matmul_w4g(x[:512], wq, ws, threads=8)
    ref = oracle.binary(oracle.unary(acc[:, 0::2].copy(), 12), acc[:, 1::2].copy(), 2) if mode else acc
    if use_res:
        ref = oracle.binary(ref, res[:512], 0)
    assert_close(outs[512], ref, what=f"64-row tile gemm mode={mode} res={use_res}")


@pytest.mark.parametrize("n_tok,H,KVH", [(1, 8, 2), (37, 8, 2), (130, 32, 8), (6, 16, 8), (3, 40, 24)])
def test_qk_rope_kv(lib, oracle, torch_dev, n_tok, H, KVH):
    """OP_QK_ROPE_KV_F16 = per-head RMSNORM2 (q_norm / k_norm), ROPE at the counter
    position, KV append into the reference ring layout; counter advances by n_tok.
    One token runs the one-workgroup kernel, more tokens the multi-token row kernel
    (partial last workgroup, 64 heads per token at most)."""
    import torch
    rng = np.random.default_rng(50 + n_tok)
    hd, pos0 = 128, 5
    nslots = 64 if pos0 + n_tok <= 64 else 256
    qkv = normal_f16(rng, n_tok, (H + 2 * KVH) * hd) * np.float16(3)
    qg = rng.uniform(0.8, 1.2, hd).astype(np.float16)
    kg = rng.uniform(0.8, 1.2, hd).astype(np.float16)
    state_bytes = nslots * KVH * hd * 4
    ring = torch.zeros(state_bytes, dtype=torch.uint8, device=torch_dev)
    count = torch.tensor([pos0], dtype=torch.int32, device=torch_dev)
    q_out = torch.empty((n_tok, H * hd), dtype=torch.float16, device=torch_dev)
    k_out = torch.empty((n_tok, KVH * hd), dtype=torch.float16, device=torch_dev)
    v_out = torch.empty((n_tok, KVH * hd), dtype=torch.float16, device=torch_dev)
    assert lib.gehtp_qk_rope_kv(ptr(to_dev(qkv, torch_dev)), n_tok, H, KVH, ptr(to_dev(qg, torch_dev)),
                                ptr(to_dev(kg, torch_dev)), 1e6, ptr(q_out), ptr(k_out), ptr(v_out), ptr(ring),
                                state_bytes, ptr(count), stream_ptr()) == 0
    _sync()
    assert int(count.item()) == pos0 + n_tok
    assert np.array_equal(from_dev(v_out), qkv[:, (H + KVH) * hd:])
    q = qkv[:, :H * hd]
    k = qkv[:, H * hd:(H + KVH) * hd]
    v = qkv[:, (H + KVH) * hd:]
    qn = oracle.rmsnorm2(q.reshape(-1, hd), qg, np.zeros(hd, np.float16)).reshape(n_tok, -1)
    kn = oracle.rmsnorm2(k.reshape(-1, hd), kg, np.zeros(hd, np.float16)).reshape(n_tok, -1)
    q_ref = oracle.rope(qn, H, hd, pos0, 1e6)
    k_ref = oracle.rope(kn, KVH, hd, pos0, 1e6)
    rq = np.abs(from_dev(q_out).view(np.int16).astype(np.int32) - q_ref.view(np.int16).astype(np.int32))
    assert rq.max() <= 1 and (rq == 0).mean() > 0.999     # RMSNorm's double sum order may flip 1 ulp
    ring_ref = oracle.KVRing(state_bytes, KVH * hd)
    for t in range(n_tok):
        ring_ref.append(from_dev(k_out)[t], v[t], pos0 + t)
    assert np.array_equal(ring.cpu().numpy(), ring_ref.buf)
    rk = np.abs(from_dev(k_out).view(np.int16).astype(np.int32) - k_ref.view(np.int16).astype(np.int32))
    assert rk.max() <= 1 and (rk == 0).mean() > 0.999


@pytest.mark.parametrize("H,KVH,pos0", [(32, 8, 100), (16, 8, 63), (8, 8, 0), (16, 2, 130),
                                        (16, 8, 4094), (32, 8, 4157), (8, 2, 8190)])   # second and third merge round
def test_attn_decode_qkv_matches_unfused(lib, oracle, torch_dev, H, KVH, pos0):
    """OP_ATTN_DECODE_QKV_F16 = OP_QK_ROPE_KV_F16 (one token) + OP_ATTN_DECODE_F16 at the
    advanced counter: same ring bytes, same counter and bit-identical outputs over three
    consecutive steps, and the attention output within the parity bar of the oracle."""
    import torch
    rng = np.random.default_rng(H * 1000 + KVH * 10 + pos0)
    hd, nslots = 128, 256 if pos0 < 250 else 12288
    kv_elems = KVH * hd
    state_bytes = nslots * kv_elems * 4
    ring_ref = oracle.KVRing(state_bytes, kv_elems)
    ks, vs = normal_f16(rng, max(pos0, 1), kv_elems), normal_f16(rng, max(pos0, 1), kv_elems)
    for t in range(pos0):
        ring_ref.append(ks[t], vs[t])
    ring_a = torch.from_numpy(ring_ref.buf.copy()).to(torch_dev)
    ring_b = ring_a.clone()
    count_a = torch.tensor([pos0], dtype=torch.int32, device=torch_dev)
    count_b = count_a.clone()
    wf = lib.gehtp_attn_decode_work_floats(nslots, H, hd)
    work_a = torch.zeros(wf, dtype=torch.float32, device=torch_dev)
    work_b = torch.zeros(wf, dtype=torch.float32, device=torch_dev)
    qg = to_dev(rng.uniform(0.8, 1.2, hd).astype(np.float16), torch_dev)
    kg = to_dev(rng.uniform(0.8, 1.2, hd).astype(np.float16), torch_dev)
    out_a = torch.empty((H, hd), dtype=torch.float16, device=torch_dev)
    out_b = torch.empty((H, hd), dtype=torch.float16, device=torch_dev)
    q_b = torch.empty((H, hd), dtype=torch.float16, device=torch_dev)
    for step in range(3):
        qkv = to_dev(normal_f16(rng, (H + 2 * KVH) * hd) * np.float16(3), torch_dev)
        assert lib.gehtp_attn_decode_qkv(ptr(qkv), H, KVH, ptr(qg), ptr(kg), 1e6, SCALE, ptr(ring_a), state_bytes,
                                         ptr(count_a), ptr(out_a), ptr(work_a), wf, stream_ptr()) == 0
        assert lib.gehtp_qk_rope_kv(ptr(qkv), 1, H, KVH, ptr(qg), ptr(kg), 1e6, ptr(q_b), None, None, ptr(ring_b),
                                    state_bytes, ptr(count_b), stream_ptr()) == 0
        n_kv = pos0 + step + 1
        assert lib.gehtp_attn_decode(ptr(q_b), ptr(ring_b), state_bytes, ptr(out_b), n_kv, H, KVH, hd, SCALE,
                                     ptr(work_b), wf, stream_ptr()) == 0
        _sync()
        assert int(count_a.item()) == int(count_b.item()) == n_kv
        assert torch.equal(ring_a, ring_b), f"step {step}: rings differ"
        assert np.array_equal(from_dev(out_a).view(np.int16), from_dev(out_b).view(np.int16)), f"step {step}"
    # the oracle over the final ring
    ring_chk = oracle.KVRing(state_bytes, kv_elems)
    ring_chk.buf[:] = ring_a.cpu().numpy()
    ring_chk.posmap[:n_kv] = np.arange(n_kv, dtype=np.uint32)
    ref = ring_chk.attn_decode(from_dev(q_b), n_kv, H, KVH, hd, SCALE)
    assert_close(from_dev(out_a), ref, what=f"decode_qkv H={H} KVH={KVH} n_kv={n_kv}")


@pytest.mark.parametrize("M,K,N,Bn", [(1, 1024, 48, 1), (2, 2050, 33, 1), (3, 700, 9, 1), (4, 2048, 8, 2), (1, 260, 8200, 1),
                                      (1, 3, 7, 1), (5, 7, 5, 1), (33, 128, 32, 1), (5, 641, 31, 1), (31, 1025, 45, 3),
                                      (64, 200, 1000, 8), (65, 1022, 4100, 1), (700, 131, 1300, 1), (1000, 64, 70, 40),
                                      (1030, 72, 8200, 1), (1030, 79, 8201, 1), (2050, 66, 4097, 2),
                                      # [K, N] GEMV of 1 or 2 rows: whole 8-row passes, then four, then the edge
                                      (1, 9728, 2560, 1), (2, 4096 + 2048 + 37, 72, 1), (1, 2048 + 1024 + 5, 8200, 1),
                                      # short K: one column per thread, and 64-square tiles in steps of 32
                                      (1, 1, 1, 1), (2, 13, 300, 1), (3, 5, 7, 1), (4, 24, 8193, 2), (1, 128, 131080, 1),
                                      (5, 32, 65, 1), (65, 31, 63, 3), (130, 9, 9, 1), (33, 33, 64, 1)])
def test_matmul_f16_tiles_and_edges(lib, torch_dev, M, K, N, Bn):
    """The tiles (32, 64 and 128 square by the grid's size; 16- and 32-column GEMV
    workgroups), their remainders in M, N and K, rows off every alignment, rows of fewer
    than 8 elements, every layout flag and a column window, against float32 products of the
    same values: the result rounds to fp16 once (2^-11), and fp32 sums of K products of
    values around 1/sqrt(K) are off by at most K 2^-24 of the sum of magnitudes. A NaN and an
    infinity in one row of A and one column of W reach that row and column alone."""
    import torch
    g = torch.Generator(device=torch_dev).manual_seed(M * 31 + K * 7 + N)
    for flags in (0, 1, 2, 3) if Bn == 1 else (4, 6):
        for n0, pad, off in ((0, 0, 0), (5, 9, 1)):   # a column window; operands starting 2 bytes off
            t0, t1, Nf = bool(flags & 1) and Bn == 1, bool(flags & 2), n0 + N + pad
            a = torch.randn((Bn, M, K), device=torch_dev, generator=g).half()
            w = (torch.randn((Bn, K, Nf), device=torch_dev, generator=g) * K ** -0.5).half()
            if M > 1:
                a[:, M // 2, K // 2] = float("nan")
                w[:, K - 1, n0 + N - 1] = float("inf")
            ab = torch.empty(a.numel() + off, dtype=torch.float16, device=torch_dev)
            wb = torch.empty(w.numel() + off, dtype=torch.float16, device=torch_dev)
            ab[off:] = (a.transpose(1, 2) if t0 else a).reshape(-1)
            wb[off:] = (w.transpose(1, 2) if t1 else w).reshape(-1)
            y = torch.full((Bn, M, Nf), 7.0, dtype=torch.float16, device=torch_dev)
            assert lib.gehtp_matmul_f16(ab.data_ptr() + 2 * off, wb.data_ptr() + 2 * off, ptr(y), M, K, Nf, n0, N,
                                        flags | (Bn << 16), stream_ptr()) == 0
            _sync()
            win, what = y[:, :, n0:n0 + N].double(), f"{M}x{K}x{N} b{Bn} f{flags} n0={n0}"
            assert (y[:, :, :n0] == 7).all() and (y[:, :, n0 + N:] == 7).all(), what
            ref = torch.stack([a[b].double() @ w[b, :, n0:n0 + N].double() for b in range(Bn)])
            mag = torch.stack([a[b].double().abs() @ w[b, :, n0:n0 + N].double().abs() for b in range(Bn)])
            ok = torch.isfinite(ref)
            assert torch.equal(torch.isnan(win), torch.isnan(ref)) and torch.equal(win[~ok & ~torch.isnan(ref)],
                                                                                   ref[~ok & ~torch.isnan(ref)]), what
            err = (win - ref)[ok].abs()
            assert (err <= ref[ok].abs() * 2 ** -11 + mag[ok] * K * 2 ** -24 + 2 ** -24).all(), (what, float(err.max()))


@pytest.mark.parametrize("M,N,K,mode,use_res,pad", [(5, 16, 64, 0, False, 0), (8, 1, 192, 0, True, 0), (9, 250, 576, 1, False, 8),
                                                    (16, 4112, 1024, 0, False, 0), (17, 6150, 2560, 1, True, 0),
                                                    (32, 12320, 128, 0, True, 8), (31, 20482, 448, 1, True, 0),
                                                    (8, 2560, 9728, 0, True, 0)])
def test_w4g_gemm_few_rows(lib, oracle, torch_dev, M, N, K, mode, use_res, pad):
    """M <= 32: 8, 16 or 32 staged rows, 1, 2, 3 or 5 column tiles per workgroup on 256 CUs
    (N up to 4096 / 8192 / 12288 / beyond), partial row and column tiles, fewer K blocks than
    waves, a half block at the end (K % 128 = 64), padded x and y rows, both epilogues.
    Against the oracle: the fp32 sums differ in order only, so an output rounds to the
    neighbouring fp16 value at most where no further op follows (one ulp, 2^-10 of the value,
    beside the order's own K 2^-24 of the summed magnitudes); an infinite activation stays in
    its row."""
    import torch
    rng = np.random.default_rng(M + N + K)
    n_out = N // 2 if mode else N
    _, wq, ws = w4g_weights(rng, N, K)
    x = normal_f16(rng, M, K + pad) * np.float16(0.25)
    res = normal_f16(rng, M, n_out)
    xd, wd, sd, rd = (to_dev(v, torch_dev) for v in (x, wq, ws, res))

    def run():
        y = torch.full((M, n_out + pad), 7.0, dtype=torch.float16, device=torch_dev)
        assert lib.gehtp_w4g_split_bytes(M, N, K) == 0
        assert lib.gehtp_w4g_fused(ptr(xd), K + pad, ptr(wd), ptr(sd), ptr(y), n_out + pad, M, N, K, None,
                                   ptr(rd) if use_res else None, n_out, mode, stream_ptr()) == 0
        _sync()
        got = from_dev(y)
        assert (got[:, n_out:] == 7).all()
        return got[:, :n_out]

    got = run()
    xc = np.ascontiguousarray(x[:, :K])
    acc = oracle.matmul_w4g(xc, wq, ws, threads=8)
    ref = oracle.binary(oracle.unary(acc[:, 0::2].copy(), 12), acc[:, 1::2].copy(), 2) if mode else acc
    if use_res:
        ref = oracle.binary(ref, res, 0)
    assert_close(got, ref, what=f"{M}x{N}x{K} mode={mode} res={use_res}")
    if not mode and not use_res:
        mag = np.abs(xc).astype(np.float64) @ np.abs(oracle.w4g_dequant(wq, ws, K).astype(np.float64)).T
        err = np.abs(got.astype(np.float64) - ref.astype(np.float64))
        assert (err <= np.abs(ref.astype(np.float64)) * 2.0 ** -10 + mag * K * 2.0 ** -24 + 2.0 ** -24).all()
    xd[M - 1, K - 1] = float("inf")
    hot = run()
    assert np.array_equal(hot[:M - 1].view(np.uint16), got[:M - 1].view(np.uint16))
    assert not np.isfinite(hot[M - 1].astype(np.float32)).all()


@pytest.mark.parametrize("M,N,K,mode,use_res", [(2, 40, 64, 0, True), (2, 6150, 2560, 1, True), (3, 4096, 192, 0, False),
                                                (3, 12290, 1024, 0, False), (4, 19456, 2560, 1, False), (4, 33, 8192, 0, True)])
def test_w4g_few_rows_norm(lib, oracle, torch_dev, M, N, K, mode, use_res):
    """2 to 4 rows with the RMSNorm inside the call: the 16-column tiles normalize the rows
    as they stage them (1, 2, 3 or 5 tiles per workgroup, K blocks fewer than waves, a half
    block at the end, the longest K the call takes). Against the oracle's RMSNorm, linear
    and epilogue."""
    import torch
    rng = np.random.default_rng(7 * M + N + K)
    n_out = N // 2 if mode else N
    _, wq, ws = w4g_weights(rng, N, K)
    x, gamma = normal_f16(rng, M, K), (rng.uniform(0.8, 1.2, K) * 0.25).astype(np.float16)
    res = normal_f16(rng, M, n_out)
    y = torch.empty((M, n_out), dtype=torch.float16, device=torch_dev)
    assert lib.gehtp_w4g_fused(ptr(to_dev(x, torch_dev)), K, ptr(to_dev(wq, torch_dev)), ptr(to_dev(ws, torch_dev)),
                               ptr(y), n_out, M, N, K, ptr(to_dev(gamma, torch_dev)),
                               ptr(to_dev(res, torch_dev)) if use_res else None, n_out, mode, stream_ptr()) == 0
    _sync()
    acc = oracle.matmul_w4g(oracle.rmsnorm2(x, gamma, np.zeros(K, np.float16)), wq, ws, threads=8)
    ref = oracle.binary(oracle.unary(acc[:, 0::2].copy(), 12), acc[:, 1::2].copy(), 2) if mode else acc
    if use_res:
        ref = oracle.binary(ref, res, 0)
    assert_close(from_dev(y), ref, what=f"norm {M}x{N}x{K} mode={mode} res={use_res}")


@pytest.mark.parametrize("rows,n", [(1, 1), (9, 2), (5, 63), (3, 64), (70, 32), (6, 129), (3, 255), (2, 257), (7, 511), (1030, 512), (4, 513), (9, 1024), (1100, 1001),
                                    (6, 2048), (5, 2049), (5, 7), (9, 768), (5, 769), (2050, 1025), (3, 1280), (3, 1281),
                                    (4, 1536), (5, 1537), (2, 1792), (3, 1793)])
def test_softmax_row_per_wave(lib, torch_dev, rows, n):
    """The row-per-wave softmax (n <= 2048: chunks of 1, 2, 4 or 8 values, 1, 2, 3, 4, 5 or 7 per lane,
    one or four rows per workgroup) and the longer rows beside it, at row lengths off every alignment, from a
    pointer 2 bytes off, in place, with -inf entries (a masked row's shape). Against float64:
    one fp16 rounding of the exponential and one of the quotient (2^-10 together), the fp32
    exponential and sum (n 2^-24) besides."""
    import torch
    g = torch.Generator(device=torch_dev).manual_seed(rows * 3 + n)
    x = (torch.randn((rows, n), device=torch_dev, generator=g) * 3).half()
    x[rows // 2, n // 2 + 1:] = float("-inf")
    for off in (0, 1):
        buf = torch.full((rows * n + off + 8,), 7.0, dtype=torch.float16, device=torch_dev)
        buf[off:off + rows * n] = x.reshape(-1)
        p = buf.data_ptr() + 2 * off
        assert lib.gehtp_softmax(p, p, rows, n, stream_ptr()) == 0
        _sync()
        assert (buf[:off] == 7).all() and (buf[off + rows * n:] == 7).all()
        got = buf[off:off + rows * n].view(rows, n).double()
        ref = torch.softmax(x.double(), -1)
        err = (got - ref).abs()
        assert (err <= ref * (2 ** -10 + (n + 16) * 2 ** -24) + 2 ** -24).all(), (off, float(err.max()))


@pytest.mark.parametrize("M,K,N", [(1, 9728, 264), (1, 12, 264), (2, 700, 1032), (4, 1100, 40), (3, 3100, 8200)])
def test_matmul_f16_gemv_special_values(lib, torch_dev, M, K, N):
    """The [K, N] GEMVs with a NaN, an infinity of each sign and 65504s in single columns of w
    (the first and last row of K, and inside): only those columns show them, the others keep
    their bits; an infinity in a's row reaches that row alone."""
    import torch
    g = torch.Generator(device=torch_dev).manual_seed(M + K + N)
    a = torch.randn((M, K), device=torch_dev, generator=g).half()
    w = (torch.randn((K, N), device=torch_dev, generator=g) * K ** -0.5).half()

    def run(a, w):
        y = torch.empty((M, N), dtype=torch.float16, device=torch_dev)
        assert lib.gehtp_matmul_f16(ptr(a), ptr(w), ptr(y), M, K, N, 0, N, 0, stream_ptr()) == 0
        _sync()
        return y

    clean, hot = run(a, w), w.clone()
    cols = [0, 9, N // 2, N - 1]
    hot[K - 1, cols[0]], hot[0, cols[1]], hot[K // 2, cols[2]], hot[:, cols[3]] = float("nan"), float("inf"), -float("inf"), 65504
    got = run(a, hot)
    keep = [j for j in range(N) if j not in cols]
    assert torch.equal(got[:, keep].view(torch.int16), clean[:, keep].view(torch.int16))
    ref = (a.double() @ hot.double()).half()   # an overflow of the fp16 result is an infinity
    for j in cols:
        assert torch.equal(torch.isnan(got[:, j]), torch.isnan(ref[:, j])) and torch.equal(torch.isinf(got[:, j]), torch.isinf(ref[:, j]))
    a2 = a.clone()
    a2[M - 1, K - 1] = float("inf")
    rows = run(a2, w)
    assert torch.equal(rows[:M - 1].view(torch.int16), clean[:M - 1].view(torch.int16)) and not torch.isfinite(rows[M - 1]).any()


@pytest.mark.parametrize("M,N,K,mode,norm", [
    (8, 20480, 64, 0, False), (8, 20496, 64, 1, False),                              # 128-column tiles / few-row kernel, K = 64
    (32, 8208, 256, 0, False), (17, 16384, 1024, 1, False), (17, 57360, 128, 0, False),   # 128-column tiles past 16 rows
    (24, 14336, 2560, 0, False), (32, 8448, 9216, 0, False),                         # their K parts, with a workspace
    (20, 32784, 320, 0, False), (5, 33000, 192, 1, False), (2, 65552, 128, 0, True),   # 3 column tiles where 2 would do
    (3, 512, 4096, 0, False), (4, 1000, 8192, 0, False), (3, 512, 8192, 1, False), (3, 9216, 8192, 0, False),   # GEMV
    (2, 64, 8192, 0, True), (2, 200, 9728, 1, True)])
def test_w4g_few_rows_forms(lib, oracle, torch_dev, M, N, K, mode, norm):
    """Up to 32 rows where the rules change kernels on 256 CUs: the GEMV, the few-row GEMM (by
    its column tiles per workgroup) and the 128-column tiles, with and without their K parts.
    Against the oracle's RMSNorm, linear and SwiGLU, and within fp32 sums of each other with
    and without a workspace."""
    import torch
    rng = np.random.default_rng(M + N + K)
    n_out = N // 2 if mode else N
    _, wq, ws = w4g_weights(rng, N, K)
    x = normal_f16(rng, M, K) * np.float16(0.25)
    gamma = (rng.uniform(0.8, 1.2, K) * 0.25).astype(np.float16)
    xd, wd, sd, gd = (to_dev(v, torch_dev) for v in (x, wq, ws, gamma))
    xr = oracle.rmsnorm2(x, gamma, np.zeros(K, np.float16)) if norm else x
    acc = oracle.matmul_w4g(xr, wq, ws, threads=8)
    ref = oracle.binary(oracle.unary(acc[:, 0::2].copy(), 12), acc[:, 1::2].copy(), 2) if mode else acc
    nb = lib.gehtp_w4g_split_bytes(M, N, K)
    assert (nb > 0) == ((M, N) in ((24, 14336), (32, 8448)))
    for work in (None, torch.empty(nb // 4, dtype=torch.float32, device=torch_dev)) if nb else (None,):
        y = torch.full((M + 1, n_out), 7.0, dtype=torch.float16, device=torch_dev)
        assert lib.gehtp_w4g_fused_ws(ptr(xd), K, ptr(wd), ptr(sd), ptr(y), n_out, M, N, K, ptr(gd) if norm else None, None,
                                      n_out, mode, ptr(work) if work is not None else None, nb if work is not None else 0,
                                      stream_ptr()) == 0
        _sync()
        got = from_dev(y)
        assert (got[M] == 7).all()
        assert_close(got[:M], ref, what=f"{M}x{N}x{K} mode={mode} norm={norm} work={work is not None}")


@pytest.mark.parametrize("n", [61, 64, 128, 256, 500, 512, 700, 1000, 1024, 1100, 1280, 1536, 1700, 1800, 2048, 2100, 2112])
def test_softmax_special_rows(lib, torch_dev, n):
    """Rows with a +inf, a NaN, all -inf, and all at the lowest finite value, between ordinary
    rows: the vector form (n a multiple of 32) scales by 0 when the sum is no positive number,
    the other divides by it, and the ordinary rows keep their bits. Rows per wave and (past
    2048 columns) per workgroup alike."""
    import torch
    g = torch.Generator(device=torch_dev).manual_seed(n)
    x = (torch.randn((9, n), device=torch_dev, generator=g) * 3).half()

    def run(x):
        y = torch.empty_like(x)
        assert lib.gehtp_softmax(ptr(x), ptr(y), x.shape[0], n, stream_ptr()) == 0
        _sync()
        return y

    clean, hot = run(x), x.clone()
    hot[1, n - 1], hot[3, n // 2], hot[5], hot[7] = float("inf"), float("nan"), float("-inf"), -65504
    got = run(hot)
    assert torch.equal(got[::2].view(torch.int16), clean[::2].view(torch.int16))
    nan = torch.zeros((9, n), dtype=torch.bool, device=torch_dev)
    nan[1, n - 1] = nan[3, n // 2] = nan[5] = True
    if n % 32:
        nan[1] = nan[3] = True
    assert torch.equal(torch.isnan(got), nan)
    assert (got[[1, 3]][~nan[[1, 3]]] == 0).all()
    assert ((got[7].double() - 1 / n).abs() <= 2 ** -10 / n + 2 ** -24).all()
