"""GPU parity tests for the prefill GEMM (tc_gemm: int8 MFMA for Q4_K / Q5_K /
Q6_K / IQ3_XXS / IQ3_S / IQ2_S / Q8_0 and, from 9 tokens, Q2_K / Q3_K / IQ4_XS;
bf16 MFMA on the pieces of fp32 x for IQ4_NL / Q5_0 / IQ2_XS; the decode kernel
over groups of tokens for the calls of those six that it keeps), through the C-ABI.

Bar: fp32 outputs within 1e-3 relative / 1e-4 absolute of the oracle (the C
restatement of the reference CPU kernels, itself bit-exact with the compiled
reference in tests/test_oracle.py). The activation quantizer the GEMM runs is
the one whose bytes are checked bit-exact in test_gpu_gemv.py.
"""
import numpy as np
import pytest

from qdata import ALL, IQ2_S, IQ2_XS, IQ4_NL, IQ4_XS, Q5_0, IQ3_S, IQ3_XXS, NAMES, Q2_K, Q3_K, Q4_K, Q5_K, Q6_K, Q8_0, close, gaussian, oracle_matmul_par, random_blocks, row_bytes, tile_edges

pytestmark = pytest.mark.gpu


def to_dev(a, dev):
    import torch
    return torch.from_numpy(np.ascontiguousarray(a)).to(dev)


def enc_weights(oracle, qt, rng, rows, cols):
    # Q4_K from N(0,1): at N(0,0.02) the reference quantizer stores most
    # scales as 0 (its fp16 conversion flushes values below 2^-13).
    return oracle.encode(qt, gaussian(rng, (rows, cols), 1.0 if qt in (Q4_K, Q5_K) else 0.02))


# (M tokens, N rows, K cols): ragged tiles, a K-split case (few output tiles),
# a single token, and a multi-tile case.
# (40, 72, 2304): K-slices of 5 and 4 superblocks (odd and even counts);
# (200, 1000, 4096): Q4_K stream-K with every tile split over 4 workgroups and
# ragged rows and tokens.
# (33, 77, 768) and (5, 129, 256): an odd number of weight units, so the
# last unit of a 2-byte-aligned format (IQ3_XXS, Q6_K, IQ3_S, IQ2_S) starts
# 4-byte aligned and its last dword load ends past the matrix.
SHAPES = [(1, 64, 256), (37, 200, 1024), (128, 256, 5120), (130, 136, 2048), (300, 384, 768), (40, 72, 2304),
          (200, 1000, 4096), (33, 77, 768), (5, 129, 256)]


MFMA_TYPES = [Q4_K, Q5_K, Q6_K, IQ3_XXS, IQ3_S, IQ2_S, Q8_0]


@pytest.mark.parametrize("M,N,K", SHAPES)
@pytest.mark.parametrize("qt", MFMA_TYPES)
def test_gemm_vs_oracle(tc, dev, oracle, qt, M, N, K):
    rng = np.random.default_rng(M * 7 + N + K + qt)
    w = enc_weights(oracle, qt, rng, N, K)
    x = gaussian(rng, (M, K))
    got = tc.gemm(qt, to_dev(w, dev), to_dev(x, dev), N, K).cpu().numpy()
    ref = oracle.matmul(qt, w, x, N, K)
    ok, worst = close(got, ref)
    assert ok, f"{NAMES[qt]} M={M} N={N} K={K}: worst err/bound {worst:.3g}"


@pytest.mark.parametrize("M", [8, 40, 64, 100])
@pytest.mark.parametrize("qt", MFMA_TYPES)
def test_gemm_token_tiles(tc, dev, oracle, qt, M):
    """Token counts around the token-tile widths the GEMM picks from M (32,
    64, 128 tokens), with a ragged last row block."""
    rng = np.random.default_rng(M * 3 + qt)
    N, K = 300, 2048
    w = enc_weights(oracle, qt, rng, N, K)
    x = gaussian(rng, (M, K))
    got = tc.gemm(qt, to_dev(w, dev), to_dev(x, dev), N, K).cpu().numpy()
    ok, worst = close(got, oracle.matmul(qt, w, x, N, K))
    assert ok, f"{NAMES[qt]} M={M}: worst err/bound {worst:.3g}"


@pytest.mark.parametrize("qt", MFMA_TYPES)
def test_gemm_random_blocks(tc, dev, oracle, qt):
    """Arbitrary block bytes (all scale/min codes, subnormal fp16 scales)."""
    rng = np.random.default_rng(99 + qt)
    M, N, K = 70, 96, 1536
    w = random_blocks(qt, rng, N, K)
    x = gaussian(rng, (M, K))
    got = tc.gemm(qt, to_dev(w, dev), to_dev(x, dev), N, K).cpu().numpy()
    ref = oracle.matmul(qt, w, x, N, K)
    ok, worst = close(got, ref)
    assert ok, worst


# From 9 tokens Q2_K, Q3_K and IQ4_XS run on the matrix cores too: one token
# past the batched path's 8, tile edges (32 / 64 / 128 tokens, 256 rows) and
# remainders, an odd number of weight units, K split over workgroups with the
# fixup launch ((200, 1000, 4096) and (130, 300, 5120)), on random block bytes.
#
# Random blocks give weights up to 2^-5 * 4064, so outputs that cancel lie
# below the fp32 rounding of their terms. The integer sums are exact on both
# sides; the fp32 sum of nb block values v_b and the at most 10 roundings that
# form each differ from the exact value by at most (nb + 10) 2^-24 sum |v_b| <=
# (nb + 10) 2^-24 |xq| . |w| on either side. (One wrong quant moves its output
# by about 1 / (8 K) of |xq| . |w|, several times that.)
@pytest.mark.parametrize("M,N,K", [(9, 64, 256), (8, 257, 768), (32, 256, 1024), (33, 77, 768), (64, 255, 512),
                                   (65, 300, 2304), (128, 512, 1280), (129, 129, 256), (200, 1000, 4096),
                                   (130, 300, 5120)])
@pytest.mark.parametrize("qt", [Q2_K, Q3_K, IQ4_XS])
def test_gemm_low_bit_mfma(tc, dev, oracle, qt, M, N, K):
    rng = np.random.default_rng(M * 5 + N + K + qt)
    w = random_blocks(qt, rng, N, K)
    x = gaussian(rng, (M, K))
    got = tc.gemm(qt, to_dev(w, dev), to_dev(x, dev), N, K).cpu().numpy()
    ref = oracle.matmul(qt, w, x, N, K)
    qs, d, _ = oracle.quantize_q8k(x.ravel())
    xa = np.abs(qs.reshape(-1, 256).astype(np.float64) * d.reshape(-1, 1)).reshape(M, K)
    wa = np.abs(oracle.dequant(qt, w, N, K).reshape(N, K).astype(np.float64))
    bound = 1e-4 + 1e-3 * np.abs(ref) + 2 * (K // 256 + 10) * 2.0**-24 * (xa @ wa.T)
    worst = (np.abs(got - ref) / bound).max()
    assert worst <= 1, f"{NAMES[qt]} M={M} N={N} K={K}: worst err/bound {worst:.3g}"


# The fp32-activation types on the bf16 matrix cores (x as three exact bf16
# pieces): from 9 tokens, tile edges and remainders, an odd number of 74-byte
# units, split tiles ((300, 7000, 2304): 84 over 256 workgroups, whole ones at
# 256 columns), activations over 12 orders of magnitude.
# Every product is exact; the fp32 sums of K / 32 block sums, each of at
# most 12 roundings, stay within (K / 32 + 12) 2^-24 |x| . |w| of the exact
# value here and in the oracle.
@pytest.mark.parametrize("M,N,K", [(9, 64, 256), (8, 257, 768), (32, 256, 1024), (33, 77, 768), (64, 255, 512),
                                   (65, 300, 2304), (128, 512, 1280), (129, 129, 256), (200, 1000, 4096),
                                   (300, 7000, 2304)])
@pytest.mark.parametrize("qt", [IQ4_NL, Q5_0, IQ2_XS])
def test_gemm_fp32_activations_mfma(tc, dev, oracle, qt, M, N, K):
    rng = np.random.default_rng(M * 3 + N + K + qt)
    w = random_blocks(qt, rng, N, K)
    x = gaussian(rng, (M, K)) * (10.0 ** rng.uniform(-6, 6, (M, 1))).astype(np.float32)
    got = tc.gemm(qt, to_dev(w, dev), to_dev(x, dev), N, K).cpu().numpy()
    rows = np.arange(N) if M * N * K < 1 << 28 else tile_edges(N, 256, 16, rng)
    wr = w.reshape(N, -1)[rows]
    ref = oracle_matmul_par(oracle, qt, wr, x, len(rows), K)
    wa = np.abs(oracle.dequant(qt, wr, len(rows), K).astype(np.float64))
    bound = 2 * (K // 32 + 12) * 2.0**-24 * (np.abs(x.astype(np.float64)) @ wa.T)
    worst = (np.abs(got[:, rows] - ref) / bound).max()
    assert worst <= 1, f"{NAMES[qt]} M={M} N={N} K={K}: worst err/bound {worst:.3g}"


# An infinite or NaN activation reaches its token's outputs and no other's.
@pytest.mark.parametrize("qt", [IQ4_NL, Q5_0, IQ2_XS])
def test_gemm_fp32_activations_nonfinite(tc, dev, oracle, qt):
    rng = np.random.default_rng(qt)
    M, N, K = 40, 96, 512
    w = random_blocks(qt, rng, N, K)
    x = gaussian(rng, (M, K))
    clean = tc.gemm(qt, to_dev(w, dev), to_dev(x, dev), N, K).cpu().numpy()
    bad = x.copy()
    bad[3, 7], bad[5, 300] = np.inf, np.nan
    got = tc.gemm(qt, to_dev(w, dev), to_dev(bad, dev), N, K).cpu().numpy()
    wf = oracle.dequant(qt, w, N, K)
    with np.errstate(invalid="ignore"):
        assert np.array_equal(got[3], np.inf * wf[:, 7], equal_nan=True)
    assert np.isnan(got[5]).all()
    keep = [m for m in range(M) if m not in (3, 5)]
    assert np.array_equal(got[keep], clean[keep])


# Q8_0 rows of an even number of 32-blocks, read in place: widths below and
# above 256, 2, 4 and 6 blocks left, every tile geometry (64 and 128 tokens, 256
# rows from 257 tokens), split tiles. A NaN or infinite scale in the next row's
# first blocks, which the last superblock's loads bring in, changes nothing.
@pytest.mark.parametrize("M,N,K", [(1, 1, 64), (9, 40, 192), (33, 130, 320), (64, 77, 448), (65, 257, 1088),
                                   (128, 300, 2880), (129, 129, 576), (257, 500, 2880), (300, 1030, 832)])
def test_gemm_q80_ragged_in_place(tc, dev, oracle, M, N, K):
    rng = np.random.default_rng(M + N + K)
    w = random_blocks(Q8_0, rng, N, K)
    x = gaussian(rng, (M, K))
    ref = oracle_matmul_par(oracle, Q8_0, w, x, N, K)
    got = tc.gemm(Q8_0, to_dev(w, dev), to_dev(x, dev), N, K).cpu().numpy()
    ok, worst = close(got, ref)
    assert ok, f"M={M} N={N} K={K}: worst err/bound {worst:.3g}"
    if N > 2:
        bad = w.reshape(N, K // 32, 34).copy()
        bad[1, 0, :2] = np.frombuffer(np.float16(np.nan).tobytes(), np.uint8)
        bad[N - 1, 1, :2] = np.frombuffer(np.float16(np.inf).tobytes(), np.uint8)
        got2 = tc.gemm(Q8_0, to_dev(bad.ravel(), dev), to_dev(x, dev), N, K).cpu().numpy()
        keep = [n for n in range(N) if n not in (1, N - 1)]
        assert np.array_equal(got2[:, keep], got[:, keep])


@pytest.mark.parametrize("S,N,K", [(8, 40, 18944), (5, 33, 18944), (4, 5000, 9216)])
@pytest.mark.parametrize("qt", ALL)
def test_few_tokens_on_the_matrix_cores(tc, dev, oracle, qt, S, N, K):
    """tc_gemv (and tc_gemm) at 8 tokens or less where the decode kernel would
    need several launches: the oracle's results, and under stream capture the
    eager call's bits, on every replay."""
    import torch
    rng = np.random.default_rng(S + N + K + qt)
    w = enc_weights(oracle, qt, rng, N, K) if N < 100 else random_blocks(qt, rng, N, K)
    x = gaussian(rng, (S, K))
    wd, xd = to_dev(w, dev), to_dev(x, dev)
    got = tc.gemv(qt, wd, xd, N, K).cpu().numpy()
    if N < 100:
        ref = oracle_matmul_par(oracle, qt, w, x, N, K)
        ok, worst = close(got, ref)
        assert ok, f"{NAMES[qt]} S={S} N={N} K={K}: worst err/bound {worst:.3g}"
        assert np.array_equal(tc.gemm(qt, wd, xd, N, K).cpu().numpy(), got) or qt in MFMA_TYPES
    out = torch.empty((S, N), device=dev)
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        tc.gemv(qt, wd, xd, N, K, out=out)
    for _ in range(3):
        out.zero_()
        graph.replay()
        torch.cuda.synchronize()
        assert np.array_equal(out.cpu().numpy(), got), NAMES[qt]


# Byte offsets of the fp16 scales of a block.
SCALES = {Q8_0: (0,), Q2_K: (80, 82), Q3_K: (108,), Q4_K: (0, 2), Q5_K: (0, 2), Q6_K: (208,)}


def even_blocks(qt, rng, rows, cols, scale=2.0**-10):
    """Random blocks whose scales lie within a factor of 3, so that every
    superblock counts alike in a sum."""
    from qdata import TYPE_SIZE
    b = random_blocks(qt, rng, rows, cols).reshape(-1, TYPE_SIZE[qt])
    for o in SCALES.get(qt, (0,)):
        b[:, o:o + 2] = rng.uniform(scale, 3 * scale, len(b)).astype(np.float16).view(np.uint8).reshape(-1, 2)
    return b.ravel()


# (20000 x 18944: tiles split over 3 workgroups; 21000 x 8192: the same with 11
# superblocks each; 10496 x 18944: over more workgroups, 12 superblocks each;
# 8192 x 8192 at 200 tokens: 4 workgroups, 8 superblocks each, summed by the last)
@pytest.mark.parametrize("qt,S,N,K", [(t, S, N, K) for t in ALL if t != Q8_0
                                      for S, N, K in [(8, 20000, 18944), (8, 21000, 8192), (8, 10496, 18944), (200, 8192, 8192)]
                                      if S == 8 or t not in MFMA_TYPES])
def test_sums_as_close_as_the_decode_kernels(tc, dev, oracle, qt, S, N, K):
    """Where the decode kernel could serve a call, the fp32 sums of the
    matrix-core kernels are no further from the 64-bit results (2-norm) than its
    own (single tokens, which always run it)."""
    import torch
    rng = np.random.default_rng(N + K + qt)
    w = even_blocks(qt, rng, N, K)
    S += S == 8 and qt not in MFMA_TYPES
    x = gaussian(rng, (S, K))
    wd, xd = to_dev(w, dev), to_dev(x, dev)
    got = tc.gemv(qt, wd, xd, N, K) if S <= 8 else tc.gemm(qt, wd, xd, N, K)
    dec = torch.cat([tc.gemv(qt, wd, xd[s:s + 1].contiguous(), N, K) for s in range(min(S, 9))])
    rows = np.sort(rng.choice(N, 4000, replace=False))
    if qt in (IQ2_XS, IQ4_NL, Q5_0):
        xa = x.astype(np.float64)
    else:
        qs, d, _ = oracle.quantize_q8k(x.ravel())
        xa = (qs.reshape(-1, 256).astype(np.float64) * d.reshape(-1, 1).astype(np.float64)).reshape(S, K)
    # (products of an fp16 scale, a 4 to 8 bit scale and a quant are exact in
    # fp32, or nearly: Q6_K, and the mins of Q2_K, Q4_K and Q5_K)
    ref = xa @ oracle.dequant(qt, w.reshape(N, -1)[rows], len(rows), K).astype(np.float64).T
    err = [np.linalg.norm(o.cpu().numpy()[:, rows] - ref[:len(o)]) / np.linalg.norm(ref[:len(o)]) for o in (got, dec)]
    print(f"{NAMES[qt]} {N}x{K}: {err[0]:.3e}, decode kernel {err[1]:.3e}")
    # (the norms over 4000 rows scatter by below 1%)
    assert err[0] <= 1.02 * err[1], (NAMES[qt], N, K, err)


LOW = [Q2_K, Q3_K, IQ4_XS, IQ4_NL, Q5_0, IQ2_XS]


# Units (tile, superblock) per workgroup of 256, chains of 8 superblocks (Q2_K,
# Q3_K, IQ4_XS up to 48 in a row) or 12: (512, 18944, 3584) 16.2, one flush, tiles
# whole and split, 128 tokens wide; (250, 16384, 12544) 24.5, two flushes, summed by
# a fixup launch or 6 workgroups' last; (40, 33000, 12544) and (20, 33000, 12544)
# 24.7, 64 and 32 tokens wide, ragged rows.
@pytest.mark.parametrize("M,N,K", [(512, 18944, 3584), (250, 16384, 12544), (40, 33000, 12544), (20, 33000, 12544)])
@pytest.mark.parametrize("qt", LOW)
def test_gemm_long_chains(tc, dev, oracle, qt, M, N, K):
    """Where a workgroup holds more superblocks of a tile than one chain of fp32
    sums, the sums that it flushes to memory and takes back; the bounds derived at
    test_gemm_low_bit_mfma and test_gemm_fp32_activations_mfma."""
    rng = np.random.default_rng(M + N + K + qt)
    w = even_blocks(qt, rng, N, K)
    x = gaussian(rng, (M, K))
    got = tc.gemm(qt, to_dev(w, dev), to_dev(x, dev), N, K).cpu().numpy()
    rows, toks = tile_edges(N, 256, 16, rng)[::3], tile_edges(M, 32, 4, rng)
    wr = w.reshape(N, -1)[rows]
    ref = oracle_matmul_par(oracle, qt, wr, x[toks], len(rows), K)
    wa = np.abs(oracle.dequant(qt, wr, len(rows), K).reshape(len(rows), K).astype(np.float64))
    if qt in (IQ4_NL, Q5_0, IQ2_XS):
        bound = 2 * (K // 32 + 12) * 2.0**-24 * (np.abs(x[toks].astype(np.float64)) @ wa.T)
    else:
        qs, d, _ = oracle.quantize_q8k(x[toks].ravel())
        xa = np.abs(qs.reshape(-1, 256).astype(np.float64) * d.reshape(-1, 1)).reshape(len(toks), K)
        bound = 2 * (K // 256 + 10) * 2.0**-24 * (xa @ wa.T)
    worst = (np.abs(got[np.ix_(toks, rows)] - ref) / bound).max()
    assert worst <= 1, f"{NAMES[qt]} M={M} N={N} K={K}: worst err/bound {worst:.3g}"
    assert np.isfinite(got).all()


@pytest.mark.parametrize("qt", [Q2_K, Q3_K, IQ4_XS])
def test_gemm_low_bit_overflow(tc, dev, oracle, qt):
    """Activations so large that block values overflow: infinities of their
    sign, also where a workgroup has more superblocks than one chain of sums
    holds (256 whole tiles of 14 superblocks), and no NaN."""
    rng = np.random.default_rng(qt + 31)
    M, N, K = 1024, 8192, 3584
    w = even_blocks(qt, rng, N, K, 2.0**(-12 if qt == IQ4_XS else -6))
    x = gaussian(rng, (M, K))
    x[3] = 0.0
    x[3, :256] = gaussian(rng, 256) * np.float32(1e38)
    got = tc.gemm(qt, to_dev(w, dev), to_dev(x, dev), N, K).cpu().numpy()[3]
    wr = w.reshape(N, -1)[:, :row_bytes(qt, 256)]
    qs, d, _ = oracle.quantize_q8k(x[3, :256])
    ref = oracle.dequant(qt, np.ascontiguousarray(wr), N, 256).astype(np.float64) @ (qs.astype(np.float64).ravel() * float(d[0]))
    top = float(np.finfo(np.float32).max)
    over = np.abs(ref) > 1.01 * top
    under = np.abs(ref) < 0.99 * top
    assert over.sum() > 100 and under.sum() > 100
    assert (got[over] == np.sign(ref[over]) * np.inf).all(), got[over][:8]
    assert np.allclose(got[under], ref[under], rtol=1e-4, atol=1e-6 * top)


@pytest.mark.parametrize("qt", LOW)
def test_gemm_captured_matches_eager(tc, dev, qt):
    """tc_gemm at 9 tokens or more of the types that the decode kernel could
    serve: every replay has the eager call's bits."""
    import torch
    rng = np.random.default_rng(qt + 77)
    M, N, K = 21, 300, 1024
    wd, xd = to_dev(random_blocks(qt, rng, N, K), dev), to_dev(gaussian(rng, (M, K)), dev)
    ref = tc.gemm(qt, wd, xd, N, K).clone()
    out = torch.empty((M, N), device=dev)
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        tc.gemm(qt, wd, xd, N, K, out=out)
    for _ in range(3):
        out.fill_(float("nan"))
        tc.gemm(qt, wd, xd, N, K)  # eager work on the same scratch
        torch.cuda.synchronize()
        graph.replay()
        torch.cuda.synchronize()
        assert torch.equal(out, ref), NAMES[qt]


def test_gemm_captured_without_scratch():
    """The same captured in a process whose scratch is still empty: the decode
    kernel over groups of 8 tokens and a remainder, the bits of tc_gemv on those
    groups."""
    import os
    import subprocess
    import sys
    here = os.path.dirname(os.path.abspath(__file__))
    code = """
import sys
sys.path[:0] = sys.argv[1:]
import numpy as np, torch, tc_hip
from qdata import gaussian, random_blocks
tc = tc_hip.Library()
rng = np.random.default_rng(5)
M, N, K = 21, 300, 1024
x = torch.from_numpy(gaussian(rng, (M, K))).cuda()
for qt in (tc_hip.Q2_K, tc_hip.Q3_K, tc_hip.IQ4_XS, tc_hip.IQ4_NL, tc_hip.Q5_0, tc_hip.IQ2_XS):
    w = torch.from_numpy(random_blocks(qt, rng, N, K)).cuda()
    ref = torch.cat([tc.gemv(qt, w, x[s:s + 8], N, K) for s in (0, 8, 16)])
    out = torch.empty_like(ref)
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        tc.gemm(qt, w, x, N, K, out=out)
    for _ in range(3):
        out.zero_()
        torch.cuda.synchronize()
        graph.replay()
        torch.cuda.synchronize()
        assert torch.equal(out, ref), qt
    print("type", qt, "ok", flush=True)
"""
    r = subprocess.run([sys.executable, "-c", code, here, os.path.join(os.path.dirname(here), "tinycoder-inference_amd")],
                       capture_output=True, text=True, timeout=100)
    assert r.returncode == 0, (r.stdout, r.stderr)


@pytest.mark.parametrize("qt", [Q2_K, Q3_K, IQ2_XS, IQ4_XS, IQ4_NL, Q5_0])
def test_gemm_exact_batched_types(tc, dev, oracle, qt):
    """The types that the reference's GEMM leaves to its exact batched path, on
    the matrix cores here (test_gemm_captured_without_scratch runs the decode
    kernel over groups of tokens)."""
    rng = np.random.default_rng(5 + qt)
    M, N, K = 21, 80, 512
    w = enc_weights(oracle, qt, rng, N, K)
    x = gaussian(rng, (M, K))
    got = tc.gemm(qt, to_dev(w, dev), to_dev(x, dev), N, K).cpu().numpy()
    ok, worst = close(got, oracle.matmul(qt, w, x, N, K))
    assert ok, worst


@pytest.mark.parametrize("M", [128, 512, 2048])
@pytest.mark.parametrize("qt,N,K", [(Q4_K, 17408, 5120), (Q4_K, 5120, 17408), (Q8_0, 17408, 5120),
                                    (Q8_0, 5120, 17408)])
def test_gemm_cfg4_full_shape(tc, dev, oracle, qt, N, K, M):
    """BASELINE config 4 at full size: both matrices, both types, M in {128,
    512, 2048}."""
    full_shape_check(tc, dev, oracle, qt, N, K, M)


@pytest.mark.parametrize("M", [128, 512])
@pytest.mark.parametrize("qt,N,K", [(qt, N, K) for qt in (Q5_K, Q6_K, IQ3_XXS, IQ3_S, IQ2_S)
                                    for N, K in ((18944, 3584), (3584, 18944))])
def test_gemm_7b_ffn_full_shape(tc, dev, oracle, qt, N, K, M):
    """The 7B FFN shapes (18944 x 3584 up, 3584 x 18944 down) for the other
    MFMA types at prefill batch sizes 128 and 512."""
    full_shape_check(tc, dev, oracle, qt, N, K, M)


def full_shape_check(tc, dev, oracle, qt, N, K, M):
    """Weights from the GPU encoder, x ~ N(0,1). The oracle checks
    the first and last row of every 64-row workgroup tile plus 32 seeded rows,
    against every token for M <= 512, and at M = 2048 the first and last token
    of every 128-token tile, the whole last token tile and 32 seeded tokens
    (tokens and rows are independent of each other, so these entries are
    exactly the full output's)."""
    import torch
    gen = torch.Generator(device=dev).manual_seed(4 + qt + N + M)
    wf = torch.randn((N, K), generator=gen, device=dev) * (1.0 if qt in (Q4_K, Q5_K) else 0.02)
    w = tc.encode(qt, wf)
    del wf
    x = torch.randn((M, K), generator=gen, device=dev)
    got = tc.gemm(qt, w, x, N, K).cpu().numpy()
    assert np.isfinite(got).all()
    rng = np.random.default_rng(M + N)
    rows = tile_edges(N, 64, 32, rng)
    toks = np.arange(M) if M <= 512 else tile_edges(M, 128, 32, rng)
    wh = w.cpu().numpy().reshape(N, row_bytes(qt, K))[rows]
    xh = x.cpu().numpy()[toks]
    ref = oracle_matmul_par(oracle, qt, wh, xh, len(rows), K)
    sub = got[np.ix_(toks, rows)]
    ok, worst = close(sub, ref)
    bad = np.argwhere(~(np.abs(sub - ref) <= 1e-4 + 1e-3 * np.abs(ref)))
    assert ok, (f"{NAMES[qt]} M={M} N={N} K={K}: worst err/bound {worst:.3g}; first bad (token, row) "
                f"{[(int(toks[i]), int(rows[j])) for i, j in bad[:5]]}")


def test_gemm_matches_gemv_small_batch(tc, dev):
    """M <= 8: the MFMA GEMM and the decode kernel agree within tolerance."""
    rng = np.random.default_rng(3)
    N, K = 300, 2048
    w = random_blocks(Q4_K, rng, N, K)
    x = gaussian(rng, (5, K))
    wd, xd = to_dev(w, dev), to_dev(x, dev)
    g = tc.gemm(Q4_K, wd, xd, N, K).cpu().numpy()
    v = tc.gemv(Q4_K, wd, xd, N, K).cpu().numpy()
    ok, worst = close(g, v)
    assert ok, worst


def test_gemm_refuses_bad_shapes(tc, dev):
    import tc_hip
    w = to_dev(np.zeros(row_bytes(Q4_K, 512) * 4, np.uint8), dev)
    x = to_dev(np.zeros((3, 500), np.float32), dev)
    with pytest.raises(tc_hip.TCError):
        tc.gemm(Q4_K, w, x, 4, 500)


def test_q80_minus128_true_product(tc, dev, oracle):
    """Q8_0 weight bytes of -128 (never written by a quantizer: q =
    round(w/d) with d = amax/127 stays in [-127, 127]): the GPU paths compute
    the true product -128 * x. The reference AVX2 kernel's sign trick
    (SIMDMatMulVecAVX2.cpp:4239-4383) cannot negate -128 and gives -128 * |x|
    instead; the oracle mirrors that, so on such rows the two differ. Pins the
    GPU's behaviour (mat-vec, the MFMA GEMM and the host entry point) against
    the exact product from the reference's own activation quantization."""
    rng = np.random.default_rng(128)
    rows, cols = 96, 1024
    w = random_blocks(Q8_0, rng, rows, cols)
    blk = w.reshape(rows, cols // 32, 34)
    q = blk[:, :, 2:].view(np.int8)
    q[rng.random(q.shape) < 0.05] = -128  # some -128 bytes in most blocks
    blk[:, :, :2] = (rng.uniform(0.5, 2.0, (rows, cols // 32, 1)) * 1e-3).astype(np.float16).view(np.uint8)
    dw = blk[:, :, :2].copy().view(np.float16).astype(np.float64)[:, :, 0]
    for S in (1, 4, 40):
        x = gaussian(rng, (S, cols))
        exact = np.zeros((S, rows))
        for s in range(S):
            xq, d8 = oracle.quantize_q8_0_act(x[s])
            isum = (q.astype(np.int64) * xq.reshape(cols // 32, 32).astype(np.int64)[None]).sum(axis=2)
            exact[s] = (isum * dw * d8.astype(np.float64)[None]).sum(axis=1)
        xd, wd = to_dev(x, dev), to_dev(w, dev)
        got = tc.gemv(Q8_0, wd, xd, rows, cols) if S <= 8 else tc.gemm(Q8_0, wd, xd, rows, cols)
        ok, worst = close(got.cpu().numpy(), exact.astype(np.float32))
        assert ok, f"S={S}: worst err/bound {worst:.3g}"
        ref = oracle.matmul(Q8_0, w, x, rows, cols)
        assert not close(ref, exact.astype(np.float32))[0], "the reference quirk should show on these rows"
