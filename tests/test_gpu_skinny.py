"""GPU: the GEMM for a handful of tokens (gemm_skinny.hip), at the sizes where it can go wrong.

One workgroup's waves split k in steps of 128 (the last step partly empty when k is not a
multiple of 128), hold 16- or 32-token tiles and 16 to 64 weight rows, and add their sums
through LDS. The plain product is checked against the oracle with the f16-weight error
model of test_gpu_gemm; the RoPE + Q8_0 and SwiGLU epilogues bit for bit against the ops
run as separate kernels, on the model of test_gpu_fused whose sums are exact in any order.
"""
import numpy as np
import pytest

import oracle
from sulimo_amd import hip
from sulimo_amd import synthetic as S
from tests.helpers import max_rel_err
from tests.test_gpu_fused import NORM_HD64, QWEN_LAYER, exact_model, run_mode
from tests.test_gpu_gemm import f16_weight_bound, run_gemm

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("M", [5, 16, 17, 24, 32, 33])
@pytest.mark.parametrize("k,m_out", [(32, 8), (96, 40), (160, 264), (2080, 72), (4128, 520)])
def test_ragged(ctx, M, k, m_out):
    rng = np.random.default_rng(100 * M + k + m_out)
    w = S.random_q4(rng, m_out, k)
    x = rng.standard_normal((M, k)).astype(np.float16)
    print(f"skinny GEMM m={M} k={k} n={m_out}", flush=True)
    y = run_gemm(ctx, w.scales, w.quants, x, m_out, k, M)
    ref = oracle.gemm_q4_0_f16_scalar_reference(w.scales, w.quants, x, m_out, k, M)
    assert np.all(np.abs(y.astype(np.float64) - ref) <= f16_weight_bound(x, w.scales, w.quants, ref))


@pytest.mark.parametrize("M,k", [(1, 33024), (2, 16480), (3, 8960), (4, 8224)])
def test_gemv_tokens_beyond_its_lds(ctx, M, k):
    """Up to 4 tokens of a k whose activations exceed the GEMV's 64 KB of LDS come here too."""
    rng = np.random.default_rng(M)
    w = S.random_q4(rng, 72, k)
    x = rng.standard_normal((M, k)).astype(np.float16)
    print(f"skinny GEMM m={M} k={k} n=72", flush=True)
    y = run_gemm(ctx, w.scales, w.quants, x, 72, k, M)
    ref = oracle.gemm_q4_0_f16_scalar_reference(w.scales, w.quants, x, 72, k, M)
    assert np.all(np.abs(y.astype(np.float64) - ref) <= f16_weight_bound(x, w.scales, w.quants, ref))


@pytest.mark.parametrize("M", [7, 23, 32])
@pytest.mark.parametrize("k,m_out", [(1536, 1536), (1536, 8960), (8960, 1536), (3072, 8192), (8192, 3072)])
def test_layer_shapes(ctx, M, k, m_out):
    """The projections of the two model shapes, each width's own split of k and columns."""
    rng = np.random.default_rng(7 * M + k + m_out)
    w = S.random_q4(rng, m_out, k)
    x = rng.standard_normal((M, k)).astype(np.float16)
    print(f"skinny GEMM m={M} k={k} n={m_out}", flush=True)
    y = run_gemm(ctx, w.scales, w.quants, x, m_out, k, M)
    assert max_rel_err(y, x.astype(np.float32) @ w.dequant_f32().T) <= 1e-2


def test_one_hot_bit_exact(ctx):
    """32 one-hot tokens read 32 columns of W^T exactly."""
    rng = np.random.default_rng(5)
    m_out, k = 264, 416
    w = S.random_q4(rng, m_out, k)
    w.quants.reshape(-1, 16)[:16] = np.arange(256, dtype=np.uint8).reshape(16, 16)
    deq = oracle.dequant_q4_0_soa(w.scales, w.quants).reshape(m_out, k)
    for c0 in range(0, k, 32):
        x = np.zeros((32, k), np.float16)
        x[np.arange(32), c0 + np.arange(32)] = 1.0
        y = run_gemm(ctx, w.scales, w.quants, x, m_out, k, 32)
        assert np.array_equal(y.view(np.uint16), deq[:, c0:c0 + 32].T.astype(np.float16).view(np.uint16))


@pytest.mark.parametrize("cfg,chunks,cap", [
    (QWEN_LAYER, [23, 16, 5, 32], 64),   # the last chunk wraps the ring (staged K/V)
    (NORM_HD64, [9, 31, 17], 48),        # Norm RoPE, head_dim 64, odd chunks, wrap
], ids=["neox_hd128", "norm_hd64"])
def test_epilogues_bit_exact_vs_separate_kernels(ctx, cfg, chunks, cap):
    hm = exact_model(cfg, 17)
    toks = S.random_tokens(18, sum(chunks), cfg.vocab)
    print(f"skinny epilogues: {cfg} chunks {chunks} capacity {cap}", flush=True)
    fused, (fk, fv) = run_mode(ctx, hm, toks, chunks, cap, unfused=False)
    plain, (pk, pv) = run_mode(ctx, hm, toks, chunks, cap, unfused=True)
    assert np.array_equal(fk[0], pk[0]) and np.array_equal(fv[0], pv[0])
    for f, p in zip(fused, plain):
        assert np.array_equal(f["q"], p["q"])
        assert np.array_equal(f["swiglu"], p["swiglu"])
        assert np.max(np.abs(f["logits"] - p["logits"])) <= 1e-3 * np.abs(p["logits"]).max()


@pytest.mark.parametrize("D", [288, 1056, 2080, 3104])
@pytest.mark.parametrize("n", [5, 33])
def test_split_reduction_of_widths_not_256(ctx, D, n):
    """Rows of 1 to 4 times 1024 columns, none a multiple of 256: the o and down projections
    split k, and their reduction adds the f32 partials, updates the residual and norms the
    row in a workgroup of its own. Against the separate kernels: the SwiGLU bytes (the FFN
    norm of the o projection's rows), the final residual, the logits (the output norm)."""
    cfg = S.ModelConfig(1, D, 1056, 8, 2, 64, 64, 512, 1e6, 1e-6, 1)
    hm = exact_model(cfg, D + n)
    toks = S.random_tokens(19, n, cfg.vocab)
    print(f"split reduction: width {D}, {n} tokens", flush=True)
    (f,), _ = run_mode(ctx, hm, toks, [n], 64, unfused=False)
    (p,), _ = run_mode(ctx, hm, toks, [n], 64, unfused=True)
    assert np.array_equal(f["swiglu"], p["swiglu"])
    # the down projection's f16 value may round one step apart (it differs from x by the
    # embedding, +-1), then x itself
    x = np.abs(p["x"])
    step = np.spacing(x + np.float16(1)).astype(np.float64) + np.spacing(x).astype(np.float64)
    assert np.all(np.abs(f["x"].astype(np.float64) - p["x"].astype(np.float64)) <= step)
    assert np.max(np.abs(f["logits"] - p["logits"])) <= 1e-3 * np.abs(p["logits"]).max()


@pytest.mark.parametrize("M,k,m_out", [(5, 32, 8), (16, 1536, 1536), (24, 96, 40), (33, 2080, 264), (64, 416, 9000),
                                       (8, 4128, 72)])
def test_no_alloc_reads_the_source_arrays(ctx, M, k, m_out):
    """The no-alloc entry point reads the weights where they are: odd block counts, ragged
    rows and each fragment count give the panel path's bits (where it does not split k)."""
    rng = np.random.default_rng(M + k + m_out)
    w = S.random_q4(rng, m_out, k)
    x = rng.standard_normal((M, k)).astype(np.float16)
    sb, qb, xb = (hip.HipBuffer.from_host(ctx, np.ascontiguousarray(a), True) for a in (w.scales, w.quants, x))
    ob = hip.HipBuffer.device_only(ctx, M * m_out * 2)
    print(f"skinny no-alloc GEMM m={M} k={k} n={m_out}", flush=True)
    hip.enqueue_gemm_q4_0_f16_noalloc(ctx, sb, qb, xb, ob, m_out, k, M)
    ctx.wait()
    y = ob.download(np.uint16, (M, m_out))
    assert np.array_equal(y, run_gemm(ctx, w.scales, w.quants, x, m_out, k, M).view(np.uint16))
