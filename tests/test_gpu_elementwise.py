"""GPU: the bandwidth operations' vector forms at their edges: totals around a thread's 8
elements, head counts that do not fill a RoPE thread's group of 4, partial rotation, and
rotation widths that take the element-wise kernel."""
import numpy as np
import pytest

import oracle
from sulimo_amd import hip
from sulimo_amd import synthetic as S
from tests.test_gpu_gemm import f16_weight_bound, run_gemm

pytestmark = pytest.mark.gpu


def up(ctx, a):
    return hip.HipBuffer.from_host(ctx, np.ascontiguousarray(a))


@pytest.mark.parametrize("total", [1, 7, 8, 9, 2047, 2048, 2049])
def test_silu_and_add_edges(ctx, total):
    rng = np.random.default_rng(total)
    g, u = ((rng.standard_normal(total + 8) * s).astype(np.float16) for s in (3, 1))
    ob = up(ctx, g)
    hip.enqueue_silu_mul(ctx, up(ctx, g), up(ctx, u), ob, total)
    got = ob.download(np.float16, g.shape)
    want = oracle.cl_silu_mul_f16(g[:total], u[:total]).astype(np.float64)
    # hardware exp2 and reciprocal (a few f32 ulps), then one f16 rounding
    assert np.all(np.abs(got[:total] - want) <= 1.01 * np.spacing(np.abs(want).astype(np.float16)).astype(np.float64))
    assert np.array_equal(got[total:], g[total:])  # nothing past the end is written
    ab = up(ctx, g)
    hip.enqueue_add(ctx, ab, up(ctx, u), total)
    got = ab.download(np.float16, g.shape)
    assert np.array_equal(got[:total], oracle.cl_add_f16(g[:total], u[:total]))
    assert np.array_equal(got[total:], g[total:])


def test_silu_vector_and_single_elements_agree(ctx):
    """Bit for bit: 7 elements run one by one, 8 as two registers of packed pairs, each of
    whose products must read its own operands."""
    rng = np.random.default_rng(40)
    for i in range(64):
        g, u = ((rng.standard_normal(8) * 4.0 ** rng.integers(-3, 3)).astype(np.float16) for _ in range(2))
        got = []
        for total in (7, 8):
            ob = up(ctx, np.zeros(8, np.float16))
            hip.enqueue_silu_mul(ctx, up(ctx, g), up(ctx, u), ob, total)
            got.append(ob.download(np.uint16, 8))
        assert np.array_equal(got[0][:7], got[1][:7]), i


@pytest.mark.parametrize("mode", [0, 1])
@pytest.mark.parametrize("heads,hd,rd,n", [(5, 64, 40, 3), (1, 128, 128, 1), (7, 64, 12, 5), (9, 32, 32, 70)])
def test_rope_partial_heads_and_widths(ctx, mode, heads, hd, rd, n):
    """Bit for bit given the device's cos/sin table (products rounded before the add)."""
    rng = np.random.default_rng(heads + rd + n)
    v = rng.standard_normal((n, heads, hd)).astype(np.float16)
    vb, tb = up(ctx, v), hip.HipBuffer.device_only(ctx, n * rd // 2 * 8)
    hip.enqueue_rope(ctx, vb, heads, hd, rd, 1e4, mode, 11, n)
    hip.rope_table(ctx, rd, 1e4, 11, n, tb)
    tab = tb.download(np.float32, (n, 1, rd // 2, 2))
    i = np.arange(rd // 2)
    i0, i1 = (2 * i, 2 * i + 1) if mode == 0 else (i, i + rd // 2)
    x = v.astype(np.float32)
    want = x.copy()
    want[:, :, i0] = x[:, :, i0] * tab[..., 0] - x[:, :, i1] * tab[..., 1]
    want[:, :, i1] = x[:, :, i0] * tab[..., 1] + x[:, :, i1] * tab[..., 0]
    assert np.array_equal(vb.download(np.float16, v.shape).view(np.uint16), want.astype(np.float16).view(np.uint16))


@pytest.mark.parametrize("M", [1, 2, 3, 4])
@pytest.mark.parametrize("k,m_out", [(8000, 40), (160, 1000), (1536, 9000)])
def test_gemv_split_stages(ctx, M, k, m_out):
    """Up to 4 tokens of a narrow matrix: the waves that share a panel's stages (16 of them,
    2 with one stage left over, and 8 with panels past the last) against the f16-weight bound."""
    rng = np.random.default_rng(M + k + m_out)
    w = S.random_q4(rng, m_out, k)
    x = rng.standard_normal((M, k)).astype(np.float16)
    y = run_gemm(ctx, w.scales, w.quants, x, m_out, k, M)
    ref = oracle.gemm_q4_0_f16_scalar_reference(w.scales, w.quants, x, m_out, k, M)
    assert np.all(np.abs(y.astype(np.float64) - ref) <= f16_weight_bound(x, w.scales, w.quants, ref))
