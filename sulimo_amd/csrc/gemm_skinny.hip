// gemm_skinny.hip - Q4_0 weight x f16 activation GEMM for a handful of tokens (m <= 64).
//
// The same product and epilogues as gemm_q4_0.hip, for the calls that are bound by
// latency: a short chat turn's projections hold 0.2-16 MB of weights, 1-3 us of HBM time,
// but a tile of that kernel walks its k stages one after another (0.3-0.5 us each) and a
// narrow projection has too few tiles to fill the chip.
//
// Here a workgroup covers few output columns and its waves split k between them, each
// wave one run of 128 k (two panel stages, a "pair") at a time, so that every load of the
// workgroup is in flight at once and the kernel costs about one memory round trip:
//  * Weights go straight to registers: a wave loads NF fragments of 16 weight rows, lane
//    l = 16 g + r one 16-byte chunk of row r, from stage g / 2 of the pair and k half
//    g % 2 of its blocks. All 32 weights of the chunk are the lane's own MFMA operands.
//  * X goes through LDS (buffer -> LDS DMA of whole 256-byte row runs, private to the
//    wave, so no barrier): read directly, the 16 rows of an A fragment would touch 64
//    cache lines per load instruction. 16-byte chunk c of row r sits at position
//    c ^ (r & 15), so the A reads are conflict free.
//  * v_mfma_f32_16x16x32_f16: lane l supplies A[row l%16] and B[col l%16] for 8 k, and
//    any 8 k serve as long as A and B agree: MFMA i of a pair takes k 64 (g/2) + 32 (i/2)
//    + 16 (i%2) + 8 (g%2) .. +7 (low nibbles for even i, high for odd).
//  * The waves' sums meet in LDS and are added in wave order; then 16 lanes x 4 rows per
//    column group run the epilogue, as in gemm_q4_0.hip.
// The weights are dequantized exactly as there (one f16 rounding of (q-8)*d), the sums
// stay in f32, and a K split across workgroups hands over f32 partials.
//
// Measured (kernel times, MI355X): Qwen2.5-1.5B projections at 23 tokens, tiled kernel ->
// this one: q/k/v with RoPE 11.1 -> 8.9 us, o 10.0 + 4.8 (RMSNorm) -> 4.3 + 4.1, gate/up
// 13.8 -> 9.5, down 8.4 + 6.0 -> 6.5 + 4.1; Llama-3.2-3B 15.4 -> 10.5, 7.4 + 8.2 -> 5.4 +
// 4.8, 22.2 -> 9.9, 7.4 + 8.2 -> 8.4 + 4.8; 1536 x 1536 alone at 8 tokens 8.0 -> 3.9. What
// is left is the launch and one memory round trip (3 us together), then the phases of a
// step that follow each other in a workgroup: loads at 64 B per clock and CU, the
// dequantization (60 VALU per fragment and step), and the sum over the waves.
//
// With SOA the weights are read from the caller's own arrays (scales [n][k/32], quants
// [n][k/32][16]) instead of a panel copy, the same bytes to the same lanes (two 8-byte
// loads and two scales each), so the sums are the same bits.
#include <algorithm>

#include "common.h"
#include "q4_mfma.h"

namespace sulimo {
namespace {

typedef float floatx4 __attribute__((ext_vector_type(4)));
typedef uint32_t u32x2 __attribute__((ext_vector_type(2)));
typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));

constexpr int kPairK = 128;      // k per wave step (two panel stages)
// Waves of a workgroup, by what its accumulators and A operands leave of the registers.
constexpr int max_waves(int MT, int NF) { return MT > 2 ? 8 : NF == 4 ? 12 : 16; }
constexpr int kMaxSplits = 8;

struct SkinnyArgs {
  GemmArgs g;
  const uint16_t *scales;  // SOA only
  const uint8_t *quants;
  int units;        // workgroups per K split
  int npairs;       // steps of 128 k
  int split_pairs;  // steps per K split
  int xrows;        // rows of X staged per step (m rounded up to 4)
};

// Output columns of one workgroup.
template <int NF, int EPI>
constexpr int unit_cols() { return EPI == EPI_SWIGLU ? 8 * NF : 16 * NF; }

template <int MT, int NF, int EPI, bool SOA>
__global__ __launch_bounds__(64 * max_waves(MT, NF)) void skinny_kernel(SkinnyArgs sa) {
  extern __shared__ __attribute__((aligned(16))) char smem[];
  const GemmArgs &a = sa.g;
  const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int nwaves = blockDim.x >> 6;
  const int r16 = lane & 15, g = lane >> 4;
  constexpr int UC = unit_cols<NF, EPI>();
  static_assert((EPI != EPI_SWIGLU && EPI != EPI_ROPE) || NF == 4, "paired panels: four fragments");

  // workgroup -> (K split, segment, unit)
  const int ks = blockIdx.y;
  int u = blockIdx.x;
  int si = 0, colbase = 0;
  for (; si < a.nseg - 1; si++) {
    const int nu = (a.seg[si].n + UC - 1) / UC;
    if (u < nu) break;
    u -= nu;
    colbase += a.seg[si].n;
  }
  const GemmSegment seg = a.seg[si];
  const int nb = a.k >> 5, nst = (nb + 1) >> 1;
  const int npanels = (seg.n + 31) / 32 * (EPI == EPI_SWIGLU ? 2 : 1);

  // The unit's panels: fragments 2j and 2j+1 are the halves of panel panel_of(j) (one
  // fragment: half u % 2). Gate / up and RoPE partners (the columns head_dim/2 apart) are
  // panels 0 and 1. hsh: log2 of the panels per half head.
  constexpr int NP = NF == 4 ? 2 : 1;
  const int hsh = EPI == EPI_ROPE ? a.rope.head_dim >> 7 : 0;  // head_dim 64 or 128
  const int hi = u & ((1 << hsh) - 1), head = u >> hsh;
  auto panel_of = [&](int j) -> int {
    if constexpr (EPI == EPI_ROPE) return (head << (hsh + 1)) + hi + (j << hsh);
    else if constexpr (NF == 1) return u >> 1;
    else return u * NP + j;
  };

  // --- per-lane buffer offsets of the weights, fixed for the kernel (the halves of a
  // panel are a constant apart) ---
  rsrc_t rq, rs;
  uint32_t qoff[NF], soff[NF];  // panels: [0, NP) used
  const int r1 = NF == 1 ? 16 * (u & 1) + r16 : r16;
  if constexpr (SOA) {
    rq = make_rsrc(sa.quants, (uint32_t)seg.n * (uint32_t)nb * 16u);
    rs = make_rsrc(sa.scales, (uint32_t)seg.n * (uint32_t)nb * 2u);
#pragma unroll
    for (int f = 0; f < NF; f++) {
      const int row = 32 * panel_of(f >> 1) + r1 + 16 * (f & 1);
      const uint32_t blk = (uint32_t)row * nb + 2u * (g >> 1);  // first block of the lane's stage
      qoff[f] = row < seg.n ? blk * 16u + 8u * (g & 1) : kOob;
      soff[f] = row < seg.n ? blk * 2u : kOob;
    }
  } else {
    rq = rs = make_rsrc(seg.panels, (uint32_t)npanels * (uint32_t)nst * (uint32_t)kQ4PanelRecord);
#pragma unroll
    for (int j = 0; j < NP; j++) {
      const int p = panel_of(j);
      const uint32_t rec = ((uint32_t)p * nst + (g >> 1)) * kQ4PanelRecord;
      qoff[j] = p < npanels ? rec + 16u * (32 * (g & 1) + r1) : kOob;
      soff[j] = p < npanels ? rec + 1024u + 4u * r1 : kOob;
    }
  }
  // Past the matrix in k (an odd count of stages or blocks ends in a partly empty pair)
  // the lane reads zeros: scale 0, weight exactly zero.
  u32x4 q[NF];
  uint32_t sc[NF];
  auto load_w = [&](int pr) __attribute__((always_inline)) {
    const bool in = 2 * pr + (g >> 1) < nst;
#pragma unroll
    for (int f = 0; f < NF; f++) {
      if constexpr (SOA) {
        const bool in1 = 4 * pr + 2 * (g >> 1) + 1 < nb;  // an odd block count ends in half a stage
        const u32x2 b0 = __builtin_amdgcn_raw_buffer_load_b64(rq, in ? qoff[f] : kOob, pr * 64, 0);
        const u32x2 b1 = __builtin_amdgcn_raw_buffer_load_b64(rq, in1 ? qoff[f] + 16u : kOob, pr * 64, 0);
        const uint32_t s0 = (uint16_t)__builtin_amdgcn_raw_buffer_load_b16(rs, in ? soff[f] : kOob, pr * 8, 0);
        const uint32_t s1 = (uint16_t)__builtin_amdgcn_raw_buffer_load_b16(rs, in1 ? soff[f] + 2u : kOob, pr * 8, 0);
        q[f] = u32x4{b0[0], b0[1], b1[0], b1[1]};
        sc[f] = s0 | s1 << 16;
      } else {
        q[f] = __builtin_amdgcn_raw_buffer_load_b128(rq, (in ? qoff[f >> 1] : kOob) + 256u * (f & 1),
                                                     pr * 2 * kQ4PanelRecord, 0);
        sc[f] = __builtin_amdgcn_raw_buffer_load_b32(rs, (in ? soff[f >> 1] : kOob) + 64u * (f & 1),
                                                     pr * 2 * kQ4PanelRecord, 0);
      }
    }
  };
  // --- X of one step: rows 4j .. 4j+3 per DMA instruction, lane = (row, position) ---
  const rsrc_t rx = make_rsrc(a.x, (uint32_t)a.m * (uint32_t)a.ldx * 2u);
  char *slot = smem + wave * sa.xrows * (kPairK * 2);
  const uint32_t xbase = (uint32_t)g * (uint32_t)a.ldx * 2u;
  const uint32_t xchunk = 16u * (r16 ^ g);  // of row 4j + g: XORed with 64 (j % 4)
  auto issue_x = [&](int pr) __attribute__((always_inline)) {
    const int left = a.k * 2 - pr * (kPairK * 2);  // bytes of the row from this step on
#pragma unroll
    for (int j = 0; j < 4 * MT; j++) {
      if (4 * j >= sa.xrows) break;
      const uint32_t c = xchunk ^ (64u * (j & 3));
      const bool in = 4 * j + g < a.m && (int)c < left;
      dma16(rx, slot + j * 1024, in ? xbase + (uint32_t)(4 * j) * (uint32_t)a.ldx * 2u + c : kOob, pr * kPairK * 2);
    }
  };

  floatx4 acc[MT][NF];
#pragma unroll
  for (int i = 0; i < MT; i++)
#pragma unroll
    for (int f = 0; f < NF; f++) acc[i][f] = floatx4{0.0f, 0.0f, 0.0f, 0.0f};

  // X rows of the A operands; rows past the staged ones repeat the last (their sums are
  // never stored)
  int xrow[MT], xsw[MT];
#pragma unroll
  for (int i = 0; i < MT; i++) {
    const int row = min(16 * i + r16, sa.xrows - 1);
    xrow[i] = row * (kPairK * 2);
    xsw[i] = 16 * (row & 15);
  }
  const int c0 = 16 * (8 * (g >> 1) + (g & 1));  // MFMA 0's chunk, in bytes
  const int p0 = ks * sa.split_pairs, p1 = min(sa.npairs, p0 + sa.split_pairs);
  // X first: the wait for it leaves the weights in flight, and each fragment is multiplied
  // as its weights land.
  auto load = [&](int pr) __attribute__((always_inline)) {
    issue_x(pr);
    __builtin_amdgcn_sched_barrier(0);
    load_w(pr);
    __builtin_amdgcn_sched_barrier(0);
  };
  int pr = p0 + wave;
  if (pr < p1) load(pr);
  // RoPE: cos/sin of the tile group this wave owns in the epilogue (see there), loaded
  // with everything else
  const int own0 = wave;
  float4 ca0{}, cb0{};
  auto rope_cs = [&](int row, int e0, float4 &ca, float4 &cb) __attribute__((always_inline)) {
    if constexpr (EPI == EPI_ROPE) {
      const int hhalf = a.rope.head_dim >> 1;
      const int idx = a.rope.mode != 0 ? e0 & (hhalf - 1) : e0 / 2;
      const float4 *cs = reinterpret_cast<const float4 *>(a.rope.cs + 2 * ((size_t)min(row, a.m - 1) * hhalf + idx));
      ca = cs[0];
      cb = cs[a.rope.mode != 0 ? 1 : 0];
    }
  };
  const int qj = lane & 3, cq4 = 4 * (r16 >> 2);
  auto rope_col = [&](int f) { return (head << (6 + hsh)) + 32 * hi + (f >> 1) * (32 << hsh) + 16 * (f & 1); };
  if constexpr (EPI == EPI_ROPE) {
    if (si < 2) rope_cs(16 * (own0 / NF) + 4 * (own0 % NF) + qj, (rope_col(g) + cq4) & ((64 << hsh) - 1), ca0, cb0);
  }
  while (pr < p1) {
    // the step's X has landed: at least the 2 NF weight loads are younger
    wait_vmcnt<2 * NF>();
    __builtin_amdgcn_sched_barrier(0);
    half8 av[MT][4];
#pragma unroll
    for (int i = 0; i < MT; i++)
#pragma unroll
      for (int s = 0; s < 4; s++) {
        const int dc = 16 * (4 * (s >> 1) + 2 * (s & 1));
        av[i][s] = *reinterpret_cast<const half8 *>(slot + xrow[i] + ((c0 + dc) ^ xsw[i]));
      }
#pragma unroll
    for (int f = 0; f < NF; f++) {
      const half2v dlo = as_h2(__builtin_amdgcn_perm(sc[f], sc[f], 0x01000100u));
      const half2v dhi = as_h2(__builtin_amdgcn_perm(sc[f], sc[f], 0x03020302u));
#pragma unroll
      for (int s = 0; s < 4; s++) {
        const half2v d2 = s < 2 ? dlo : dhi;
        const uint32_t x = s < 2 ? q[f][0] : q[f][2], y = s < 2 ? q[f][1] : q[f][3];
        half2v w0, w1, w2, w3;
        if (s & 1) {
          dq4<true>(x & 0xF0F0F0F0u, d2, w0, w1);
          dq4<true>(y & 0xF0F0F0F0u, d2, w2, w3);
        } else {
          dq4<false>(x & 0x0F0F0F0Fu, d2, w0, w1);
          dq4<false>(y & 0x0F0F0F0Fu, d2, w2, w3);
        }
        const half8 b = half8{w0[0], w0[1], w1[0], w1[1], w2[0], w2[1], w3[0], w3[1]};
#pragma unroll
        for (int i = 0; i < MT; i++) acc[i][f] = __builtin_amdgcn_mfma_f32_16x16x32_f16(av[i][s], b, acc[i][f], 0, 0, 0);
      }
    }
    pr += nwaves;
    if (pr < p1) {
      // every A operand of the step has left the slot
      asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
      __builtin_amdgcn_sched_barrier(0);
      load(pr);
    }
  }

  // --- the waves' sums meet in LDS (over the X slots). A 16-row tile is 4 NF groups of 16
  // lanes, group (f, gg) = rows 4gg .. +3 of fragment f's columns; an owner wave adds 4
  // groups over the waves, in wave order, and runs the epilogue for them. ---
  float4 *red = reinterpret_cast<float4 *>(smem);
  lds_barrier();
#pragma unroll
  for (int i = 0; i < MT; i++)
#pragma unroll
    for (int f = 0; f < NF; f++)
      red[((i * nwaves + wave) * NF + f) * 64 + lane] = float4{acc[i][f][0], acc[i][f][1], acc[i][f][2], acc[i][f][3]};
  lds_barrier();
  for (int o = wave; o < MT * NF; o += nwaves) {
    const int i = o / NF;  // 16-row tile
    const int id = 4 * (o % NF) + g, f = id % NF, gg = id / NF;
    const float4 *red_t = red + (size_t)i * nwaves * NF * 64;
    float4 v = red_t[f * 64 + 16 * gg + r16];
#pragma unroll 4
    for (int w = 1; w < nwaves; w++) {
      const float4 t = red_t[(w * NF + f) * 64 + 16 * gg + r16];
      v.x += t.x;
      v.y += t.y;
      v.z += t.z;
      v.w += t.w;
    }
    // the lane's column before the quad transpose, and row / first column after it
    const int row = 16 * i + 4 * gg + qj;
    if constexpr (EPI == EPI_SWIGLU) {
      // gate fragments (lanes 0-31) and up fragments (lanes 32-63), f16-rounded first
      const float gv[4] = {(float)(_Float16)v.x, (float)(_Float16)v.y, (float)(_Float16)v.z, (float)(_Float16)v.w};
      float s[4];
#pragma unroll
      for (int e = 0; e < 4; e++) s[e] = silu_mul(gv[e], __shfl_xor(gv[e], 32, 64));
      const uint2 w = quad_t16(pack_h2(s[0], s[1]), pack_h2(s[2], s[3]), qj);
      const int col = UC * u + 16 * (f & 1) + cq4;
      if (lane < 32 && row < a.m && col < seg.n) {
        _Float16 *dst = reinterpret_cast<_Float16 *>(seg.out) + (size_t)row * seg.ldo + seg.col0 + col;
        if (((seg.ldo | seg.col0) & 3) == 0 && ((uintptr_t)seg.out & 7) == 0 && col + 4 <= seg.n) {
          *reinterpret_cast<uint2 *>(dst) = w;
        } else {
          const uint32_t ww[2] = {w.x, w.y};
          for (int e = 0; e < 4 && col + e < seg.n; e++)
            reinterpret_cast<uint16_t *>(dst)[e] = (uint16_t)(ww[e >> 1] >> (16 * (e & 1)));
        }
      }
    } else if constexpr (EPI == EPI_ROPE) {
      // RoPE + Q8_0 K/V store: the values and rounding points of gemm_q4_0.hip's RoPE
      // epilogue. Lanes 0-31 hold 32 columns of the first half of a head, lanes 32-63
      // the columns head_dim/2 further: a Q8_0 block is half a wave, NeoX partners are
      // lanes l and l ^ 32.
      const GemmRope &rp = a.rope;
      const int hd = rp.head_dim;
      const bool neox = rp.mode != 0, rotate = si < 2;
      const int fcol = rope_col(f);  // fragment's first column
      const float b = seg.bias ? seg.bias[fcol + r16] : 0.0f;
      const int col = fcol + cq4, e0 = col & (hd - 1);
      float4 ca = ca0, cb = cb0;
      if (rotate && o != own0) rope_cs(row, e0, ca, cb);
      const uint2 xv = quad_t16(pack_h2(v.x + b, v.y + b), pack_h2(v.z + b, v.w + b), qj);
      const half2v x01 = as_h2(xv.x), x23 = as_h2(xv.y);
      const float x[4] = {(float)x01[0], (float)x01[1], (float)x23[0], (float)x23[1]};
      float out[4] = {x[0], x[1], x[2], x[3]};
      if (rotate && neox) {
        const half2v p01 = as_h2((uint32_t)__shfl_xor((int)xv.x, 32, 64)), p23 = as_h2((uint32_t)__shfl_xor((int)xv.y, 32, 64));
        const float p[4] = {(float)p01[0], (float)p01[1], (float)p23[0], (float)p23[1]};
        const float cc[4] = {ca.x, ca.z, cb.x, cb.z}, ss[4] = {ca.y, ca.w, cb.y, cb.w};
#pragma unroll
        for (int j = 0; j < 4; j++)
          out[j] = lane < 32 ? rot_sub(x[j], cc[j], p[j], ss[j]) : rot_add(p[j], ss[j], x[j], cc[j]);
      } else if (rotate) {
        const float cc[2] = {ca.x, ca.z}, ss[2] = {ca.y, ca.w};
#pragma unroll
        for (int j = 0; j < 4; j += 2) {
          out[j] = rot_sub(x[j], cc[j / 2], x[j + 1], ss[j / 2]);
          out[j + 1] = rot_add(x[j], ss[j / 2], x[j + 1], cc[j / 2]);
        }
      }
      const bool ok = row < a.m;
      if (si == 0) {
        if (ok)
          *reinterpret_cast<uint2 *>(reinterpret_cast<_Float16 *>(seg.out) + (size_t)row * seg.ldo + seg.col0 + col) =
              uint2{pack_h2(out[0], out[1]), pack_h2(out[2], out[3])};
        continue;
      }
      float amax = fmaxf(fmaxf(fabsf(out[0]), fabsf(out[1])), fmaxf(fabsf(out[2]), fabsf(out[3])));
#pragma unroll
      for (int sh = 4; sh <= 16; sh *= 2) amax = fmaxf(amax, __shfl_xor(amax, sh, 64));
      const float d = amax / 127.0f;
      const float id = d != 0.0f ? 1.0f / d : 0.0f;
      float qc[4];
#pragma unroll
      for (int j = 0; j < 4; j++) qc[j] = fminf(fmaxf(roundf(out[j] * id), -128.0f), 127.0f);
      const int kvh = head, e = e0;
      if (ok) {
        int slot_i = rp.slot0 + row;
        if (slot_i >= rp.wrap) slot_i %= rp.wrap;
        uint8_t *blk = (si == 1 ? rp.k_dst : rp.v_dst) + (size_t)slot_i * rp.row_bytes +
                       (size_t)(kvh * (hd >> 5) + (e >> 5)) * 34;
        if ((e & 31) == 0) *reinterpret_cast<_Float16 *>(blk) = (_Float16)d;
        uint16_t *codes = reinterpret_cast<uint16_t *>(blk + 2 + (e & 31));  // 2-byte aligned
#pragma unroll
        for (int j = 0; j < 4; j += 2)
          codes[j / 2] = (uint16_t)((uint8_t)(int8_t)(int)qc[j] | ((uint16_t)(uint8_t)(int8_t)(int)qc[j + 1] << 8));
      }
      if (!rp.win.k) continue;
      // window entries f16(code * f16(d))
      const float dq = (float)(_Float16)d;
      const uint2 w = uint2{pack_h2(qc[0] * dq, qc[1] * dq), pack_h2(qc[2] * dq, qc[3] * dq)};
      if (si == 1) {
        if (ok)
          *reinterpret_cast<uint2 *>(reinterpret_cast<_Float16 *>(rp.win.k) +
                                     ((size_t)kvh * rp.win.pad + rp.win.j0 + row) * hd + e) = w;
      } else {
        // back to one column per lane: column fcol + r16, tokens t0 .. t0+3
        const uint2 wt = quad_t16(w.x, w.y, qj);
        const int t0 = 16 * i + 4 * gg, cv = fcol + r16;
        if (t0 >= a.m) continue;
        _Float16 *vrow = reinterpret_cast<_Float16 *>(rp.win.vt) + (size_t)cv * rp.win.vst;
        const int j = rp.win.j0 + t0;
        if ((j & 3) == 0 && t0 + 3 < a.m) {
          *reinterpret_cast<uint2 *>(vrow + window_vt_col(j)) = wt;  // 4 consecutive columns
        } else {
          const uint32_t ww[2] = {wt.x, wt.y};
          for (int jj = 0; jj < 4 && t0 + jj < a.m; jj++)
            reinterpret_cast<uint16_t *>(vrow)[window_vt_col(j + jj)] = (uint16_t)(ww[jj >> 1] >> (16 * (jj & 1)));
        }
      }
    } else {
      const int fcol = (NF == 1 ? 16 * u : UC * u + 16 * f);
      if constexpr (EPI == EPI_F16 || EPI == EPI_F32) {
        if (seg.bias) {
          const float b = fcol + r16 < seg.n ? seg.bias[fcol + r16] : 0.0f;
          v = float4{v.x + b, v.y + b, v.z + b, v.w + b};
        }
      }
      const int col = fcol + cq4;
      const bool in = row < a.m && col < seg.n;
      if constexpr (EPI == EPI_F16) {
        const uint2 w = quad_t16(pack_h2(v.x, v.y), pack_h2(v.z, v.w), qj);
        if (in) {
          _Float16 *dst = reinterpret_cast<_Float16 *>(seg.out) + (size_t)row * seg.ldo + seg.col0 + col;
          if (((seg.ldo | seg.col0) & 3) == 0 && ((uintptr_t)seg.out & 7) == 0 && col + 4 <= seg.n) {
            *reinterpret_cast<uint2 *>(dst) = w;
          } else {
            const uint32_t ww[2] = {w.x, w.y};
            for (int e = 0; e < 4 && col + e < seg.n; e++)
              reinterpret_cast<uint16_t *>(dst)[e] = (uint16_t)(ww[e >> 1] >> (16 * (e & 1)));
          }
        }
      } else {
        if constexpr (EPI == EPI_RESID)  // x += f16(acc)
          v = float4{(float)(_Float16)v.x, (float)(_Float16)v.y, (float)(_Float16)v.z, (float)(_Float16)v.w};
        const float4 w = quad_t32(v.x, v.y, v.z, v.w, qj);
        if (in) {
          float *dst;
          bool vec;
          if constexpr (EPI == EPI_PART) {  // f32 partials, rows 4-column aligned (checked by the planner)
            dst = a.part + ((size_t)ks * a.m + row) * a.ldp + colbase + col;
            vec = col + 4 <= seg.n;
          } else {
            dst = reinterpret_cast<float *>(seg.out) + (size_t)row * seg.ldo + seg.col0 + col;
            vec = ((seg.ldo | seg.col0) & 3) == 0 && ((uintptr_t)seg.out & 15) == 0 && col + 4 <= seg.n;
          }
          if (vec) {
            float4 o4 = w;
            if constexpr (EPI == EPI_RESID) {
              const float4 old = *reinterpret_cast<const float4 *>(dst);
              o4 = float4{old.x + w.x, old.y + w.y, old.z + w.z, old.w + w.w};
            }
            *reinterpret_cast<float4 *>(dst) = o4;
          } else {
            const float ww[4] = {w.x, w.y, w.z, w.w};
            for (int e = 0; e < 4 && col + e < seg.n; e++) dst[e] = EPI == EPI_RESID ? dst[e] + ww[e] : ww[e];
          }
        }
      }
    }
  }
}

int unit_cols_of(const GemmArgs &a, int nf) { return a.epi == EPI_SWIGLU ? 8 * nf : 16 * nf; }

int units_of(const GemmArgs &a, int nf) {
  const int uc = unit_cols_of(a, nf);
  int u = 0;
  for (int i = 0; i < a.nseg; i++) u += (a.seg[i].n + uc - 1) / uc;
  return u;
}

int pairs_of(const GemmArgs &a) { return (a.k + kPairK - 1) / kPairK; }

template <int MT, int NF, int EPI, bool SOA>
int32_t launch_skinny_t(const SkinnyArgs &sa, int splits, hipStream_t s, LaunchStamp st) {
  // One step per wave where LDS holds the waves' X, the steps spread evenly over them
  // otherwise. Up to one workgroup per CU may take the CU's whole LDS. More workgroups
  // than CUs must run side by side (a second round costs the kernel's whole latency
  // again): four waves each (gate/up of 280 workgroups: at 23 tokens 9.6 us against 11.2
  // with six and 12.7 with twelve, at 40 tokens 11.4 against 14.7; of 256 workgroups: at 23
  // tokens 10.2 with twelve and 12.2 with four, at 40 12.4 and 14.7).
  const int slot = sa.xrows * kPairK * 2;
  const bool alone = sa.units * splits <= device_cu_count();
  constexpr int kRoomAlone = 156 << 10, kRoomShared = 76 << 10, kWavesShared = 4;
  constexpr int kTiles = NF * MT * 1024;  // bytes of one wave's sums, which meet in LDS
  static_assert(max_waves(MT, NF) * kTiles <= kRoomAlone && kWavesShared * kTiles <= kRoomShared, "the waves' sums fit");
  const size_t room = alone ? kRoomAlone : kRoomShared;
  const int most = std::max(1, std::min({alone ? max_waves(MT, NF) : kWavesShared, (int)(room / slot)}));
  const int iters = (sa.split_pairs + most - 1) / most;
  const int waves = (sa.split_pairs + iters - 1) / iters;
  const size_t lds = (size_t)waves * std::max(slot, kTiles);
  launch_stamped(skinny_kernel<MT, NF, EPI, SOA>, dim3((unsigned)sa.units, (unsigned)splits), dim3(64 * waves), lds, s,
                 st.start, st.stop, sa);
  const hipError_t e = hipGetLastError();
  return e == hipSuccess ? SULIMO_HIP_OK : hip_fail(e, "skinny_kernel launch");
}

template <int NF, int EPI, bool SOA = false>
int32_t launch_skinny_mt(const SkinnyArgs &sa, int splits, hipStream_t s, LaunchStamp st) {
  switch ((sa.g.m + 15) / 16) {
    case 1: return launch_skinny_t<1, NF, EPI, SOA>(sa, splits, s, st);
    case 2: return launch_skinny_t<2, NF, EPI, SOA>(sa, splits, s, st);
    case 3: return launch_skinny_t<3, NF, EPI, SOA>(sa, splits, s, st);
    default: return launch_skinny_t<4, NF, EPI, SOA>(sa, splits, s, st);
  }
}

SkinnyArgs skinny_args(const GemmArgs &a, int nf, int *splits) {
  SkinnyArgs sa{};
  sa.g = a;
  sa.units = units_of(a, nf);
  sa.npairs = pairs_of(a);
  sa.split_pairs = (sa.npairs + *splits - 1) / *splits;
  *splits = (sa.npairs + sa.split_pairs - 1) / sa.split_pairs;
  sa.xrows = (a.m + 3) / 4 * 4;
  return sa;
}

}  // namespace

// Token counts and widths the skinny kernel takes from the tiled one: up to 64 tokens (48
// with the RoPE epilogue, whose units of 64 columns leave few workgroups: 12.7 us against
// 11.4 tiled at 64, 11.0 against 11.5 at 48; at 64 tokens the others still gain, the two
// models' shapes: gate/up 13.9 and 14.8 us against 17.3 and 27.0 tiled, o and down with
// their norm 10.2 to 18.5 against 10.8 to 21.9, single f16 projections 6.0 to 14.9 against
// 9.0 to 15.1; more tokens than four tiles of 16 rows are not built), and few enough
// columns that a unit of 64 leaves at most two workgroups per CU (beyond that each CU would
// read X again and again, and the tiles of the other kernel fill the chip).
bool skinny_fits(const GemmArgs &a) {
  if (a.m < 1 || a.m > kSkinnyMaxTokens || a.ldx % 8) return false;
  if (a.epi == EPI_ROPE) {
    if (a.m > kSkinnyMaxRopeTokens) return false;
    if (a.rope.head_dim != 64 && a.rope.head_dim != 128) return false;
    for (int i = 0; i < a.nseg; i++)
      if (a.seg[i].n % a.rope.head_dim) return false;
  }
  return units_of(a, 4) <= 2 * device_cu_count();
}

// A residual GEMM's reduction takes the place of the RMSNorm launch after it, so it splits
// until the workgroups fill the CUs (at least three steps each). A plain f16 one pays a
// launch for it: only long k of few columns at more than 16 tokens (1536 x 8960 at 37
// tokens: 10.1 us against 11.6 unsplit, 12.9 tiled; at 8 tokens 8.7 against 7.6; 3072 x
// 8192, where two splits fill the CUs, 12.6 against 11.9).
int skinny_splits(const GemmArgs &a, bool unbounded) {
  if (a.epi != EPI_RESID && a.epi != EPI_F16) return 1;
  for (int i = 0; i < a.nseg; i++)
    if (a.seg[i].n % 4 || a.seg[i].ldo % 4 || a.seg[i].col0 % 4) return 1;
  // the reductions of f32 partials with the norm hold rows of up to 4096 columns (256 CUs
  // leave no wider matrix a split)
  if (a.epi == EPI_RESID && a.seg[0].n > 4096) return 1;
  const int pairs = pairs_of(a);
  int splits = std::min({kMaxSplits, device_cu_count() / std::max(1, units_of(a, 2)), (pairs + 2) / 3});
  if (splits < 2 || (a.epi == EPI_F16 && (a.m <= 16 || pairs < 32 || splits < 4))) return 1;
  skinny_args(a, 2, &splits);
  size_t cols = 0;
  for (int i = 0; i < a.nseg; i++) cols += a.seg[i].n;
  if (!unbounded && (!a.part || (size_t)splits * a.m * cols * 4 > a.part_bytes)) return 1;
  return splits;
}

namespace {
// 16 columns per workgroup while that leaves no CU a second one, else 32, else 64.
int fragments_of(const GemmArgs &a) {
  const int cus = device_cu_count();
  return units_of(a, 1) <= cus ? 1 : units_of(a, 2) <= 2 * cus ? 2 : 4;
}
}  // namespace

int32_t launch_skinny_soa(const GemmArgs &a, const uint16_t *scales, const uint8_t *quants, hipStream_t s) {
  if (a.epi != EPI_F16 || a.nseg != 1 || !skinny_fits(a))
    return fail(SULIMO_HIP_ERR_INVALID_ARGUMENT, "not a GEMM the skinny kernel reads from the source arrays");
  const int nf = fragments_of(a);
  int one = 1;
  SkinnyArgs sa = skinny_args(a, nf, &one);
  sa.scales = scales;
  sa.quants = quants;
  return nf == 1   ? launch_skinny_mt<1, EPI_F16, true>(sa, 1, s, LaunchStamp{})
         : nf == 2 ? launch_skinny_mt<2, EPI_F16, true>(sa, 1, s, LaunchStamp{})
                   : launch_skinny_mt<4, EPI_F16, true>(sa, 1, s, LaunchStamp{});
}

int32_t launch_skinny(const GemmArgs &a, hipStream_t s, LaunchStamp st) {
  int one = 1;
  if (a.epi == EPI_PART) {
    int splits = a.splits;
    const SkinnyArgs sa = skinny_args(a, 2, &splits);
    return launch_skinny_mt<2, EPI_PART>(sa, splits, s, st);
  }
  if (a.epi == EPI_SWIGLU) return launch_skinny_mt<4, EPI_SWIGLU>(skinny_args(a, 4, &one), 1, s, st);
  if (a.epi == EPI_ROPE) return launch_skinny_mt<4, EPI_ROPE>(skinny_args(a, 4, &one), 1, s, st);
  const int nf = fragments_of(a);
  const SkinnyArgs sa = skinny_args(a, nf, &one);
#define SULIMO_SKINNY(EPI)                                   \
  return nf == 1   ? launch_skinny_mt<1, EPI>(sa, 1, s, st)  \
         : nf == 2 ? launch_skinny_mt<2, EPI>(sa, 1, s, st)  \
                   : launch_skinny_mt<4, EPI>(sa, 1, s, st);
  switch (a.epi) {
    case EPI_F16: SULIMO_SKINNY(EPI_F16)
    case EPI_F32: SULIMO_SKINNY(EPI_F32)
    case EPI_RESID: SULIMO_SKINNY(EPI_RESID)
    default: return fail(SULIMO_HIP_ERR_INVALID_ARGUMENT, "unknown GEMM epilogue");
  }
#undef SULIMO_SKINNY
}

}  // namespace sulimo
