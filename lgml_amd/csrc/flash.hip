// Attention over strided K / V views with an explicit additive mask: the
// semantics of graph:flash_attn (src/lgml.c:2121-2170), i.e.
// ggml_flash_attn_ext's softmax(scale q k^T [softcap] + slope * mask) v.
// It serves callers whose K / V are plain (n_kv, Hkv * D) rows rather than
// this library's block pool (the paged path is attn.hip).
//
// The rows of a KV head are its T * G (token, query head) pairs, 16 to a
// wave. A workgroup is KW groups of RW waves: the waves of a group take
// consecutive row tiles over the same cells, the groups take the 64- (or 32-)
// cell tiles in turn (tile i is group i % KW's), and their states are merged
// in group order at the end. Per tile a group stages K as rows and V
// transposed in LDS, from registers that were loaded while the tile before
// was computed; a wave computes S^T = K Q^T with 16x16x32 f16 MFMAs, an
// online softmax in f32 (a lane owns one row), and O^T += V^T P^T.
//
// K and V are exact f16; Q and P enter the MFMAs as f16 hi + lo pairs, with
// the largest of a row near f16's (Q by a power of two per row, so any f32
// row fits; P FA_P times as large, O with it, and l in the end: the factor
// cancels) and the low parts FA_LO times as large again, with products
// of their own: a pair carries 22 bits of every value down to 2^-28 of the
// row's largest, and what is lost below is at most 2^-51 of that. (With the
// largest at 1 and one sum for both, q values below 2^-14 of it lost bits: rows
// with one value 2^14 to 2^22 times the others, where K is 0, were wrong by up
// to 24%. P below 2^-25 was 0 in O but counted in l, and one cell 16 above
// 2048 others made 4% to 20% of the result wrong; P 2^15 times as large alone
// leaves up to 8e-6 there.) The MFMA's k index over 32 cells is taken in the
// order (quad, tile of 16, i): a lane's own S^T values then are its B operand
// of the second product, with no trip through LDS, and V^T is stored in that
// order of cells.
//
// An infinity in Q or K has no pair: its products with the low parts are NaN
// where the score is an infinity (-inf drops the cell; with a softcap it is
// one of +- softcap). A row that ends with a sum that is not a number is
// therefore computed again from f32 products (exact_row), whichever it holds.
// (At the end it costs other calls up to 1.5%; scoring the tile again where it
// happens took registers of the loop, 512 x 2048 cells 69 -> 72 us.)
//
// A masked cell (mask -inf, or past n_kv) adds nothing whatever K and V
// hold there: its score is set, and a V value that is not finite is stored
// as 0 for the MFMAs and added afterwards to the rows that do see its cell.
//
// What bounds it: the f16 MFMAs (twice the products' flops for the hi + lo
// pairs) and the softmax's VALU, which overlap only in part (the two waves of
// a SIMD run in step). 32 / 8 heads of 128, 512 rows over 2048 cells under a
// causal mask: 69 us, 218 TFLOP/s of the products (2458 us with one wave per
// query row and head, each column's dot product in VALU; 66 with P's low
// parts unscaled and added in the MFMAs).
#include <math.h>

#include "common.h"

namespace lgmlh {

constexpr int FA_MAX_D = 256;
constexpr float FA_LOG2E = 1.4426950408889634f;
constexpr float FA_P = 32768.0f, FA_LO = 4096.0f;  // the scales of P and of a low part

// ALiBi slope of head h (1 without max_bias): with n the largest power of
// two <= H, heads below n take (2^(-max_bias / n))^(h + 1), the others
// (2^(-max_bias / 2 / n))^(2 (h - n) + 1).
__device__ __forceinline__ float alibi(int h, int H, float max_bias) {
  if (max_bias <= 0.0f) return 1.0f;
  int n = 1;
  while (n * 2 <= H) n *= 2;
  const float m0 = powf(2.0f, -max_bias / (float)n);
  const float m1 = powf(2.0f, -(max_bias / 2.0f) / (float)n);
  return h < n ? powf(m0, (float)(h + 1)) : powf(m1, (float)(2 * (h - n) + 1));
}

// Vectors of memory that need not be aligned to their size (Q, V, mask and
// out start anywhere their elements may; the hardware loads such addresses,
// and aligned ones as fast as ever).
typedef float f32x2 __attribute__((ext_vector_type(2)));
typedef u32x4 u32x4_u __attribute__((aligned(2)));
typedef u32x2 u32x2_u __attribute__((aligned(2)));

struct FlashArgs {
  const float *q;
  const uint16_t *k, *v, *mask;
  float *out;
  int H, T, D, G, n_kv, mask_heads, mask_rows;
  int64_t k_rs, k_hs, v_rs, v_hs;
  float scale, max_bias, softcap;
};

// Row rr of KV head kvh by one wave, from f32 products: a cell per lane, then
// D / 64 output values per lane.
__device__ void exact_row(const FlashArgs &A, int kvh, uint32_t rr) {
  const int t = rr / (uint32_t)A.G, h = kvh * A.G + rr % (uint32_t)A.G, lane = threadIdx.x & 63;
  const float slope = alibi(h, A.H, A.max_bias);
  const float *qr = A.q + ((int64_t)h * A.T + t) * A.D;
  const uint16_t *mr = A.mask ? A.mask + ((int64_t)(h % A.mask_heads) * A.mask_rows + t) * A.n_kv
                              : nullptr;
  const uint16_t *kb = A.k + (int64_t)kvh * A.k_hs, *vb = A.v + (int64_t)kvh * A.v_hs;
  const float sc = A.softcap > 0.0f ? A.scale / A.softcap : A.scale;
  float m = -INFINITY, l = 0.0f, o[FA_MAX_D / 64];
#pragma unroll
  for (int i = 0; i < FA_MAX_D / 64; i++) o[i] = 0.0f;
  for (int j0 = 0; j0 < A.n_kv; j0 += 64) {
    const int j = j0 + lane;
    const float mv = j >= A.n_kv ? -INFINITY : mr ? h2f(mr[j]) : 0.0f;
    float s = -INFINITY;
    if (mv != -INFINITY) {
      const uint16_t *kr = kb + (int64_t)j * A.k_rs;
      float a = 0.0f;
#pragma unroll 4
      for (int d = 0; d < A.D; d += 8) {
        const u32x4 w = *(const u32x4 *)(kr + d);
#pragma unroll
        for (int e = 0; e < 4; e++) {
          a = fmaf(qr[d + 2 * e], h2f((uint16_t)(w[e] & 0xffffu)), a);
          a = fmaf(qr[d + 2 * e + 1], h2f((uint16_t)(w[e] >> 16)), a);
        }
      }
      a *= sc;
      if (A.softcap > 0.0f) a = A.softcap * tanhf(a);
      s = a + slope * mv;
    }
    float mt = s;
    for (int x = 32; x > 0; x >>= 1) mt = fmaxf(mt, __shfl_xor(mt, x));
    const float mn = fmaxf(m, mt), mu = mn == -INFINITY ? 0.0f : mn;
    const float corr = expf(m - mu), p = expf(s - mu);  // 0 at -inf
    float ps = p;
    for (int x = 32; x > 0; x >>= 1) ps += __shfl_xor(ps, x);
    l = l * corr + ps;
#pragma unroll
    for (int i = 0; i < FA_MAX_D / 64; i++) o[i] *= corr;
    const int nj = min(A.n_kv - j0, 64);
#pragma unroll 1
    for (int j1 = 0; j1 < nj; j1 += 4) {  // four cells' values in flight
      uint16_t x[4][FA_MAX_D / 64];
#pragma unroll
      for (int c = 0; c < 4; c++) {
        const uint16_t *vr = vb + (int64_t)(j0 + min(j1 + c, nj - 1)) * A.v_rs;
#pragma unroll
        for (int i = 0; i < FA_MAX_D / 64; i++) x[c][i] = lane + 64 * i < A.D ? vr[lane + 64 * i] : 0;
      }
#pragma unroll
      for (int c = 0; c < 4; c++) {
        const float pj = __shfl(p, j1 + c);
        if (pj == 0.0f || j1 + c >= nj) continue;  // wave-uniform
#pragma unroll
        for (int i = 0; i < FA_MAX_D / 64; i++) o[i] = fmaf(pj, h2f(x[c][i]), o[i]);
      }
    }
    m = mn;
  }
  float *orow = A.out + ((int64_t)t * A.H + h) * A.D;
  const float inv = l == 0.0f ? 0.0f : 1.0f / l;
#pragma unroll
  for (int i = 0; i < FA_MAX_D / 64; i++)
    if (lane + 64 * i < A.D) orow[lane + 64 * i] = o[i] * inv;
}

// Calls of few cells: a wave per row.
__global__ void __launch_bounds__(64) flash_row_kernel(FlashArgs A) {
  exact_row(A, blockIdx.y, blockIdx.x);
}

// DP: the head size padded to the MFMA step (zeros past D); BC: cells per
// tile.
template <int DP, int BC, int RW, int KW>
__global__ void __launch_bounds__(RW *KW * 64, 1) flash_attn_kernel(FlashArgs A) {
  constexpr int KS = DP / 32, DT = DP / 16, CT = BC / 16, CJ = BC / 32;
  constexpr int KROW = DP + 8, VROW = BC + 8;  // f16 per LDS row: conflict-free 16-row reads
  // A group of one wave takes its K fragments straight from memory.
  constexpr bool KLDS = RW > 1;
  constexpr int KT = KLDS ? BC * KROW : 0, VT = DP * VROW, NT = RW * 64;
  constexpr int KU = (BC * (DP / 8) + NT - 1) / NT;        // 16-byte K pieces per thread
  constexpr int VU = ((BC / 4) * (DP / 8) + NT - 1) / NT;  // V pieces of 4 cells x 8 values
  constexpr int NB = KLDS ? 2 : 1;                         // stages
  constexpr int STAGE = NB * KW * (KT + VT) * 2;           // bytes
  constexpr int STATE = KW > 1 ? KW * RW * 16 * (DP + 2) * 4 : 0;
  __shared__ __align__(16) uint8_t lds[STAGE > STATE ? STAGE : STATE];
  __shared__ uint32_t bad[3][KW][2];  // cells of a tile with a V value that is not finite

  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int kw = wave / RW, rw = wave % RW;
  const int gt = threadIdx.x - kw * NT;  // thread of the group
  uint16_t *const stage0 = (uint16_t *)lds + kw * NB * (KT + VT);
  auto kl_of = [&](int it) { return stage0 + (NB == 2 ? (it & 1) * (KT + VT) : 0); };
  const int D = A.D, kvh = blockIdx.x;
  const int r16 = lane & 15, quad = lane >> 4;
  // (rows past 2^31 fit a GPU: 32-bit, but unsigned)
  const uint32_t G = A.G, rows = A.T * G;
  const uint32_t rr = ((blockIdx.z * gridDim.y + blockIdx.y) * RW + rw) * 16 + r16;
  const bool rvalid = rr < rows;
  const int t = (rvalid ? rr : 0) / G, h = kvh * A.G + (rvalid ? rr : 0) % G;
  const float slope = alibi(h, A.H, A.max_bias);
  const uint16_t *mr = A.mask ? A.mask + ((int64_t)(h % A.mask_heads) * A.mask_rows + t) * A.n_kv
                              : nullptr;
  const uint16_t *kb = A.k + (int64_t)kvh * A.k_hs, *vb = A.v + (int64_t)kvh * A.v_hs;
  const int ntiles = (A.n_kv + BC - 1) / BC;

  if (threadIdx.x < 6 * KW) (&bad[0][0][0])[threadIdx.x] = 0;

  // Q fragments: row rr scaled by a power of two that brings its largest |q| to
  // [2^14, 2^15), hi + lo.
  f16x8 qh[KS], ql[KS];
  float qscale;
  {
    const float *qr = A.q + ((int64_t)h * A.T + t) * D;
    float x[KS][8], mx = 0.0f;
#pragma unroll
    for (int ks = 0; ks < KS; ks++) {
      const int d0 = ks * 32 + quad * 8;
      f32x4 a = {0, 0, 0, 0}, b = a;
      if (d0 < D && rvalid) {
        a = *(const f32x4_u *)(qr + d0);
        b = *(const f32x4_u *)(qr + d0 + 4);
      }
#pragma unroll
      for (int e = 0; e < 4; e++) {
        x[ks][e] = a[e];
        x[ks][4 + e] = b[e];
      }
#pragma unroll
      for (int e = 0; e < 8; e++) mx = fmaxf(mx, fabsf(x[ks][e]));
    }
    mx = fmaxf(mx, __shfl_xor(mx, 16));
    mx = fmaxf(mx, __shfl_xor(mx, 32));
    // (rows below 2^-112 by the power of that)
    const int ex = min(max((int)(__builtin_bit_cast(uint32_t, mx) >> 23), 15), 254);
    const float inv = __builtin_bit_cast(float, (uint32_t)(268 - ex) << 23);
    qscale = __builtin_bit_cast(float, (uint32_t)(ex - 14) << 23);
#pragma unroll
    for (int ks = 0; ks < KS; ks++)
#pragma unroll
      for (int e = 0; e < 8; e++) {
        const float v = x[ks][e] * inv;
        qh[ks][e] = (f16)v;
        ql[ks][e] = (f16)((v - (float)qh[ks][e]) * FA_LO);
      }
  }
  // with a softcap the scale goes inside the tanh: softcap tanh(s (scale / softcap))
  const float sc = (A.softcap > 0.0f ? A.scale / A.softcap : A.scale) * qscale;

  // A tile's K rows, V pieces and mask values in registers. Cells past n_kv
  // repeat the last one and are masked. In whole tiles a thread's rows are
  // fixed distances from its first, so that its addresses take one add each.
  u32x4 kr[KU], vr[VU][4];
  u32x2 mk[CT];  // 4 cells of f16 bits (taken apart only when they are used)
  constexpr bool KSTEP = !KLDS || NT % (DP / 8) == 0;
  static_assert(NT % (BC / 4) == 0, "a thread's V pieces are of the same cells");
  auto k_row = [&](int u) { return KLDS ? (gt + u * NT) / (DP / 8) : u / KS * 16 + r16; };
  auto k_col = [&](int u) { return KLDS ? (gt + u * NT) % (DP / 8) * 8 : u % KS * 32 + quad * 8; };
  const int vc0 = gt % (BC / 4) * 4;
  auto v_col = [&](int u) { return (gt + u * NT) / (BC / 4) * 8; };
  const uint16_t *const kp0 = kb + (int64_t)k_row(0) * A.k_rs + k_col(0);
  const uint16_t *const vp0 = vb + (int64_t)vc0 * A.v_rs + v_col(0);
  auto load_k = [&](int tile) {
    const int j0 = tile * BC, jl = A.n_kv - 1;
    if (KSTEP && D == DP && j0 + BC <= A.n_kv) {
      const uint16_t *p = kp0 + (int64_t)j0 * A.k_rs;
#pragma unroll
      for (int u = 0; u < KU; u++)
        kr[u] = KLDS ? *(const u32x4 *)(p + (int64_t)(u * (NT / (DP / 8))) * A.k_rs)
                     : *(const u32x4 *)(p + (int64_t)(u / KS * 16) * A.k_rs + u % KS * 32);
      return;
    }
#pragma unroll
    for (int u = 0; u < KU; u++) {
      const int d0 = k_col(u);
      kr[u] = *(const u32x4 *)(kb + (int64_t)min(j0 + k_row(u), jl) * A.k_rs + (d0 < D ? d0 : 0));
      if (d0 >= D) kr[u] = u32x4{0, 0, 0, 0};
    }
  };
  auto load_vm = [&](int tile) {
    const int j0 = tile * BC, jl = A.n_kv - 1;
    if (D == DP && VU * NT == BC / 4 * (DP / 8) && j0 + BC <= A.n_kv) {
      const uint16_t *p = vp0 + (int64_t)j0 * A.v_rs;
#pragma unroll
      for (int u = 0; u < VU; u++)
#pragma unroll
        for (int i = 0; i < 4; i++)
          vr[u][i] = *(const u32x4_u *)(p + i * A.v_rs + u * (NT / (BC / 4)) * 8);
    } else {
#pragma unroll
      for (int u = 0; u < VU; u++) {
        const uint16_t *s = vb + (v_col(u) < D ? v_col(u) : 0);
#pragma unroll
        for (int i = 0; i < 4; i++)
          vr[u][i] = *(const u32x4_u *)(s + (int64_t)min(j0 + vc0 + i, jl) * A.v_rs);
      }
    }
    if (mr && j0 + BC <= A.n_kv) {
#pragma unroll
      for (int ct = 0; ct < CT; ct++) mk[ct] = *(const u32x2_u *)(mr + j0 + ct * 16 + quad * 4);
    } else {
#pragma unroll
      for (int ct = 0; ct < CT; ct++) {
        uint32_t b[4];
#pragma unroll
        for (int i = 0; i < 4; i++) {
          const int j = j0 + ct * 16 + quad * 4 + i;
          b[i] = j > jl ? 0xfc00u : mr ? mr[min(j, jl)] : 0u;
        }
        mk[ct] = u32x2{b[0] | (b[1] << 16), b[2] | (b[3] << 16)};
      }
    }
  };
  // The registers of a tile to LDS: K rows, V transposed (4 cells of a value
  // are 8 bytes).
  auto store = [&](int it) {
    uint16_t *const kl = kl_of(it), *const vl = kl + KT;
    if constexpr (KLDS) {
#pragma unroll
      for (int u = 0; u < KU; u++) {
        if (k_row(u) < BC) *(u32x4 *)(kl + k_row(u) * KROW + k_col(u)) = kr[u];
      }
    }
#pragma unroll
    for (int u = 0; u < VU; u++) {
      const int c0 = vc0, d0 = v_col(u);
      uint32_t nf = 0;  // bits 15, 31: an exponent of all ones
#pragma unroll
      for (int i = 0; i < 4; i++)
#pragma unroll
        for (int e = 0; e < 4; e++) nf |= (vr[u][i][e] & 0x7fff7fffu) + 0x04000400u;
      if (__builtin_expect((nf & 0x80008000u) != 0, 0)) {
#pragma unroll
        for (int i = 0; i < 4; i++) {
          bool any = false;
#pragma unroll
          for (int e = 0; e < 4; e++) {
            const uint32_t w = vr[u][i][e], f = ((w & 0x7fff7fffu) + 0x04000400u) & 0x80008000u;
            any = any || f;
            vr[u][i][e] = w & ~((f >> 15) * 0xffffu);
          }
          if (any) atomicOr(&bad[it % 3][kw][(c0 + i) >> 5], 1u << ((c0 + i) & 31));
        }
      }
      // cell c of a tile of 32 at place (c % 16 / 4) * 8 + c / 16 * 4 + c % 4
      const int place = (c0 & ~31) + ((c0 & 15) >> 2) * 8 + ((c0 >> 4) & 1) * 4;
      if (d0 < DP)
#pragma unroll
        for (int e = 0; e < 8; e++) {
          const uint32_t s = (e & 1) ? 0x07060302u : 0x05040100u;
          const u32x2 w = {__builtin_amdgcn_perm(vr[u][1][e >> 1], vr[u][0][e >> 1], s),
                           __builtin_amdgcn_perm(vr[u][3][e >> 1], vr[u][2][e >> 1], s)};
          *(u32x2 *)(vl + (d0 + e) * VROW + place) = w;
        }
    }
  };

  f32x4 o[DT];
#pragma unroll
  for (int i = 0; i < DT; i++) o[i] = f32x4{0, 0, 0, 0};
  float m = -INFINITY, l = 0.0f;

  // S^T of a tile.
  f32x4 st[CT];
  auto scores = [&](const uint16_t *kl) {
    // K fragments of a step over D are read while the one before multiplies
    f16x8 kf[2][CT];
    auto read = [&](int ks, f16x8(&f)[CT]) {
#pragma unroll
      for (int ct = 0; ct < CT; ct++)
        f[ct] = KLDS ? *(const f16x8 *)(kl + (ct * 16 + r16) * KROW + ks * 32 + quad * 8)
                     : __builtin_bit_cast(f16x8, kr[(ct * KS + ks) % KU]);
    };
    f32x4 low[CT];  // FA_LO times the products with the low parts
    const f32x4 z = {0, 0, 0, 0};
    read(0, kf[0]);
#pragma unroll
    for (int ks = 0; ks < KS; ks++) {
      if (ks + 1 < KS) read(ks + 1, kf[(ks + 1) & 1]);
      __builtin_amdgcn_sched_barrier(0);
#pragma unroll
      for (int ct = 0; ct < CT; ct++)
        st[ct] = __builtin_amdgcn_mfma_f32_16x16x32_f16(kf[ks & 1][ct], qh[ks], ks ? st[ct] : z, 0, 0, 0);
#pragma unroll
      for (int ct = 0; ct < CT; ct++)
        low[ct] = __builtin_amdgcn_mfma_f32_16x16x32_f16(kf[ks & 1][ct], ql[ks], ks ? low[ct] : z, 0, 0, 0);
      __builtin_amdgcn_sched_barrier(0);
    }
#pragma unroll
    for (int ct = 0; ct < CT; ct++) st[ct] += low[ct] * (1.0f / FA_LO);
  };
  // The softmax of a tile (its mask values in mc) and its products with V.
  auto compute = [&](int tile, int it, const uint16_t *vl, const u32x2 (&mc)[CT]) {
#pragma unroll
    for (int ct = 0; ct < CT; ct++) st[ct] *= sc;
    if (A.softcap > 0.0f) {
#pragma unroll 1
      for (int ct = 0; ct < CT; ct++) {
        f32x4 x = st[0];
#pragma unroll
        for (int i = 0; i < 4; i++) x[i] = A.softcap * tanhf(x[i]);
        // the tiles rotate through st[0], so that no register is indexed
#pragma unroll
        for (int c2 = 0; c2 + 1 < CT; c2++) st[c2] = st[c2 + 1];
        st[CT - 1] = x;
      }
    }
    uint32_t any = 0;
#pragma unroll
    for (int ct = 0; ct < CT; ct++) any |= mc[ct][0] | mc[ct][1];
    if (__builtin_amdgcn_ballot_w64(any != 0)) {  // else every mask value of the tile is 0
#pragma unroll
      for (int ct = 0; ct < CT; ct++)
#pragma unroll
        for (int i = 0; i < 4; i++) {
          const float b = h2f((uint16_t)(mc[ct][i >> 1] >> (16 * (i & 1))));
          st[ct][i] = b == -INFINITY ? -INFINITY : st[ct][i] + slope * b;
        }
    }
    float mx = -INFINITY;
#pragma unroll
    for (int ct = 0; ct < CT; ct++)
#pragma unroll
      for (int i = 0; i < 4; i++) mx = fmaxf(mx, st[ct][i]);
    mx = fmaxf(mx, __shfl_xor(mx, 16));
    mx = fmaxf(mx, __shfl_xor(mx, 32));
    const float m_new = fmaxf(m, mx);
    const float m_use = m_new == -INFINITY ? 0.0f : m_new;
    float rs = 0.0f;
#pragma unroll
    for (int ct = 0; ct < CT; ct++)
#pragma unroll
      for (int i = 0; i < 4; i++) {
        st[ct][i] = __builtin_amdgcn_exp2f((st[ct][i] - m_use) * FA_LOG2E);  // exp2(-inf) = 0
        rs += st[ct][i];
      }
    rs += __shfl_xor(rs, 16);
    rs += __shfl_xor(rs, 32);
    if (__builtin_amdgcn_ballot_w64(m_new != m)) {
      const float alpha = __builtin_amdgcn_exp2f((m - m_use) * FA_LOG2E);  // 0 while m is -inf
      l *= alpha;
#pragma unroll
      for (int dt = 0; dt < DT; dt++) o[dt] *= alpha;
    }
    l += rs;
    m = m_new;
    f16x8 ph[CJ], pl[CJ];
#pragma unroll
    for (int j = 0; j < CJ; j++)
#pragma unroll
      for (int e = 0; e < 8; e += 2) {
        const f32x2 p = {st[2 * j + (e >> 2)][e & 3] * FA_P,
                         st[2 * j + (e >> 2)][(e & 3) + 1] * FA_P};
        const f16x2 hi = __builtin_convertvector(p, f16x2);
        const f32x2 r = {(p[0] - (float)hi[0]) * FA_LO, (p[1] - (float)hi[1]) * FA_LO};
        const f16x2 lo = __builtin_convertvector(r, f16x2);
        ph[j][e] = hi[0];
        ph[j][e + 1] = hi[1];
        pl[j][e] = lo[0];
        pl[j][e + 1] = lo[1];
      }
    f16x8 vf[2][CJ];
    auto read = [&](int dt, f16x8(&f)[CJ]) {
#pragma unroll
      for (int j = 0; j < CJ; j++)
        f[j] = *(const f16x8 *)(vl + (dt * 16 + r16) * VROW + j * 32 + quad * 8);
    };
    // two tiles of D at a time, the next two read meanwhile; their products
    // with the low parts (FA_LO times too large) are added a turn later
    static_assert(DT % 2 == 0, "d tiles in pairs");
    f16x8 vg[2][CJ];
    f32x4 lf[2], lg[2];
    auto add_low = [&](int dt) {
      const int b = dt >> 1 & 1;
      o[dt] += lf[b] * (1.0f / FA_LO);
      o[dt + 1] += lg[b] * (1.0f / FA_LO);
    };
    read(0, vf[0]);
    read(1, vg[0]);
#pragma unroll
    for (int dt = 0; dt < DT; dt += 2) {
      const int b = dt >> 1 & 1;
      if (dt + 2 < DT) {
        read(dt + 2, vf[b ^ 1]);
        read(dt + 3, vg[b ^ 1]);
      }
      __builtin_amdgcn_sched_barrier(0);
#pragma unroll
      for (int j = 0; j < CJ; j++) {
        const f32x4 z = {0, 0, 0, 0};
        o[dt] = __builtin_amdgcn_mfma_f32_16x16x32_f16(vf[b][j], ph[j], o[dt], 0, 0, 0);
        o[dt + 1] = __builtin_amdgcn_mfma_f32_16x16x32_f16(vg[b][j], ph[j], o[dt + 1], 0, 0, 0);
        lf[b] = __builtin_amdgcn_mfma_f32_16x16x32_f16(vf[b][j], pl[j], j ? lf[b] : z, 0, 0, 0);
        lg[b] = __builtin_amdgcn_mfma_f32_16x16x32_f16(vg[b][j], pl[j], j ? lg[b] : z, 0, 0, 0);
      }
      if (dt > 0) add_low(dt - 2);
      __builtin_amdgcn_sched_barrier(0);
    }
    add_low(DT - 2);
    // V values that are not finite, to the rows that see their cells
    for (int w = 0; w < 2; w++) {
      uint32_t b = __builtin_amdgcn_readfirstlane(bad[it % 3][kw][w]);
      for (; b; b &= b - 1) {
        const int c = 32 * w + __builtin_ctz(b);
        float p = 0.0f;
#pragma unroll
        for (int ct = 0; ct < CT; ct++)
#pragma unroll
          for (int i = 0; i < 4; i++)
            if (c == ct * 16 + (c & 12) + i) p = st[ct][i];
        p = __shfl(p, ((c & 12) >> 2) * 16 + r16) * FA_P;
        const uint16_t *vs = vb + (int64_t)min(tile * BC + c, A.n_kv - 1) * A.v_rs;
#pragma unroll
        for (int dt = 0; dt < DT; dt++)
#pragma unroll
          for (int i = 0; i < 4; i++) {
            const int d = dt * 16 + quad * 4 + i;
            const uint16_t x = d < D ? vs[d] : 0;
            if (p != 0.0f && (x & 0x7c00) == 0x7c00) o[dt][i] += p * h2f(x);
          }
      }
    }
  };

  // Tile it * KW + kw: its registers go to LDS, the next tile's loads go out,
  // then it is computed. All groups take the same number of turns. A group of
  // one wave needs no barrier: its LDS operations complete in order.
  auto turn_barrier = [&]() {
    if constexpr (KLDS)
      lds_sync();
    else
      asm volatile("" ::: "memory");
  };
  // Loads are unconditional: tiles past the last repeat its last cell, all
  // masked. With two stages a tile is computed from one while the next
  // tile's registers, loaded meanwhile, wait for the other: one barrier a
  // turn.
  const int turns = (ntiles + KW - 1) / KW;
  lds_sync();  // bad starts at zero
  u32x2 mc[CT];
  auto take_mask = [&]() {
#pragma unroll
    for (int ct = 0; ct < CT; ct++) mc[ct] = mk[ct];
  };
  if (turns > 0) {
    load_k(kw);
    load_vm(kw);
    if constexpr (KLDS) {
      store(0);
      take_mask();
      load_k(KW + kw);
      load_vm(KW + kw);
    }
  }
  for (int it = 0; it < turns; it++) {
    const int tile = it * KW + kw;
    turn_barrier();
    if constexpr (!KLDS) {
      store(it);
      take_mask();
      load_vm(tile + KW);
      turn_barrier();
    }
    if (gt < 2) bad[(it + 2) % 3][kw][gt] = 0;  // read last in the turn before
    const uint16_t *const kl = kl_of(it), *const vl = kl + KT;
    bool seen = false;
#pragma unroll
    for (int ct = 0; ct < CT; ct++)
      seen = seen || mc[ct][0] != 0xfc00fc00u || mc[ct][1] != 0xfc00fc00u;
    // a tile that no row of the wave sees adds nothing
    const bool some = __builtin_amdgcn_ballot_w64(seen && rvalid) != 0;
    if (!KLDS || some) scores(kl);
    if constexpr (!KLDS) load_k(tile + KW);
    if (some) compute(tile, it, vl, mc);
    if constexpr (KLDS) {
      store(it + 1);
      take_mask();
      load_k(tile + 2 * KW);
      load_vm(tile + 2 * KW);
    }
  }

  if constexpr (KW > 1) {
    // the groups' states of a row tile, merged in group order
    float *const sl = (float *)lds;
    auto state = [&](int g) { return sl + (g * RW + rw) * 16 * (DP + 2); };
    lds_sync();
    {
      float *s = state(kw);
#pragma unroll
      for (int dt = 0; dt < DT; dt++) *(f32x4 *)(s + (dt * 64 + lane) * 4) = o[dt];
      if (quad == 0) {
        s[16 * DP + r16] = m;
        s[16 * DP + 16 + r16] = l;
      }
    }
    lds_sync();
    if (kw != 0) return;
    float M = -INFINITY;
#pragma unroll
    for (int g = 0; g < KW; g++) M = fmaxf(M, state(g)[16 * DP + r16]);
    const float mu = M == -INFINITY ? 0.0f : M;
    l = 0.0f;
#pragma unroll
    for (int dt = 0; dt < DT; dt++) o[dt] = f32x4{0, 0, 0, 0};
#pragma unroll
    for (int g = 0; g < KW; g++) {
      const float *s = state(g);
      const float w = __builtin_amdgcn_exp2f((s[16 * DP + r16] - mu) * FA_LOG2E);
      l += s[16 * DP + 16 + r16] * w;
#pragma unroll
      for (int dt = 0; dt < DT; dt++) o[dt] += *(const f32x4 *)(s + (dt * 64 + lane) * 4) * w;
    }
  }
  if (rvalid && l == l) {
    // a row with every cell masked gives zeros
    const float inv = l == 0.0f ? 0.0f : 1.0f / (l * FA_P);
    float *orow = A.out + ((int64_t)t * A.H + h) * D;
#pragma unroll
    for (int dt = 0; dt < DT; dt++) {
      const int d0 = dt * 16 + quad * 4;
      if (d0 >= D) continue;
      *(f32x4_u *)(orow + d0) = o[dt] * inv;
    }
  }
  uint32_t lost = (uint32_t)__builtin_amdgcn_ballot_w64(rvalid && l != l) & 0xffffu;
#pragma unroll 1
  for (; lost; lost &= lost - 1)
    exact_row(A, kvh, ((blockIdx.z * gridDim.y + blockIdx.y) * RW + rw) * 16 + __builtin_ctz(lost));
}

template <int DP, int BC, int RW, int KW>
static void launch_flash(const FlashArgs &A, int n_head_kv, hipStream_t st) {
  const int64_t tiles = ((int64_t)A.T * A.G + RW * 16 - 1) / (RW * 16);
  const int64_t gy = tiles < 65535 ? tiles : 65535;  // the most a grid takes in y
  hipLaunchKernelGGL((flash_attn_kernel<DP, BC, RW, KW>),
                     dim3((unsigned)n_head_kv, (unsigned)gy, (unsigned)((tiles + gy - 1) / gy)),
                     dim3(RW * KW * 64), 0, st, A);
}

// The split of a call: RW row tiles of 16 share a workgroup's K and V, KW
// groups share its cells. From 96 workgroups of 64 rows up, four row tiles
// (one wave per SIMD and group) in two groups (one past 128, whose stages
// fill LDS). Below, most CUs would stay idle: one row tile per workgroup,
// its cells over 8 waves (4 past 128, whose registers take a SIMD each),
// K straight from memory. (32 / 8 heads of 128, 2048 cells: 200 rows, 104
// workgroups of 64 rows, 70 us; 100 rows as 16-row workgroups 40.6; one row
// 36.9, 670 in the wave-per-row kernel before.) A single 32-cell tile
// needs one wave: nothing to merge. And a wave per row where the cells are fewer than
// a tile's setup takes: up to 4 cells of 2048 rows in all (in us, a tile / a
// wave per row: one row of 32 heads of 64 over 4 cells 5.3 / 4.0, of 256 10.0 /
// 6.4, 64 rows of 8 heads of 16 4.8 / 4.0; 512 rows of 8 heads of 16 4.9 / 5.4),
// for heads past 32 up to 8 cells of 512 rows (one row of 32 heads of 64 over 8
// 5.3 / 4.8, 12 5.3 / 5.7; 64 rows of 32 heads over 8 5.6 / 5.8).
template <int DP>
static void flash_for(const FlashArgs &A, int n_head_kv, hipStream_t st) {
  const int64_t rows = (int64_t)A.T * A.G * n_head_kv;
  if (A.n_kv <= 4 ? rows <= 2048 : A.n_kv <= 8 && DP >= 64 && rows <= 512) {
    hipLaunchKernelGGL(flash_row_kernel, dim3((unsigned)(A.T * A.G), (unsigned)n_head_kv), dim3(64),
                       0, st, A);
    return;
  }
  const int64_t tiles = ((int64_t)A.T * A.G + 63) / 64 * n_head_kv;
  constexpr int WIDE = DP <= 128 ? 2 : 1, SPLIT = DP <= 128 ? 8 : 4;
  if (tiles >= 96)
    launch_flash<DP, 64, 4, WIDE>(A, n_head_kv, st);
  else if (A.n_kv > 32)
    launch_flash<DP, 32, 1, SPLIT>(A, n_head_kv, st);
  else
    launch_flash<DP, 32, 1, 1>(A, n_head_kv, st);
}

}  // namespace lgmlh

using namespace lgmlh;

extern "C" int lgmlh_flash_attn(const float *q, int n_head, int n_tokens, int head_dim,
                                const uint16_t *k, const uint16_t *v, int n_head_kv, int n_kv,
                                int64_t k_row_stride, int64_t k_head_stride,
                                int64_t v_row_stride, int64_t v_head_stride,
                                const uint16_t *mask, int mask_heads, int mask_rows, float scale,
                                float max_bias, float softcap, float *out, void *stream) {
  if (!q || !k || !v || !out || n_head <= 0 || n_head_kv <= 0 || n_head % n_head_kv ||
      n_tokens < 0 || n_kv < 0 || head_dim <= 0 || head_dim > FA_MAX_D || head_dim % 8 ||
      k_row_stride % 8 || k_head_stride % 8 || v_row_stride < 0 || v_head_stride < 0 ||
      k_row_stride < 0 || k_head_stride < 0 || ((uintptr_t)k & 15) || softcap < 0.0f) {
    set_error("flash_attn: bad arguments (head size %d: a multiple of 8 up to %d; K rows "
              "16-byte aligned)", head_dim, FA_MAX_D);
    return LGMLH_EINVAL;
  }
  if (mask && (mask_heads <= 0 || n_head % mask_heads || mask_rows < n_tokens)) {
    set_error("flash_attn: mask shape mismatch");
    return LGMLH_EINVAL;
  }
  if (!mask && max_bias > 0.0f) {
    set_error("max_bias needs a mask");
    return LGMLH_EINVAL;
  }
  if (n_tokens == 0) return LGMLH_OK;
  const FlashArgs A{q, k, v, mask, out, n_head, n_tokens, head_dim, n_head / n_head_kv, n_kv,
                    mask ? mask_heads : 1, mask_rows, k_row_stride, k_head_stride, v_row_stride,
                    v_head_stride, scale, max_bias, softcap};
  hipStream_t st = as_stream(stream);
  if (head_dim <= 32)
    flash_for<32>(A, n_head_kv, st);
  else if (head_dim <= 64)
    flash_for<64>(A, n_head_kv, st);
  else if (head_dim <= 96)
    flash_for<96>(A, n_head_kv, st);
  else if (head_dim <= 128)
    flash_for<128>(A, n_head_kv, st);
  else if (head_dim <= 192)
    flash_for<192>(A, n_head_kv, st);
  else
    flash_for<256>(A, n_head_kv, st);
  return hip_check(hipGetLastError(), "flash_attn");
}
