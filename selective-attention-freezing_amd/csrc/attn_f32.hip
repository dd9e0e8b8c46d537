// float32 inputs: the reference's IEEE-dot contract (kernel/fused_attn.py:36-37,
// :128-140; tests at 2e-5 forward / 2e-4 backward, kernel/test_fused_attn.py:188-190).
//
// The 16-bit MFMA kernels round scores, P and products to their input type;
// fp32 q/k/v run here on v_mfma_f32_32x32x2_f32, whose inputs, products and
// sums are fp32 throughout (157 TFLOP/s, twice the vector ALUs' fp32 rate,
// and one LDS or memory operand per 4096 flops).
//
// Every kernel gives a workgroup one 32-row tile of its output (queries for
// out and dQ, keys for dK / dV) and its 4 waves every fourth 32-row block of
// the other axis; the waves share nothing until their accumulators (and the
// softmax's running max and sum) are merged through LDS at the end, so the
// block loop has no barrier and the causal work of a tile is spread over
// four SIMDs.  A block's operands come straight from memory into registers
// (each is used by one wave only), each product's loads issued one product
// (2048 cycles at hd 64) ahead into the registers the previous one freed:
//   RowFrag  lane (m, g) holds elements 8t + 4g + 0..3 of row m: one 16-byte
//            load feeds four MFMAs (k = the lane half, so four MFMAs walk
//            the eight columns in the order 0|4, 1|5, 2|6, 3|7 in both operands)
//   ColFrag  lane (m, g) holds columns NE m + 0..NE-1 of rows 8a + 4g + r:
//            the A operand of an accumulator tile e whose rows are the
//            columns NE m + e
// The 32x32 product's accumulator register i of lane (n, g) is row
// 8 (i / 4) + 4 g + i % 4 of column n, which is exactly the B operand
// (rows 8a + r of half 0 and 8a + 4 + r of half 1) of the second product
// over ColFrag row i: P and dS never leave their registers.
//
// Bound by the matrix pipe: at B=4, 12 heads (9 live), T=1000, hd 64 the
// forward + backward takes 297 us against 1759 us on the vector ALUs
// (64 x 64 tiles in LDS, one workgroup per tile); the forward alone at B=8,
// 12 live heads, T=2000 runs at 115 TFLOP/s (25 before).
//
//   live heads     online softmax in base 2 (scale sm_scale log2 e), output
//                  divided by the row sum, LSE = m + log2(l) as the MFMA path
//   dense heads    P read from the (P, S, S) buffer (fp32 / bf16 / fp16)
//   decomposed     P = exp(alpha_j + rho_{i-j} - z_i) in fp32
//                  (closed-form heads run here through their decomposed
//                  buffers)
//   backward       dQ per query tile, which also writes delta = rowsum(out *
//                  dout); dK / dV per key tile (live heads); dV = P^T dO per
//                  key tile (frozen heads)
#include <type_traits>

#include "saf_kernels.h"

namespace saf {

namespace {

constexpr int kW = 4;   // waves of a workgroup
constexpr int kR = 32;  // rows of an output tile and of a block

template <int HD> struct F32Shape {
  static constexpr int NE = HD / 32;       // accumulator tiles (columns NE m + e)
  static constexpr int NT = HD / 8;        // 16-byte row pieces per lane
  static constexpr int LD = HD + 4;        // LDS pitch of a merged tile's rows (floats)
  // operand fragments of a tile held in LDS: [NT][64 lanes] x 16 bytes
  static constexpr int FRAG = kR * HD;     // floats
  static constexpr int MERGE = kW * kR * LD;
  // whole blocks of operands fit the registers beside the accumulators up to
  // hd 128; above, they are loaded piece by piece next to their use
  static constexpr bool kWhole = HD <= 128;
};

__device__ __forceinline__ f32x16_t mfma2(float a, float b, f32x16_t c) {
  return __builtin_amdgcn_mfma_f32_32x32x2f32(a, b, c, 0, 0, 0);
}

typedef unsigned u32x2_t __attribute__((ext_vector_type(2)));
typedef unsigned u32x3_t __attribute__((ext_vector_type(3)));
typedef unsigned u32x4_t __attribute__((ext_vector_type(4)));

// Keeps the compiler's scheduler from moving loads across: left alone it sank
// each load next to its use (with a full wait) to save registers.
#define SAF_PIN() __builtin_amdgcn_sched_barrier(0)

__device__ __forceinline__ float4 buf_load4(__amdgpu_buffer_rsrc_t r, int off) {
  return __builtin_bit_cast(float4, __builtin_amdgcn_raw_buffer_load_b128(r, off, 0, 0));
}

// Descriptor over the HD-float rows r0 .. T - 1 of a tensor with row pitch st:
// it ends with the last row's last element, so rows closer than HD (a tensor
// expanded over T: st = 0; overlapping windows) are read whole too.  Rows past
// T then read whatever lies before that end; their cells are masked or dropped.
template <int HD>
__device__ __forceinline__ __amdgpu_buffer_rsrc_t tile_rsrc(const float* base, int64_t st, int r0, int T_len) {
  return span_rsrc(base + (int64_t)r0 * st, r0 < T_len ? ((int64_t)(T_len - 1 - r0) * st + HD) * 4 : (int64_t)0);
}

// Rows r0 .. r0 + 31 of a (T, st) fp32 tensor as a row operand.
template <int HD, bool WHOLE = F32Shape<HD>::kWhole> struct RowFrag {
  static constexpr int NT = F32Shape<HD>::NT;
  float4 r[WHOLE ? NT : 1];
  __amdgpu_buffer_rsrc_t rsrc;
  __device__ __forceinline__ void load(const float* base, int64_t st, int r0, int T_len, int off) {
    rsrc = tile_rsrc<HD>(base, st, r0, T_len);
    if constexpr (WHOLE) {
      SAF_PIN();
#pragma unroll
      for (int t = 0; t < NT; ++t) r[t] = buf_load4(rsrc, off + 32 * t);
      SAF_PIN();
    }
  }
  // acc[row][n] += sum_d rows[row][d] b[n][d], b's fragments in LDS
  __device__ __forceinline__ f32x16_t dot(const float4* b, int lane, int off, f32x16_t acc) const {
#pragma unroll
    for (int t0 = 0; t0 < NT; t0 += 4) {
      float4 a[4];
#pragma unroll
      for (int u = 0; u < 4; ++u) a[u] = WHOLE ? r[WHOLE ? t0 + u : 0] : buf_load4(rsrc, off + 32 * (t0 + u));
#pragma unroll
      for (int u = 0; u < 4; ++u) {
        const float4 q = b[(t0 + u) * 64 + lane];
        acc = mfma2(a[u].x, q.x, acc);
        acc = mfma2(a[u].y, q.y, acc);
        acc = mfma2(a[u].z, q.z, acc);
        acc = mfma2(a[u].w, q.w, acc);
      }
      SAF_PIN();  // bounds the b fragments held ahead
    }
    return acc;
  }
};
// this lane's byte offset of a row operand
__device__ __forceinline__ int row_off(int64_t st, int lane) { return (int)((lane & 31) * st * 4) + 16 * (lane >> 5); }

// Rows r0 .. r0 + 31 of a (T, st) fp32 tensor as a column operand.
template <int HD, bool WHOLE = F32Shape<HD>::kWhole> struct ColFrag {
  static constexpr int NE = F32Shape<HD>::NE;
  float c[WHOLE ? 16 : 1][NE];
  __amdgpu_buffer_rsrc_t rsrc;
  __device__ __forceinline__ static void row(__amdgpu_buffer_rsrc_t rs, float (&d)[NE], int off) {
    if constexpr (NE == 1) {
      d[0] = __uint_as_float(__builtin_amdgcn_raw_buffer_load_b32(rs, off, 0, 0));
    } else if constexpr (NE == 2) {
      const u32x2_t w = __builtin_amdgcn_raw_buffer_load_b64(rs, off, 0, 0);
      d[0] = __uint_as_float(w[0]);
      d[1] = __uint_as_float(w[1]);
    } else if constexpr (NE == 3) {
      const u32x3_t w = __builtin_amdgcn_raw_buffer_load_b96(rs, off, 0, 0);
#pragma unroll
      for (int e = 0; e < 3; ++e) d[e] = __uint_as_float(w[e]);
    } else {
#pragma unroll
      for (int u = 0; u < NE / 4; ++u) {
        const u32x4_t w = __builtin_amdgcn_raw_buffer_load_b128(rs, off + 16 * u, 0, 0);
#pragma unroll
        for (int e = 0; e < 4; ++e) d[4 * u + e] = __uint_as_float(w[e]);
      }
    }
  }
  __device__ __forceinline__ void load(const float* base, int64_t st, int r0, int T_len, int off) {
    rsrc = tile_rsrc<HD>(base, st, r0, T_len);
    if constexpr (WHOLE) {
      SAF_PIN();
      // the sixteen row offsets are formed here each time: held across the
      // loop they cost sixteen registers per operand and spilled
      asm volatile("" : "+v"(off));
#pragma unroll
      for (int i = 0; i < 16; ++i) row(rsrc, c[i], off + (8 * (i >> 2) + (i & 3)) * (int)(st * 4));
      SAF_PIN();
    }
  }
  // o[e][column][n] += sum_row rows[row][NE column + e] w[row][n]
  __device__ __forceinline__ void axpy(f32x16_t (&o)[NE], const float (&w)[16], int64_t st, int off) const {
#pragma unroll
    for (int i = 0; i < 16; ++i) {
      float d[NE];
      if constexpr (WHOLE) {
#pragma unroll
        for (int e = 0; e < NE; ++e) d[e] = c[WHOLE ? i : 0][e];
      } else {
        row(rsrc, d, off + (8 * (i >> 2) + (i & 3)) * (int)(st * 4));
      }
#pragma unroll
      for (int e = 0; e < NE; ++e) o[e] = mfma2(d[e], w[i], o[e]);
      if constexpr (!WHOLE)
        if (i % 4 == 3) SAF_PIN();
    }
  }
};
// this lane's byte offset of a column operand
template <int HD> __device__ __forceinline__ int col_off(int64_t st, int lane) {
  return (int)((lane >> 5) * 4 * st * 4) + (lane & 31) * F32Shape<HD>::NE * 4;
}

// Row of accumulator register i of lane half g within a 32-row block.
__device__ __forceinline__ int acc_row(int i, int g) { return 8 * (i >> 2) + 4 * g + (i & 3); }

// The tile's own 32 rows as B fragments in LDS, each wave a quarter of the pieces.
template <int HD>
__device__ __forceinline__ void stage_tile(float4* dst, const float* base, int64_t st, int r0, int T_len, int wave,
                                           int lane) {
  const __amdgpu_buffer_rsrc_t r = tile_rsrc<HD>(base, st, r0, T_len);
  for (int t = wave; t < F32Shape<HD>::NT; t += kW) dst[t * 64 + lane] = buf_load4(r, row_off(st, lane) + 32 * t);
}

// This wave's accumulators into its (32, HD) slab of the merge buffer, times f.
template <int HD>
__device__ __forceinline__ void put_tile(float* sm, const f32x16_t (&o)[F32Shape<HD>::NE], float f, int wave, int lane) {
  constexpr int NE = F32Shape<HD>::NE, LD = F32Shape<HD>::LD;
  float* row = sm + (wave * kR + (lane & 31)) * LD + NE * 4 * (lane >> 5);
#pragma unroll
  for (int a = 0; a < 4; ++a) {
    float w[4 * NE];  // columns NE (8a + 4g) + 0 .. 4 NE - 1
#pragma unroll
    for (int r = 0; r < 4; ++r)
#pragma unroll
      for (int e = 0; e < NE; ++e) w[NE * r + e] = o[e][4 * a + r] * f;
#pragma unroll
    for (int u = 0; u < NE; ++u)
      *reinterpret_cast<float4*>(row + 8 * NE * a + 4 * u) = make_float4(w[4 * u], w[4 * u + 1], w[4 * u + 2], w[4 * u + 3]);
  }
}

// The four waves' slabs summed and stored: rows r0 .. of dst, times scale
// (per row where row_scale is given).  Rows past T are dropped.
template <int HD>
__device__ __forceinline__ void store_sum(const float* sm, float* dst, int64_t st, int r0, int T_len, float scale,
                                          const float* row_scale, int tid) {
  constexpr int V4 = HD / 4, LD = F32Shape<HD>::LD;
  for (int idx = tid; idx < kR * V4; idx += 64 * kW) {
    const int r = idx / V4, c = idx % V4;
    if (r0 + r >= T_len) continue;
    float4 s = *reinterpret_cast<const float4*>(sm + r * LD + 4 * c);
#pragma unroll
    for (int w = 1; w < kW; ++w) {
      const float4 x = *reinterpret_cast<const float4*>(sm + (w * kR + r) * LD + 4 * c);
      s.x += x.x; s.y += x.y; s.z += x.z; s.w += x.w;
    }
    const float f = row_scale != nullptr ? row_scale[r] : scale;
    // 8-byte stores: the outputs' rows are only 8-byte aligned by contract
    float2* o = reinterpret_cast<float2*>(dst + (int64_t)(r0 + r) * st + 4 * c);
    o[0] = make_float2(s.x * f, s.y * f);
    o[1] = make_float2(s.z * f, s.w * f);
  }
}

// Pattern inputs of frozen heads.  The element reads take any strides and
// storage type, with indexes clamped into the buffers (the cells they stand
// for are masked); FAST kernels (fp32 buffers with unit inner strides, every
// model's layout) read four neighbours per 16-byte load instead: 4 loads per
// 16 cells in place of 16, each of which cost a 64-bit address and a type
// switch.
struct FrozenCells {
  const void* patt;
  const void* alpha;
  const void* rho;
  const void* z;
  int patt_dtype, a_dtype, r_dtype, z_dtype, T_len;
  int64_t prow0, p_si, p_sj, a0, a_ss, r0, r_ss, z0, z_ss;
  template <typename P> __device__ __forceinline__ void init(const P& p, int ph) {
    patt = p.patt; alpha = p.alpha; rho = p.rho; z = p.z;
    patt_dtype = p.patt_dtype; a_dtype = p.a_dtype; r_dtype = p.r_dtype; z_dtype = p.z_dtype;
    prow0 = (int64_t)ph * p.p_sh; p_si = p.p_si; p_sj = p.p_sj;
    a0 = (int64_t)ph * p.a_sh; a_ss = p.a_ss;
    r0 = (int64_t)ph * p.r_sh; r_ss = p.r_ss;
    z0 = (int64_t)ph * p.z_sh; z_ss = p.z_ss;
    T_len = p.T;
  }
  __device__ __forceinline__ float cell(int i, int j) const {
    return load_as_f32(patt, prow0 + (int64_t)min(i, T_len - 1) * p_si + (int64_t)min(j, T_len - 1) * p_sj, patt_dtype);
  }
  __device__ __forceinline__ float alpha_at(int j) const {
    return load_as_f32(alpha, a0 + (int64_t)min(j, T_len - 1) * a_ss, a_dtype);
  }
  __device__ __forceinline__ float rho_at(int d) const {
    return load_as_f32(rho, r0 + (int64_t)min(max(d, 0), T_len - 1) * r_ss, r_dtype);
  }
  __device__ __forceinline__ float z_at(int i) const {
    return load_as_f32(z, z0 + (int64_t)min(i, T_len - 1) * z_ss, z_dtype);
  }
  __device__ __forceinline__ __amdgpu_buffer_rsrc_t vec(const void* v, int64_t off) const {
    return rows_rsrc(reinterpret_cast<const float*>(v) + off, (int64_t)1, 0, T_len);
  }
  // the pattern from row i0 < T to column T - 1 of row T - 1 (FAST: the host
  // has checked that 32 rows fit 32-bit offsets)
  __device__ __forceinline__ __amdgpu_buffer_rsrc_t rows(int i0) const {
    return span_rsrc(reinterpret_cast<const float*>(patt) + prow0 + (int64_t)i0 * p_si,
                     ((int64_t)(T_len - 1 - i0) * p_si + T_len) * 4);
  }
  // alpha + rho - z with the rounding error of the sum carried (TwoSum):
  // where P matters z is close to alpha + rho, so (s - z) is exact and the
  // exponent keeps its low bits even for logits of scale 100+
  __device__ __forceinline__ static float prob(float a, float r, float zi) {
    const float s = a + r;
    const float bp = s - a;
    const float e = (a - (s - bp)) + (r - bp);
    // -inf logits (masked keys, windows): exact zeros
    return expf(__builtin_isfinite(s) ? (s - zi) + e : s - zi);
  }
};

__device__ __forceinline__ void put4(float (&d)[16], int a, float4 w) {
  d[4 * a] = w.x; d[4 * a + 1] = w.y; d[4 * a + 2] = w.z; d[4 * a + 3] = w.w;
}

// One fp32 statistic of the 16 rows this lane's accumulator registers hold,
// rows r0 .. r0 + 31 of a vector with stride st (rows past T read as 0 or as
// row T - 1; their cells are masked).
__device__ __forceinline__ void load_stat(float (&d)[16], const float* base, int64_t st, int r0, int T_len, int g) {
  if (st == 1) {
    const __amdgpu_buffer_rsrc_t r = rows_rsrc(base, (int64_t)1, r0, T_len);
#pragma unroll
    for (int a = 0; a < 4; ++a) put4(d, a, buf_load4(r, 32 * a + 16 * g));
  } else {
#pragma unroll
    for (int i = 0; i < 16; ++i) d[i] = base[(int64_t)min(r0 + acc_row(i, g), T_len - 1) * st];
  }
  SAF_PIN();
}

// ---- forward -------------------------------------------------------------

template <int HD>
__global__ __launch_bounds__(256) void f32_live_kernel(const FlashParams p) {
  using Sh = F32Shape<HD>;
  constexpr int NE = Sh::NE;
  __shared__ __align__(16) float sm[Sh::MERGE > Sh::FRAG ? Sh::MERGE : Sh::FRAG];
  __shared__ float sm_m[kW][kR], sm_l[kW][kR], sm_inv[kR];
  const int tid = threadIdx.x, lane = tid & 63, n = lane & 31, g = lane >> 5;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int T_len = p.T, nqt = (T_len + kR - 1) / kR, nbh = p.B * p.n_slots;
  const int qt = nqt - 1 - (int)(blockIdx.x / nbh);  // heaviest first
  const int bh = (int)(blockIdx.x % nbh);
  const int b = bh / p.n_slots, slot = bh % p.n_slots;
  const int h = p.out_head[slot], q0 = qt * kR, q = q0 + n;
  const float* kbase = reinterpret_cast<const float*>(p.k) + b * p.k_sb + (int64_t)p.k_head[slot] * p.k_sh;
  const float* vbase = reinterpret_cast<const float*>(p.v) + b * p.v_sb + (int64_t)p.v_head[slot] * p.v_sh;
  float4* const qf = reinterpret_cast<float4*>(sm);
  stage_tile<HD>(qf, reinterpret_cast<const float*>(p.q) + b * p.q_sb + (int64_t)p.q_head[slot] * p.q_sh, p.q_st, q0,
                 T_len, wave, lane);
  const int ko = row_off(p.k_st, lane), vo = col_off<HD>(p.v_st, lane);
  RowFrag<HD> kf;
  ColFrag<HD> vf;
  // a block past the diagonal loads nothing (an empty descriptor)
  auto lim = [&](int jb) { return jb <= qt ? T_len : 0; };
  kf.load(kbase, p.k_st, kR * wave, lim(wave), ko);
  vf.load(vbase, p.v_st, kR * wave, lim(wave), vo);
  __syncthreads();
  float m = -INFINITY, l = 0.f;
  f32x16_t o[NE];
#pragma unroll
  for (int e = 0; e < NE; ++e) o[e] = zero16();
  for (int jb = wave; jb <= qt; jb += kW) {
    const f32x16_t s = kf.dot(qf, lane, ko, zero16());
    kf.load(kbase, p.k_st, kR * (jb + kW), lim(jb + kW), ko);
    float x[16], mx = -INFINITY;
#pragma unroll
    for (int i = 0; i < 16; ++i) x[i] = s[i] * p.scale_log2;
    if (jb == qt) {
#pragma unroll
      for (int i = 0; i < 16; ++i) x[i] = kR * jb + acc_row(i, g) <= q ? x[i] : -INFINITY;
    }
#pragma unroll
    for (int i = 0; i < 16; ++i) mx = fmaxf(mx, x[i]);
    const float m_new = fmaxf(m, half_swap_max(mx));
    const float corr = m_new == -INFINITY ? 1.f : fast_exp2(m - m_new);
    float sum = 0.f;
#pragma unroll
    for (int i = 0; i < 16; ++i) {
      x[i] = m_new == -INFINITY ? 0.f : fast_exp2(x[i] - m_new);
      sum += x[i];
    }
    l = l * corr + half_swap_sum(sum);
    m = m_new;
#pragma unroll
    for (int e = 0; e < NE; ++e)
#pragma unroll
      for (int i = 0; i < 16; ++i) o[e][i] *= corr;
    vf.axpy(o, x, p.v_st, vo);
    vf.load(vbase, p.v_st, kR * (jb + kW), lim(jb + kW), vo);
  }
  if (g == 0) {
    sm_m[wave][n] = m;
    sm_l[wave][n] = l;
  }
  __syncthreads();  // every wave has read Q: its LDS becomes the merge buffer
  float M = sm_m[0][n];
#pragma unroll
  for (int w = 1; w < kW; ++w) M = fmaxf(M, sm_m[w][n]);
  float L = 0.f;
#pragma unroll
  for (int w = 0; w < kW; ++w) {
    const float mw = sm_m[w][n];
    L += mw == -INFINITY ? 0.f : sm_l[w][n] * fast_exp2(mw - M);
  }
  put_tile<HD>(sm, o, m == -INFINITY ? 0.f : fast_exp2(m - M), wave, lane);
  if (wave == 0 && g == 0) {
    sm_inv[n] = L > 0.f ? 1.f / L : 1.f;
    if (p.lse != nullptr && q < T_len)
      p.lse[b * p.l_sb + (int64_t)h * p.l_sh + (int64_t)q * p.l_st] = M + __log2f(L > 0.f ? L : 1.f);
  }
  __syncthreads();
  store_sum<HD>(sm, reinterpret_cast<float*>(p.out) + b * p.o_sb + (int64_t)h * p.o_sh, p.o_st, q0, T_len, 1.f, sm_inv,
                tid);
}

// out = P V of frozen heads (DENSE: P from the pattern buffer, else rebuilt);
// the next block's pattern inputs are fetched before the current product.
template <int HD, bool DENSE, bool FAST>
__global__ __launch_bounds__(256) void f32_frozen_kernel(const FrozenParams p) {
  using Sh = F32Shape<HD>;
  constexpr int NE = Sh::NE;
  __shared__ __align__(16) float sm[Sh::MERGE];
  const int tid = threadIdx.x, lane = tid & 63, n = lane & 31, g = lane >> 5;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int T_len = p.T, nqt = (T_len + kR - 1) / kR, nbh = p.B * p.n_slots;
  const int qt = nqt - 1 - (int)(blockIdx.x / nbh);
  const int bh = (int)(blockIdx.x % nbh);
  const int b = bh / p.n_slots, slot = bh % p.n_slots;
  const int q0 = qt * kR, q = q0 + n;
  const float* vbase = reinterpret_cast<const float*>(p.v) + b * p.v_sb + (int64_t)p.v_head[slot] * p.v_sh;
  FrozenCells P;
  P.init(p, p.pat_head[slot]);
  const int vo = col_off<HD>(p.v_st, lane);
  ColFrag<HD> vf;
  float u[16], w[16];  // dense: pattern cells; decomposed: alpha_j and rho_{q-j}
  const __amdgpu_buffer_rsrc_t pr = P.rows(q0), ar = P.vec(P.alpha, P.a0), rr = P.vec(P.rho, P.r0);
  auto fetch = [&](int jb) {
    const int j0 = kR * jb + 4 * g;  // keys j0 + 8a + r
    if (FAST && (DENSE || jb < qt)) {
      // below the diagonal block every distance is >= 1, so the four
      // distances q - j0 - 8a - 3 .. - 0 are one load; columns and distances
      // past T belong to masked cells or dropped rows (they read the next
      // row's values or zeros)
#pragma unroll
      for (int a = 0; a < 4; ++a) {
        if constexpr (DENSE) {
          put4(u, a, buf_load4(pr, (int)(n * P.p_si * 4) + 4 * (j0 + 8 * a)));
        } else {
          put4(u, a, buf_load4(ar, 4 * (j0 + 8 * a)));
          const float4 t = buf_load4(rr, 4 * (q - j0 - 8 * a - 3));
          put4(w, a, make_float4(t.w, t.z, t.y, t.x));
        }
      }
    } else {
#pragma unroll
      for (int i = 0; i < 16; ++i) {
        const int j = kR * jb + acc_row(i, g);
        if constexpr (DENSE) {
          u[i] = P.cell(q, j);
        } else {
          u[i] = P.alpha_at(j);
          w[i] = P.rho_at(q - j);
        }
      }
    }
    SAF_PIN();
  };
  auto lim = [&](int jb) { return jb <= qt ? T_len : 0; };
  if (wave <= qt) fetch(wave);
  vf.load(vbase, p.v_st, kR * wave, lim(wave), vo);
  const float zq = DENSE ? 0.f : P.z_at(q);
  f32x16_t o[NE];
#pragma unroll
  for (int e = 0; e < NE; ++e) o[e] = zero16();
  for (int jb = wave; jb <= qt; jb += kW) {
    float x[16];
#pragma unroll
    for (int i = 0; i < 16; ++i) x[i] = DENSE ? u[i] : FrozenCells::prob(u[i], w[i], zq);
    if (jb == qt) {
#pragma unroll
      for (int i = 0; i < 16; ++i) x[i] = kR * jb + acc_row(i, g) <= q ? x[i] : 0.f;
    }
    if (jb + kW <= qt) fetch(jb + kW);
    vf.axpy(o, x, p.v_st, vo);
    vf.load(vbase, p.v_st, kR * (jb + kW), lim(jb + kW), vo);
  }
  put_tile<HD>(sm, o, 1.f, wave, lane);
  __syncthreads();
  store_sum<HD>(sm, reinterpret_cast<float*>(p.out) + b * p.o_sb + (int64_t)p.out_head[slot] * p.o_sh, p.o_st, q0,
                T_len, 1.f, nullptr, tid);
}

// ---- backward ------------------------------------------------------------

// Waves per SIMD of the dQ and dK / dV kernels: two up to hd 64 (left to the
// compiler they took 270 to 340 registers and ran one), so one wave's softmax
// and loads run beside the other's products.
constexpr int f32_bwd_waves(int hd) { return hd <= 64 ? 2 : 1; }

// dQ of one query tile; its prologue forms delta = rowsum(out * dout) of the
// tile's rows and stores it for the dK / dV kernel, which runs after it.
template <int HD>
__global__ __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(f32_bwd_waves(HD), f32_bwd_waves(HD))))
void f32_bwd_dq_kernel(const BwdParams p) {
  using Sh = F32Shape<HD>;
  constexpr int NE = Sh::NE, NT = Sh::NT;
  __shared__ __align__(16) float sm[Sh::MERGE > 2 * Sh::FRAG ? Sh::MERGE : 2 * Sh::FRAG];
  __shared__ float sm_d[kW][kR];
  const int tid = threadIdx.x, lane = tid & 63, n = lane & 31, g = lane >> 5;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int T_len = p.T, nqt = (T_len + kR - 1) / kR, nbh = p.B * p.n_live;
  const int qt = nqt - 1 - (int)(blockIdx.x / nbh);
  const int bh = (int)(blockIdx.x % nbh);
  const int b = bh / p.n_live, slot = bh % p.n_live;
  const int h = p.out_head[slot], qs = p.q_head[slot], q0 = qt * kR, q = q0 + n;
  const float* kbase = reinterpret_cast<const float*>(p.k) + b * p.k_sb + (int64_t)qs * p.k_sh;
  const float* vbase = reinterpret_cast<const float*>(p.v) + b * p.v_sb + (int64_t)h * p.v_sh;
  float4* const qf = reinterpret_cast<float4*>(sm);
  float4* const gf = reinterpret_cast<float4*>(sm + Sh::FRAG);
  stage_tile<HD>(qf, reinterpret_cast<const float*>(p.q) + b * p.q_sb + (int64_t)qs * p.q_sh, p.q_st, q0, T_len, wave,
                 lane);
  const int ko = row_off(p.k_st, lane), vo = row_off(p.v_st, lane), co = col_off<HD>(p.k_st, lane);
  auto lim = [&](int jb) { return jb <= qt ? T_len : 0; };
  RowFrag<HD> kf, vf;
  ColFrag<HD> kc;
  {
    const __amdgpu_buffer_rsrc_t gr =
        tile_rsrc<HD>(reinterpret_cast<const float*>(p.dout) + b * p.do_sb + (int64_t)h * p.do_sh, p.do_st, q0, T_len);
    const __amdgpu_buffer_rsrc_t orr =
        tile_rsrc<HD>(reinterpret_cast<const float*>(p.out) + b * p.o_sb + (int64_t)h * p.o_sh, p.o_st, q0, T_len);
    float acc = 0.f;
    for (int t = wave; t < NT; t += kW) {
      const float4 d = buf_load4(gr, row_off(p.do_st, lane) + 32 * t);
      const float4 y = buf_load4(orr, row_off(p.o_st, lane) + 32 * t);
      gf[t * 64 + lane] = d;
      acc = fmaf(d.x, y.x, fmaf(d.y, y.y, fmaf(d.z, y.z, fmaf(d.w, y.w, acc))));
    }
    acc = half_swap_sum(acc);
    if (g == 0) sm_d[wave][n] = acc;
  }
  kf.load(kbase, p.k_st, kR * wave, lim(wave), ko);
  vf.load(vbase, p.v_st, kR * wave, lim(wave), vo);
  const float lse =
      q < T_len ? p.lse[b * p.l_sb + (int64_t)h * p.l_sh + (int64_t)q * p.l_st] : 0.f;
  __syncthreads();
  const float dl = (sm_d[0][n] + sm_d[1][n]) + (sm_d[2][n] + sm_d[3][n]);
  if (wave == 0 && g == 0 && q < T_len) p.delta[((int64_t)b * p.n_live + slot) * T_len + q] = dl;
  f32x16_t acc[NE];
#pragma unroll
  for (int e = 0; e < NE; ++e) acc[e] = zero16();
  for (int jb = wave; jb <= qt; jb += kW) {
    const f32x16_t s = kf.dot(qf, lane, ko, zero16());
    kc.load(kbase, p.k_st, kR * jb, T_len, co);
    const f32x16_t dp = vf.dot(gf, lane, vo, zero16());
    kf.load(kbase, p.k_st, kR * (jb + kW), lim(jb + kW), ko);
    float x[16];
#pragma unroll
    for (int i = 0; i < 16; ++i) x[i] = s[i] * p.scale_log2 - lse;
    if (jb == qt) {
#pragma unroll
      for (int i = 0; i < 16; ++i) x[i] = (q < T_len && kR * jb + acc_row(i, g) <= q) ? x[i] : -INFINITY;
    }
#pragma unroll
    for (int i = 0; i < 16; ++i) x[i] = fast_exp2(x[i]) * (dp[i] - dl);
    kc.axpy(acc, x, p.k_st, co);
    vf.load(vbase, p.v_st, kR * (jb + kW), lim(jb + kW), vo);
  }
  __syncthreads();
  put_tile<HD>(sm, acc, 1.f, wave, lane);
  __syncthreads();
  store_sum<HD>(sm, reinterpret_cast<float*>(p.dq) + b * p.dq_sb + (int64_t)qs * p.dq_sh, p.dq_st, q0, T_len,
                p.sm_scale, nullptr, tid);
}

// dK / dV of one key tile of a live head: S = Q K^T and dP = dO V^T with the
// keys in the lanes, so the query's LSE and delta are per register.
template <int HD>
__global__ __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(f32_bwd_waves(HD), f32_bwd_waves(HD))))
void f32_bwd_kv_kernel(const BwdParams p) {
  using Sh = F32Shape<HD>;
  constexpr int NE = Sh::NE;
  __shared__ __align__(16) float sm[Sh::MERGE > 2 * Sh::FRAG ? Sh::MERGE : 2 * Sh::FRAG];
  const int tid = threadIdx.x, lane = tid & 63, n = lane & 31, g = lane >> 5;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int T_len = p.T, nqt = (T_len + kR - 1) / kR, nbh = p.B * p.n_live;
  const int kt = (int)(blockIdx.x / nbh);  // heaviest (most queries) first
  const int bh = (int)(blockIdx.x % nbh);
  const int b = bh / p.n_live, slot = bh % p.n_live;
  const int h = p.out_head[slot], qs = p.q_head[slot], k0 = kt * kR, key = k0 + n;
  const float* qbase = reinterpret_cast<const float*>(p.q) + b * p.q_sb + (int64_t)qs * p.q_sh;
  const float* gbase = reinterpret_cast<const float*>(p.dout) + b * p.do_sb + (int64_t)h * p.do_sh;
  const float* lse = p.lse + b * p.l_sb + (int64_t)h * p.l_sh;
  const float* delta = p.delta + ((int64_t)b * p.n_live + slot) * T_len;
  float4* const kf = reinterpret_cast<float4*>(sm);
  float4* const vf = reinterpret_cast<float4*>(sm + Sh::FRAG);
  stage_tile<HD>(kf, reinterpret_cast<const float*>(p.k) + b * p.k_sb + (int64_t)qs * p.k_sh, p.k_st, k0, T_len, wave,
                 lane);
  stage_tile<HD>(vf, reinterpret_cast<const float*>(p.v) + b * p.v_sb + (int64_t)h * p.v_sh, p.v_st, k0, T_len, wave,
                 lane);
  const int qo = row_off(p.q_st, lane), go = row_off(p.do_st, lane);
  const int qco = col_off<HD>(p.q_st, lane), gco = col_off<HD>(p.do_st, lane);
  auto lim = [&](int ib) { return ib < nqt ? T_len : 0; };
  RowFrag<HD> qr, gr;
  ColFrag<HD> qc, gc;
  qr.load(qbase, p.q_st, kR * (kt + wave), lim(kt + wave), qo);
  gr.load(gbase, p.do_st, kR * (kt + wave), lim(kt + wave), go);
  __syncthreads();
  f32x16_t dk[NE], dv[NE];
#pragma unroll
  for (int e = 0; e < NE; ++e) {
    dk[e] = zero16();
    dv[e] = zero16();
  }
  for (int ib = kt + wave; ib < nqt; ib += kW) {
    // dP's chain starts from -delta of each register's query
    float ls[16], dl[16];
    load_stat(ls, lse, p.l_st, kR * ib, T_len, g);
    load_stat(dl, delta, 1, kR * ib, T_len, g);
    const f32x16_t s = qr.dot(kf, lane, qo, zero16());
    gc.load(gbase, p.do_st, kR * ib, T_len, gco);
    f32x16_t dp;
#pragma unroll
    for (int i = 0; i < 16; ++i) dp[i] = -dl[i];
    dp = gr.dot(vf, lane, go, dp);
    qc.load(qbase, p.q_st, kR * ib, T_len, qco);
    float x[16], y[16];
#pragma unroll
    for (int i = 0; i < 16; ++i) x[i] = s[i] * p.scale_log2 - ls[i];
    if (ib == kt || ib == nqt - 1) {
#pragma unroll
      for (int i = 0; i < 16; ++i) {
        const int q = kR * ib + acc_row(i, g);
        x[i] = (key <= q && q < T_len) ? x[i] : -INFINITY;
      }
    }
#pragma unroll
    for (int i = 0; i < 16; ++i) {
      x[i] = fast_exp2(x[i]);
      y[i] = x[i] * dp[i];
    }
    gc.axpy(dv, x, p.do_st, gco);
    qr.load(qbase, p.q_st, kR * (ib + kW), lim(ib + kW), qo);
    qc.axpy(dk, y, p.q_st, qco);
    gr.load(gbase, p.do_st, kR * (ib + kW), lim(ib + kW), go);
  }
  __syncthreads();
  put_tile<HD>(sm, dv, 1.f, wave, lane);
  __syncthreads();
  store_sum<HD>(sm, reinterpret_cast<float*>(p.dv) + b * p.dv_sb + (int64_t)h * p.dv_sh, p.dv_st, k0, T_len, 1.f,
                nullptr, tid);
  __syncthreads();
  put_tile<HD>(sm, dk, 1.f, wave, lane);
  __syncthreads();
  store_sum<HD>(sm, reinterpret_cast<float*>(p.dk) + b * p.dk_sb + (int64_t)qs * p.dk_sh, p.dk_st, k0, T_len,
                p.sm_scale, nullptr, tid);
}

// dV = P^T dO of one key tile of a frozen head (KIND 1 dense, 2 decomposed).
template <int HD, int KIND, bool FAST>
__global__ __launch_bounds__(256) void f32_bwd_frozen_kernel(const BwdParams p) {
  using Sh = F32Shape<HD>;
  constexpr int NE = Sh::NE;
  __shared__ __align__(16) float sm[Sh::MERGE];
  const int tid = threadIdx.x, lane = tid & 63, n = lane & 31, g = lane >> 5;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int T_len = p.T, nqt = (T_len + kR - 1) / kR, nbf = p.B * p.n_frozen;
  const int kt = (int)(blockIdx.x / nbf);
  const int bf = (int)(blockIdx.x % nbf);
  const int b = bf / p.n_frozen, fs = bf % p.n_frozen;
  if (p.f_kind[fs] != KIND) return;
  const int h = p.f_head[fs], k0 = kt * kR, key = k0 + n;
  const float* gbase = reinterpret_cast<const float*>(p.dout) + b * p.do_sb + (int64_t)h * p.do_sh;
  FrozenCells P;
  P.init(p, p.pat_head[fs]);
  const int gco = col_off<HD>(p.do_st, lane);
  ColFrag<HD> gc;
  float u[16], w[16];  // dense: pattern cells; decomposed: rho_{i-key} and z_i
  const __amdgpu_buffer_rsrc_t rr = P.vec(P.rho, P.r0), zr = P.vec(P.z, P.z0);
  auto fetch = [&](int ib) {
    const int i0 = kR * ib + 4 * g;  // queries i0 + 8a + r
    if (FAST && KIND == 1) {
      const __amdgpu_buffer_rsrc_t pr = P.rows(kR * ib);
#pragma unroll
      for (int i = 0; i < 16; ++i)
        u[i] = __uint_as_float(
            __builtin_amdgcn_raw_buffer_load_b32(pr, acc_row(i, g) * (int)(P.p_si * 4) + 4 * key, 0, 0));
    } else if (FAST && ib > kt) {  // every distance is >= 1
#pragma unroll
      for (int a = 0; a < 4; ++a) {
        put4(u, a, buf_load4(rr, 4 * (i0 + 8 * a - key)));
        put4(w, a, buf_load4(zr, 4 * (i0 + 8 * a)));
      }
    } else {
#pragma unroll
      for (int i = 0; i < 16; ++i) {
        const int q = kR * ib + acc_row(i, g);
        if constexpr (KIND == 1) {
          u[i] = P.cell(q, key);
        } else {
          u[i] = P.rho_at(q - key);
          w[i] = P.z_at(q);
        }
      }
    }
    SAF_PIN();
  };
  auto lim = [&](int ib) { return ib < nqt ? T_len : 0; };
  if (kt + wave < nqt) fetch(kt + wave);
  gc.load(gbase, p.do_st, kR * (kt + wave), lim(kt + wave), gco);
  const float ak = KIND == 1 ? 0.f : P.alpha_at(key);
  f32x16_t dv[NE];
#pragma unroll
  for (int e = 0; e < NE; ++e) dv[e] = zero16();
  for (int ib = kt + wave; ib < nqt; ib += kW) {
    float x[16];
#pragma unroll
    for (int i = 0; i < 16; ++i) x[i] = KIND == 1 ? u[i] : FrozenCells::prob(ak, u[i], w[i]);
    if (ib == kt || ib == nqt - 1) {
#pragma unroll
      for (int i = 0; i < 16; ++i) {
        const int q = kR * ib + acc_row(i, g);
        x[i] = (key <= q && q < T_len) ? x[i] : 0.f;
      }
    }
    if (ib + kW < nqt) fetch(ib + kW);
    gc.axpy(dv, x, p.do_st, gco);
    gc.load(gbase, p.do_st, kR * (ib + kW), lim(ib + kW), gco);
  }
  put_tile<HD>(sm, dv, 1.f, wave, lane);
  __syncthreads();
  store_sum<HD>(sm, reinterpret_cast<float*>(p.dv) + b * p.dv_sb + (int64_t)h * p.dv_sh, p.dv_st, k0, T_len, 1.f,
                nullptr, tid);
}

// FAST pattern reads: fp32 buffers, unit inner strides, a pattern row pitch
// that 32-bit offsets of a row block can hold.
template <typename P>
bool cells_fast(const P& p, bool dense) {
  if (dense)
    return p.patt_dtype == kF32 && p.p_sj == 1 && p.p_si >= 0 && p.p_si * 4 < kMaxRowBytes;
  return p.a_dtype == kF32 && p.r_dtype == kF32 && p.z_dtype == kF32 && p.a_ss == 1 && p.r_ss == 1 && p.z_ss == 1;
}

template <int HD>
hipError_t f32_fwd_hd(const FlashParams* fp, const FrozenParams* zp, int mode, hipStream_t s) {
  if (fp != nullptr) {
    const dim3 grid((unsigned)((int64_t)((fp->T + kR - 1) / kR) * fp->n_slots * fp->B));
    hipLaunchKernelGGL((f32_live_kernel<HD>), grid, dim3(64 * kW), 0, s, *fp);
  } else {
    const dim3 grid((unsigned)((int64_t)((zp->T + kR - 1) / kR) * zp->n_slots * zp->B));
    const bool fast = cells_fast(*zp, mode == 0);
    if (mode == 0 && fast)
      hipLaunchKernelGGL((f32_frozen_kernel<HD, true, true>), grid, dim3(64 * kW), 0, s, *zp);
    else if (mode == 0)
      hipLaunchKernelGGL((f32_frozen_kernel<HD, true, false>), grid, dim3(64 * kW), 0, s, *zp);
    else if (fast)
      hipLaunchKernelGGL((f32_frozen_kernel<HD, false, true>), grid, dim3(64 * kW), 0, s, *zp);
    else
      hipLaunchKernelGGL((f32_frozen_kernel<HD, false, false>), grid, dim3(64 * kW), 0, s, *zp);
  }
  return hipGetLastError();
}

template <int HD>
hipError_t f32_bwd_hd(const BwdParams& p, int which, hipStream_t s) {
  const int64_t nt = (p.T + kR - 1) / kR;
  const dim3 live((unsigned)(nt * p.n_live * p.B)), frozen((unsigned)(nt * p.n_frozen * p.B));
  switch (which) {
    case 1:
      hipLaunchKernelGGL((f32_bwd_dq_kernel<HD>), live, dim3(64 * kW), 0, s, p);
      break;
    case 2:
      hipLaunchKernelGGL((f32_bwd_kv_kernel<HD>), live, dim3(64 * kW), 0, s, p);
      break;
    default: {
      bool kind[3] = {false, false, false};
      for (int i = 0; i < p.n_frozen; ++i) kind[p.f_kind[i]] = true;
      if (kind[1] && cells_fast(p, true))
        hipLaunchKernelGGL((f32_bwd_frozen_kernel<HD, 1, true>), frozen, dim3(64 * kW), 0, s, p);
      else if (kind[1])
        hipLaunchKernelGGL((f32_bwd_frozen_kernel<HD, 1, false>), frozen, dim3(64 * kW), 0, s, p);
      if (kind[2] && cells_fast(p, false))
        hipLaunchKernelGGL((f32_bwd_frozen_kernel<HD, 2, true>), frozen, dim3(64 * kW), 0, s, p);
      else if (kind[2])
        hipLaunchKernelGGL((f32_bwd_frozen_kernel<HD, 2, false>), frozen, dim3(64 * kW), 0, s, p);
      break;
    }
  }
  return hipGetLastError();
}

template <typename F>
hipError_t by_hd(int hd, F&& f) {
  switch (hd) {
    case 32: return f(std::integral_constant<int, 32>());
    case 64: return f(std::integral_constant<int, 64>());
    case 96: return f(std::integral_constant<int, 96>());
    case 128: return f(std::integral_constant<int, 128>());
    case 256: return f(std::integral_constant<int, 256>());
    default: return hipErrorInvalidValue;
  }
}

}  // namespace

hipError_t launch_f32_live(const FlashParams& p, int hd, hipStream_t s) {
  if (p.n_slots == 0 || p.T == 0 || p.B == 0) return hipSuccess;
  return by_hd(hd, [&](auto c) { return f32_fwd_hd<decltype(c)::value>(&p, nullptr, 0, s); });
}

hipError_t launch_f32_frozen(const FrozenParams& p, int hd, int mode, hipStream_t s) {
  if (p.n_slots == 0 || p.T == 0 || p.B == 0) return hipSuccess;
  return by_hd(hd, [&](auto c) { return f32_fwd_hd<decltype(c)::value>(nullptr, &p, mode, s); });
}

hipError_t launch_f32_bwd(const BwdParams& p, int hd, int which, hipStream_t s) {
  if (p.T == 0 || p.B == 0 || (which < 3 ? p.n_live == 0 : p.n_frozen == 0)) return hipSuccess;
  return by_hd(hd, [&](auto c) { return f32_bwd_hd<decltype(c)::value>(p, which, s); });
}

}  // namespace saf
