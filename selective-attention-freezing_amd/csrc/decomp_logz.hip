// Row normalisers of decomposed patterns on gfx950:
//   z[h, i] = logsumexp_{j <= i} (alpha[h, j] + rho[h, i - j]),  i < S
// (/root/reference/kernel/fused_attn.py:101-116 decomposed_logz, which the
// reference computes in chunks of materialised (H, rows, S) logits; the model
// calls it at freeze time, nanogpt/model.py freeze_heads_decomposed, and
// fused_mixed_attn calls it per call when alpha comes without z, :690-694).
//
// exp2 of a sum of two vectors' elements is a product of two exp2s, so the sum
// over j is a convolution: per chunk of kLzChunk keys a work-group forms
// a'_j = 2^(alpha_j - A) and r'_d = 2^(rho_d - R) once (A, R the maxima over the
// chunk's keys and over the distances it can meet; log2 units), and each of
// its 256 rows then costs one fp32 FMA per key instead of an add, a maximum, a
// subtraction and an exp2.  Lane l owns rows 4 l .. 4 l + 3, and per 4 keys its
// 16 products need 7 distances: one 16-byte LDS read slides the window (r' by
// 16-byte lanes, conflict-free; a' is a broadcast).  The 8 waves split a
// chunk's keys; a chunk's sums start from zero and join the row's total scaled
// by 2^(A + R - M), M the running maximum of A + R, so no sum runs over more
// than a chunk's share of terms.
//
// Every factor is <= 1 and the products of a row are lost only below 2^-126 of
// the scale M: at most S 2^-126 in all.  A row whose total is below 2^-80 (its
// own keys lie far below the chunk's maxima, or all are -inf, or a value is
// not finite) sends its 64-row block to the direct form: 16 logits at a time
// folded into a running (max, sum) per lane.
//
// Bound by FMA issue (S(S+1)/2 per head; HBM traffic is 3 S 4 bytes):
// H=12, S=8192: 135 us (one exp2 per logit) -> 30 us; S=16384: 321 -> 74 us.
#include "saf_kernels.h"

namespace saf {

constexpr int kLzRows = 256;           // rows (outputs) of a work-group
constexpr int kLzWaves = 8;
constexpr int kLzThreads = 64 * kLzWaves;
constexpr int kLzChunk = 2048;         // keys per chunk
constexpr int kLzWin = kLzChunk + kLzRows;
constexpr int kLzDirect = 1024;        // direct form: keys per chunk
constexpr int kLzGroup = 16;
constexpr int kLzNA = kLzChunk / kLzThreads;                       // staged values per thread
constexpr int kLzNW = (kLzWin + kLzThreads - 1) / kLzThreads;
static_assert(kLzDirect % (kLzWaves * kLzGroup) == 0, "chunk must split into whole groups per wave");
constexpr float kLzLow = 8.271806125530277e-25f;  // 2^-80
constexpr float kLn2 = 0.6931471805599453f;

// Maxima of x and y over the work-group (each wave's through `red`).
__device__ __forceinline__ void group_max2(float& x, float& y, float (*red)[kLzWaves], int lane, int w) {
  x = wave_max(x);
  y = wave_max(y);
  if (lane == 0) {
    red[0][w] = x;
    red[1][w] = y;
  }
  __syncthreads();
#pragma unroll
  for (int q = 0; q < kLzWaves; ++q) {
    x = fmaxf(x, red[0][q]);
    y = fmaxf(y, red[1][q]);
  }
}

// acc[r] += sum over steps of 4 terms of as[t + u] * win(r, u), the window
// sliding by 4 elements per step.  UP: the window moves up with t (win index
// 3 + u - r), else down (3 + r - u); p is this lane's first low quad.
template <bool UP>
__device__ __forceinline__ void slide(float (&acc)[4], const float* as, const float* p, int t0, int t1) {
  float4 lo, hi;
  if (UP) lo = *reinterpret_cast<const float4*>(p + t0);
  else hi = *reinterpret_cast<const float4*>(p + 4 - t0);
#pragma unroll 4
  for (int t = t0; t < t1; t += 4) {
    if (UP) hi = *reinterpret_cast<const float4*>(p + 4 + t);
    else lo = *reinterpret_cast<const float4*>(p - t);
    const float4 a4 = *reinterpret_cast<const float4*>(as + t);
    const float a[4] = {a4.x, a4.y, a4.z, a4.w};
    const float win[8] = {lo.x, lo.y, lo.z, lo.w, hi.x, hi.y, hi.z, hi.w};
#pragma unroll
    for (int u = 0; u < 4; ++u)
#pragma unroll
      for (int r = 0; r < 4; ++r) acc[r] = fmaf(a[u], win[UP ? 3 + u - r : 3 + r - u], acc[r]);
    if (UP) lo = hi;
    else hi = lo;
  }
}

__global__ __launch_bounds__(kLzThreads) void decomp_logz_kernel(const LogzParams p) {
  __shared__ __align__(16) float as[kLzChunk];
  __shared__ __align__(16) float rs[kLzWin];
  __shared__ float part[kLzWaves][kLzRows];
  __shared__ float red[2][kLzWaves];
  __shared__ int low[kLzRows / 64];

  const float ninf = -__builtin_inff();
  const int S = p.S;
  const int nblk = (S + kLzRows - 1) / kLzRows;
  const int i0 = (nblk - 1 - (int)blockIdx.x) * kLzRows;  // heaviest first
  const int h = blockIdx.y;
  const int tid = threadIdx.x, lane = tid & 63, w = __builtin_amdgcn_readfirstlane(tid >> 6);
  const float* alpha = p.alpha + (int64_t)h * p.a_hs;
  const float* rho = p.rho + (int64_t)h * p.r_hs;
  const int jend = min(i0 + kLzRows, S);  // keys any row of the block can see

  float M = ninf, tot[4] = {0.f, 0.f, 0.f, 0.f};
  float av[kLzNA], rv[kLzNW];
  auto load = [&](int j0) {  // this thread's share of a chunk's keys and window
    const int dlo = i0 - j0 - kLzChunk + 1;  // distance of window element 0
#pragma unroll
    for (int k = 0; k < kLzNA; ++k) {
      const int j = j0 + tid + k * kLzThreads;
      av[k] = j < jend ? alpha[j] : ninf;
    }
#pragma unroll
    for (int k = 0; k < kLzNW; ++k) {
      const int x = tid + k * kLzThreads, d = dlo + x;
      rv[k] = (x < kLzWin && d >= 0 && d < S) ? rho[d] : ninf;
    }
  };
  load(0);
  for (int j0 = 0; j0 < jend; j0 += kLzChunk) {
    float A = ninf, R = ninf;
#pragma unroll
    for (int k = 0; k < kLzNA; ++k) A = fmaxf(A, av[k] *= kLog2e);
#pragma unroll
    for (int k = 0; k < kLzNW; ++k) R = fmaxf(R, rv[k] *= kLog2e);
    group_max2(A, R, red, lane, w);  // its barrier: the previous chunk is consumed
    const float sc = A + R;
    if (sc != ninf) {
#pragma unroll
      for (int k = 0; k < kLzNA; ++k) as[tid + k * kLzThreads] = fast_exp2(av[k] - A);
#pragma unroll
      for (int k = 0; k < kLzNW; ++k)
        if (tid + k * kLzThreads < kLzWin) rs[tid + k * kLzThreads] = fast_exp2(rv[k] - R);
    }
    __syncthreads();
    load(j0 + kLzChunk);  // lands while the products run
    __builtin_amdgcn_sched_barrier(0);
    if (sc == ninf) continue;  // every logit of the chunk is -inf
    const int n = min(kLzChunk, jend - j0);
    const int quota = ((n + kLzWaves - 1) / kLzWaves + 3) / 4 * 4;  // keys past n are zero
    float acc[4] = {0.f, 0.f, 0.f, 0.f};
    // window element of (row 4 lane + r, key t): 4 lane + r + kLzChunk - 1 - t
    const int n4 = (n + 3) / 4 * 4;
    slide<false>(acc, as, rs + 4 * lane + kLzChunk - 4, min(w * quota, n4), min((w + 1) * quota, n4));
    const float Mn = fmaxf(M, sc), f0 = fast_exp2(M - Mn), f1 = fast_exp2(sc - Mn);
#pragma unroll
    for (int r = 0; r < 4; ++r) tot[r] = fmaf(acc[r], f1, tot[r] * f0);
    M = Mn;
  }
#pragma unroll
  for (int r = 0; r < 4; ++r) part[w][4 * lane + r] = tot[r];
  if (tid < kLzRows / 64) low[tid] = 0;
  __syncthreads();
  if (tid < kLzRows && i0 + tid < S) {
    float s = 0.f;
#pragma unroll
    for (int q = 0; q < kLzWaves; ++q) s += part[q][tid];
    if (s >= kLzLow)
      p.z[(int64_t)h * p.z_hs + i0 + tid] = (M + log2f(s)) * kLn2;
    else
      low[tid >> 6] = 1;
  }
  __syncthreads();

  // direct form of the 64-row blocks with a low row
  for (int b = 0; b < kLzRows / 64; ++b) {
    if (!low[b]) continue;
    const int b0 = i0 + 64 * b, bend = min(b0 + 64, S);
    float m = ninf, s = 0.f;
    for (int j0 = 0; j0 < bend; j0 += kLzDirect) {
      const int dlo = b0 - j0 - kLzDirect + 1;
      __syncthreads();  // previous chunk fully consumed
      for (int t = tid; t < kLzDirect; t += kLzThreads) as[t] = j0 + t < bend ? alpha[j0 + t] * kLog2e : ninf;
      for (int t = tid; t < kLzDirect + 63; t += kLzThreads) {
        const int d = dlo + t;
        rs[t] = (d >= 0 && d < S) ? rho[d] * kLog2e : ninf;
      }
      __syncthreads();
      const int tw0 = w * (kLzDirect / kLzWaves);
      const int tw1 = min(tw0 + kLzDirect / kLzWaves, bend - j0);
      const int rbase = lane + kLzDirect - 1;
      for (int t = tw0; t < tw1; t += kLzGroup) {
        float x[kLzGroup];
        float gm = ninf;
#pragma unroll
        for (int k = 0; k < kLzGroup; ++k) {
          x[k] = as[t + k] + rs[rbase - t - k];
          gm = fmaxf(gm, x[k]);
        }
        const float mn = fmaxf(m, gm);
        if (mn == ninf) continue;  // every logit so far is -inf: nothing to add
        float acc = s * fast_exp2(m - mn);
#pragma unroll
        for (int k = 0; k < kLzGroup; ++k) acc += fast_exp2(x[k] - mn);
        s = acc;
        m = mn;
      }
    }
    part[w][lane] = m;
    part[w][64 + lane] = s;
    __syncthreads();
    if (w == 0 && b0 + lane < S) {
      float mx = part[0][lane];
#pragma unroll
      for (int q = 1; q < kLzWaves; ++q) mx = fmaxf(mx, part[q][lane]);
      float zi = ninf;
      if (mx != ninf) {
        float sum = 0.f;
#pragma unroll
        for (int q = 0; q < kLzWaves; ++q) sum += part[q][64 + lane] * fast_exp2(part[q][lane] - mx);
        zi = (mx + log2f(sum)) * kLn2;
      }
      p.z[(int64_t)h * p.z_hs + b0 + lane] = zi;
    }
    __syncthreads();
  }
}

hipError_t launch_decomp_logz(const LogzParams& p, hipStream_t s) {
  const int nblk = (p.S + kLzRows - 1) / kLzRows;
  hipLaunchKernelGGL(decomp_logz_kernel, dim3(nblk, p.H), dim3(kLzThreads), 0, s, p);
  return hipGetLastError();
}


// ---- backward of the row normalisers ------------------------------------------
//   dalpha[h, j] = sum_{i >= j} gz[h, i] exp(alpha[h, j] + rho[h, i - j] - z[h, i])
//   drho[h, d]   = sum_{i >= d} gz[h, i] exp(alpha[h, i - d] + rho[h, d] - z[h, i])
// (the derivative of z = logsumexp_{j<=i}(alpha_j + rho_{i-j}); every term is
// gz_i times a probability <= 1).  Both are one sweep over the rows i >= o of an
// output index o: o's own logit part (alpha_j for dalpha, rho_d for drho) times a
// correlation of w_i = gz_i 2^(-z_i) with the other vector's exponentials at
// i - o, in the forward's layout: per chunk of rows w' = gz_i 2^(-z_i - W) and
// o' = 2^(other - O) (W, O the maxima over the chunk's rows and over the elements
// it can meet), 4 outputs per lane, one FMA per pair, and the chunk's sums join
// the output's total times 2^(own + O + W).  A product lost below 2^-126 is then
// worth at most 2^(own + O + W - 126) |gz_i|: chunks where own + O + W exceeds
// kLzScale for some output (logits whose maxima lie far above every pair's
// value) or is not finite run the direct form, one exp2 per pair, and so do
// chunks with a gz that is not finite: the zero that stands for a pair outside
// the triangle would turn it into NaN for outputs o > i that the row does not
// reach.  Rows whose z is -inf (every logit -inf) contribute nothing.
// H=12, S=8192: 264 us (one exp2 per pair) -> 49 us.
constexpr float kLzScale = 40.f;

__global__ __launch_bounds__(kLzThreads) void decomp_logz_bwd_kernel(const LogzBwdParams p) {
  __shared__ __align__(16) float as[kLzChunk];  // w' (direct form: gz)
  __shared__ __align__(16) float es[kLzChunk];  // direct form: -z log2 e
  __shared__ __align__(16) float ws[kLzWin];    // o' (direct form: other log2 e)
  __shared__ float part[kLzWaves][kLzRows];
  __shared__ float red[2][kLzWaves];

  const float ninf = -__builtin_inff();
  const int S = p.S;
  const int o0 = (int)blockIdx.x * kLzRows;   // heaviest first
  const int h = blockIdx.y;
  const bool dr = blockIdx.z == 1;             // 0: dalpha, 1: drho
  const int tid = threadIdx.x, lane = tid & 63, w = __builtin_amdgcn_readfirstlane(tid >> 6);
  const float* alpha = p.alpha + (int64_t)h * p.a_hs;
  const float* rho = p.rho + (int64_t)h * p.r_hs;
  const float* own = dr ? rho : alpha;       // logit part indexed by the output
  const float* other = dr ? alpha : rho;     // logit part indexed by i - o
  float fixed[4], fmx = ninf;
#pragma unroll
  for (int r = 0; r < 4; ++r) {
    const int o = o0 + 4 * lane + r;
    fixed[r] = o < S ? own[o] * kLog2e : ninf;
    fmx = fmaxf(fmx, fixed[r]);
  }
  fmx = wave_max(fmx);  // every wave holds the same 256 outputs

  float tot[4] = {0.f, 0.f, 0.f, 0.f};
  float gv[kLzNA], ev[kLzNA], ov[kLzNW];
  auto load = [&](int c0) {  // this thread's share of a chunk's rows and window
    const int tlo = c0 - o0 - (kLzRows - 1);   // smallest i - o of the chunk
#pragma unroll
    for (int k = 0; k < kLzNA; ++k) {
      const int i = c0 + tid + k * kLzThreads;
      ev[k] = i < S ? p.z[(int64_t)h * p.z_hs + i] : ninf;
      gv[k] = i < S ? p.gz[(int64_t)h * p.g_hs + i] : 0.f;
    }
#pragma unroll
    for (int k = 0; k < kLzNW; ++k) {
      const int x = tid + k * kLzThreads, d = tlo + x;
      ov[k] = (x < kLzWin && d >= 0 && d < S) ? other[d] : ninf;
    }
  };
  load(o0);
  for (int c0 = o0; c0 < S; c0 += kLzChunk) {
    float W = ninf, O = ninf;
#pragma unroll
    for (int k = 0; k < kLzNA; ++k) {
      const bool none = ev[k] == ninf;  // z of a row without a share
      gv[k] = none ? 0.f : gv[k];
      ev[k] = none ? ninf : -ev[k] * kLog2e;
      W = fmaxf(W, __builtin_isfinite(gv[k]) ? ev[k] : -ninf);
    }
#pragma unroll
    for (int k = 0; k < kLzNW; ++k) O = fmaxf(O, ov[k] *= kLog2e);
    group_max2(W, O, red, lane, w);  // its barrier: the previous chunk is consumed
    const float sc = O + W;
    const bool fast = fmx + sc <= kLzScale;  // false where not comparable
#pragma unroll
    for (int k = 0; k < kLzNA; ++k) {
      const int t = tid + k * kLzThreads;
      // a row without a share (ev -inf) adds nothing whatever the maxima are
      as[t] = fast ? (ev[k] == ninf ? 0.f : gv[k] * fast_exp2(ev[k] - W)) : gv[k];
      if (!fast) es[t] = ev[k];
    }
#pragma unroll
    for (int k = 0; k < kLzNW; ++k) {
      const int x = tid + k * kLzThreads;
      if (x < kLzWin) ws[x] = fast ? (ov[k] == ninf ? 0.f : fast_exp2(ov[k] - O)) : ov[k];
    }
    __syncthreads();
    load(c0 + kLzChunk);  // lands while the products run
    __builtin_amdgcn_sched_barrier(0);
    const int n = min(kLzChunk, S - c0);
    const int quota = ((n + kLzWaves - 1) / kLzWaves + 3) / 4 * 4;  // rows past n are zero
    const int n4 = (n + 3) / 4 * 4, t0 = min(w * quota, n4), t1 = min((w + 1) * quota, n4);
    float acc[4] = {0.f, 0.f, 0.f, 0.f};
    // window element of (output 4 lane + r, row t): t - 4 lane - r + kLzRows - 1
    if (fast) {
      slide<true>(acc, as, ws + kLzRows - 4 - 4 * lane, t0, t1);
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        const float c = fixed[r] + sc;
        tot[r] = fmaf(acc[r], c == ninf ? 0.f : fast_exp2(c), tot[r]);
      }
    } else {
      for (int t = t0; t < min(t1, n); ++t)
#pragma unroll
        for (int r = 0; r < 4; ++r) {
          const float x = fixed[r] + ws[t - 4 * lane - r + kLzRows - 1] + es[t];
          if (x != ninf) acc[r] = fmaf(as[t], fast_exp2(x), acc[r]);
        }
#pragma unroll
      for (int r = 0; r < 4; ++r) tot[r] += acc[r];
    }
  }
#pragma unroll
  for (int r = 0; r < 4; ++r) part[w][4 * lane + r] = tot[r];
  __syncthreads();
  if (tid < kLzRows && o0 + tid < S) {
    float s = 0.f;
#pragma unroll
    for (int q = 0; q < kLzWaves; ++q) s += part[q][tid];
    (dr ? p.drho + (int64_t)h * p.dr_hs : p.dalpha + (int64_t)h * p.da_hs)[o0 + tid] = s;
  }
}

hipError_t launch_decomp_logz_bwd(const LogzBwdParams& p, hipStream_t s) {
  const int nblk = (p.S + kLzRows - 1) / kLzRows;
  hipLaunchKernelGGL(decomp_logz_bwd_kernel, dim3(nblk, p.H, 2), dim3(kLzThreads), 0, s, p);
  return hipGetLastError();
}

}  // namespace saf
