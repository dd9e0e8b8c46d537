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
// The two factors carry 2^52 each, so that a chunk's sums stay below 2^128 and
// factors are lost only below 2^-178 of their maximum, products below 2^-230 of
// the scale M: at most S 2^-178 of it in all.  A row whose total is below 2^-132
// (its own keys lie far below the chunk's maxima, or all are -inf, or a value is
// not finite) sends its work-group through the direct form too: the same sweep
// with 8 logits at a time folded into a row's running (max, sum), one exp2 per
// pair.  H=12, us, one exp2 per logit always / a direct form from 2^-80 on, of one
// 64-row block at a time with two LDS reads per pair / now: logits of scale 20
// S=2048 18 / 37 / 12, S=8192 130 / 212 / 64; of scale 40, where most groups run both
// forms, S=2048 17 / - / 14, S=8192 130 / - / 133.
//
// Bound by FMA issue (S(S+1)/2 per head; HBM traffic is 3 S 4 bytes):
// H=12, S=8192: 135 us (one exp2 per logit) -> 23 us; S=16384: 321 -> 61 us.
#include "saf_kernels.h"

namespace saf {

constexpr int kLzRows = 256;           // rows (outputs) of a work-group (64 where these are few: launch)
constexpr int kLzWaves = 8;
constexpr int kLzThreads = 64 * kLzWaves;
constexpr int kLzChunk = 2048;         // keys per chunk
constexpr int kLzWin = kLzChunk + kLzRows;
constexpr int kLzNA = kLzChunk / kLzThreads;                       // staged values per thread
constexpr int kLzNW = (kLzWin + kLzThreads - 1) / kLzThreads;
constexpr int kLzBias = 52;                       // forward: exponent added to a' and to r'
constexpr float kLzLow = 3.725290298461914e-09f;  // 2^-28: 2^-132 of the scale and both biases
constexpr float kLn2 = 0.6931471805599453f;

// Maxima of x[0 .. N) over the work-group (each wave's through `red`).
template <int N>
__device__ __forceinline__ void group_max(float (&x)[N], float (*red)[kLzWaves], int lane, int w) {
#pragma unroll
  for (int i = 0; i < N; ++i) {
    x[i] = wave_max(x[i]);
    if (lane == 0) red[i][w] = x[i];
  }
  __syncthreads();
#pragma unroll
  for (int i = 0; i < N; ++i)
#pragma unroll
    for (int q = 0; q < kLzWaves; ++q) x[i] = fmaxf(x[i], red[i][q]);
}

// A NaN counts as +inf in a maximum that scales: what it scales is then NaN too.
__device__ __forceinline__ float top(float m, float x) { return fmaxf(m, x != x ? __builtin_inff() : x); }

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

// The direct forms of the two sweeps.  CHECK: a pair outside the triangle (win
// -inf; backward: a logit of -inf) adds nothing even where its other factor is
// not finite; without it such a pair is finite + -inf, or a finite g times 0.
//
// (m[r], s[r]): running maximum and sum of 2^(x - m) over x = as[t + u] + win(r, u).
template <bool CHECK>
__device__ __forceinline__ void slide_lse(float (&m)[4], float (&s)[4], const float* as, const float* p, int t0,
                                          int t1) {
  float4 w0 = *reinterpret_cast<const float4*>(p + 4 - t0);
  for (int t = t0; t < t1; t += 8) {
    const float4 w1 = *reinterpret_cast<const float4*>(p - t), w2 = *reinterpret_cast<const float4*>(p - t - 4);
    const float4 a4 = *reinterpret_cast<const float4*>(as + t), b4 = *reinterpret_cast<const float4*>(as + t + 4);
    const float a[8] = {a4.x, a4.y, a4.z, a4.w, b4.x, b4.y, b4.z, b4.w};
    const float win[12] = {w2.x, w2.y, w2.z, w2.w, w1.x, w1.y, w1.z, w1.w, w0.x, w0.y, w0.z, w0.w};
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      float x[8], mn = m[r];
#pragma unroll
      for (int u = 0; u < 8; ++u) {
        const float v = win[7 + r - u];
        x[u] = CHECK && v == -__builtin_inff() ? v : a[u] + v;
        mn = fmaxf(mn, x[u]);
      }
      const float ref = mn == -__builtin_inff() ? 0.f : mn;  // nothing but -inf so far (or NaN, which stays)
      float acc = s[r] * fast_exp2(m[r] - ref);
#pragma unroll
      for (int u = 0; u < 8; ++u) acc += fast_exp2(x[u] - ref);
      s[r] = acc;
      m[r] = mn;
    }
    w0 = w2;
  }
}

// acc[r] += sum of g[t] 2^(fixed[r] + win(r, t) + e[t]), the window moving up.
template <bool CHECK>
__device__ __forceinline__ void slide_exp(float (&acc)[4], const float* g, const float* e, const float* p,
                                          const float (&fixed)[4], int t0, int t1) {
  float4 lo = *reinterpret_cast<const float4*>(p + t0);
#pragma unroll 2
  for (int t = t0; t < t1; t += 4) {
    const float4 hi = *reinterpret_cast<const float4*>(p + 4 + t);
    const float4 g4 = *reinterpret_cast<const float4*>(g + t), e4 = *reinterpret_cast<const float4*>(e + t);
    const float gt[4] = {g4.x, g4.y, g4.z, g4.w}, et[4] = {e4.x, e4.y, e4.z, e4.w};
    const float win[8] = {lo.x, lo.y, lo.z, lo.w, hi.x, hi.y, hi.z, hi.w};
#pragma unroll
    for (int u = 0; u < 4; ++u)
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        const float x = fixed[r] + win[3 + u - r] + et[u];
        const float v = fmaf(gt[u], fast_exp2(x), acc[r]);
        acc[r] = CHECK && x == -__builtin_inff() ? acc[r] : v;
      }
    lo = hi;
  }
}

// 2^(x + kLzBias) of x <= 0, down to x = -178.
__device__ __forceinline__ float biased_exp2(float x) {
  const float n = __builtin_rintf(fmaxf(x, -200.f));
  return __builtin_ldexpf(fast_exp2(x - n), (int)n + kLzBias);
}

// ROWS rows per work-group, 256 or 64: 64 lanes cover them (4 each) LG times over,
// each time with another share of the keys.
template <int ROWS>
__global__ __launch_bounds__(kLzThreads) void decomp_logz_kernel(const LogzParams p) {
  constexpr int LG = kLzRows / ROWS, kUnits = kLzWaves * LG;  // shares of a chunk's keys
  constexpr int kWin = kLzChunk + ROWS, kNW = (kWin + kLzThreads - 1) / kLzThreads;
  static_assert(kUnits * ROWS <= kWin, "the direct form's row maxima fit the window");
  __shared__ __align__(16) float as[kLzChunk];
  __shared__ __align__(16) float rs[kWin];
  __shared__ float part[kUnits][ROWS];
  __shared__ float red[2][kLzWaves];

  const float ninf = -__builtin_inff();
  const int S = p.S;
  const int nblk = (S + ROWS - 1) / ROWS;
  const int h = blockIdx.x % p.H;
  const int i0 = (nblk - 1 - (int)(blockIdx.x / p.H)) * ROWS;  // heaviest first
  const int tid = threadIdx.x, lane = tid & 63, w = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int rl = lane % (ROWS / 4), unit = w * LG + lane / (ROWS / 4);
  const float* alpha = p.alpha + (int64_t)h * p.a_hs;
  const float* rho = p.rho + (int64_t)h * p.r_hs;
  const int jend = min(i0 + ROWS, S);  // keys any row of the block can see

  float M = ninf, tot[4] = {0.f, 0.f, 0.f, 0.f};
  float av[kLzNA], rv[kNW];
  auto load = [&](int j0) {  // this thread's share of a chunk's keys and window
    const int dlo = i0 - j0 - kLzChunk + 1;  // distance of window element 0
#pragma unroll
    for (int k = 0; k < kLzNA; ++k) {
      const int j = j0 + tid + k * kLzThreads;
      av[k] = j < jend ? alpha[j] : ninf;
    }
#pragma unroll
    for (int k = 0; k < kNW; ++k) {
      const int x = tid + k * kLzThreads, d = dlo + x;
      rv[k] = (x < kWin && d >= 0 && d < S) ? rho[d] : ninf;
    }
  };
  load(0);
  for (int j0 = 0; j0 < jend; j0 += kLzChunk) {
    float mx[2] = {ninf, ninf};
#pragma unroll
    for (int k = 0; k < kLzNA; ++k) mx[0] = top(mx[0], av[k] *= kLog2e);
#pragma unroll
    for (int k = 0; k < kNW; ++k) mx[1] = top(mx[1], rv[k] *= kLog2e);
    group_max(mx, red, lane, w);  // its barrier: the previous chunk is consumed
    const float A = mx[0], R = mx[1], sc = A + R;
    if (sc != ninf) {
#pragma unroll
      for (int k = 0; k < kLzNA; ++k) as[tid + k * kLzThreads] = biased_exp2(av[k] - A);
#pragma unroll
      for (int k = 0; k < kNW; ++k)
        if (tid + k * kLzThreads < kWin) rs[tid + k * kLzThreads] = biased_exp2(rv[k] - R);
    }
    __syncthreads();
    load(j0 + kLzChunk);  // lands while the products run
    __builtin_amdgcn_sched_barrier(0);
    if (sc == ninf) continue;  // every logit of the chunk is -inf
    const int n = min(kLzChunk, jend - j0);
    const int quota = ((n + kUnits - 1) / kUnits + 3) / 4 * 4;  // keys past n are zero
    float acc[4] = {0.f, 0.f, 0.f, 0.f};
    // window element of (row 4 rl + r, key t): 4 rl + r + kLzChunk - 1 - t
    const int n4 = (n + 3) / 4 * 4;
    slide<false>(acc, as, rs + 4 * rl + kLzChunk - 4, min(unit * quota, n4), min((unit + 1) * quota, n4));
    const float Mn = fmaxf(M, sc), f0 = fast_exp2(M - Mn), f1 = fast_exp2(sc - Mn);
#pragma unroll
    for (int r = 0; r < 4; ++r) tot[r] = fmaf(acc[r], f1, tot[r] * f0);
    M = Mn;
  }
#pragma unroll
  for (int r = 0; r < 4; ++r) part[unit][4 * rl + r] = tot[r];
  __syncthreads();
  bool low = false;  // of this thread's row (the first ROWS threads)
  if (tid < ROWS && i0 + tid < S) {
    float s = 0.f;
#pragma unroll
    for (int q = 0; q < kUnits; ++q) s += part[q][tid];
    low = !(s >= kLzLow && s < __builtin_inff());  // NaN included
    const float e = (float)(__builtin_amdgcn_frexp_expf(s) - 2 * kLzBias);
    if (!low) p.z[(int64_t)h * p.z_hs + i0 + tid] = (M + (e + log2f(__builtin_amdgcn_frexp_mantf(s)))) * kLn2;
  }
  if (!__syncthreads_or(low)) return;

  // direct form, for the low rows
  float m[4] = {ninf, ninf, ninf, ninf}, s[4] = {0.f, 0.f, 0.f, 0.f};
  load(0);
  for (int j0 = 0; j0 < jend; j0 += kLzChunk) {
    bool odd = false;  // a key that the pairs outside the triangle must not see
#pragma unroll
    for (int k = 0; k < kLzNA; ++k) odd |= !(av[k] < __builtin_inff());
    const bool check = __syncthreads_or(odd);  // also: the previous chunk is consumed
#pragma unroll
    for (int k = 0; k < kLzNA; ++k) as[tid + k * kLzThreads] = av[k] * kLog2e;
#pragma unroll
    for (int k = 0; k < kNW; ++k)
      if (tid + k * kLzThreads < kWin) rs[tid + k * kLzThreads] = rv[k] * kLog2e;
    __syncthreads();
    load(j0 + kLzChunk);
    const int n = min(kLzChunk, jend - j0), n8 = (n + 7) / 8 * 8;  // keys past n are -inf
    const int quota = ((n + kUnits - 1) / kUnits + 7) / 8 * 8;
    const int t0 = min(unit * quota, n8), t1 = min((unit + 1) * quota, n8);
    const float* const win = rs + 4 * rl + kLzChunk - 4;
    if (t0 < t1) {
      if (check)
        slide_lse<true>(m, s, as, win, t0, t1);
      else
        slide_lse<false>(m, s, as, win, t0, t1);
    }
  }
  __syncthreads();
  float* const pm = rs;  // [unit][row] maxima
#pragma unroll
  for (int r = 0; r < 4; ++r) {
    pm[unit * ROWS + 4 * rl + r] = m[r];
    part[unit][4 * rl + r] = s[r];
  }
  __syncthreads();
  if (low) {
    float mx = ninf, sum = 0.f;
#pragma unroll
    for (int q = 0; q < kUnits; ++q) mx = fmaxf(mx, pm[q * ROWS + tid]);
    const float ref = mx == ninf ? 0.f : mx;
#pragma unroll
    for (int q = 0; q < kUnits; ++q) sum += part[q][tid] * fast_exp2(pm[q * ROWS + tid] - ref);
    p.z[(int64_t)h * p.z_hs + i0 + tid] = (ref + log2f(sum)) * kLn2;  // log2f(0): no key at all, -inf
  }
}

hipError_t launch_decomp_logz(const LogzParams& p, hipStream_t s) {
  const int nblk = (p.S + kLzRows - 1) / kLzRows;
  // Heads first: a CU's second work-group is lighter than its first.  64 rows
  // where 256 would leave CUs without a work-group.  256 / 64, us, learned logits
  // and scale 40 (both forms): 12 heads S=2048 (96 groups of 256) 7.1 / 6.3 and 29.6
  // / 14.2, S=4096 (192) 11.6 / 10.6 and 57 / 33; 24 heads S=3072 (288) 10.8 / 12.4
  // and 46 / 36, S=8192 (768) 31 / 46 and 199 / 182.
  if ((int64_t)nblk * p.H < p.n_cu)
    hipLaunchKernelGGL(decomp_logz_kernel<64>, dim3((unsigned)p.H * ((p.S + 63) / 64)), dim3(kLzThreads), 0, s, p);
  else
    hipLaunchKernelGGL(decomp_logz_kernel<kLzRows>, dim3((unsigned)p.H * nblk), dim3(kLzThreads), 0, s, p);
  return hipGetLastError();
}


// ---- backward of the row normalisers ------------------------------------------
//   dalpha[h, j] = sum_{i >= j} gz[h, i] exp(alpha[h, j] + rho[h, i - j] - z[h, i])
//   drho[h, d]   = sum_{i >= d} gz[h, i] exp(alpha[h, i - d] + rho[h, d] - z[h, i])
// (the derivative of z = logsumexp_{j<=i}(alpha_j + rho_{i-j}); every term is
// gz_i times a probability <= 1).  Both are one sweep over the rows i >= o of an
// output index o: o's own logit part (alpha_j for dalpha, rho_d for drho) times a
// correlation of w_i = gz_i 2^(-z_i) with the other vector's exponentials at
// i - o, in the forward's layout: per chunk of rows w' = gz_i 2^(-z_i - W - G) and
// o' = 2^(other - O) (W, O the maxima over the chunk's rows and over the elements
// it can meet, 2^G the power of two at its largest |gz|), 4 outputs per lane, one
// FMA per pair, and the chunk's sums join the output's total times 2^(own + O + W
// + G).  A product lost below 2^-126 is then worth at most 2^(own + O + W - 125)
// of that |gz|: chunks where own + O + W exceeds kLzScale for some output (logits
// whose maxima lie far above every pair's value) or is not finite run the direct
// form, one exp2 per pair over the same sliding window, and so do chunks with a
// gz that is not finite: the zero that stands for a pair outside the triangle
// would turn it into NaN for outputs o > i that the row does not reach.  Rows
// whose z is -inf (every logit -inf) contribute nothing.
// H=12, S=8192: 264 us (one exp2 per pair) -> 35 us; with logits of scale 20 (all
// direct) forward + backward 370 us before, 610 with a direct form that read the
// window by elements, 215 now.
constexpr float kLzScale = 40.f;

__global__ __launch_bounds__(kLzThreads) void decomp_logz_bwd_kernel(const LogzBwdParams p) {
  __shared__ __align__(16) float as[kLzChunk];  // w' (direct form: gz)
  __shared__ __align__(16) float es[kLzChunk];  // direct form: -z log2 e
  __shared__ __align__(16) float ws[kLzWin];    // o' (direct form: other log2 e)
  __shared__ float part[kLzWaves][kLzRows];
  __shared__ float red[3][kLzWaves];

  const float ninf = -__builtin_inff();
  const int S = p.S;
  const int o0 = (int)(blockIdx.x / (2 * p.H)) * kLzRows;  // heaviest first
  const int h = (int)(blockIdx.x % (2 * p.H)) >> 1;
  const bool dr = blockIdx.x & 1;                          // 0: dalpha, 1: drho
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
    float mx[3] = {ninf, ninf, 0.f};
#pragma unroll
    for (int k = 0; k < kLzNA; ++k) {
      const bool none = ev[k] == ninf;  // z of a row without a share
      gv[k] = none ? 0.f : gv[k];
      ev[k] = none ? ninf : -ev[k] * kLog2e;
      mx[0] = fmaxf(mx[0], __builtin_isfinite(gv[k]) ? ev[k] : -ninf);
      mx[2] = fmaxf(mx[2], fabsf(gv[k]));
    }
#pragma unroll
    for (int k = 0; k < kLzNW; ++k) mx[1] = fmaxf(mx[1], ov[k] *= kLog2e);
    group_max(mx, red, lane, w);  // its barrier: the previous chunk is consumed
    const float W = mx[0], O = mx[1], sc = O + W;
    const int G = __builtin_amdgcn_frexp_expf(mx[2]);
    const bool fast = fmx + sc <= kLzScale;  // false where not comparable
#pragma unroll
    for (int k = 0; k < kLzNA; ++k) {
      const int t = tid + k * kLzThreads;
      // a row without a share (ev -inf) adds nothing whatever the maxima are
      as[t] = fast ? (ev[k] == ninf ? 0.f : __builtin_ldexpf(gv[k], -G) * fast_exp2(ev[k] - W)) : gv[k];
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
    const float* const win = ws + kLzRows - 4 - 4 * lane;
    if (fast) {
      slide<true>(acc, as, win, t0, t1);
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        const float c = fixed[r] + sc;
        tot[r] += __builtin_ldexpf(acc[r] * (c == ninf ? 0.f : fast_exp2(c)), G);
      }
    } else {
      if (W == -ninf)  // a gz that is not finite
        slide_exp<true>(acc, as, es, win, fixed, t0, t1);
      else
        slide_exp<false>(acc, as, es, win, fixed, t0, t1);
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
  hipLaunchKernelGGL(decomp_logz_bwd_kernel, dim3(2u * p.H * nblk), dim3(kLzThreads), 0, s, p);
  return hipGetLastError();
}

}  // namespace saf
