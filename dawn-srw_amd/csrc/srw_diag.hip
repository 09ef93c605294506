// srw_diag.hip -- training diagnostics: of a stored score matrix, the tiled
// family's per-token and per-unit statistics (v41:434-483, 519-552); of those
// statistics, the result tuple's values (v41:588-635); and the operands'
// bf16 casts.

#include <math.h>

#include "srw_internal.hpp"
#include "srw_mfma_util.hpp"

namespace srw {

namespace {

typedef uint32_t u32x2_t __attribute__((ext_vector_type(2)));

constexpr int kDgRows = 32;    // rows per wave: one unit_part block
constexpr int kDgUnits = 256;  // units per wave: four per lane

// One wave per (32 rows, 256 units).  A wave instruction covers one row's
// 256 units (a lane four of them), so that
//   * a unit's statistics stay in its lane's registers over the rows,
//   * the counts are wave masks of a compare, counted on the scalar unit,
//   * the row's sums and maximum are left per lane for 16 rows and then
//     reduced together (reduce_scatter16: one exchange per value and row).
// Bound: the vector ALU, ~38 instructions per score (three transcendentals:
// exp and rcp of the gate, log of g log g); the scores are read once, 2 bytes
// each.  A kernel of its own rather than a part of the gate kernel's
// epilogue, which one wave per SIMD runs with nothing beside it.
struct DgRow {
  float s3, s4, glogg, smax;
};

template <bool FULL>
__device__ __attribute__((always_inline)) inline void diag_wave(const TiledDiagArgs& p, int64_t rb, int64_t ct,
                                                                int lane) {
  const int64_t u0 = ct * kDgUnits + 4 * lane;
  const int64_t r0 = rb * kDgRows;
  const float c_exp = p.exp_scale, eps = p.gp.eps, maxi = p.gp.maxi;
  const bool col_ok = FULL || u0 < p.N64;
  bool ok[4];
#pragma unroll
  for (int e = 0; e < 4; ++e) ok[e] = FULL || u0 + e < p.N;
  float su[4] = {0.f, 0.f, 0.f, 0.f};
  float mx[4] = {-INFINITY, -INFINITY, -INFINITY, -INFINITY};
#pragma unroll 1
  for (int half = 0; half < 2; ++half) {
    const int64_t rh = r0 + 16 * half;
    if (rh >= p.Tv) break;
    u32x2_t sv[16];
#pragma unroll
    for (int i = 0; i < 16; ++i) {
      const int64_t t = rh + i < p.Tv ? rh + i : p.Tv - 1;
      sv[i] = col_ok ? *reinterpret_cast<const u32x2_t*>(p.S + t * p.N64 + u0) : u32x2_t{0u, 0u};
    }
    float s3[16], s4[16], gl[16], sm[16];
    int c_sb = 0, c_73 = 0, c_cap = 0;  // lane reversed(i): row i's counts, two 16-bit halves each
#pragma unroll
    for (int i = 0; i < 16; ++i) {
      const int64_t t = rh + i < p.Tv ? rh + i : p.Tv - 1;
      const float tau = p.tau[t];
      const float tau_thr = tau + p.gp.thr;
      const float k_exp = -tau_thr * c_exp;
      const float tau_cut = tau_thr + p.gp.cut;
      const bool row = rh + i < p.Tv;  // uniform
      float a3 = 0.f, a4 = 0.f, ag = 0.f, am = -INFINITY;
      int n_strong = 0, n_bound = 0, n_075 = 0, n_030 = 0, n_cap = 0;
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        const uint32_t w = sv[i][e >> 1];
        const float s = (e & 1) ? hi_f32(w) : lo_f32(w);
        const GateElem g = gate_elem(s, c_exp, k_exp, tau_cut, eps, maxi);
        const float arg = __uint_as_float(g.sign), aa = fabsf(arg);
        const float s2 = s * s;
        a3 = fmaf(s2, s, a3);  // zero past N
        a4 = fmaf(s2, s2, a4);
        const float gg = FULL || ok[e] ? g.g : 0.f;
        ag = fmaf(gg, __builtin_amdgcn_logf(gg + 1e-8f), ag);
        am = fmaxf(am, FULL || ok[e] ? s : -INFINITY);
        // act > 0.9 <=> arg < -log2 9 and so on (the sigmoid's exact inverse)
        n_strong += __builtin_popcountll(__ballot((FULL || ok[e]) && arg < -3.169925001442312f));
        n_bound += __builtin_popcountll(__ballot((FULL || ok[e]) && aa < 3.169925001442312f));
        n_075 += __builtin_popcountll(__ballot((FULL || ok[e]) && aa < 4.247927513443585f));
        n_030 += __builtin_popcountll(__ballot((FULL || ok[e]) && aa < 2.0f));
        n_cap += __builtin_popcountll(__ballot((FULL || ok[e]) && g.inten >= p.gp.cap_thresh));
        if (row) {
          su[e] += s;
          mx[e] = fmaxf(mx[e], s - tau);
        }
      }
      s3[i] = a3;
      s4[i] = a4;
      gl[i] = ag;
      sm[i] = am;
      // the lane that reduce_scatter16 leaves row i in
      const int li = 8 * (i & 1) + 4 * ((i >> 1) & 1) + 2 * ((i >> 2) & 1) + ((i >> 3) & 1);
      c_sb = lane == li ? n_strong | (n_bound << 16) : c_sb;
      c_73 = lane == li ? n_075 | (n_030 << 16) : c_73;
      c_cap = lane == li ? n_cap : c_cap;
      __builtin_amdgcn_sched_barrier(0);  // one row at a time: bounded registers
    }
    auto add = [](float x, float y) { return x + y; };
    auto mxf = [](float x, float y) { return fmaxf(x, y); };
    reduce_scatter16(s3, lane, add);
    reduce_scatter16(s4, lane, add);
    reduce_scatter16(gl, lane, add);
    reduce_scatter16(sm, lane, mxf);
    const float t3 = s3[0] + __shfl_xor(s3[0], 32), t4 = s4[0] + __shfl_xor(s4[0], 32);
    const float tg = gl[0] + __shfl_xor(gl[0], 32), tm = fmaxf(sm[0], __shfl_xor(sm[0], 32));
    const int64_t t = rh + 8 * (lane & 1) + 4 * ((lane >> 1) & 1) + 2 * ((lane >> 2) & 1) + ((lane >> 3) & 1);
    if (lane < 16 && t < p.Tv) {
      float4* q = reinterpret_cast<float4*>(p.part + (ct * p.Tv + t) * kTokPartDiag);
      q[0] = make_float4(t3, t4, 0.f, 0.f);
      q[1] = make_float4(tm, static_cast<float>(c_sb & 0xffff), static_cast<float>(c_sb >> 16),
                         static_cast<float>(c_73 & 0xffff));
      q[2] = make_float4(static_cast<float>(c_73 >> 16), static_cast<float>(c_cap), tg * 0.69314718055994531f, 0.f);
    }
  }
  if (p.unit_part) {
#pragma unroll
    for (int e = 0; e < 4; ++e)
      if (ok[e]) p.unit_part[rb * p.N + u0 + e] = make_float2(su[e], mx[e]);
  }
}

__global__ __launch_bounds__(256) void tiled_diag_kernel(TiledDiagArgs p) {
  const int lane = threadIdx.x & 63;
  const int64_t rb = static_cast<int64_t>(blockIdx.x) * 4 + __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int64_t ct = blockIdx.y;
  if (rb * kDgRows >= p.Tv) return;
  if ((ct + 1) * kDgUnits <= p.N) diag_wave<true>(p, rb, ct, lane);
  else diag_wave<false>(p, rb, ct, lane);
}

// A row's slots over the 256-unit slices, in a fixed order: thread (c, grp)
// of a workgroup sums float4 c of the [Tv][3] float4s over slices grp mod 4
// with eight loads in flight; the four groups combine in LDS in order.
__global__ __launch_bounds__(256) void tiled_diag_sum_kernel(TiledDiagArgs p, int CT) {
  __shared__ float4 red[4][64];
  const int c = threadIdx.x & 63, grp = threadIdx.x >> 6;
  const int64_t n = p.Tv * 3;
  const int64_t i = static_cast<int64_t>(blockIdx.x) * 64 + c;
  const int64_t il = i < n ? i : n - 1;
  const float4* col = reinterpret_cast<const float4*>(p.part) + il;
  const bool has_max = il % 3 == 1;  // TP_SMAX is the first float of the row's second float4
  float4 acc = has_max ? make_float4(-INFINITY, 0.f, 0.f, 0.f) : make_float4(0.f, 0.f, 0.f, 0.f);
  auto join = [&](float4& a, const float4& q) {
    a.x = has_max ? fmaxf(a.x, q.x) : a.x + q.x;
    a.y += q.y;
    a.z += q.z;
    a.w += q.w;
  };
  int s = grp;
  for (; s + 28 < CT; s += 32) {
    float4 q[8];
#pragma unroll
    for (int k = 0; k < 8; ++k) q[k] = col[(s + 4 * k) * n];
#pragma unroll
    for (int k = 0; k < 8; ++k) join(acc, q[k]);
  }
  for (; s < CT; s += 4) join(acc, col[s * n]);
  red[grp][c] = acc;
  __syncthreads();
  if (grp != 0 || i >= n) return;
#pragma unroll
  for (int g = 1; g < 4; ++g) join(acc, red[g][c]);
  const int64_t t = i / 3;
  if (i % 3 == 0) {
    if (p.token_diag) {
      p.token_diag[t * SRW_TDIAG_COUNT + SRW_TDIAG_SUM_S3] = acc.x;
      p.token_diag[t * SRW_TDIAG_COUNT + SRW_TDIAG_SUM_S4] = acc.y;
    }
  } else {
    *reinterpret_cast<float4*>(p.tok_sum + t * kTokPartDiag + 4 * (i % 3)) = acc;
  }
}

// ---------------------------------------------------------------------------
// The result tuple's per-token values and scalars (v41:588-635, :862-907;
// v401:343-367, :525-553).  As torch operations on the [T, R] and [N] columns
// they were ~70 launches of 2-5 us each, more than the layer's own kernels at
// the small pools (a paired step at N = 1 580, T = 4 096: 905 -> 519 us with
// these two launches and the operands' casts in one; the Know pool's 2 131 ->
// 1 846).  Here: workgroups over the tokens, then the units, each
// leaving its sums in double; one workgroup joins them in workgroup order.
// ---------------------------------------------------------------------------
enum {
  DS_STD, DS_G, DS_NA, DS_NA2, DS_TAU, DS_075, DS_030, DS_SKEW, DS_ENT, DS_INT, DS_KURT, DS_CAP,  // over rows
  DS_PN, DS_PN2, DS_PEN, DS_DEAD,                                                                 // over units
  DS_IMAX,                                                                                        // a maximum
  DS_COUNT
};
constexpr int kDsBlocks = 256;  // at most this many workgroups (rows and units together)
static_assert(kDsBlocks * DS_COUNT * sizeof(double) <= SRW_DSUM_WORKSPACE_BYTES, "partials fit the workspace");

struct DsumParams {
  const float* gate_sum;
  const int32_t* n_active;
  const float* td;
  const float* ud;
  srw_diag_out_t out;
  double* part;  // [blocks][DS_COUNT]
  int64_t T, N;
  int R, v401, row_blocks, blocks;
  float dead_threshold;
};

__device__ inline double wave_sum_d(double v) {
#pragma unroll
  for (int o = 32; o > 0; o >>= 1) v += __shfl_xor(v, o);
  return v;
}
// torch's max: a NaN stays
__device__ inline double max_nan(double a, double b) { return a != a || a > b ? a : b; }

__global__ __launch_bounds__(256) void diag_rows_units_kernel(DsumParams p) {
  double v[DS_COUNT];
#pragma unroll
  for (int k = 0; k < DS_COUNT; ++k) v[k] = k == DS_IMAX ? -INFINITY : 0.0;
  const double N = static_cast<double>(p.N);
  const float nf = static_cast<float>(p.N);
  if (static_cast<int>(blockIdx.x) < p.row_blocks) {
    for (int64_t t = static_cast<int64_t>(blockIdx.x) * 256 + threadIdx.x; t < p.T; t += 256LL * p.row_blocks) {
      float tok[SRW_DSUM_TOKEN_COUNT] = {0.f, 0.f, 0.f, 0.f, 0.f};
      for (int r = 0; r < p.R; ++r) {
        const int64_t i = t * p.R + r;
        const float* td = p.td + i * SRW_TDIAG_COUNT;
        const float g = p.gate_sum[i], na = static_cast<float>(p.n_active[i]);
        tok[SRW_DSUM_ACTIVE_FRAC] += na / nf;
        tok[SRW_DSUM_GATE_MAX] += td[SRW_TDIAG_GATE_MAX];
        tok[SRW_DSUM_STRONG_FRAC] += td[SRW_TDIAG_N_STRONG] / nf;
        tok[SRW_DSUM_BOUNDARY_FRAC] += td[SRW_TDIAG_N_BOUNDARY] / nf;
        tok[SRW_DSUM_Z_MEAN_ACTIVE] += (p.v401 ? td[SRW_TDIAG_INT_SUM] : g) / (na + 1e-8f);
        // moments -> skew / kurtosis (v41:466-474)
        const double m = td[SRW_TDIAG_S_MEAN], sd = td[SRW_TDIAG_S_STD];
        const double c3 = td[SRW_TDIAG_SUM_S3] / N, c4 = td[SRW_TDIAG_SUM_S4] / N;
        v[DS_STD] += sd;
        v[DS_G] += g;
        v[DS_NA] += na;
        v[DS_NA2] += static_cast<double>(na) * na;
        v[DS_TAU] += td[SRW_TDIAG_TAU];
        const float act = p.v401 ? na + 1e-8f : (na < 1.0f ? 1.0f : na);  // v41:599, v401:349
        v[DS_075] += td[SRW_TDIAG_N_BAND075] / act;
        v[DS_030] += td[SRW_TDIAG_N_BAND030] / act;
        v[DS_SKEW] += (c3 - 3.0 * m * sd * sd - m * m * m) / (sd * sd * sd + 1e-8);
        v[DS_KURT] += (c4 - 4.0 * m * c3 + 6.0 * m * m * sd * sd + 3.0 * m * m * m * m) / (sd * sd * sd * sd + 1e-8);
        // entropy (v41:611-618; v401:360-363)
        float ent;
        if (p.v401) {
          const float ge = g + 1e-8f;
          ent = -td[SRW_TDIAG_G_LOG_G] / ge + logf(ge);
        } else {
          const float ge = g < 1e-6f ? 1e-6f : g;
          ent = -(g > 1e-6f ? td[SRW_TDIAG_G_LOG_G] : 0.f) / ge + logf(ge);
          ent = isfinite(ent) ? ent : 0.f;
        }
        v[DS_ENT] += ent;
        v[DS_INT] += td[SRW_TDIAG_INT_SUM];
        v[DS_CAP] += td[SRW_TDIAG_N_INT_CAP];
        v[DS_IMAX] = max_nan(td[SRW_TDIAG_INT_MAX], v[DS_IMAX]);
      }
      const float inv = p.R == 2 ? 0.5f : 1.0f;
#pragma unroll
      for (int k = 0; k < SRW_DSUM_TOKEN_COUNT; ++k)
        if (p.out.token[k]) p.out.token[k][t] = tok[k] * inv;
    }
  } else {
    const int nb = p.blocks - p.row_blocks;
    const float rows = static_cast<float>(p.T * p.R);
    for (int64_t n = (static_cast<int64_t>(blockIdx.x) - p.row_blocks) * 256 + threadIdx.x; n < p.N; n += 256LL * nb) {
      const float pn = p.ud[n * SRW_UDIAG_COUNT + SRW_UDIAG_SCORE_SUM] / rows;   // mean score (v41:445-447)
      const bool dead = p.ud[n * SRW_UDIAG_COUNT + SRW_UDIAG_GATE_MAX] < p.dead_threshold;
      v[DS_PN] += pn;
      v[DS_PN2] += static_cast<double>(pn) * pn;
      // relu(-pn) * dead, a product: a NaN or -inf mean gives NaN also times 0 (v41:548-552)
      v[DS_PEN] += (pn != pn ? pn : (pn < 0.f ? -pn : 0.f)) * (dead ? 1.f : 0.f);
      v[DS_DEAD] += dead ? 1.0 : 0.0;
    }
  }
  __shared__ double red[4][DS_COUNT];
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
#pragma unroll
  for (int k = 0; k < DS_COUNT; ++k) {
    double x = v[k];
    if (k == DS_IMAX) {
#pragma unroll
      for (int o = 32; o > 0; o >>= 1) x = max_nan(x, __shfl_xor(x, o));
    } else {
      x = wave_sum_d(x);
    }
    if (lane == 0) red[wave][k] = x;
  }
  __syncthreads();
  if (threadIdx.x < DS_COUNT) {
    const int k = threadIdx.x;
    double x = red[0][k];
    for (int w = 1; w < 4; ++w) x = k == DS_IMAX ? max_nan(x, red[w][k]) : x + red[w][k];
    p.part[static_cast<int64_t>(blockIdx.x) * DS_COUNT + k] = x;
  }
}

// One wave per sum: its workgroups' partials in a fixed order, then the tuple.
__global__ __launch_bounds__(1024) void diag_scalars_kernel(DsumParams p) {
  __shared__ double tot[DS_COUNT];
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  for (int k = wave; k < DS_COUNT; k += 16) {
    double x = k == DS_IMAX ? -INFINITY : 0.0;
    for (int b = lane; b < p.blocks; b += 64) {
      const double q = p.part[static_cast<int64_t>(b) * DS_COUNT + k];
      x = k == DS_IMAX ? max_nan(q, x) : x + q;
    }
    if (k == DS_IMAX) {
#pragma unroll
      for (int o = 32; o > 0; o >>= 1) x = max_nan(x, __shfl_xor(x, o));
    } else {
      x = wave_sum_d(x);
    }
    if (lane == 0) tot[k] = x;
  }
  __syncthreads();
  if (threadIdx.x != 0) return;
  const double rows = static_cast<double>(p.T) * p.R, N = static_cast<double>(p.N);
  double s[SRW_DSUM_SCALAR_COUNT];
  const double mean = tot[DS_PN] / N, var = tot[DS_PN2] / N - mean * mean;
  s[SRW_DSUM_SCORE_LB] = var / (mean * mean + var + 1e-2);                       // v41:477-483
  s[SRW_DSUM_SCORE_STD] = tot[DS_STD] / rows;
  s[SRW_DSUM_GATE_SUM] = tot[DS_G] / rows;
  s[SRW_DSUM_ACTIVE_N] = tot[DS_NA] / rows;
  s[SRW_DSUM_TAU] = tot[DS_TAU] / rows;
  s[SRW_DSUM_Z_LT_075] = tot[DS_075] / rows;
  s[SRW_DSUM_Z_LT_030] = tot[DS_030] / rows;
  s[SRW_DSUM_SKEW] = tot[DS_SKEW] / rows;
  const double na = tot[DS_NA] / rows, na_var = tot[DS_NA2] / rows - na * na;    // counts: exact sums
  s[SRW_DSUM_ACTIVE_STD] = sqrt(na_var > 0.0 ? na_var : 0.0);
  s[SRW_DSUM_ENTROPY] = tot[DS_ENT] / rows;
  s[SRW_DSUM_INT_SUM] = tot[DS_INT] / rows;
  s[SRW_DSUM_KURT] = tot[DS_KURT] / rows;
  s[SRW_DSUM_DEAD_PENALTY] = tot[DS_PEN];
  s[SRW_DSUM_DEAD_COUNT] = tot[DS_DEAD];
  s[SRW_DSUM_INT_MAX] = tot[DS_IMAX];
  s[SRW_DSUM_INT_CAP] = tot[DS_CAP] / (rows * N);
#pragma unroll
  for (int k = 0; k < SRW_DSUM_SCALAR_COUNT; ++k)
    if (p.out.scalar[k]) *p.out.scalar[k] = static_cast<float>(s[k]);
}

// ---------------------------------------------------------------------------
// fp32 -> bf16 casts of several arrays in one launch, 16 bytes stored per
// thread and step where the array allows; bound by HBM.
// ---------------------------------------------------------------------------
constexpr int kCastBlock = 256 * 8;  // elements per workgroup
struct CastParams {
  const float* src[SRW_MAX_CAST];
  uint16_t* dst[SRW_MAX_CAST];
  int64_t count[SRW_MAX_CAST];
  int64_t start[SRW_MAX_CAST + 1];  // first workgroup of each array
  int n;
};
__global__ __launch_bounds__(256) void cast_bf16_kernel(CastParams p) {
  int i = 0;
  for (int k = 1; k < p.n; ++k) i += static_cast<int64_t>(blockIdx.x) >= p.start[k] ? 1 : 0;
  const float* src = p.src[i];
  uint16_t* dst = p.dst[i];
  const int64_t k = (static_cast<int64_t>(blockIdx.x) - p.start[i]) * kCastBlock + 8 * threadIdx.x;
  const int64_t left = p.count[i] - k;
  if (left <= 0) return;
  const bool wide = ((reinterpret_cast<uintptr_t>(src) | reinterpret_cast<uintptr_t>(dst)) & 15) == 0;
  if (left >= 8 && wide) {
    const float4 a = *reinterpret_cast<const float4*>(src + k), b = *reinterpret_cast<const float4*>(src + k + 4);
    *reinterpret_cast<u32x4_t*>(dst + k) =
        u32x4_t{pack_bf16(a.x, a.y), pack_bf16(a.z, a.w), pack_bf16(b.x, b.y), pack_bf16(b.z, b.w)};
  } else {
    for (int e = 0; e < 8 && e < left; ++e) dst[k + e] = f32_to_bf16_bits(src[k + e]);
  }
}

}  // namespace

hipError_t diag_summary(const srw_desc_t& d, const srw_outputs_t& o, const srw_diag_out_t& out, double* part,
                        hipStream_t s) {
  DsumParams p{};
  p.gate_sum = o.gate_sum;
  p.n_active = o.n_active;
  p.td = o.token_diag;
  p.ud = o.unit_diag;
  p.out = out;
  p.part = part;
  p.T = d.T;
  p.N = d.n_units;
  p.R = d.n_routes;
  p.v401 = d.gate == SRW_GATE_GELU_V401;
  p.dead_threshold = d.dead_threshold;
  const int64_t rb = (d.T + 255) / 256, ub = (d.n_units + 255) / 256;
  p.row_blocks = static_cast<int>(rb < kDsBlocks / 2 ? rb : kDsBlocks / 2);
  p.blocks = p.row_blocks + static_cast<int>(ub < kDsBlocks / 2 ? ub : kDsBlocks / 2);
  hipLaunchKernelGGL(diag_rows_units_kernel, dim3(static_cast<unsigned>(p.blocks)), dim3(256), 0, s, p);
  hipError_t e = hipGetLastError();
  if (e != hipSuccess) return e;
  hipLaunchKernelGGL(diag_scalars_kernel, dim3(1), dim3(1024), 0, s, p);
  return hipGetLastError();
}

hipError_t cast_bf16(int n, const float* const* src, uint16_t* const* dst, const int64_t* count, hipStream_t s) {
  CastParams p{};
  p.n = n;
  for (int i = 0; i < n; ++i) {
    p.src[i] = src[i];
    p.dst[i] = dst[i];
    p.count[i] = count[i];
    p.start[i + 1] = p.start[i] + (count[i] + kCastBlock - 1) / kCastBlock;
  }
  if (p.start[n] == 0) return hipSuccess;
  if (p.start[n] > 0x7fffffff) return hipErrorInvalidValue;
  hipLaunchKernelGGL(cast_bf16_kernel, dim3(static_cast<unsigned>(p.start[n])), dim3(256), 0, s, p);
  return hipGetLastError();
}

hipError_t tiled_diag(const TiledDiagArgs& a, hipStream_t s) {
  static_assert(kTokPartDiag == 12 && TP_SMAX == 4 && TP_GLOGG == 10, "three float4s per row");
  const int64_t rbs = (a.Tv + kDgRows - 1) / kDgRows;
  const int CT = static_cast<int>((a.N + kDgUnits - 1) / kDgUnits);
  hipLaunchKernelGGL(tiled_diag_kernel, dim3(static_cast<unsigned>((rbs + 3) / 4), static_cast<unsigned>(CT)),
                     dim3(256), 0, s, a);
  hipError_t e = hipGetLastError();
  if (e != hipSuccess) return e;
  hipLaunchKernelGGL(tiled_diag_sum_kernel, dim3(static_cast<unsigned>((a.Tv * 3 + 63) / 64)), dim3(256), 0, s, a, CT);
  return hipGetLastError();
}

}  // namespace srw
