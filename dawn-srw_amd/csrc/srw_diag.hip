// srw_diag.hip -- training diagnostics of a stored score matrix: the tiled
// family's per-token and per-unit statistics (v41:434-483, 519-552).

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

}  // namespace

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
