// srw_model.hip -- the decode step of the DAWN model around the SRW calls
// (v41:1772-1828, 1914-1957), for decode-sized batches.
//
// As separate float32 operations a layer was ~45 launches beside its SRW
// calls' eight (router products, casts, cache writes, transposed copies of the
// whole KV cache for the batched products); the step was bound by their
// launches.  Here a layer has four: LayerNorm + router, attention over the
// cache, expand_O + residual, LayerNorm + router; the residual add of the Know
// output rides on the next LayerNorm.  Everything stays float32 where the
// reference computes float32.

#include <math.h>

#include "srw_internal.hpp"
#include "srw_mfma_util.hpp"

namespace srw {

namespace {

typedef float f32x4_t __attribute__((ext_vector_type(4)));

constexpr int kDh = 64;  // head width

// Dense layer on 16-row x 16-column tiles of v_mfma_f32_16x16x4_f32, the four
// waves of a workgroup splitting K and joined in LDS: a decode step's [B, D]
// x [D, C] product is a few MFLOP, so what counts is the number of workgroups
// (B / 16 x C / 16) and one round trip for each wave's loads, all of which
// are issued before any is used.  With LN every workgroup normalises its 16
// rows itself (the rows come from L2); column tile 0 writes what others need.
struct DenseParams {
  const float* x;          // [T, D]
  const uint16_t* add;     // [T, D] bf16: x + float(add) * add_scale[0] is the input row; or null
  const float* add_scale;
  float* x_out;            // [T, D]: the summed rows (with add)
  const float* ln_scale;   // [D] (LN)
  const float* ln_bias;
  uint16_t* n0;            // [T, D] bf16 normalised rows, or null
  uint16_t* n1;            // a second copy, or null
  const float* w;          // [D, cols]
  const float* b;          // [cols] or null
  int cols;
  const float* w2;         // [D, cols2]: a last tile of at most 16 columns, or cols2 = 0
  const float* b2;
  int cols2;
  uint16_t* h0;            // columns [0, split0) of w: h0[t * split0 + c], the rest h1[t * (cols - split0) + c - split0]
  uint16_t* h1;
  int split0;
  float* t0;               // columns [0, split2) of w2: t0[t * split2 + c], the rest t1
  float* t1;
  int split2;
  float* res;              // no LN: res[t * cols + c] += the product, in float32
  int64_t T;
};

template <int NI, bool LN>  // D = 64 NI
__global__ __launch_bounds__(256) void rows_dense_kernel(DenseParams p) {
  constexpr int D = 64 * NI;
  __shared__ float rs[2][4][16];
  __shared__ float red[4][64][4];
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const int r = lane & 15, g = lane >> 4;
  const int64_t row = static_cast<int64_t>(blockIdx.y) * 16 + r;
  const int64_t t = row < p.T ? row : p.T - 1;
  const bool second = static_cast<int>(blockIdx.x) * 16 >= p.cols;  // the w2 tile
  const float* w = second ? p.w2 : p.w;
  const int ld = second ? p.cols2 : p.cols;
  const int c0 = second ? 0 : static_cast<int>(blockIdx.x) * 16;
  const int col = c0 + r < ld ? c0 + r : ld - 1;
  const int k0 = wave * 16 * NI + 4 * g;  // the lane's k: k0 + 16 s + c
  float a[NI][4], wv[NI][4];
#pragma unroll
  for (int s = 0; s < NI; ++s) {
    const float4 q = *reinterpret_cast<const float4*>(p.x + t * D + k0 + 16 * s);
    a[s][0] = q.x;
    a[s][1] = q.y;
    a[s][2] = q.z;
    a[s][3] = q.w;
  }
  uint2 ad[NI];
  if (LN && p.add) {
#pragma unroll
    for (int s = 0; s < NI; ++s) ad[s] = *reinterpret_cast<const uint2*>(p.add + t * D + k0 + 16 * s);
  }
#pragma unroll
  for (int s = 0; s < NI; ++s)
#pragma unroll
    for (int c = 0; c < 4; ++c) wv[s][c] = w[static_cast<int64_t>(k0 + 16 * s + c) * ld + col];
  if constexpr (LN) {
    const bool first = blockIdx.x == 0 && row < p.T;
    if (p.add) {
      const float sc = p.add_scale[0];
#pragma unroll
      for (int s = 0; s < NI; ++s) {
        a[s][0] += lo_f32(ad[s].x) * sc;
        a[s][1] += hi_f32(ad[s].x) * sc;
        a[s][2] += lo_f32(ad[s].y) * sc;
        a[s][3] += hi_f32(ad[s].y) * sc;
        if (first)
          *reinterpret_cast<float4*>(p.x_out + t * D + k0 + 16 * s) = make_float4(a[s][0], a[s][1], a[s][2], a[s][3]);
      }
    }
    // mean, then the variance about it (v41:321-324), over the four lane
    // groups and the four waves
    float v = 0.f;
#pragma unroll
    for (int s = 0; s < NI; ++s) v += (a[s][0] + a[s][1]) + (a[s][2] + a[s][3]);
    v += __shfl_xor(v, 16);
    v += __shfl_xor(v, 32);
    if (g == 0) rs[0][wave][r] = v;
    __syncthreads();
    const float mean = ((rs[0][0][r] + rs[0][1][r]) + (rs[0][2][r] + rs[0][3][r])) / D;
    v = 0.f;
#pragma unroll
    for (int s = 0; s < NI; ++s)
#pragma unroll
      for (int c = 0; c < 4; ++c) v += (a[s][c] - mean) * (a[s][c] - mean);
    v += __shfl_xor(v, 16);
    v += __shfl_xor(v, 32);
    if (g == 0) rs[1][wave][r] = v;
    __syncthreads();
    const float rstd = 1.0f / sqrtf(((rs[1][0][r] + rs[1][1][r]) + (rs[1][2][r] + rs[1][3][r])) / D + 1e-6f);
#pragma unroll
    for (int s = 0; s < NI; ++s) {
      const float4 ls = *reinterpret_cast<const float4*>(p.ln_scale + k0 + 16 * s);
      const float4 lb = *reinterpret_cast<const float4*>(p.ln_bias + k0 + 16 * s);
      a[s][0] = (a[s][0] - mean) * rstd * ls.x + lb.x;
      a[s][1] = (a[s][1] - mean) * rstd * ls.y + lb.y;
      a[s][2] = (a[s][2] - mean) * rstd * ls.z + lb.z;
      a[s][3] = (a[s][3] - mean) * rstd * ls.w + lb.w;
      if (first) {
        const uint2 n = make_uint2(pack_bf16(a[s][0], a[s][1]), pack_bf16(a[s][2], a[s][3]));
        if (p.n0) *reinterpret_cast<uint2*>(p.n0 + t * D + k0 + 16 * s) = n;
        if (p.n1) *reinterpret_cast<uint2*>(p.n1 + t * D + k0 + 16 * s) = n;
      }
    }
  }
  f32x4_t acc = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
  for (int s = 0; s < NI; ++s)
#pragma unroll
    for (int c = 0; c < 4; ++c) acc = __builtin_amdgcn_mfma_f32_16x16x4f32(a[s][c], wv[s][c], acc, 0, 0, 0);
  // acc[v] of lane (r, g): row 4 g + v, column r of the tile
#pragma unroll
  for (int v = 0; v < 4; ++v) red[wave][16 * g + r][v] = acc[v];
  __syncthreads();
  const int oc = threadIdx.x & 15, orow = threadIdx.x >> 4;
  const int src = 16 * (orow >> 2) + oc, sv = orow & 3;
  const float sum = (red[0][src][sv] + red[1][src][sv]) + (red[2][src][sv] + red[3][src][sv]);
  const int64_t to = static_cast<int64_t>(blockIdx.y) * 16 + orow;
  const int co = c0 + oc;
  if (to >= p.T || co >= ld) return;
  if constexpr (LN) {
    if (second) {
      const float y = sum + p.b2[co];
      if (co < p.split2) p.t0[to * p.split2 + co] = y;
      else p.t1[to * (ld - p.split2) + co - p.split2] = y;
    } else {
      const uint16_t y = static_cast<uint16_t>(pack_bf16(sum + p.b[co], 0.f));
      if (co < p.split0) p.h0[to * p.split0 + co] = y;
      else p.h1[to * (ld - p.split0) + co - p.split0] = y;
    }
  } else {
    p.res[to * ld + co] += sum;
  }
}

// Last LayerNorm: out = LN(x + float(add) * scale), one wave per row.
template <int NI>
__global__ __launch_bounds__(256) void final_norm_kernel(const float* x, const uint16_t* add, const float* add_scale,
                                                         const float* ln_scale, const float* ln_bias, float* out,
                                                         int64_t T) {
  constexpr int D = 64 * NI;
  const int lane = threadIdx.x & 63;
  const int64_t t = static_cast<int64_t>(blockIdx.x) * 4 + (threadIdx.x >> 6);
  if (t >= T) return;
  const float sc = add_scale[0];
  float a[NI];
  float v = 0.f;
#pragma unroll
  for (int i = 0; i < NI; ++i) {
    a[i] = x[t * D + lane + 64 * i] + bf16_to_f32(add[t * D + lane + 64 * i]) * sc;
    v += a[i];
  }
  const float mean = wave_sum(v) / D;
  v = 0.f;
#pragma unroll
  for (int i = 0; i < NI; ++i) v += (a[i] - mean) * (a[i] - mean);
  const float rstd = 1.0f / sqrtf(wave_sum(v) / D + 1e-6f);
#pragma unroll
  for (int i = 0; i < NI; ++i)
    out[t * D + lane + 64 * i] = (a[i] - mean) * rstd * ln_scale[lane + 64 * i] + ln_bias[lane + 64 * i];
}

// One token's attention per (sequence, head) (v41:1800-1815): q, k, v are the
// SRW outputs times their pool scales; k and v also go into the caches at
// position pos.  32 groups of 16 lanes (a lane four of the 64 columns) take
// the cached positions 32 apart, each with its own running maximum, sum and
// output (no barrier in the loop); they join in LDS.  Bound by the cache
// stream, 512 bytes per (head, position): eight positions' keys and values a
// group are requested together.
struct AttnParams {
  const uint16_t* qk;  // [B, 2, H 64] bf16
  const uint16_t* v;   // [B, H 64]
  const float* qk_scale;
  const float* v_scale;
  float* ck;           // [B, H, max_seq, 64] of the layer
  float* cv;
  float* out;          // [B, H 64]
  int H;
  int64_t max_seq, pos;
};
constexpr int kAtThreads = 512, kAtGroups = kAtThreads / 16, kAtChunk = 8;

__device__ inline float sum16(float v) {
  v += __shfl_xor(v, 1);
  v += __shfl_xor(v, 2);
  v += __shfl_xor(v, 4);
  v += __shfl_xor(v, 8);
  return v;
}

__global__ __launch_bounds__(kAtThreads) void decode_attn_kernel(AttnParams p) {
  __shared__ float gm[kAtGroups], gl[kAtGroups], ga[kAtGroups][kDh];
  const int h = blockIdx.x;
  const int64_t b = blockIdx.y;
  const int c = threadIdx.x & 15, grp = threadIdx.x >> 4;
  const int64_t D = static_cast<int64_t>(p.H) * kDh;
  auto load4 = [&](const uint16_t* src, float sc) {
    const uint2 q = *reinterpret_cast<const uint2*>(src + h * kDh + 4 * c);
    return make_float4(lo_f32(q.x) * sc, hi_f32(q.x) * sc, lo_f32(q.y) * sc, hi_f32(q.y) * sc);
  };
  const float sqk = p.qk_scale[0];
  const float4 q = load4(p.qk + b * 2 * D, sqk);
  float* ck = p.ck + (b * p.H + h) * p.max_seq * kDh + 4 * c;
  float* cv = p.cv + (b * p.H + h) * p.max_seq * kDh + 4 * c;
  // scores in units of log2: 2^s
  constexpr float kScale = 0.125f * 1.4426950408889634f;
  auto dot = [&](const float4& k) { return sum16((q.x * k.x + q.y * k.y) + (q.z * k.z + q.w * k.w)) * kScale; };
  float m = -INFINITY, l = 0.f;
  float4 acc = make_float4(0.f, 0.f, 0.f, 0.f);
  if (grp == 0) {  // the new position
    const float4 k = load4(p.qk + b * 2 * D + D, sqk), v = load4(p.v + b * D, p.v_scale[0]);
    *reinterpret_cast<float4*>(ck + p.pos * kDh) = k;
    *reinterpret_cast<float4*>(cv + p.pos * kDh) = v;
    m = dot(k);
    l = 1.f;
    acc = v;
  }
  for (int64_t p0 = grp; p0 < p.pos; p0 += kAtGroups * kAtChunk) {
    float4 k[kAtChunk], v[kAtChunk];
#pragma unroll
    for (int j = 0; j < kAtChunk; ++j) {
      const int64_t at = p0 + kAtGroups * j;
      k[j] = *reinterpret_cast<const float4*>(ck + (at < p.pos ? at : p0) * kDh);
    }
#pragma unroll
    for (int j = 0; j < kAtChunk; ++j) {
      const int64_t at = p0 + kAtGroups * j;
      v[j] = *reinterpret_cast<const float4*>(cv + (at < p.pos ? at : p0) * kDh);
    }
    float s[kAtChunk], mn = m;
#pragma unroll
    for (int j = 0; j < kAtChunk; ++j) {
      s[j] = dot(k[j]);
      if (p0 + kAtGroups * j < p.pos) mn = fmaxf(mn, s[j]);
    }
    const float w = m == mn ? 1.f : __builtin_amdgcn_exp2f(m - mn);
    l *= w;
    acc.x *= w;
    acc.y *= w;
    acc.z *= w;
    acc.w *= w;
#pragma unroll
    for (int j = 0; j < kAtChunk; ++j) {
      // a score of -inf has weight 0 whatever the group's maximum
      const float e = p0 + kAtGroups * j < p.pos && s[j] != -INFINITY ? __builtin_amdgcn_exp2f(s[j] - mn) : 0.f;
      l += e;
      acc.x = fmaf(e, p0 + kAtGroups * j < p.pos ? v[j].x : 0.f, acc.x);
      acc.y = fmaf(e, p0 + kAtGroups * j < p.pos ? v[j].y : 0.f, acc.y);
      acc.z = fmaf(e, p0 + kAtGroups * j < p.pos ? v[j].z : 0.f, acc.z);
      acc.w = fmaf(e, p0 + kAtGroups * j < p.pos ? v[j].w : 0.f, acc.w);
    }
    m = mn;
  }
  if (c == 0) {
    gm[grp] = m;
    gl[grp] = l;
  }
  *reinterpret_cast<float4*>(&ga[grp][4 * c]) = acc;
  __syncthreads();
  if (threadIdx.x >= kDh) return;
  float mm = gm[0];
#pragma unroll
  for (int i = 1; i < kAtGroups; ++i) mm = fmaxf(mm, gm[i]);
  float ls = 0.f, o = 0.f;
#pragma unroll
  for (int i = 0; i < kAtGroups; ++i) {
    // a group without positions has l = 0 and m = -inf
    const float w = gl[i] == 0.f ? 0.f : __builtin_amdgcn_exp2f(gm[i] - mm);
    ls += gl[i] * w;
    o += ga[i][threadIdx.x] * w;
  }
  p.out[b * D + h * kDh + threadIdx.x] = o / ls;
}

template <int NI>
srw_status_t step(const srw_dawn_step_t& s, const srw_desc_t* descs_in, hipStream_t st) {
  const int64_t B = s.B, D = s.d_model, dr = s.d_route;
  auto bf = [](const void* q) { return static_cast<uint16_t*>(const_cast<void*>(q)); };
  auto fl = [](const float* q) { return const_cast<float*>(q); };
  const srw_tensors_t &tq = s.tensors[0], &tv = s.tensors[1], &tk = s.tensors[2];
  srw_desc_t descs[3] = {descs_in[0], descs_in[1], descs_in[2]};
  const unsigned rt = static_cast<unsigned>((B + 15) / 16);
  float *cur = s.x, *alt = s.x_alt;
  const auto* know_out = static_cast<const uint16_t*>(s.outs[2].out);
  srw_status_t e;
  for (int i = 0; i < s.n_layers; ++i) {
    const srw_dawn_layer_t& ly = s.layers[i];
    DenseParams a{};
    a.x = cur;
    if (i > 0) {  // the previous layer's Know output (v41:1175)
      a.add = know_out;
      a.add_scale = s.know_scale;
      a.x_out = alt;
      float* x = cur;
      cur = alt;
      alt = x;
    }
    a.ln_scale = ly.norm1_scale;
    a.ln_bias = ly.norm1_bias;
    a.n0 = bf(tq.x);
    a.n1 = bf(tv.x);
    a.w = s.proj_attn_w;
    a.b = s.proj_attn_b;
    a.cols = static_cast<int>(3 * dr);
    a.w2 = s.tau_attn_w;
    a.b2 = s.tau_attn_b;
    a.cols2 = 3;
    a.h0 = bf(tq.h);
    a.h1 = bf(tv.h);
    a.split0 = static_cast<int>(2 * dr);
    a.t0 = fl(tq.tau_offset);
    a.t1 = fl(tv.tau_offset);
    a.split2 = 2;
    a.T = B;
    hipLaunchKernelGGL((rows_dense_kernel<NI, true>), dim3(static_cast<unsigned>(a.cols / 16 + 1), rt), dim3(256), 0,
                       st, a);
    if (hipGetLastError() != hipSuccess) return SRW_EHIP;
    const bool cached = i > 0;
    for (int k = 0; k < 3; ++k)
      if (cached || (k < 2 ? s.qkv_cached : s.know_cached)) descs[k].flags |= SRW_FLAG_POOL_CACHED;
    if ((e = srw_forward_batch(2, descs, s.tensors, s.outs, s.ws_qkv, s.ws_qkv_bytes, st)) != SRW_OK) return e;
    if (s.path_qkv) *s.path_qkv = srw_last_path();
    AttnParams t{};
    t.qk = static_cast<const uint16_t*>(s.outs[0].out);
    t.v = static_cast<const uint16_t*>(s.outs[1].out);
    t.qk_scale = s.qk_scale;
    t.v_scale = s.v_scale;
    t.ck = s.cache_k + i * B * s.max_seq * D;
    t.cv = s.cache_v + i * B * s.max_seq * D;
    t.out = s.attn;
    t.H = s.n_heads;
    t.max_seq = s.max_seq;
    t.pos = s.pos;
    hipLaunchKernelGGL(decode_attn_kernel, dim3(static_cast<unsigned>(s.n_heads), static_cast<unsigned>(B)),
                       dim3(kAtThreads), 0, st, t);
    if (hipGetLastError() != hipSuccess) return SRW_EHIP;
    DenseParams o{};
    o.x = s.attn;
    o.w = ly.expand_o;
    o.cols = static_cast<int>(D);
    o.res = cur;
    o.T = B;
    hipLaunchKernelGGL((rows_dense_kernel<NI, false>), dim3(static_cast<unsigned>(D / 16), rt), dim3(256), 0, st, o);
    if (hipGetLastError() != hipSuccess) return SRW_EHIP;
    DenseParams k{};
    k.x = cur;
    k.ln_scale = ly.norm2_scale;
    k.ln_bias = ly.norm2_bias;
    k.n0 = bf(tk.x);
    k.w = s.proj_know_w;
    k.b = s.proj_know_b;
    k.cols = static_cast<int>(dr);
    k.w2 = s.tau_know_w;
    k.b2 = s.tau_know_b;
    k.cols2 = 1;
    k.h0 = bf(tk.h);
    k.split0 = static_cast<int>(dr);
    k.t0 = fl(tk.tau_offset);
    k.split2 = 1;
    k.T = B;
    hipLaunchKernelGGL((rows_dense_kernel<NI, true>), dim3(static_cast<unsigned>(k.cols / 16 + 1), rt), dim3(256), 0,
                       st, k);
    if (hipGetLastError() != hipSuccess) return SRW_EHIP;
    if ((e = srw_forward(&descs[2], &tk, &s.outs[2], s.ws_know, s.ws_know_bytes, st)) != SRW_OK) return e;
  }
  hipLaunchKernelGGL(final_norm_kernel<NI>, dim3(static_cast<unsigned>((B + 3) / 4)), dim3(256), 0, st, cur, know_out,
                     s.know_scale, s.norm_scale, s.norm_bias, s.normed, B);
  return hipGetLastError() == hipSuccess ? SRW_OK : SRW_EHIP;
}

}  // namespace

bool dawn_step_supports(const srw_dawn_step_t& s) {
  return (s.d_model == 384 || s.d_model == 128) && s.d_model == static_cast<int64_t>(s.n_heads) * kDh &&
         s.d_route % 16 == 0 && s.d_route > 0 && s.B > 0 && s.B <= 65535;
}

srw_status_t dawn_decode_step(const srw_dawn_step_t& s, hipStream_t st) {
  return s.d_model == 384 ? step<6>(s, s.descs, st) : step<2>(s, s.descs, st);
}

}  // namespace srw
