// srw_split_f32.hip -- the fp32 family's three GEMMs on the fp16 matrix cores,
// each fp32 operand as the sum of two fp16 numbers.
//
// An operand row is scaled by a power of two (its largest element into [2^14,
// 2^15)) and each element x becomes hi = f16(x), lo = f16(x - hi): 22
// significant bits, elements below 2^-16 of the row's largest losing them
// gradually (2^-40 of it absolute).  x.y = hi.hi' + hi.lo' + lo.hi' then costs three
// v_mfma_f32_32x32x16_f16 of 32 cycles for 16 k where v_mfma_f32_32x32x2_f32
// costs eight of 64.  Products are exact in fp32 and a k-step of 16 adds to the
// accumulator once, so against 64 bits a dot of K = 384 is off by 1.7e-7 of
// its norm, the fp32 MFMA's chain of 192 additions by 2.5e-7 (K = 128: 1.1 and
// 1.4e-7; K = 1024: 2.6 and 4.0e-7; below 128 the split is the less exact one,
// so those widths keep the fp32 kernels).
//
// Scales: one per row of x, h, E and R, taken out of the accumulator in the
// epilogue; one per unit's W row, taken out of P (k of the write GEMM); and one
// per row of P, set from a bound before the gate kernel runs: the row's
// largest gate (the gate of its largest score) times |x| max |r_n| / scale
// (Cauchy), taken out of the write GEMM's accumulator.
//
// Rows with an infinity, a NaN or a largest element outside 2^+-26, and pools
// whose units' |r| |w| differ by more than 2^8, set a flag on the device; the split kernels then leave at once and the fp32 kernels,
// which are launched behind them and otherwise leave at once, do the call:
// infinities and NaNs come out as products of fp32 numbers give them.
//
// fp32 srw_inference of the Know pool (T = 4 096, N = 25 200, d 384): 2 295 ->
// 1 051 us, its error against 64 bits 9.2e-7 -> 7.4e-7; score kernel 781 -> 340
// us, gate 949 -> 450, write 664 -> 252 (0.95 PFLOP/s of fp16 products), the
// operands' splitting 26 -> 73.
//
// A split row has the fp32 row's size and lines: per 32 k one 128-byte line,
// 32 hi then 32 lo.  So the tiles, the LDS ring and the swizzle are the fp32
// kernels' own, and P replaces the scores in place.

#include <math.h>

#include "srw_internal.hpp"
#include "srw_mfma_util.hpp"

namespace srw {

namespace {

typedef _Float16 f16x8_t __attribute__((ext_vector_type(8)));
typedef _Float16 f16x2_t __attribute__((ext_vector_type(2)));
typedef uint32_t u32x2_t __attribute__((ext_vector_type(2)));

constexpr int kSThreads = 256;
constexpr int kSK = 32;                      // k per stage: one 128-byte line per row
constexpr int kSGroupBytes = 32 * kSK * 4;   // 32 rows

__device__ inline f32x16_t mfma_h(u32x4_t a, u32x4_t b, f32x16_t c) {
  return __builtin_amdgcn_mfma_f32_32x32x16_f16(__builtin_bit_cast(f16x8_t, a), __builtin_bit_cast(f16x8_t, b), c, 0,
                                                 0, 0);
}
// two scaled floats -> (hi pair, lo pair)
__device__ inline void split2(float a, float b, uint32_t& hi, uint32_t& lo) {
  const f16x2_t h = __builtin_convertvector((f32x2_t{a, b}), f16x2_t);
  const float ra = a - static_cast<float>(h[0]), rb = b - static_cast<float>(h[1]);
  const f16x2_t l = __builtin_convertvector((f32x2_t{ra, rb}), f16x2_t);
  hi = __builtin_bit_cast(uint32_t, h);
  lo = __builtin_bit_cast(uint32_t, l);
}
// the power of two that brings m into [2^14, 2^15), and its inverse
__device__ inline float pow2(int e) { return __uint_as_float(static_cast<uint32_t>(e + 127) << 23); }
__device__ inline int exponent(float m) { return static_cast<int>((__float_as_uint(m) >> 23) & 0xff) - 127; }
// range of a row's largest element: three inverse scales multiply within fp32
constexpr int kTop = 14, kRange = 26;

// ---------------------------------------------------------------------------
// rows -> split rows, one wave per row
// ---------------------------------------------------------------------------
struct SplitRows {
  const float* src;  // [rows, K]
  char* dst;         // [rows][K / 32][64 B hi | 64 B lo], or null: the scales only
  float* inv;        // [rows] 1 / scale
  float* norm;       // [rows] |row|, or null
  int* flag;         // set to 1 where a row is not finite or out of range
  int64_t rows, K;
};
struct SplitRowsParams {
  SplitRows a[5];
  int start[6];  // first workgroup (four rows each) of each array
  int n;
};

__global__ __launch_bounds__(256) void split_rows_kernel(SplitRowsParams p) {
  int i = 0;
  for (int k = 1; k < p.n; ++k) i += static_cast<int>(blockIdx.x) >= p.start[k] ? 1 : 0;
  const SplitRows& q = p.a[i];
  const int lane = threadIdx.x & 63;
  const int64_t row = (static_cast<int64_t>(blockIdx.x) - p.start[i]) * 4 + (threadIdx.x >> 6);
  if (row >= q.rows) return;
  const float2* src = reinterpret_cast<const float2*>(q.src + row * q.K);
  char* dst = q.dst + row * q.K * 4;
  const int64_t pairs = q.K / 2;
  constexpr int kRegs = 8;  // rows up to 1024 elements stay in registers
  float2 v[kRegs];
  float m = 0.f, ss = 0.f;
  bool nan = false;
  auto look = [&](const float2& x) {
    m = fmaxf(m, fmaxf(fabsf(x.x), fabsf(x.y)));
    nan = nan || x.x != x.x || x.y != x.y;
    ss += x.x * x.x + x.y * x.y;
  };
#pragma unroll
  for (int j = 0; j < kRegs; ++j) {
    v[j] = lane + 64 * j < pairs ? src[lane + 64 * j] : make_float2(0.f, 0.f);
  }
#pragma unroll
  for (int j = 0; j < kRegs; ++j) look(v[j]);
  for (int64_t k = lane + 64 * kRegs; k < pairs; k += 64) look(src[k]);
  m = wave_max(m);
  const int e = exponent(m);
  const bool bad = __any(nan) || (m > 0.f && (e > kRange || e < -kRange));  // an infinity's exponent is 128
  const float s = m > 0.f && !bad ? pow2(kTop - e) : 1.f;
  ss = q.norm ? wave_sum(ss) : 0.f;
  if (lane == 0) {
    q.inv[row] = 1.f / s;
    if (q.norm) q.norm[row] = sqrtf(ss);
    if (bad) *q.flag = 1;  // every writer writes the same
  }
  if (!q.dst) return;
  auto put = [&](int64_t pair, const float2& x) {
    uint32_t hi, lo;
    split2(x.x * s, x.y * s, hi, lo);
    char* at = dst + (pair >> 4) * 128 + (pair & 15) * 4;
    *reinterpret_cast<uint32_t*>(at) = hi;
    *reinterpret_cast<uint32_t*>(at + 64) = lo;
  };
#pragma unroll
  for (int j = 0; j < kRegs; ++j)
    if (lane + 64 * j < pairs) put(lane + 64 * j, v[j]);
  for (int64_t k = lane + 64 * kRegs; k < pairs; k += 64) put(k, src[k]);
}

// W [N, D] -> W^T split [D][N64 / 32][64 B hi | 64 B lo] with the units' scales
// (1 / iw), zero past N: 32 units x 64 columns per workgroup, turned over in LDS
__global__ __launch_bounds__(256) void split_wt_kernel(const float* __restrict__ W, char* __restrict__ WT,
                                                       const float* __restrict__ iw, int64_t N, int64_t N64,
                                                       int64_t D) {
  __shared__ float tile[32][65];
  const int64_t n0 = static_cast<int64_t>(blockIdx.x) * 32, d0 = static_cast<int64_t>(blockIdx.y) * 64;
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
#pragma unroll
  for (int k = 0; k < 8; ++k) {
    const int r = wave + 4 * k;
    const int64_t n = n0 + r, d = d0 + lane;
    tile[r][lane] = n < N && d < D ? W[n * D + d] / iw[n] : 0.f;  // powers of two: exact
  }
  __syncthreads();
  // thread (column c, pairs 4 q .. 4 q + 3)
  const int c = threadIdx.x >> 2, q = threadIdx.x & 3;
  if (d0 + c >= D) return;
  u32x4_t hi, lo;
#pragma unroll
  for (int k = 0; k < 4; ++k) {
    uint32_t a, b;
    split2(tile[8 * q + 2 * k][c], tile[8 * q + 2 * k + 1][c], a, b);
    hi[k] = a;
    lo[k] = b;
  }
  char* at = WT + (d0 + c) * N64 * 4 + (n0 / 32) * 128 + q * 16;
  *reinterpret_cast<u32x4_t*>(at) = hi;
  *reinterpret_cast<u32x4_t*>(at + 64) = lo;
}

// irw[n] = ir[n] iw[n], what the gate kernel takes out of x.r and puts into P (0
// past N), and the largest and smallest non-zero |r_n| iw[n] (non-negative
// floats order like their bits; the smallest as 0x7f800000 - bits)
__global__ __launch_bounds__(256) void split_factor_kernel(const float* ir, const float* iw, const float* rnorm,
                                                           float* irw, unsigned* rmax, int64_t N, int64_t N64) {
  const int64_t n = static_cast<int64_t>(blockIdx.x) * 256 + threadIdx.x;
  float m = 0.f;
  if (n < N64) irw[n] = n < N ? ir[n] * iw[n] : 0.f;
  if (n < N) m = rnorm[n] * iw[n];
  const float top = wave_max(m), low = -wave_max(m > 0.f ? -m : -INFINITY);
  if ((threadIdx.x & 63) == 0 && top > 0.f) {
    atomicMax(rmax, __float_as_uint(top));
    atomicMax(rmax + 1, 0x7f800000u - __float_as_uint(low));
  }
}

// ---------------------------------------------------------------------------
// main loop
// ---------------------------------------------------------------------------
__device__ inline int sswz(int u) { return (u & 7) ^ ((u >> 3) & 1); }

template <int G>
struct SOpnd {
  const char* base;  // byte address of memory row row0 / div, k = 0 (uniform)
  uint32_t off[G];   // per-lane byte offsets from base: row and swizzled piece
};
template <int G>
__device__ inline SOpnd<G> make_sopnd(const char* p, int64_t ld, int64_t row0, int64_t rows, int div, int wave,
                                      int lane) {
  SOpnd<G> o;
  // a unit tile may lie past the last row (the slices come in pairs)
  const int64_t base_row = (row0 < rows ? row0 : rows - 1) / div;
  o.base = p + base_row * ld * 4;
  const int r8 = lane >> 3;
  const int piece = (lane & 7) ^ r8 ^ (wave & 1);  // sswz(8 wave + r8) = r8 ^ (wave & 1)
#pragma unroll
  for (int i = 0; i < G; ++i) {
    int64_t row = row0 + 32 * i + 8 * wave + r8;
    row = row < rows ? row : rows - 1;
    o.off[i] = static_cast<uint32_t>(((row / div - base_row) * ld + 4 * piece) * 4);
  }
  return o;
}

// acc[i][j] += A rows (32 (ga0 + i) ..) . B rows (32 (gb0 + j) ..)^T over nk
// 32-wide k blocks from k0, in two k-steps of 16 a block: a step's fragments
// (hi and lo of each row group: piece 2 m + h of the line, and 4 further) are
// read while the other step's MFMAs run, the low-order products first.
template <int GA, int GB, int MI, int MJ>
__device__ inline void sgemm_loop(f32x16_t (&acc)[MI][MJ], const SOpnd<GA>& A, const SOpnd<GB>& B, int64_t k0, int nk,
                                  char* lds, int ga0, int gb0, int wave, int lane) {
  constexpr int kOpA = GA * kSGroupBytes, kStage = (GA + GB) * kSGroupBytes;
  const int u = lane & 31, h = lane >> 5;
  int le[4];  // [m][hi, lo]
#pragma unroll
  for (int m = 0; m < 4; ++m)
    le[m] = (u >> 3) * 1024 + (u & 7) * 128 + (((2 * (m >> 1) + h + 4 * (m & 1)) ^ sswz(u)) * 16);
  auto issue = [&](int b, char* stage) {
    const int64_t kbyte = (k0 + static_cast<int64_t>(b) * kSK) * 4;
#pragma unroll
    for (int q = 0; q < GA; ++q) g2lds16(A.base + kbyte + A.off[q], stage + q * kSGroupBytes + wave * 1024);
#pragma unroll
    for (int q = 0; q < GB; ++q) g2lds16(B.base + kbyte + B.off[q], stage + kOpA + q * kSGroupBytes + wave * 1024);
  };
  auto read = [&](const char* st, int m, u32x4_t (&fa)[MI][2], u32x4_t (&fb)[MJ][2]) {
#pragma unroll
    for (int x = 0; x < 2; ++x) {
#pragma unroll
      for (int g = 0; g < MI; ++g)
        fa[g][x] = *reinterpret_cast<const u32x4_t*>(st + (ga0 + g) * kSGroupBytes + le[2 * m + x]);
#pragma unroll
      for (int g = 0; g < MJ; ++g)
        fb[g][x] = *reinterpret_cast<const u32x4_t*>(st + kOpA + (gb0 + g) * kSGroupBytes + le[2 * m + x]);
    }
  };
  auto steps = [&](const u32x4_t (&fa)[MI][2], const u32x4_t (&fb)[MJ][2]) {
#pragma unroll
    for (int x = 0; x < 3; ++x)  // hi.lo, lo.hi, hi.hi
#pragma unroll
      for (int q = 0; q < MI * MJ; ++q)
        acc[q / MJ][q % MJ] = mfma_h(fa[q / MJ][x == 1], fb[q % MJ][x == 0], acc[q / MJ][q % MJ]);
  };
  auto landed = [&](int kb) {
    constexpr int kN = GA + GB;  // loads of block kb + 1, still in flight
    if (kb + 1 < nk)
      __builtin_amdgcn_s_waitcnt(0x0F70 | (kN & 0xF) | ((kN >> 4) << 14));  // vmcnt(GA + GB)
    else
      wait_vm0();
    barrier_lds();
  };
  u32x4_t fa0[MI][2], fb0[MJ][2], fa1[MI][2], fb1[MJ][2];
  issue(0, lds);
  if (nk > 1) issue(1, lds + kStage);
  landed(0);
  read(lds, 0, fa0, fb0);
  for (int kb = 0; kb < nk; ++kb) {
    char* st = lds + (kb & 1) * kStage;
    read(st, 1, fa1, fb1);
    steps(fa0, fb0);
    barrier_lds();  // no wave reads block kb's stage any more
    if (kb + 2 < nk) issue(kb + 2, st);
    if (kb + 1 < nk) {
      landed(kb + 1);
      read(lds + ((kb + 1) & 1) * kStage, 0, fa0, fb0);
    }
    steps(fa1, fb1);
  }
}

__device__ inline bool stile_of(int nrow, int ncol, int& rt, int& ct) {
  const int x = blockIdx.x & 7, k = blockIdx.x >> 3;
  ct = (k / nrow) * 8 + x;
  rt = k % nrow;
  return ct < ncol;
}

// ---------------------------------------------------------------------------
// score and gate kernels: tiles of 128 units x 128 tokens, 2 x 2 waves of 64 x
// 64 (64 KB of LDS: two workgroups per CU, one's epilogue beside the other's
// MFMAs).  The epilogues work on each 32 x 32 block turned over in LDS, lane l
// holding rows (tokens) 8 k + l / 8, units 4 (l % 8) .. + 3: eight lanes read and
// write a row's whole 128-byte line.  In the accumulator's layout an access
// touches 32 rows of 32 bytes each (256 x 64 tiles so: score 380 us and gate
// 696 at T = 4 096, N = 25 200, d 384, against the write kernel's 217).
// ---------------------------------------------------------------------------
constexpr int kPatchRow = 36;                       // floats: 32 and a shift of four banks
constexpr int kPatchBytes = 32 * kPatchRow * 4;
constexpr int kTileGroups = 4, kMI = 2, kMJ = 2;    // 128 rows a side; 64 x 64 a wave
constexpr int kLdsTile = 2 * 2 * kTileGroups * kSGroupBytes;

// the block's element [4 k + c]: row 8 k + l / 8, column 4 (l % 8) + c
__device__ inline void turn(f32x16_t& a, float* patch, int lane) {
  const int u = lane & 31, h = lane >> 5;
#pragma unroll
  for (int b = 0; b < 4; ++b)
    *reinterpret_cast<float4*>(patch + u * kPatchRow + 8 * b + 4 * h) =
        make_float4(a[4 * b], a[4 * b + 1], a[4 * b + 2], a[4 * b + 3]);
  __builtin_amdgcn_wave_barrier();
#pragma unroll
  for (int k = 0; k < 4; ++k) {
    const float4 q = *reinterpret_cast<const float4*>(patch + (8 * k + (lane >> 3)) * kPatchRow + 4 * (lane & 7));
    a[4 * k] = q.x;
    a[4 * k + 1] = q.y;
    a[4 * k + 2] = q.z;
    a[4 * k + 3] = q.w;
  }
  __builtin_amdgcn_wave_barrier();
}
// over the eight lanes of a row
template <class Op>
__device__ inline float row8(float v, int lane, Op op) {
  v = op(v, lane_xor<1>(v, lane));
  v = op(v, lane_xor<2>(v, lane));
  return op(v, lane_xor<4>(v, lane));
}
__device__ inline uint32_t or8(uint32_t m, int lane) {
  auto x = [&](uint32_t w, float f) { return w | __float_as_uint(f); };
  m = x(m, lane_xor<1>(__uint_as_float(m), lane));
  m = x(m, lane_xor<2>(__uint_as_float(m), lane));
  return x(m, lane_xor<4>(__uint_as_float(m), lane));
}

__global__ __launch_bounds__(kSThreads, 2) void split_stats_kernel(SplitArgs p) {
  extern __shared__ __attribute__((aligned(1024))) char lds[];
  __shared__ float part[2][128][4];  // per wave row and token: count, sum, second moment, maximum
  if (p.flags[0] | p.flags[1]) return;
  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int wa = wave >> 1, wb = wave & 1;
  int rt, ct;
  if (!stile_of(p.RT, p.CT, rt, ct)) return;
  const int64_t u0 = static_cast<int64_t>(ct) * 128, v0 = static_cast<int64_t>(rt) * 128;
  f32x16_t acc[kMI][kMJ];
#pragma unroll
  for (int i = 0; i < kMI; ++i)
#pragma unroll
    for (int j = 0; j < kMJ; ++j) acc[i][j] = f32x16_t{};
  {
    const SOpnd<4> A = make_sopnd<4>(p.e, p.dr, u0, p.N, 1, wave, lane);
    const SOpnd<4> B = make_sopnd<4>(p.h, p.dr, v0, p.Tv, 1, wave, lane);
    sgemm_loop(acc, A, B, 0, static_cast<int>(p.dr / kSK), lds, kMI * wa, kMJ * wb, wave, lane);
  }
  barrier_lds();  // every wave has read the last stage
  float* patch = reinterpret_cast<float*>(lds + wave * kPatchBytes);
  const int64_t uw = u0 + 64 * wa + 4 * (lane & 7);  // the lane's first unit
  const int64_t nleft = p.N - uw;
  const int64_t nrow = p.N - (u0 + 64 * wa);
  const float cnt = static_cast<float>(nrow <= 0 ? 0 : (nrow < 64 ? nrow : 64));
  auto add = [](float a, float b) { return a + b; };
  auto mxf = [](float a, float b) { return fmaxf(a, b); };
  float4 ie[kMI];
#pragma unroll
  for (int i = 0; i < kMI; ++i)
    ie[i] = *reinterpret_cast<const float4*>(p.ie + (uw + 32 * i < p.N64 ? uw + 32 * i : 0));
#pragma unroll
  for (int j = 0; j < kMJ; ++j) {
    const int r0 = 64 * wb + 32 * j + (lane >> 3);  // token 8 k further for each k
    float ih[4], s1[4], s2[4], sm[4];
#pragma unroll
    for (int k = 0; k < 4; ++k) {
      const int64_t t = v0 + r0 + 8 * k;
      ih[k] = p.ih[t < p.Tv ? t : p.Tv - 1];
      s1[k] = s2[k] = 0.f;
      sm[k] = -INFINITY;
    }
#pragma unroll
    for (int i = 0; i < kMI; ++i) {
      turn(acc[i][j], patch, lane);
      const float ies[4] = {ie[i].x, ie[i].y, ie[i].z, ie[i].w};
#pragma unroll
      for (int k = 0; k < 4; ++k) {
        const int64_t t = v0 + r0 + 8 * k;
        float q[4];
#pragma unroll
        for (int c = 0; c < 4; ++c) {
          const bool ok = 32 * i + c < nleft;
          const float sc = acc[i][j][4 * k + c] * ih[k] * ies[c];
          q[c] = ok ? sc : 0.f;
          sm[k] = fmaxf(sm[k], ok ? sc : -INFINITY);
          s1[k] += q[c];
          s2[k] += q[c] * q[c];
          acc[i][j][4 * k + c] = q[c];
        }
        if (t < p.Tv && uw + 32 * i < p.N64)
          *reinterpret_cast<float4*>(p.S + t * p.N64 + uw + 32 * i) = make_float4(q[0], q[1], q[2], q[3]);
      }
    }
#pragma unroll
    for (int k = 0; k < 4; ++k) {
      s1[k] = row8(s1[k], lane, add);
      sm[k] = row8(sm[k], lane, mxf);
    }
    if (p.centred) {  // sum (s - mean)^2 over the wave's 64 units (v41:1719-1721), merged below and by kTauChan
#pragma unroll
      for (int k = 0; k < 4; ++k) {
        const float mu = cnt > 0.f ? s1[k] / cnt : 0.f;
        s2[k] = 0.f;
#pragma unroll
        for (int i = 0; i < kMI; ++i)
#pragma unroll
          for (int c = 0; c < 4; ++c) {
            const float d = 32 * i + c < nleft ? acc[i][j][4 * k + c] - mu : 0.f;
            s2[k] += d * d;
          }
      }
    }
#pragma unroll
    for (int k = 0; k < 4; ++k) {
      s2[k] = row8(s2[k], lane, add);
      if ((lane & 7) == 0)
        *reinterpret_cast<float4*>(part[wa][r0 + 8 * k]) = make_float4(cnt, s1[k], s2[k], sm[k]);
    }
  }
  __syncthreads();
  const int64_t t = v0 + threadIdx.x;
  if (threadIdx.x < 128 && t < p.Tv) {
    const float4 a = *reinterpret_cast<const float4*>(part[0][threadIdx.x]);
    const float4 b = *reinterpret_cast<const float4*>(part[1][threadIdx.x]);
    float s2 = a.z + b.z;
    if (p.centred && b.x > 0.f) {  // Chan et al.'s merge of the two halves
      const float d = b.y / b.x - a.y / a.x;
      s2 += d * d * (a.x * b.x / (a.x + b.x));
    }
    const int64_t sl = static_cast<int64_t>(ct) * p.Tv + t;
    *reinterpret_cast<float2*>(p.mom + 2 * sl) = make_float2(a.y + b.y, s2);
    p.smax[sl] = fmaxf(a.w, b.w);
  }
}

// ---------------------------------------------------------------------------
// scale of each row of P: 64 rows per workgroup, four groups of slices
// ---------------------------------------------------------------------------
__global__ __launch_bounds__(256) void split_scale_kernel(SplitArgs p, int slices) {
  __shared__ float red[4][64];
  const int c = threadIdx.x & 63, grp = threadIdx.x >> 6;
  const int64_t t = static_cast<int64_t>(blockIdx.x) * 64 + c;
  const int64_t tl = t < p.Tv ? t : p.Tv - 1;
  float m = -INFINITY;
#pragma unroll 8
  for (int s = grp; s < slices; s += 4) m = fmaxf(m, p.smax[s * p.Tv + tl]);
  red[grp][c] = m;
  __syncthreads();
  if (grp != 0 || t >= p.Tv) return;
  m = fmaxf(fmaxf(red[0][c], red[1][c]), fmaxf(red[2][c], red[3][c]));
  const GateParams& g = p.gp;
  float gmax;
  if (p.sstd) {
    gmax = fmaxf((m - p.tau[t]) / p.sstd[t], 0.f);
  } else if (g.sharp > 0.f && g.eps >= 0.f && g.maxi >= 0.f) {  // non-decreasing in the score
    const float mg = (m - p.tau[t]) - g.thr;
    gmax = (g.eps + fminf(fmaxf(mg - g.cut, 0.f), g.maxi)) / (1.f + __builtin_amdgcn_exp2f(-g.sharp * 1.4426950408889634f * mg));
  } else {
    gmax = fabsf(g.eps) + fabsf(g.maxi);
  }
  // units whose |r| |w| lie far below others' would lose digits of P to the
  // row's one scale: such pools go to the fp32 kernels
  const float top = __uint_as_float(p.rmax[0]), low = __uint_as_float(0x7f800000u - p.rmax[1]);
  if (low < top * 0x1p-8f) p.flags[0] = 1;
  const float bound = 1.01f * gmax * p.xnorm[t / p.routes] * __uint_as_float(*p.rmax);
  if (bound < 1.2676506e30f) {  // 2^100
    const int e = exponent(bound);
    p.sp[t] = bound > 0.f ? pow2(kTop - (e < -100 ? -100 : e)) : 1.f;
  } else {  // a NaN threshold makes the row NaN whatever its scale; a finite bound this large does not fit
    p.sp[t] = 1.f;
    if (!(gmax != gmax)) p.flags[0] = 1;
  }
}

// ---------------------------------------------------------------------------
// gate: XR of a tile, the gate of the stored scores, split P over S in place
// (a wave reads a line of scores whole before it writes the line)
// ---------------------------------------------------------------------------
template <bool GL>
__global__ __launch_bounds__(kSThreads, 2) void split_gate_kernel(SplitArgs p) {
  extern __shared__ __attribute__((aligned(1024))) char lds[];
  __shared__ float part[2][128][4];  // per wave row and token: sum gate, sum intensity, active count
  if (p.flags[0] | p.flags[1]) return;
  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int wa = wave >> 1, wb = wave & 1;
  int rt, ct;
  if (!stile_of(p.RT, p.CT, rt, ct)) return;
  const int64_t u0 = static_cast<int64_t>(ct) * 128, v0 = static_cast<int64_t>(rt) * 128;
  f32x16_t acc[kMI][kMJ];
#pragma unroll
  for (int i = 0; i < kMI; ++i)
#pragma unroll
    for (int j = 0; j < kMJ; ++j) acc[i][j] = f32x16_t{};
  {
    const SOpnd<4> A = make_sopnd<4>(p.r, p.D, u0, p.N, 1, wave, lane);
    const SOpnd<4> B = make_sopnd<4>(p.x, p.D, v0, p.Tv, p.routes, wave, lane);
    sgemm_loop(acc, A, B, 0, static_cast<int>(p.D / kSK), lds, kMI * wa, kMJ * wb, wave, lane);
  }
  barrier_lds();
  float* patch = reinterpret_cast<float*>(lds + wave * kPatchBytes);
  const int64_t uw = u0 + 64 * wa + 4 * (lane & 7);
  const int64_t nleft = p.N - uw;
  const float k_exp2 = -p.gp.sharp * 1.4426950408889634f;   // e^(-sharpness m) = 2^(m k_exp2)
  auto add = [](float a, float b) { return a + b; };
  float4 fr[kMI];
#pragma unroll
  for (int i = 0; i < kMI; ++i)
    fr[i] = *reinterpret_cast<const float4*>(p.irw + (uw + 32 * i < p.N64 ? uw + 32 * i : 0));
#pragma unroll
  for (int j = 0; j < kMJ; ++j) {
    const int r0 = 64 * wb + 32 * j + (lane >> 3);
    float4 sv[kMI][4];
    float tau[4], sd[4], ix[4], sp[4], gs[4], is[4];
    int na[4];
#pragma unroll
    for (int k = 0; k < 4; ++k) {
      const int64_t t = v0 + r0 + 8 * k, tc = t < p.Tv ? t : p.Tv - 1;
#pragma unroll
      for (int i = 0; i < kMI; ++i)
        sv[i][k] = uw + 32 * i < p.N64 ? *reinterpret_cast<const float4*>(p.S + tc * p.N64 + uw + 32 * i)
                                       : float4{0.f, 0.f, 0.f, 0.f};
      tau[k] = p.tau[tc];
      sd[k] = GL ? p.sstd[tc] : 1.f;
      ix[k] = p.ix[tc / p.routes];
      sp[k] = p.sp[tc];
      gs[k] = is[k] = 0.f;
      na[k] = 0;
    }
#pragma unroll
    for (int i = 0; i < kMI; ++i) {
      turn(acc[i][j], patch, lane);
      const float f[4] = {fr[i].x, fr[i].y, fr[i].z, fr[i].w};
      u32x2_t hi[4], lo[4];
#pragma unroll
      for (int k = 0; k < 4; ++k) {
        const float e[4] = {sv[i][k].x, sv[i][k].y, sv[i][k].z, sv[i][k].w};
        const int64_t t = v0 + r0 + 8 * k;
        uint32_t m = 0;
        float o[4];
#pragma unroll
        for (int c = 0; c < 4; ++c) {
          // margin, sigmoid through the hardware exp2 (within 2 ulp of expf),
          // intensity and gate in the reference's order (v41:1723-1728)
          const bool ok = 32 * i + c < nleft;  // units past N count for nothing
          float gate;
          if constexpr (GL) {
            const GeluOut go = gate_gelu_v401(e[c], tau[k], sd[k]);
            gate = ok ? go.gate : 0.f;
            is[k] += ok && go.z > 0.f ? go.z : 0.f;
            m |= gate > 0.f ? 1u << c : 0u;
          } else {
            const float margin = (e[c] - tau[k]) - p.gp.thr;
            const float act = __builtin_amdgcn_rcpf(1.0f + __builtin_amdgcn_exp2f(margin * k_exp2));
            const float inten = p.gp.eps + fminf(fmaxf(margin - p.gp.cut, 0.0f), p.gp.maxi);
            gate = ok ? act * inten : 0.f;
            is[k] += ok ? inten : 0.f;
            m |= ok && act > 0.5f ? 1u << c : 0u;
          }
          gs[k] += gate;
          if (p.G && t < p.Tv && ok) p.G[t * p.N + uw + 32 * i + c] = gate;
          o[c] = (gate * sp[k]) * (acc[i][j][4 * k + c] * (ix[k] * f[c]));  // P = gate * xr (v41:1735), scaled
        }
        uint32_t h0, h1, l0, l1;
        split2(o[0], o[1], h0, l0);
        split2(o[2], o[3], h1, l1);
        hi[k] = u32x2_t{h0, h1};
        lo[k] = u32x2_t{l0, l1};
        na[k] += __builtin_popcount(m);
        m = or8(m << (4 * (lane & 7)), lane);
        const int64_t word = (u0 + 64 * wa + 32 * i) / 32;
        if (p.mask32 && (lane & 7) == 0 && t < p.Tv && word < p.mask_words32) p.mask32[t * p.mask_words32 + word] = m;
      }
      __builtin_amdgcn_sched_barrier(0);  // every score of the lines has been used
#pragma unroll
      for (int k = 0; k < 4; ++k) {
        const int64_t t = v0 + r0 + 8 * k;
        if (t < p.Tv && uw + 32 * i < p.N64) {
          char* line = reinterpret_cast<char*>(p.S + t * p.N64 + u0 + 64 * wa + 32 * i) + 8 * (lane & 7);
          *reinterpret_cast<u32x2_t*>(line) = hi[k];
          *reinterpret_cast<u32x2_t*>(line + 64) = lo[k];
        }
      }
    }
#pragma unroll
    for (int k = 0; k < 4; ++k) {
      const float g = row8(gs[k], lane, add), in = row8(is[k], lane, add);
      const float n = row8(static_cast<float>(na[k]), lane, add);
      if ((lane & 7) == 0) *reinterpret_cast<float4*>(part[wa][r0 + 8 * k]) = make_float4(g, in, n, 0.f);
    }
  }
  __syncthreads();
  const int64_t t = v0 + threadIdx.x;
  if (threadIdx.x < 128 && t < p.Tv) {
    const float4 a = *reinterpret_cast<const float4*>(part[0][threadIdx.x]);
    const float4 b = *reinterpret_cast<const float4*>(part[1][threadIdx.x]);
    *reinterpret_cast<float4*>(p.tok_part + (static_cast<int64_t>(ct) * p.Tv + t) * 4) =
        make_float4(a.x + b.x, a.y + b.y, a.z + b.z, 0.f);
  }
}

// ---------------------------------------------------------------------------
// write: partial [Tv, D] of one split of the units, in fp32
// ---------------------------------------------------------------------------
template <int GA, int GB, int MI, int MJ>
__global__ __launch_bounds__(kSThreads, 1) void split_write_kernel(SplitArgs p) {
  static_assert(GA % MI == 0 && GB % MJ == 0 && (GA / MI) * (GB / MJ) == kSThreads / 64,
                "one accumulator block per wave");
  extern __shared__ __attribute__((aligned(1024))) char lds[];
  if (p.flags[0] | p.flags[1]) return;
  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  constexpr int WB = GB / MJ;
  const int wa = wave / WB, wb = wave % WB, u = lane & 31, h = lane >> 5;
  // XCD x (blockIdx % 8) takes W8 consecutive (token tile, split) pairs, each
  // with its column tiles in a row
  const int x = blockIdx.x & 7, k = blockIdx.x >> 3;
  const int dt = k % p.WDT;
  const int w = x * p.W8 + k / p.WDT;
  if (k / p.WDT >= p.W8 || w >= p.WRT * p.WS) return;
  const int rt = w % p.WRT, split = w / p.WRT;
  const int64_t kb0 = static_cast<int64_t>(p.nkb) * split / p.WS, kb1 = static_cast<int64_t>(p.nkb) * (split + 1) / p.WS;
  const int64_t v0 = static_cast<int64_t>(rt) * 32 * GA, d0 = static_cast<int64_t>(dt) * 32 * GB;
  const SOpnd<GA> A = make_sopnd<GA>(reinterpret_cast<const char*>(p.S), p.N64, v0, p.Tv, 1, wave, lane);
  const SOpnd<GB> B = make_sopnd<GB>(p.wt, p.N64, d0, p.D, 1, wave, lane);
  f32x16_t acc[MI][MJ];
#pragma unroll
  for (int i = 0; i < MI; ++i)
#pragma unroll
    for (int j = 0; j < MJ; ++j) acc[i][j] = f32x16_t{};
  sgemm_loop(acc, A, B, kb0 * kSK, static_cast<int>(kb1 - kb0), lds, MI * wa, MJ * wb, wave, lane);
  float* dst = p.out_part + static_cast<int64_t>(split) * p.Tv * p.D;
#pragma unroll
  for (int i = 0; i < MI; ++i) {
#pragma unroll
    for (int v = 0; v < 16; ++v) {
      const int64_t t = v0 + 32 * (MI * wa + i) + 8 * (v >> 2) + 4 * h + (v & 3);
      if (t >= p.Tv) continue;
      const float is = 1.f / p.sp[t];
#pragma unroll
      for (int j = 0; j < MJ; ++j) {
        const int64_t d = d0 + 32 * (MJ * wb + j) + u;
        if (d < p.D) dst[t * p.D + d] = acc[i][j][v] * is;
      }
    }
  }
}

}  // namespace

hipError_t split_prepare(const SplitArgs& a, const SplitSources& q, bool pool, hipStream_t s) {
  hipError_t e;
  // flags[0]: tokens, flags[1]: pool; rmax behind them
  if ((e = fill_f32(reinterpret_cast<float*>(a.flags), pool ? 4 : 1, 0.f, s)) != hipSuccess) return e;
  SplitRowsParams p{};
  auto add = [&](const float* src, const char* dst, const float* inv, const float* norm, int flag, int64_t rows,
                 int64_t K) {
    p.a[p.n] = SplitRows{src, const_cast<char*>(dst), const_cast<float*>(inv), const_cast<float*>(norm),
                         a.flags + flag, rows, K};
    p.start[p.n + 1] = p.start[p.n] + static_cast<int>((rows + 3) / 4);
    ++p.n;
  };
  add(q.x, a.x, a.ix, a.xnorm, 0, a.Tv / a.routes, a.D);
  if (a.h != a.x) add(q.h, a.h, a.ih, nullptr, 0, a.Tv, a.dr);
  if (pool) {
    add(q.e, a.e, a.ie, nullptr, 1, a.N, a.dr);
    add(q.r, a.r, q.ir, q.rnorm, 1, a.N, a.D);
    add(q.w, nullptr, q.iw, nullptr, 1, a.N, a.D);
  }
  hipLaunchKernelGGL(split_rows_kernel, dim3(static_cast<unsigned>(p.start[p.n])), dim3(256), 0, s, p);
  if ((e = hipGetLastError()) != hipSuccess) return e;
  if (!pool) return hipSuccess;
  hipLaunchKernelGGL(split_factor_kernel, dim3(static_cast<unsigned>((a.N64 + 255) / 256)), dim3(256), 0, s, q.ir,
                     q.iw, q.rnorm, const_cast<float*>(a.irw), a.rmax, a.N, a.N64);
  if ((e = hipGetLastError()) != hipSuccess) return e;
  hipLaunchKernelGGL(split_wt_kernel, dim3(static_cast<unsigned>(a.N64 / 32), static_cast<unsigned>((a.D + 63) / 64)),
                     dim3(256), 0, s, q.w, const_cast<char*>(a.wt), q.iw, a.N, a.N64, a.D);
  return hipGetLastError();
}

namespace {
hipError_t lds_of(const void* fn, int bytes) {
  return hipFuncSetAttribute(fn, hipFuncAttributeMaxDynamicSharedMemorySize, bytes);
}
}  // namespace

hipError_t split_stats(const SplitArgs& a, hipStream_t s) {
  const auto fn = split_stats_kernel;
  hipError_t e = lds_of(reinterpret_cast<const void*>(fn), kLdsTile);
  if (e != hipSuccess) return e;
  hipLaunchKernelGGL(fn, dim3(static_cast<unsigned>(8 * a.RT * ((a.CT + 7) / 8))), dim3(kSThreads), kLdsTile, s, a);
  return hipGetLastError();
}

hipError_t split_gate(const SplitArgs& a, hipStream_t s) {
  hipLaunchKernelGGL(split_scale_kernel, dim3(static_cast<unsigned>((a.Tv + 63) / 64)), dim3(256), 0, s, a, a.CT);
  hipError_t e = hipGetLastError();
  if (e != hipSuccess) return e;
  const auto fn = a.sstd ? split_gate_kernel<true> : split_gate_kernel<false>;
  if ((e = lds_of(reinterpret_cast<const void*>(fn), kLdsTile)) != hipSuccess) return e;
  dominant_kernel_begin(s);
  hipLaunchKernelGGL(fn, dim3(static_cast<unsigned>(8 * a.RT * ((a.CT + 7) / 8))), dim3(kSThreads), kLdsTile, s, a);
  dominant_kernel_end(s);
  return hipGetLastError();
}

hipError_t split_write(const SplitArgs& a, bool w192, hipStream_t s) {
  const auto fn = w192 ? split_write_kernel<4, 6, 2, 3> : split_write_kernel<8, 8, 4, 4>;
  const int lds = w192 ? 2 * (4 + 6) * kSGroupBytes : 2 * (8 + 8) * kSGroupBytes;
  hipError_t e = lds_of(reinterpret_cast<const void*>(fn), lds);
  if (e != hipSuccess) return e;
  hipLaunchKernelGGL(fn, dim3(static_cast<unsigned>(8 * a.WDT * a.W8)), dim3(kSThreads), lds, s, a);
  return hipGetLastError();
}

}  // namespace srw
