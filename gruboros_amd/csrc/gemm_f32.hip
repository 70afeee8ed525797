// fp32 matrix products on the bf16 matrix cores, to fp32 accuracy: the
// nn.Linear products of an fp32 model (reference mingru/minGRU.py:45,71;
// mingru/minLM.py:17-23,75,138) and of their autograd backward.
//
//   C[m, n] (=|+=) epilogue(sum_k A(m, k) B(k, n))
//
// with mg_gemm's epilogues in fp32: bias, bias + GELU (keeping the
// pre-activation for the backward) and the GELU gradient, applied where a sum
// is complete (the tile's store, or the K-split reduction). The FeedForward's
// GELU and its gradient were passes of their own (30 us of 430 at [4096, 512]
// x 2048).
//
// Each fp32 value is split into three bf16 limbs h + m + l == x (h = bf16(x),
// m = bf16(x - h), l = bf16(x - h - m); the differences are exact in fp32),
// and the six limb products down to 2^-16 relative (hh, mh, hm, mm, lh, hl)
// are accumulated in fp32 by v_mfma_f32_16x16x32_bf16; the dropped ones are
// below 2^-24.
//
// The split happens between global memory and LDS: a workgroup loads fp32
// tiles into registers, splits them there and writes the three limb tiles.
// Before, a pass over memory wrote each operand as six bf16 segments (4 bytes
// read, 12 written per element, at about 2.3 TB/s) and a plain bf16 product
// ran over a 6-fold K. At the fp32 layers of [4096, 512] activations those
// passes were 40% of the GPU time, and the 6-fold K read every limb tile
// twice. Here an operand is read as it is, each limb tile is in LDS once and
// serves two of the six products, and a layer's product is one launch.
//
// What bounds it: per 32 k a 128 x 128 tile takes 1536 cycles of MFMA and about
// 900 of vector work (the split) on each SIMD, and about 1520 of LDS traffic on
// the CU (147 KB of fragments, 48 KB of limbs written); a k-tile measures 1.4 us
// or about 2900. A 256 x 128 tile (64 x 64 per wave) halves the LDS traffic per
// flop but spilled 11 to 30 registers and measured 15-25% slower.
// Measured (MI355X, forward / dX / dW of an fp32 [4096, 512] -> 1024 layer):
// 31 / 34 + 6 / 32 + 5 us with the K-split reductions, against 77 / 88 / 93 us
// with the split passes; error against fp64 1.3e-7 (before: 3.1e-7), since the
// five small products keep an accumulator of their own.

#include <algorithm>

#include "mg_common.h"

namespace mg {
namespace gemm_f32 {

typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef __bf16 bf16x2 __attribute__((ext_vector_type(2)));
typedef float f32x2 __attribute__((ext_vector_type(2)));
typedef float f32x4v __attribute__((ext_vector_type(4)));
typedef short s16x4 __attribute__((ext_vector_type(4)));
typedef __attribute__((address_space(3))) s16x4 lds_s16x4;

constexpr int BM = 128, BN = 128, BK = 32;
constexpr int kThreads = 512;             // eight waves, 2 x 4, each 64 rows x 32 columns
constexpr int NV = 2;                     // float4 per thread, operand and k-tile
constexpr int kLimb = 128 * BK * 2;       // bytes of one limb of an operand tile
constexpr int kSide = 3 * kLimb;          // h, m, l
constexpr int kCUs = 256;

struct Params {
  const float* A;
  const float* B;
  float* C;
  const float* bias;
  float* aux;   // BIAS_GELU: receives the pre-activation (nullable); GELU_GRAD: holds it
  float* part;  // split partials: one dense [M, N] slice per split
  int64_t lda, ldb, ldc, ldaux;
  int M, N, K;
  int tiles_m, tiles_n, kt_per_split;
  int accumulate, epilogue;
};

// gelu'(x) with the device library's erff and expf: the fp32 path keeps fp32
// accuracy (mg_common.h's gelu_grad is a 1.5e-7 approximation for bf16 results).
__device__ __forceinline__ float gelu_grad_f32(float x) {
  return 0.5f * (1.0f + erff(x * 0.70710678118654752f)) + x * (expf(-0.5f * x * x) * 0.39894228040143268f);
}

// What happens to four consecutive sums of row m before they are stored at C.
__device__ __forceinline__ void finish(const Params& p, int64_t m, int64_t c, f4 x) {
  float* cp = p.C + m * p.ldc + c;
  if (p.bias) {
    const f4 bv = io4<float>::load(p.bias + c);
#pragma unroll
    for (int e = 0; e < 4; ++e) x.v[e] += bv.v[e];
  }
  if (p.epilogue == MG_EPI_BIAS_GELU) {
    if (p.aux) io4<float>::store(p.aux + m * p.ldaux + c, x);
#pragma unroll
    for (int e = 0; e < 4; ++e) x.v[e] = gelu(x.v[e]);
  } else if (p.epilogue == MG_EPI_GELU_GRAD) {
    const f4 a = io4<float>::load(p.aux + m * p.ldaux + c);
#pragma unroll
    for (int e = 0; e < 4; ++e) x.v[e] *= gelu_grad_f32(a.v[e]);
  }
  if (p.accumulate) {
    const f4 old = io4<float>::load(cp);
#pragma unroll
    for (int e = 0; e < 4; ++e) x.v[e] = old.v[e] + x.v[e];
  }
  io4<float>::store(cp, x);
}

// (x0, x1) -> their three limbs as packed bf16 pairs. The conversions round
// to nearest; x - h and x - h - m are exact.
__device__ __forceinline__ void split2(float x0, float x1, uint32_t& h, uint32_t& m, uint32_t& l) {
  h = __builtin_bit_cast(uint32_t, __builtin_convertvector((f32x2{x0, x1}), bf16x2));
  const float r0 = x0 - __uint_as_float(h << 16), r1 = x1 - __uint_as_float(h & 0xffff0000u);
  m = __builtin_bit_cast(uint32_t, __builtin_convertvector((f32x2{r0, r1}), bf16x2));
  const float s0 = r0 - __uint_as_float(m << 16), s1 = r1 - __uint_as_float(m & 0xffff0000u);
  l = __builtin_bit_cast(uint32_t, __builtin_convertvector((f32x2{s0, s1}), bf16x2));
}

__device__ __forceinline__ int tr_swz(int r) { return (((r & 3) << 1) | ((r >> 1) & 1)) ^ (((r >> 3) & 1) << 2); }

// One operand's side of the pipeline: a k-tile of 128 rows, NV float4 per thread.
//   K-contiguous (element (row, k) at p + row * ld + k): thread t takes 4 k of
//     rows 64 i + t / 8; a limb tile is [128 rows][32 k] (64-byte rows, 16-byte
//     chunk c of row r at c ^ ((r >> 2) & 3)), a fragment one 16-byte read;
//   MN-contiguous (element (row, k) at p + k * ld + row): thread t takes 4 rows
//     of one k-row per load; a limb tile is [32 k][128 rows] (32-byte segment s of
//     k-row r at s ^ tr_swz(r)), a fragment two LDS transpose reads.
// In both, the 16 lanes of a read group hit distinct banks.
template <bool KMAJ>
struct Side;

template <>
struct Side<true> {
  const float* p;
  int left;    // rows from the thread's first to the operand's end
  int kc;      // the thread's first k within the k-tile
  uint32_t w;  // LDS byte offset of its first 8-byte limb word (64 rows on: the same swizzle)
  uint32_t f;  // LDS byte offset of the wave's first fragment
  __device__ __forceinline__ void init(const float* base, int64_t ld, int r0, int rmax, int wr, int k0, int tid, int lane) {
    kc = (tid & 7) * 4;
    const int r1 = tid >> 3;
    left = rmax - r0 - r1;
    p = base + static_cast<int64_t>(r0 + r1) * ld + k0 + kc;
    w = static_cast<uint32_t>(r1 * 64 + ((((tid & 7) >> 1) ^ ((r1 >> 2) & 3)) << 4) + (tid & 1) * 8);
    const int r = wr + (lane & 15);
    f = static_cast<uint32_t>(r * 64 + (((lane >> 4) ^ ((r >> 2) & 3)) << 4));
  }
  // the k-tile's values; zero past the rows and past krem k (nothing is accessed there)
  __device__ __forceinline__ void load(float4 (&v)[NV], int krem, int64_t ld) const {
#pragma unroll
    for (int i = 0; i < NV; ++i)
      v[i] = 64 * i < left && kc < krem ? *reinterpret_cast<const float4*>(p + 64 * i * ld)
                                        : make_float4(0.0f, 0.0f, 0.0f, 0.0f);
  }
  __device__ __forceinline__ void advance(int64_t) { p += BK; }
  __device__ __forceinline__ uint32_t word(int i) const { return w + 4096u * i; }
  __device__ __forceinline__ bf16x8 frag(const char* tile, int limb, int I) const {
    return *reinterpret_cast<const bf16x8*>(tile + limb * kLimb + f + I * 1024);
  }
};

template <>
struct Side<false> {
  static constexpr int kStep = BK / NV;  // k-rows between a thread's loads (the swizzle repeats)
  const float* p;
  bool ok;
  int kr;
  uint32_t w;       // LDS byte offset of the thread's first 8-byte limb word
  uint32_t f, swz;  // the lane's k-row address and its swizzle
  int seg;          // the wave's first 16-row block
  __device__ __forceinline__ void init(const float* base, int64_t ld, int r0, int rmax, int wr, int k0, int tid, int lane) {
    kr = tid >> 5;
    const int c = tid & 31;
    ok = r0 + 4 * c < rmax;
    p = base + static_cast<int64_t>(k0 + kr) * ld + (ok ? r0 + 4 * c : 0);
    w = static_cast<uint32_t>(kr * 256 + (((c >> 2) ^ tr_swz(kr)) << 5) + (c & 3) * 8);
    // lane 4 j + q of 16-lane group g addresses k-row 8 g + j, rows 4 q .. 4 q + 3 of a 16-row block
    const int g = lane >> 4, j = (lane >> 2) & 3, q = lane & 3;
    f = static_cast<uint32_t>((8 * g + j) * 256 + 8 * q);
    swz = static_cast<uint32_t>(tr_swz(8 * g + j));
    seg = wr >> 4;
  }
  __device__ __forceinline__ void load(float4 (&v)[NV], int krem, int64_t ld) const {
#pragma unroll
    for (int i = 0; i < NV; ++i)
      v[i] = ok && kr + kStep * i < krem ? *reinterpret_cast<const float4*>(p + kStep * i * ld)
                                         : make_float4(0.0f, 0.0f, 0.0f, 0.0f);
  }
  __device__ __forceinline__ void advance(int64_t ld) { p += BK * ld; }
  __device__ __forceinline__ uint32_t word(int i) const { return w + static_cast<uint32_t>(kStep * 256 * i); }
  __device__ __forceinline__ bf16x8 frag(const char* tile, int limb, int I) const {
    const char* a = tile + limb * kLimb + f + ((static_cast<uint32_t>(seg + I) ^ swz) << 5);
    const s16x4 lo = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_s16x4*)(a));
    const s16x4 hi = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_s16x4*)(a + 4 * 256));
    return __builtin_bit_cast(bf16x8, __builtin_shufflevector(lo, hi, 0, 1, 2, 3, 4, 5, 6, 7));
  }
};

__device__ __forceinline__ void put(char* tile, uint32_t w, const float4& v) {
  uint2 h, m, l;
  split2(v.x, v.y, h.x, m.x, l.x);
  split2(v.z, v.w, h.y, m.y, l.y);
  *reinterpret_cast<uint2*>(tile + w) = h;
  *reinterpret_cast<uint2*>(tile + kLimb + w) = m;
  *reinterpret_cast<uint2*>(tile + 2 * kLimb + w) = l;
}

// Workgroups go round robin over the 8 XCDs (each with its own L2): each XCD
// takes a contiguous range of tiles, walked in groups of 8 tile rows.
__device__ __forceinline__ void tile_of(int pid, int tiles_m, int tiles_n, int& tm, int& tn) {
  const int nt = tiles_m * tiles_n;
  if ((nt & 7) == 0) pid = (pid & 7) * (nt >> 3) + (pid >> 3);
  const int per_group = 8 * tiles_n, group = pid / per_group, first = group * 8;
  const int gsize = min(tiles_m - first, 8), in_group = pid - group * per_group;
  tm = first + in_group % gsize;
  tn = in_group / gsize;
}

// Two LDS stages; while k-tile t is multiplied, k-tile t + 1 (in registers
// since the iteration before) is split into the other stage and k-tile t + 2
// is requested. One barrier per k-tile. Waves w and w + 4 share a SIMD: one
// multiplies first and splits then, the other the other way round, so the
// matrix core and the vector unit of a SIMD are both busy.
template <bool AK, bool BKM, bool SPLIT>
__global__ __launch_bounds__(kThreads) void gemm_f32_kernel(Params p) {
  constexpr int NB = 2;  // 16-column blocks per wave
  __shared__ __attribute__((aligned(16))) char lds[2][2 * kSide];
  const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int wm = (wave >> 2) * 64, wn = (wave & 3) * 32;
  int tm, tn;
  tile_of(blockIdx.x, p.tiles_m, p.tiles_n, tm, tn);
  const int m0 = tm * BM, n0 = tn * BN;
  const int nkt = (p.K + BK - 1) / BK;
  const int kt0 = blockIdx.y * p.kt_per_split;
  const int n = min(nkt - kt0, p.kt_per_split);
  int krem = p.K - kt0 * BK;  // k left from the next tile to load

  Side<AK> a;
  Side<BKM> b;
  a.init(p.A, p.lda, m0, p.M, wm, kt0 * BK, tid, lane);
  b.init(p.B, p.ldb, n0, p.N, wn, kt0 * BK, tid, lane);
  // hh in acc, the five smaller products in low: they round at 2^-8 of acc's
  // magnitude there, and acc takes one rounding per 32 k
  f32x4v acc[4][NB], low[4][NB];
#pragma unroll
  for (int i = 0; i < 4; ++i)
#pragma unroll
    for (int j = 0; j < NB; ++j) acc[i][j] = low[i][j] = f32x4v{0.0f, 0.0f, 0.0f, 0.0f};

  float4 va[NV], vb[NV];
  auto fetch = [&]() __attribute__((always_inline)) {
    a.load(va, krem, p.lda);
    b.load(vb, krem, p.ldb);
    a.advance(p.lda);
    b.advance(p.ldb);
    krem -= BK;
  };
  auto store = [&](char* st) __attribute__((always_inline)) {
#pragma unroll
    for (int i = 0; i < NV; ++i) {
      put(st, a.word(i), va[i]);
      put(st + kSide, b.word(i), vb[i]);
    }
  };
  fetch();
  store(lds[0]);
  fetch();
  __syncthreads();
  auto multiply = [&](const char* cur) __attribute__((always_inline)) {
    // A's fragments one 16-row block ahead of the MFMAs that use them
    bf16x8 fa[2][3], fb[3][NB];
#pragma unroll
    for (int q = 0; q < 3; ++q) fa[0][q] = a.frag(cur, q, 0);
#pragma unroll
    for (int q = 0; q < 3; ++q)
#pragma unroll
      for (int j = 0; j < NB; ++j) fb[q][j] = b.frag(cur + kSide, q, j);
    // (limb of A, limb of B): hh, then mh, hm, mm, lh, hl
    constexpr int kLa[6] = {0, 1, 0, 1, 2, 0}, kLb[6] = {0, 0, 1, 1, 0, 2};
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      if (i < 3) {
#pragma unroll
        for (int q = 0; q < 3; ++q) fa[(i + 1) & 1][q] = a.frag(cur, q, i + 1);
      }
      __builtin_amdgcn_sched_barrier(0);
#pragma unroll
      for (int q = 0; q < 6; ++q)
#pragma unroll
        for (int j = 0; j < NB; ++j) {
          f32x4v& d = q == 0 ? acc[i][j] : low[i][j];
          d = __builtin_amdgcn_mfma_f32_16x16x32_bf16(fb[kLb[q]][j], fa[i & 1][kLa[q]], d, 0, 0, 0);
        }
    }
  };
  auto refill = [&](int t) __attribute__((always_inline)) {
    if (t + 1 < n) {
      store(lds[(t + 1) & 1]);
      if (t + 2 < n) fetch();
    }
  };
  if (wave < 4) {
    for (int t = 0; t < n; ++t) {
      multiply(lds[t & 1]);
      __builtin_amdgcn_sched_barrier(0);
      refill(t);
      __syncthreads();
    }
  } else {
    for (int t = 0; t < n; ++t) {
      refill(t);
      __builtin_amdgcn_sched_barrier(0);
      multiply(lds[t & 1]);
      __syncthreads();
    }
  }
#pragma unroll
  for (int i = 0; i < 4; ++i)
#pragma unroll
    for (int j = 0; j < NB; ++j) acc[i][j] += low[i][j];

  // lane l: row 16 i + (l & 15), columns 16 j + 4 (l >> 4) .. + 3
  const int hq = lane >> 4;
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    const int m = m0 + wm + 16 * i + (lane & 15);
#pragma unroll
    for (int j = 0; j < NB; ++j) {
      const int c = n0 + wn + 16 * j + 4 * hq;
      if (m >= p.M || c >= p.N) continue;
      f4 x;
#pragma unroll
      for (int e = 0; e < 4; ++e) x.v[e] = acc[i][j][e];
      if constexpr (SPLIT)
        io4<float>::store(p.part + (static_cast<int64_t>(blockIdx.y) * p.M + m) * p.N + c, x);
      else
        finish(p, m, c, x);
    }
  }
}

// The partials' sum in split order, finished as an unsplit tile's
__global__ __launch_bounds__(256) void reduce_kernel(Params p, int S) {
  const int64_t n4 = static_cast<int64_t>(p.M) * (p.N / 4), slice = static_cast<int64_t>(p.M) * p.N;
  for (int64_t i = blockIdx.x * static_cast<int64_t>(blockDim.x) + threadIdx.x; i < n4;
       i += static_cast<int64_t>(gridDim.x) * blockDim.x) {
    const int64_t m = i / (p.N / 4), c = (i % (p.N / 4)) * 4;
    const float* q = p.part + m * p.N + c;
    f4 sum = io4<float>::load(q);
#pragma unroll 4
    for (int s = 1; s < S; ++s) {
      const f4 v = io4<float>::load(q + s * slice);
#pragma unroll
      for (int e = 0; e < 4; ++e) sum.v[e] += v.v[e];
    }
    finish(p, m, c, sum);
  }
}

struct Plan {
  int kt_per_split, splits;
};

// Split along K: the count that takes the least time in a model of one
// workgroup per CU, fitted to MI355X timings of 0.1 to 137 GFLOP products. A
// round of workgroups takes 1.4 us per k-tile plus about 6 us to start and to
// write; the partials' extra pass takes 3 us for its launch and its bytes
// (written and read back) at about 4 TB/s. At least 4 k-tiles per split.
// [4096, 512] x [512, 2048]: 62 us split in two against 96 whole; with 256
// tiles or more (4096 x 1024 x 512: 31 us) whole is faster.
inline Plan plan(int M, int N, int K, bool deterministic) {
  const int64_t tiles = int64_t((M + BM - 1) / BM) * ((N + BN - 1) / BN);
  const int nkt = std::max((K + BK - 1) / BK, 1);
  Plan best{nkt, 1};
  double least = 1e300;
  for (int s = 1; s <= 64 && (s == 1 || (!deterministic && nkt / s >= 4)); ++s) {
    const int kt = (nkt + s - 1) / s, ys = (nkt + kt - 1) / kt;
    double cost = double((tiles * ys + kCUs - 1) / kCUs) * (kt * 1.4 + 6.0);
    if (ys > 1) cost += 3.0 + double(ys) * M * N * 8.0 / 4e6;
    if (cost < least) least = cost, best = Plan{kt, ys};
  }
  return best;
}

inline size_t ws_bytes(const Plan& pl, int M, int N) {
  return pl.splits <= 1 ? 0 : static_cast<size_t>(pl.splits) * M * N * sizeof(float);
}

template <bool AK, bool BKM>
int launch(const Params& p, const Plan& pl, hipStream_t s) {
  const dim3 grid(p.tiles_m * p.tiles_n, pl.splits);
  if (pl.splits > 1) hipLaunchKernelGGL((gemm_f32_kernel<AK, BKM, true>), grid, dim3(kThreads), 0, s, p);
  else hipLaunchKernelGGL((gemm_f32_kernel<AK, BKM, false>), grid, dim3(kThreads), 0, s, p);
  return check_launch("mg_gemm_f32");
}

}  // namespace gemm_f32
}  // namespace mg

using namespace mg;

extern "C" size_t mg_gemm_f32_workspace_bytes(int M, int N, int K, int flags) {
  if (M < 1 || N < 1 || K < 1) return 0;
  return gemm_f32::ws_bytes(gemm_f32::plan(M, N, K, flags & MG_GEMM_DETERMINISTIC), M, N);
}

extern "C" int mg_gemm_f32(int a_layout, const float* A, int64_t lda, int b_layout, const float* B, int64_t ldb, int M,
                           int N, int K, int epilogue, const float* bias, float* aux, int64_t ldaux, float* C, int64_t ldc,
                           int flags, void* workspace, size_t workspace_bytes, void* stream) {
  const char* fn = "mg_gemm_f32";
  if (flags & ~(MG_GEMM_ACCUMULATE | MG_GEMM_DETERMINISTIC)) return fail(MG_ERR_ARG, "%s: unknown flags %d", fn, flags);
  if (!A || !B || !C) return fail(MG_ERR_ARG, "%s: null operand", fn);
  if (M < 0 || N < 0 || K < 0) return fail(MG_ERR_ARG, "%s: negative size", fn);
  if ((a_layout != MG_KCONTIG && a_layout != MG_MNCONTIG) || (b_layout != MG_KCONTIG && b_layout != MG_MNCONTIG))
    return fail(MG_ERR_ARG, "%s: bad layout code", fn);
  const bool ak = a_layout == MG_KCONTIG, bk = b_layout == MG_KCONTIG;
  if (N % 4 || (!ak && M % 4) || ((ak || bk) && K % 4))
    return fail(MG_ERR_ARG, "%s: M=%d N=%d K=%d (N and every contiguous dimension a multiple of 4)", fn, M, N, K);
  if (lda % 4 || ldb % 4 || ldc % 4 || lda < (ak ? K : M) || ldb < (bk ? K : N) || ldc < N)
    return fail(MG_ERR_ARG, "%s: leading dimensions must cover a row and be multiples of 4", fn);
  if (!aligned(A, 16) || !aligned(B, 16) || !aligned(C, 16) || (bias && !aligned(bias, 16)))
    return fail(MG_ERR_ARG, "%s: operands must be 16-byte aligned", fn);
  if (epilogue < MG_EPI_NONE || epilogue > MG_EPI_GELU_GRAD) return fail(MG_ERR_ARG, "%s: bad epilogue %d", fn, epilogue);
  const bool biased = epilogue == MG_EPI_BIAS || epilogue == MG_EPI_BIAS_GELU;
  if (biased != (bias != nullptr)) return fail(MG_ERR_ARG, "%s: a bias with the bias epilogues, none without", fn);
  if (epilogue == MG_EPI_GELU_GRAD && !aux) return fail(MG_ERR_ARG, "%s: the GELU gradient needs aux", fn);
  if (aux && (ldaux < N || ldaux % 4 || !aligned(aux, 16))) return fail(MG_ERR_ARG, "%s: aux rows of N, 16-byte aligned", fn);
  if ((flags & MG_GEMM_ACCUMULATE) && epilogue != MG_EPI_NONE)
    return fail(MG_ERR_ARG, "%s: no epilogue when accumulating", fn);
  if (M == 0 || N == 0 || (K == 0 && (flags & MG_GEMM_ACCUMULATE))) return MG_OK;
  if (int64_t((M + 127) / 128) * ((N + 127) / 128) >= (int64_t(1) << 31)) return fail(MG_ERR_ARG, "%s: too many tiles", fn);
  gemm_f32::Plan pl = gemm_f32::plan(M, N, K, (flags & MG_GEMM_DETERMINISTIC) || !workspace);
  gemm_f32::Params p{};
  if (pl.splits > 1) {
    const size_t need = gemm_f32::ws_bytes(pl, M, N);
    if (workspace_bytes < need)
      return fail(MG_ERR_WORKSPACE, "%s: workspace %zu bytes < required %zu (mg_gemm_f32_workspace_bytes)", fn,
                  workspace_bytes, need);
    if (!aligned(workspace, 16)) return fail(MG_ERR_ARG, "%s: workspace not 16-byte aligned", fn);
    p.part = static_cast<float*>(workspace);
  }
  p.A = A; p.B = B; p.C = C; p.bias = bias; p.aux = aux;
  p.epilogue = epilogue;
  p.lda = lda; p.ldb = ldb; p.ldc = ldc; p.ldaux = ldaux;
  p.M = M; p.N = N; p.K = K;
  p.tiles_m = (M + gemm_f32::BM - 1) / gemm_f32::BM;
  p.tiles_n = (N + gemm_f32::BN - 1) / gemm_f32::BN;
  p.kt_per_split = pl.kt_per_split;
  p.accumulate = flags & MG_GEMM_ACCUMULATE ? 1 : 0;
  hipStream_t s = static_cast<hipStream_t>(stream);
  const int rc = ak ? (bk ? gemm_f32::launch<true, true>(p, pl, s) : gemm_f32::launch<true, false>(p, pl, s))
                    : (bk ? gemm_f32::launch<false, true>(p, pl, s) : gemm_f32::launch<false, false>(p, pl, s));
  if (rc || pl.splits <= 1) return rc;
  const int64_t n4 = int64_t(M) * (N / 4);
  hipLaunchKernelGGL(gemm_f32::reduce_kernel, dim3(static_cast<int>(std::min<int64_t>((n4 + 255) / 256, 2048))), dim3(256), 0,
                     s, p, pl.splits);
  return check_launch(fn);
}
