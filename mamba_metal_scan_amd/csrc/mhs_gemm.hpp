// fp32 matrix products on the bf16 matrix cores for gfx950:
//   C[m,n] = sum_k A(m,k) B(n,k)      (+ C, or a split-K partial)
// with fp32 operands in memory and fp32 results.
//
// Each fp32 value is split into three bf16 parts, x = x0 + x1 + x2 (x0 = x
// rounded to bf16, x1 = (x - x0) rounded, x2 the rest: 24 bits in all, the
// differences are exact), and the product takes the six partial products
// whose weight reaches fp32's last bit:
//   x0 y0 + (x0 y1 + x1 y0) + (x0 y2 + x1 y1 + x2 y0);
// the dropped x1 y2, x2 y1 and x2 y2 are below 2^-26 |x y|. A bf16 MFMA
// multiplies exactly and adds in fp32. Six bf16 products at 2.5 PFLOP/s
// against one fp32 product at 157 TFLOP/s: 2.6 times the rate at the peaks.
//
// The MFMA rounds its sum down, towards -inf: with the k tiles' sums formed
// by MFMAs and added exactly rounded, the results of a 8192 x 1464 x 1432
// product of normal operands (rms 38) are low by 3.0e-6 on average, at an rms
// error of 7.4e-6, and sums over time (the gradients of the biases, B and C)
// then add these up. So A is negated, and the running sum with it, every
// kGemmFlip k tiles: the roundings of neighbouring runs cancel (mean error
// 1e-8, rms 2.2e-5; an fp32 rocBLAS product 5e-9 and 2.6e-5).
//
// Range: with x1 about 2^-9 x and x2 2^-18 x, values down to 2^-110 keep all
// 24 bits (below, the parts run into the subnormals). A thread ORs the leading
// parts that it stages; where all of them lie below 2^-95 and not all are
// zero, the block computes its tile again with fp32 MFMAs (plain_products). A
// smaller value among larger ones of its row loses what is below their last
// bits; values below 2^-134, among themselves too, count as zeros. Infinities,
// NaN and values that round to a bf16 infinity make the element's sum NaN or
// infinite: a wave that ends with such an element computes its part of the
// tile again likewise.
#pragma once

#include "mhs_common.hpp"

namespace mhs {

typedef __bf16 bf16x2 __attribute__((ext_vector_type(2)));
typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef float f32x2 __attribute__((ext_vector_type(2)));
typedef float f32x16 __attribute__((ext_vector_type(16)));

struct GemmArgs {
  const float* A;   // K-major: (M, K) rows lda apart; else (K, M) rows lda apart
  const float* B;   // K-major: (N, K) rows ldb apart; else (K, N) rows ldb apart
  float* C;         // (M, N) rows ldc apart; split-K: partials (splits, M, N)
  int M, N, K;
  long long lda, ldb, ldc;
  int kt_per_split;   // 16-deep k tiles per split
  int accumulate;     // C += (one split only)
  int grid_m, grid_n;
};

constexpr int kGemmBK = 16;       // k depth of a tile: one 32x32x16 MFMA
constexpr int kGemmThreads = 256; // 4 waves
constexpr int kGemmTile = 128, kGemmSmallTile = 64;
constexpr int kGemmFlip = 4;      // k tiles between changes of sign (see below)
constexpr int kGemmPad = 64;      // bytes between the halves of an LDS plane

// One operand's LDS tile: three bf16 planes, each [2 halves][R rows][8 k]
// (a lane's MFMA operand is one 16-byte read; 32 lanes read 512 contiguous
// bytes), the second half 64 bytes further: eight lanes writing both halves of
// four rows then hit all 32 banks (SQ_LDS_BANK_CONFLICT 0; with 0 or 128 bytes
// 8 cycles per write).
__host__ __device__ constexpr int gemm_half_bytes(int R) { return R * 16 + kGemmPad; }
__host__ __device__ constexpr int gemm_plane_bytes(int R) { return 2 * gemm_half_bytes(R); }
__host__ __device__ constexpr int gemm_lds_bytes(int BM, int BN) {
  return 2 * 3 * (gemm_plane_bytes(BM) + gemm_plane_bytes(BN));
}

// 8 consecutive k of one row, split: the three parts as 16-byte operands.
// seen: the leading parts ORed in.
__device__ __forceinline__ void split8(const float (&v)[8], bf16x8 (&p)[3], unsigned& seen) {
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    f32x2 r = {v[2 * i], v[2 * i + 1]};
#pragma unroll
    for (int q = 0; q < 3; ++q) {
      const bf16x2 h = __builtin_convertvector(r, bf16x2);
      p[q][2 * i] = h[0];
      p[q][2 * i + 1] = h[1];
      const unsigned u = __builtin_bit_cast(unsigned, h);
      if (q == 0) seen |= u;
      if (q < 2) {
        r[0] -= __uint_as_float(u << 16);
        r[1] -= __uint_as_float(u & 0xffff0000u);
      }
    }
  }
}

// Whether the two bf16's of `seen`, an OR of parts, have exponents below
// 2^-95's and are not both zero (of exponent fields below 32 and others, the OR
// tells which: no sum carries).
__device__ __forceinline__ bool all_tiny(unsigned seen) {
  seen = (seen | seen >> 16) & 0x7fffu;
  return seen != 0 && seen < (32u << 7);
}

// The staging of one operand's R x 16 tile: one task per thread, a task being
// 8 consecutive k of one row. K-major memory: two 16-byte loads; otherwise
// eight 4-byte loads, consecutive lanes on consecutive rows. R = 128: every
// thread has a task of each operand; R = 64: the first half of the threads
// stage A, the second half B (LATE), whole waves.
template <int R, bool KMAJOR, bool LATE>
struct GemmLoader {
  static constexpr int T = 1;
  static constexpr bool kAll = R * 2 == kGemmThreads;
  static_assert(kAll || R * 4 == kGemmThreads, "one task of one or of each operand");
  __device__ __forceinline__ static bool mine() {
    const int w0 = __builtin_amdgcn_readfirstlane(threadIdx.x);
    return kAll || (LATE ? w0 >= R * 2 : w0 < R * 2);
  }
  const float* base;   // of the block's rows, at its first k
  long long ld;
  int width;           // rows from the block's first to the operand's last
  unsigned off[T];     // byte offset of the task at k tile 0, or kOOB
  int kpos[T];         // first k of the task within a tile
  int lds[T];          // byte offset in a plane
  unsigned seen = 0;   // the leading parts staged so far, ORed
  __device__ __forceinline__ GemmLoader(const float* p, long long ld_, int r0, int rows,
                                        long long k_first)
      : ld(ld_), width(rows - r0) {
    base = KMAJOR ? p + (long long)r0 * ld_ + k_first : p + k_first * ld_ + r0;
#pragma unroll
    for (int i = 0; i < T; ++i) {
      const int t = threadIdx.x - (!kAll && LATE ? R * 2 : 0);
      const int row = KMAJOR ? t >> 1 : t % R;
      const int half = KMAJOR ? t & 1 : t / R;
      kpos[i] = 8 * half;
      lds[i] = half * gemm_half_bytes(R) + row * 16;
      off[i] = mine() && r0 + row < rows
                   ? (KMAJOR ? 4u * ((unsigned)row * (unsigned)ld_ + 8u * half)
                             : 4u * ((unsigned)(8 * half) * (unsigned)ld_ + (unsigned)row))
                   : kOOB;
    }
  }
  // k tile kt (relative to the block's first), `left` the k's from there to
  // the split's end: k's at or past it read as zero (K-major: by their
  // offset; otherwise the resource ends with the last k's row, and ld >=
  // rows puts every later k past its end).
  __device__ __forceinline__ void load(float (&v)[T][8], int kt, int left) const {
    if (!mine()) return;
    if constexpr (KMAJOR) {
      const GBuf g(base + (long long)kt * kGemmBK, left > 0 ? kOOB - 1u : 0u);
#pragma unroll
      for (int i = 0; i < T; ++i) {
#pragma unroll
        for (int h = 0; h < 2; ++h) {   // K a multiple of 4: whole float4s
          const unsigned o = kpos[i] + 4 * h < left ? off[i] + 16u * h : kOOB;
          typedef unsigned u4 __attribute__((ext_vector_type(4)));
          const u4 t = __builtin_bit_cast(u4, __builtin_amdgcn_raw_buffer_load_b128(g.r, o, 0, 0));
#pragma unroll
          for (int e = 0; e < 4; ++e) v[i][4 * h + e] = __uint_as_float(t[e]);
        }
      }
    } else {
      const unsigned ld4 = 4u * (unsigned)ld;
      const GBuf g(base + (long long)kt * kGemmBK * ld,
                   left > 0 ? (unsigned)(min(left, kGemmBK) - 1) * ld4 + 4u * (unsigned)width
                            : 0u);
#pragma unroll
      for (int i = 0; i < T; ++i) {
        unsigned o = off[i];
#pragma unroll
        for (int e = 0; e < 8; ++e, o += ld4) v[i][e] = g.ld(o);
      }
    }
  }
  __device__ __forceinline__ void store(char* tile, const float (&w)[T][8], unsigned sign) {
    if (!mine()) return;
#pragma unroll
    for (int i = 0; i < T; ++i) {
      float v[8];
#pragma unroll
      for (int e = 0; e < 8; ++e) v[e] = __uint_as_float(__float_as_uint(w[i][e]) ^ sign);
      bf16x8 p[3];
      split8(v, p, seen);
#pragma unroll
      for (int q = 0; q < 3; ++q)
        *reinterpret_cast<bf16x8*>(tile + q * gemm_plane_bytes(R) + lds[i]) = p[q];
    }
  }
};

// 4 of the 8 k's from k of row r of one operand (rows rows, k's below k_end):
// the lane's operands of 4 fp32 MFMAs, lanes 32-63 taking the second 4 k's.
template <bool KMAJOR>
__device__ __forceinline__ void load_plain(float (&v)[4], const float* p, long long ld, int r,
                                           int rows, int k, int k_end) {
  k += 4 * ((threadIdx.x >> 5) & 1);
#pragma unroll
  for (int t = 0; t < 4; ++t) v[t] = 0.f;
  if (r >= rows || k >= k_end) return;
  if constexpr (KMAJOR) {   // K a multiple of 4: a whole float4
    f4_to(v, *reinterpret_cast<const float4*>(p + (long long)r * ld + k));
  } else {
#pragma unroll
    for (int t = 0; t < 4; ++t)
      if (k + t < k_end) v[t] = p[(long long)(k + t) * ld + r];
  }
}

// The wave's FM x FN fragments from row m, column n, over k's k_first ..
// k_end - 1, with fp32 MFMAs from global memory: a lane's operands are row (or
// column) lane % 32, k lane / 32, and the sum's elements lie as the bf16
// products' do. For the waves that meet infinities, NaN or parts that
// overflow; bound by the fp32 matrix rate. 8192 x 1464 x 1432 of NaN: 490 to 560 us
// with the bf16 products before it, against 21 to 32 ms by a serial fma loop
// per element and 265 us by the library.
template <bool AK, bool BK, int FM, int FN>
__device__ __forceinline__ void plain_products(f32x16 (&acc)[FM][FN], const GemmArgs& g, int m,
                                               int n, int k_first, int k_end) {
  m += threadIdx.x & 31;
  n += threadIdx.x & 31;
#pragma unroll
  for (int i = 0; i < FM; ++i)
#pragma unroll
    for (int j = 0; j < FN; ++j)
#pragma unroll
      for (int e = 0; e < 16; ++e) acc[i][j][e] = 0.f;
#pragma unroll 1
  for (int k = k_first; k < k_end; k += 8) {
    float a[FM][4], b[FN][4];
#pragma unroll
    for (int i = 0; i < FM; ++i) load_plain<AK>(a[i], g.A, g.lda, m + 32 * i, g.M, k, k_end);
#pragma unroll
    for (int j = 0; j < FN; ++j) load_plain<BK>(b[j], g.B, g.ldb, n + 32 * j, g.N, k, k_end);
#pragma unroll
    for (int t = 0; t < 4; ++t)
#pragma unroll
      for (int i = 0; i < FM; ++i)
#pragma unroll
        for (int j = 0; j < FN; ++j)
          acc[i][j] = __builtin_amdgcn_mfma_f32_32x32x2f32(a[i][t], b[j][t], acc[i][j], 0, 0, 0);
  }
}

// One 128 x 128 tile per block, 2 x 2 waves of 64 x 64 (or 64 x 64 of 32 x 32,
// for products of few tiles), k 16 deep and double
// buffered: while a wave multiplies a tile it splits the next one into the
// other buffer and loads the one after it into registers.
// Bound by the matrix cores at the power limit: per k tile a wave issues 24
// MFMAs (768 cycles of its SIMD's matrix core) beside 96 VALU (the split) and
// 12 + 6 LDS accesses of 1 KB; SQ_VALU_MFMA_BUSY_CYCLES 66% of the CU cycles
// at 1.6-1.8 GHz (2.4 nominal), three blocks per CU. Measured, against the
// fp32 library product, us (TFLOP/s of fp32 work):
//   NT 8192 x 1464 x 1432   195 (176) / 310       NN 8192 x 1432 x 1464  191 / 307
//   NT 8192 x 2864 x 640    171 (176) / 255       TN 1464 x 1432 x 8192  215 / 349
//   NT 8192 x 32768 x 640  1850 (186) / 2490      TN 32768 x 640 x 8192 1640 / 2260
// i.e. 1.05-1.2 PFLOP/s of bf16, what an 8192^3 bf16 library product reaches
// here (1.25). 256 x 128 tiles (two blocks per CU, a quarter fewer LDS reads)
// were within 4% either way; each k tile's products summed from zero and then
// added (a third of the error) took 8% longer.
template <bool AK, bool BK, int TILE>
__global__ void __launch_bounds__(kGemmThreads, TILE == kGemmTile ? 3 : 4)
gemm3_kernel(GemmArgs g) {
  constexpr int BM = TILE, BN = TILE;
  constexpr int FM = BM / 64, FN = BN / 64;   // 32 x 32 fragments per wave
  extern __shared__ float lds_f[];
  char* const lds = reinterpret_cast<char*>(lds_f);
  constexpr int PA = gemm_plane_bytes(BM), PB = gemm_plane_bytes(BN);
  constexpr int BUF = 3 * (PA + PB);
  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  // Blocks go round the 8 XCDs: each XCD takes a contiguous run of tiles,
  // so that the rows of A and B it shares stay in its own L2.
  const int tiles = g.grid_m * g.grid_n;
  const int xcd = blockIdx.x & 7, per = tiles >> 3, rem = tiles & 7;
  const int tile = xcd * per + min(xcd, rem) + (blockIdx.x >> 3);
  const int m0 = tile / g.grid_n * BM, n0 = tile % g.grid_n * BN;
  const int k_first = blockIdx.y * g.kt_per_split * kGemmBK;
  const int k_len = min(g.K - k_first, g.kt_per_split * kGemmBK);
  const int nk = (k_len + kGemmBK - 1) / kGemmBK;

  GemmLoader<BM, AK, false> la(g.A, g.lda, m0, g.M, k_first);
  GemmLoader<BN, BK, true> lb(g.B, g.ldb, n0, g.N, k_first);
  float va[la.T][8], vb[lb.T][8];
  f32x16 acc[FM][FN];
#pragma unroll
  for (int i = 0; i < FM; ++i)
#pragma unroll
    for (int j = 0; j < FN; ++j)
#pragma unroll
      for (int e = 0; e < 16; ++e) acc[i][j][e] = 0.f;

  la.load(va, 0, k_len);
  lb.load(vb, 0, k_len);
  la.store(lds, va, 0u);
  lb.store(lds + 3 * PA, vb, 0u);
  la.load(va, 1, k_len - kGemmBK);
  lb.load(vb, 1, k_len - kGemmBK);
  __syncthreads();

  const int wm = wave >> 1, wn = wave & 1;
  const int fa = (lane >> 5) * gemm_half_bytes(BM) + (wm * (BM / 2) + (lane & 31)) * 16;
  const int fb = 3 * PA + (lane >> 5) * gemm_half_bytes(BN) + (wn * (BN / 2) + (lane & 31)) * 16;
  unsigned sign = 0u;   // of the A staged for tile kt, and of acc
  for (int kt = 0; kt < nk; ++kt) {
    const unsigned next = sign ^ (kt % kGemmFlip == kGemmFlip - 1 ? 0x80000000u : 0u);
    if (kt > 0 && kt % kGemmFlip == 0) {
#pragma unroll
      for (int i = 0; i < FM; ++i)
#pragma unroll
        for (int j = 0; j < FN; ++j)
#pragma unroll
          for (int e = 0; e < 16; ++e) acc[i][j][e] = -acc[i][j][e];
    }
    const char* buf = lds + (kt & 1) * BUF;
    bf16x8 b[FN][3];
#pragma unroll
    for (int q = 0; q < 3; ++q)
#pragma unroll
      for (int j = 0; j < FN; ++j)
        b[j][q] = *reinterpret_cast<const bf16x8*>(buf + fb + q * PB + j * 32 * 16);
#pragma unroll
    for (int i = 0; i < FM; ++i) {
      bf16x8 a[3];
#pragma unroll
      for (int q = 0; q < 3; ++q)
        a[q] = *reinterpret_cast<const bf16x8*>(buf + fa + q * PA + i * 32 * 16);
      // The six products, smallest first, the fragments of a row in turn (a
      // product does not wait for the one before it).
      constexpr int PQ[6][2] = {{2, 0}, {0, 2}, {1, 1}, {1, 0}, {0, 1}, {0, 0}};
#pragma unroll
      for (int q = 0; q < 6; ++q)
#pragma unroll
        for (int j = 0; j < FN; ++j)
          acc[i][j] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(a[PQ[q][0]], b[j][PQ[q][1]],
                                                              acc[i][j], 0, 0, 0);
      if (i == 0) {
        // The next tile into the other buffer (last read before the previous
        // barrier), and the loads of the one after it.
        char* nbuf = lds + ((kt + 1) & 1) * BUF;
        la.store(nbuf, va, next);
        lb.store(nbuf + 3 * PA, vb, 0u);
        la.load(va, kt + 2, k_len - (kt + 2) * kGemmBK);
        lb.load(vb, kt + 2, k_len - (kt + 2) * kGemmBK);
      }
    }
    __syncthreads();
    sign = next;
  }
  if ((nk - 1) / kGemmFlip & 1)
#pragma unroll
    for (int i = 0; i < FM; ++i)
#pragma unroll
      for (int j = 0; j < FN; ++j)
#pragma unroll
        for (int e = 0; e < 16; ++e) acc[i][j][e] = -acc[i][j][e];

  float odd = 0.f;   // NaN once an element is not finite
#pragma unroll
  for (int i = 0; i < FM; ++i)
#pragma unroll
    for (int j = 0; j < FN; ++j)
#pragma unroll
      for (int e = 0; e < 16; ++e) odd = __builtin_fmaf(acc[i][j][e], 0.f, odd);
  // (The loop ended on a barrier: LDS is free.)
  if (lane == 0) lds_f[wave] = 0.f;
  if (all_tiny(la.seen) || all_tiny(lb.seen)) lds_f[wave] = 1.f;
  __syncthreads();
  const float4 tiny = *reinterpret_cast<const float4*>(lds_f);
  if (__builtin_amdgcn_ballot_w64(odd != odd || tiny.x + tiny.y + tiny.z + tiny.w != 0.f) != 0)
    plain_products<AK, BK>(acc, g, m0 + wm * (BM / 2), n0 + wn * (BN / 2), k_first,
                           k_first + k_len);

  // A fragment's element e of lane l: row 8 (e / 4) + 4 (l / 32) + e % 4,
  // column l % 32.
  float* const cb = g.C + (long long)blockIdx.y * g.M * g.ldc;
#pragma unroll
  for (int i = 0; i < FM; ++i) {
#pragma unroll
    for (int j = 0; j < FN; ++j) {
      const int n = n0 + wn * (BN / 2) + j * 32 + (lane & 31);
      const int mb = m0 + wm * (BM / 2) + i * 32 + 4 * (lane >> 5);
#pragma unroll
      for (int e = 0; e < 16; ++e) {
        const int m = mb + 8 * (e / 4) + e % 4;
        if (m < g.M && n < g.N) {
          float* p = cb + (long long)m * g.ldc + n;
          *p = g.accumulate ? *p + acc[i][j][e] : acc[i][j][e];
        }
      }
    }
  }
}

// out = the rows of a, then b, then c: float4s, na + nb + nc of them.
template <int UNUSED = 0>
__global__ void __launch_bounds__(256)
concat3_kernel(const float4* __restrict__ a, const float4* __restrict__ b,
               const float4* __restrict__ c, float4* __restrict__ out, long long na, long long nb,
               long long nc) {
  const long long i = (long long)blockIdx.x * 256 + threadIdx.x;
  if (i < na) out[i] = a[i];
  else if (i < na + nb) out[i] = b[i - na];
  else if (i < na + nb + nc) out[i] = c[i - na - nb];
}

__device__ __forceinline__ float add(float a, float b) { return a + b; }
__device__ __forceinline__ float4 add(float4 a, float4 b) {
  return make_float4(a.x + b.x, a.y + b.y, a.z + b.z, a.w + b.w);
}

// out (M, N; rows ldc apart) = the sum of the split-K partials (splits, M,
// N), in split order (+ out). V: float4 (N and ldc in float4s; rows 16-byte
// aligned), or float for any width.
template <class V>
__global__ void __launch_bounds__(256)
gemm_reduce_kernel(const V* __restrict__ part, V* __restrict__ out, int splits, long long M,
                   int N, long long ldc, int accumulate) {
  const long long n = M * N;
  for (long long i = (long long)blockIdx.x * 256 + threadIdx.x; i < n;
       i += (long long)gridDim.x * 256) {
    const long long at = ldc == N ? i : i / N * ldc + i % N;
    V s = part[i];
    for (int k = 1; k < splits; ++k) s = add(s, part[k * n + i]);
    if (accumulate) s = add(s, out[at]);
    out[at] = s;
  }
}

}  // namespace mhs
