// One recurrent token of the whole TinyMamba for gfx950 (the reference's step
// in pure torch, mamba_metal/model.py:228-256, :289-298): per block
//   in    x | z = in_proj(rms_norm(x));  xc = silu(conv(window, x));  the
//         window moves on by x
//   proj  dt = dt_min + (dt_max - dt_min) sigmoid(dt_proj(xc));  B, C
//   state h <- exp(-dt softplus(A)) h + dt xc B;  g = (C h + D_skip) silu(z)
//   out   x <- x + out_proj(g)
// then logits = head(rms_norm(x)). Four launches a block: the norm, the conv
// step and the gates ride along in the products that feed or need them.
//
// The products have `batch` columns (1 .. tens): they are bound by reading
// each weight once (314 MB for 79.5 M parameters, 65 us at 4.8 TB/s) and, at
// these sizes, by the launches. A wave computes RW rows of the weight for NB
// batch rows: the lanes read 16 bytes each of the rows (every weight byte is
// read once per NB batch rows, coalesced) and sum their products over the
// wave at the end, in a fixed order. All loads of a wave, the epilogue's
// included, are issued before the first is waited for: at batch 4 a launch
// takes 3.5 to 6.7 us (traced; 2.3 an empty one), 1.5 of it for the 7.3 MB of
// in_proj. Measured at the 80M model, batch 4: 3684 us a token by module
// calls, 307 with the loads of each pass waited for in turn, 273 so.
#pragma once

#include "mhs_common.hpp"
#include "mhs_conv.hpp"
#include "mhs_norm.hpp"

namespace mhs {

enum DecodeKind { kDecIn = 0, kDecProj = 1, kDecOut = 2, kDecHead = 3 };

struct DecodeArgs {
  const float* x;    // (batch, K): the product's input rows
  const float* w;    // (rows, K); kDecProj: dt_proj, then B_proj, C_proj
  const float* w_b;
  const float* w_c;
  const float* norm_w;   // kDecIn, kDecHead: the norm before the product
  float eps;
  int batch, K, rows;
  int D, N;              // d_inner, d_state (kDecIn, kDecProj)
  float* out;            // kDecIn: xc; kDecProj: dt; kDecOut: x; kDecHead: logits
  float* out2;           // kDecIn: z; kDecProj: B (batch, N), then C
  const float* bias;     // kDecProj: dt_proj's
  float dt_lo, dt_span;
  const float* res;      // kDecOut: the residual stream's x
  // kDecIn: the conv window (batch, D, taps - 1), any strides, and the next
  // one (contiguous); taps >= 2.
  const float* conv_w;
  const float* conv_b;
  const float* conv;
  long long conv_sb, conv_sd, conv_sk;
  float* conv_next;
  int taps;
};

// The sum over the wave's 64 lanes, in every lane (fixed order).
__device__ __forceinline__ float wave_total(float v) {
  v = group_sum<16>(v);
  const auto a = __builtin_amdgcn_permlane16_swap(__float_as_uint(v), __float_as_uint(v), false,
                                                 false);
  v = __uint_as_float(a[0]) + __uint_as_float(a[1]);
  const auto b = __builtin_amdgcn_permlane32_swap(__float_as_uint(v), __float_as_uint(v), false,
                                                 false);
  return __uint_as_float(b[0]) + __uint_as_float(b[1]);
}

__device__ __forceinline__ float dot4(const float4& a, const float4& b, float s) {
  s = __builtin_fmaf(a.x, b.x, s);
  s = __builtin_fmaf(a.y, b.y, s);
  s = __builtin_fmaf(a.z, b.z, s);
  return __builtin_fmaf(a.w, b.w, s);
}

__device__ __forceinline__ float4 ld4(const GBuf& g, unsigned byte_off) {
  typedef unsigned u4 __attribute__((ext_vector_type(4)));
  const u4 t = __builtin_bit_cast(u4, __builtin_amdgcn_raw_buffer_load_b128(g.r, byte_off, 0, 0));
  return make_float4(__uint_as_float(t[0]), __uint_as_float(t[1]), __uint_as_float(t[2]),
                     __uint_as_float(t[3]));
}

// What the product's element (weight row n, batch row b) becomes. fetch()
// loads what that takes before the product, so that its latency is hidden
// there; store() finishes the element.
template <int KIND>
struct DecodeEpilogue {
  float win[KIND == kDecIn ? kConvMaxK - 1 : 1], cw[KIND == kDecIn ? kConvMaxK : 1], c0;
  // b < batch, n < rows. Loads without branches (each would wait for its own):
  // taps past the kernel's read tap 0, rows of z the last channel.
  __device__ __forceinline__ void fetch(const DecodeArgs& a, int b, int n) {
    if constexpr (KIND == kDecIn) {
      const int d = min(n, a.D - 1);
      c0 = a.conv_b[d];
      const float* w = a.conv + b * a.conv_sb + d * a.conv_sd;
      const float* c = a.conv_w + (size_t)d * a.taps;
#pragma unroll
      for (int k = 0; k < kConvMaxK; ++k) cw[k] = c[k < a.taps ? k : 0];
#pragma unroll
      for (int k = 0; k < kConvMaxK - 1; ++k) win[k] = w[(k < a.taps - 1 ? k : 0) * a.conv_sk];
    } else if constexpr (KIND == kDecProj) {
      c0 = a.bias[min(n, a.D - 1)];
    } else if constexpr (KIND == kDecOut) {
      c0 = a.res[(size_t)b * a.rows + n];
    }
  }
  __device__ __forceinline__ void store(const DecodeArgs& a, int b, int n, float v) {
    if constexpr (KIND == kDecIn) {
      if (n >= a.D) {
        a.out2[(size_t)b * a.D + n - a.D] = v;
        return;
      }
      float pre = c0, last = cw[1];
      float* next = a.conv_next + ((size_t)b * a.D + n) * (a.taps - 1);
#pragma unroll
      for (int k = 0; k < kConvMaxK - 1; ++k) {
        if (k < a.taps - 1) {
          pre = __builtin_fmaf(cw[k], win[k], pre);
          if (k > 0) next[k - 1] = win[k];
        }
        if (k == a.taps - 2) last = cw[k + 1];
      }
      next[a.taps - 2] = v;
      pre = __builtin_fmaf(last, v, pre);
      a.out[(size_t)b * a.D + n] = pre * sigmoid_f(pre);
    } else if constexpr (KIND == kDecProj) {
      if (n < a.D) {
        a.out[(size_t)b * a.D + n] = gate_dt(v + c0, a.dt_lo, a.dt_span);
      } else {
        const int c = n - a.D >= a.N;
        a.out2[((size_t)c * a.batch + b) * a.N + n - a.D - c * a.N] = v;
      }
    } else if constexpr (KIND == kDecOut) {
      a.out[(size_t)b * a.rows + n] = c0 + v;
    } else {
      a.out[(size_t)b * a.rows + n] = v;
    }
  }
};

// rows of the weight: wave (blockIdx.x * 4 + wave) takes RW of them, U 16-byte
// loads of each in flight per lane. K a multiple of 4, pointers 16-byte
// aligned.
template <int KIND, int NB, int RW, int U>
__global__ void __launch_bounds__(256) decode_product_kernel(DecodeArgs a) {
  constexpr bool NORM = KIND == kDecIn || KIND == kDecHead;
  const int lane = threadIdx.x & 63;
  const int n0 = (blockIdx.x * 4 + __builtin_amdgcn_readfirstlane(threadIdx.x >> 6)) * RW;
  if (n0 >= a.rows) return;   // whole waves
  // Rows through buffer resources of their own length: lanes past a row's end
  // read zero.
  const float* wr[RW];
#pragma unroll
  for (int r = 0; r < RW; ++r) {
    const int n = min(n0 + r, a.rows - 1);
    wr[r] = a.w + (size_t)n * a.K;
    if constexpr (KIND == kDecProj) {
      if (n >= a.D + a.N) wr[r] = a.w_c + (size_t)(n - a.D - a.N) * a.K;
      else if (n >= a.D) wr[r] = a.w_b + (size_t)(n - a.D) * a.K;
    }
  }
  const unsigned row_bytes = 4u * (unsigned)a.K;
  const GBuf gn(NORM ? a.norm_w : a.w, NORM ? row_bytes : 0u);
  for (int b0 = 0; b0 < a.batch; b0 += NB) {
    // Lane r * NB + b takes element (n0 + r, b0 + b).
    const int er = lane / NB, eb = b0 + lane % NB;
    const bool emit = lane < RW * NB && n0 + er < a.rows && eb < a.batch;
    DecodeEpilogue<KIND> epi;
    epi.fetch(a, min(eb, a.batch - 1), min(n0 + min(er, RW - 1), a.rows - 1));
    float acc[RW][NB], ss[NB];
#pragma unroll
    for (int b = 0; b < NB; ++b) {
      ss[b] = 0.f;
#pragma unroll
      for (int r = 0; r < RW; ++r) acc[r][b] = 0.f;
    }
    for (unsigned c = 16u * lane; __builtin_amdgcn_readfirstlane(c) < row_bytes;
         c += 1024u * U) {
      float4 wv[U][RW], nv[U];
#pragma unroll
      for (int u = 0; u < U; ++u) {
#pragma unroll
        for (int r = 0; r < RW; ++r) wv[u][r] = ld4(GBuf(wr[r], row_bytes), c + 1024u * u);
        if constexpr (NORM) nv[u] = ld4(gn, c + 1024u * u);
      }
      float4 xs[NB][U];
#pragma unroll
      for (int b = 0; b < NB; ++b) {
        const GBuf gx(a.x + (size_t)(b0 + b) * a.K, b0 + b < a.batch ? row_bytes : 0u);
#pragma unroll
        for (int u = 0; u < U; ++u) xs[b][u] = ld4(gx, c + 1024u * u);
      }
      step_fence();   // every load issued before the first is waited for
#pragma unroll
      for (int b = 0; b < NB; ++b) {
#pragma unroll
        for (int u = 0; u < U; ++u) {
          float4 xv = xs[b][u];
          if constexpr (NORM) {
            ss[b] = dot4(xv, xv, ss[b]);
            xv = make_float4(xv.x * nv[u].x, xv.y * nv[u].y, xv.z * nv[u].z, xv.w * nv[u].w);
          }
#pragma unroll
          for (int r = 0; r < RW; ++r) acc[r][b] = dot4(wv[u][r], xv, acc[r][b]);
        }
      }
    }
    float mine = 0.f;
#pragma unroll
    for (int b = 0; b < NB; ++b) {
      float rs = 1.f;
      if constexpr (NORM)
        rs = 1.f / __fsqrt_rn(__builtin_fmaf(wave_total(ss[b]), 1.f / (float)a.K, a.eps));
#pragma unroll
      for (int r = 0; r < RW; ++r) {
        const float v = wave_total(acc[r][b]) * rs;
        if (lane == r * NB + b) mine = v;
      }
    }
    if (emit) epi.store(a, eb, n0 + er, mine);
  }
}

// softplus(v) = max(v, 0) + log1p(u), u = e^-|v|, with the hardware's exp2,
// log2 and reciprocal: log1p(u) = u log(w) / (w - 1), w = 1 + u rounded (the
// rounding of w cancels; Goldberg's form), u itself where w is 1.
__device__ __forceinline__ float softplus_hw(float v) {
  const float u = exp2_hw(-fabsf(v) * kLog2e);
  const float w = 1.f + u, t = w - 1.f;
  const float l = __builtin_amdgcn_logf(w) * kLn2;
  return fmaxf(v, 0.f) + (t == 0.f ? u : u * l * __builtin_amdgcn_rcpf(t));
}

// The state step and the output gate: h (batch, D, N) in place, g (batch, D).
// A group of LPC lanes owns one channel; lane q of it the states q, q + LPC,
// ... (coalesced over the group); LPC = 4 for N 4 and up, else 1.
template <int LPC>
__global__ void __launch_bounds__(256)
decode_state_kernel(float* __restrict__ h, const float* __restrict__ xc,
                    const float* __restrict__ dt, const float* __restrict__ a_raw,
                    const float* __restrict__ Bm, const float* __restrict__ Cm,
                    const float* __restrict__ dskip, const float* __restrict__ z,
                    float* __restrict__ g, int batch, int D, int N) {
  const long long gid = (long long)blockIdx.x * 256 + threadIdx.x;
  const long long ch = gid / LPC;          // (b, d)
  const int q = (int)(gid % LPC);
  const bool valid = ch < (long long)batch * D;
  float part = 0.f;
  if (valid) {
    const int b = (int)(ch / D), d = (int)(ch % D);
    const float dtv = dt[ch], bx = dtv * xc[ch];
    const float* ar = a_raw + (size_t)d * N;
    const float* br = Bm + (size_t)b * N;
    const float* cr = Cm + (size_t)b * N;
    float* hr = h + ch * N;
#pragma unroll 4
    for (int n = q; n < N; n += LPC) {
      const float v = __builtin_fmaf(exp2_hw(-dtv * kLog2e * softplus_hw(ar[n])), hr[n],
                                     br[n] * bx);
      hr[n] = v;
      part = __builtin_fmaf(cr[n], v, part);
    }
  }
  part = group_sum<LPC>(part);
  if (valid && q == 0) {
    const float zv = z[ch];
    g[ch] = (part + dskip[(int)(ch % D)]) * (zv * sigmoid_f(zv));
  }
}

}  // namespace mhs
