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
// wave at the end, in a fixed order.
#pragma once

#include "mhs_common.hpp"
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

// What the product's element (weight row n, batch row b) becomes.
template <int KIND>
__device__ __forceinline__ void decode_store(const DecodeArgs& a, int b, int n, float v) {
  if constexpr (KIND == kDecIn) {
    if (n >= a.D) {
      a.out2[(size_t)b * a.D + n - a.D] = v;
      return;
    }
    float pre = a.conv_b[n];
    const float* win = a.conv + b * a.conv_sb + n * a.conv_sd;
    float* next = a.conv_next + ((size_t)b * a.D + n) * (a.taps - 1);
    const float* cw = a.conv_w + (size_t)n * a.taps;
    for (int k = 0; k < a.taps - 1; ++k) {
      const float t = win[k * a.conv_sk];
      pre = __builtin_fmaf(cw[k], t, pre);
      if (k > 0) next[k - 1] = t;
    }
    next[a.taps - 2] = v;
    pre = __builtin_fmaf(cw[a.taps - 1], v, pre);
    a.out[(size_t)b * a.D + n] = pre * sigmoid_f(pre);
  } else if constexpr (KIND == kDecProj) {
    if (n < a.D) {
      a.out[(size_t)b * a.D + n] = gate_dt(v + a.bias[n], a.dt_lo, a.dt_span);
    } else {
      const int c = n - a.D >= a.N;
      a.out2[((size_t)c * a.batch + b) * a.N + n - a.D - c * a.N] = v;
    }
  } else if constexpr (KIND == kDecOut) {
    a.out[(size_t)b * a.rows + n] = a.res[(size_t)b * a.rows + n] + v;
  } else {
    a.out[(size_t)b * a.rows + n] = v;
  }
}

// rows of the weight: wave (blockIdx.x * 4 + wave) takes RW of them. K a
// multiple of 4, pointers 16-byte aligned.
template <int KIND, int NB, int RW>
__global__ void __launch_bounds__(256) decode_product_kernel(DecodeArgs a) {
  constexpr bool NORM = KIND == kDecIn || KIND == kDecHead;
  constexpr int U = 2;   // 16-byte loads of a row in flight per lane and pass
  const int lane = threadIdx.x & 63;
  const int n0 = (blockIdx.x * 4 + __builtin_amdgcn_readfirstlane(threadIdx.x >> 6)) * RW;
  if (n0 >= a.rows) return;   // whole waves
  const int K4 = a.K >> 2;
  const float4* wr[RW];
#pragma unroll
  for (int r = 0; r < RW; ++r) {
    const int n = min(n0 + r, a.rows - 1);
    const float* p = a.w + (size_t)n * a.K;
    if constexpr (KIND == kDecProj) {
      if (n >= a.D + a.N) p = a.w_c + (size_t)(n - a.D - a.N) * a.K;
      else if (n >= a.D) p = a.w_b + (size_t)(n - a.D) * a.K;
    }
    wr[r] = reinterpret_cast<const float4*>(p);
  }
  for (int b0 = 0; b0 < a.batch; b0 += NB) {
    float acc[RW][NB], ss[NB];
#pragma unroll
    for (int b = 0; b < NB; ++b) {
      ss[b] = 0.f;
#pragma unroll
      for (int r = 0; r < RW; ++r) acc[r][b] = 0.f;
    }
    for (int c = 0; c < K4; c += 64 * U) {
      float4 wv[U][RW], nv[U];
#pragma unroll
      for (int u = 0; u < U; ++u) {
        const int i = c + 64 * u + lane;
#pragma unroll
        for (int r = 0; r < RW; ++r) wv[u][r] = i < K4 ? wr[r][i] : f4_zero();
        if constexpr (NORM)
          nv[u] = i < K4 ? reinterpret_cast<const float4*>(a.norm_w)[i] : f4_zero();
      }
#pragma unroll
      for (int u = 0; u < U; ++u) {
        const int i = c + 64 * u + lane;
#pragma unroll
        for (int b = 0; b < NB; ++b) {
          float4 xv = i < K4 && b0 + b < a.batch
                          ? reinterpret_cast<const float4*>(a.x + (size_t)(b0 + b) * a.K)[i]
                          : f4_zero();
          if constexpr (NORM) {
            ss[b] = dot4(xv, xv, ss[b]);
            xv = make_float4(xv.x * nv[u].x, xv.y * nv[u].y, xv.z * nv[u].z, xv.w * nv[u].w);
          }
#pragma unroll
          for (int r = 0; r < RW; ++r) acc[r][b] = dot4(wv[u][r], xv, acc[r][b]);
        }
      }
    }
    // Lane r * NB + b takes element (n0 + r, b0 + b).
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
    const int r = lane / NB, b = b0 + lane % NB;
    if (lane < RW * NB && n0 + r < a.rows && b < a.batch) decode_store<KIND>(a, b, n0 + r, mine);
  }
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
      const float v = __builtin_fmaf(exp2_hw(-dtv * kLog2e * softplus_f(ar[n])), hr[n],
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
