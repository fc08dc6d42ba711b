// Shared pieces of the GEMMs on fragment-order operands (lx_gemm_fs.hip,
// lx_gemm_ft.hip): arguments, and the epilogues on an accumulator quad.
#pragma once

#include "lx_common.hpp"
#include "lx_gemm_common.hpp"
#include "lx_internal.hpp"

namespace lx {

struct FsArgs {
  const void* A;  // fragment order, or fp32 rows (lda)
  long lda;
  unsigned a_bytes;
  const void* Wf;  // wfrag_pack
  unsigned w_bytes;
  const float* bias;
  float* Y;
  long ldy, slice_stride;
  int M, N, K, tiles_m, tiles_n, slices;
  // kEpiNeox (q|k|v heads of 64): rotary on the first rope_heads heads, q columns
  // to Y, the k and v columns to the caches' row m
  int q_cols, kv_cols, rope_heads;
  const float* rope_cs;  // per position 32 cosines, then 32 sines
  float *k_cache, *v_cache;
};

constexpr int kEpiNeox = 100;  // internal epilogue beside LX_EPI_*
// Fewest 128 x 128 tiles (times K slices) per 256 CUs that linear_ft runs as such, else 128
// x 64 (M = 1000, N = 3072: 192 tiles 27.8 against 32.2 us; M = 256, N = 9728: 152 tiles
// 25.5 / 31.3; M = 1000, N = 2048: 128 tiles 26.0 / 21.6).
constexpr int kFtWideTiles = 150;

// lx_linear_bx of few rows (fp32 or packed, fp32 or packed output, one slice, arguments
// checked) on the few-row kernel; the choice depends on the shape alone, so fp32 and
// packed operands give the same bits.  false: not taken.
bool linear_fs_rows(const lx_linear_bx& g, const EpiArgs& ep, hipStream_t stream, int* rc);
// Three products; outputs and epilogues as linear_fs, without the gated residual.
int linear_ft(FsArgs a, int out, const EpiArgs& ep, hipStream_t s);

__device__ __forceinline__ sbf16x8 frag_bf(uintx4_t v) { return __builtin_bit_cast(sbf16x8, v); }

// What the epilogue of columns n .. n + 3 of row m reads: bias, gate, the residual
// and the rotary angles.  Loaded ahead of the K loop where registers allow.
struct FsEpiIn {
  float4 b, g, y;
  float a0, a1;
};
template <int EPI, int OUT>
__device__ __forceinline__ FsEpiIn fs_epi_load(const FsArgs& a, const EpiArgs& ep, int m, int n) {
  FsEpiIn in;
  in.b = in.g = in.y = make_float4(0.f, 0.f, 0.f, 0.f);
  in.a0 = in.a1 = 0.0f;
  if (OUT == FS_OUT_PARTIAL) return in;
  if (a.bias) in.b = *reinterpret_cast<const float4*>(a.bias + n);
  if (EPI == LX_EPI_GATED_RESID)
    in.g = *reinterpret_cast<const float4*>(ep.gate + (long)(m / ep.rows_per_batch) *
                                                          ep.gate_stride + n);
  if (EPI == LX_EPI_GATED_RESID || EPI == LX_EPI_RESID)
    in.y = *reinterpret_cast<const float4*>(a.Y + (long)m * a.ldy + n);
  if (EPI == LX_EPI_ROPE_PARTIAL && n < ep.sections * ep.section &&
      n % ep.section < ep.rot_dim) {
    const float p = (float)ep.pos[m % ep.rows_per_batch];
    const int i = (n % ep.section) >> 1;
    in.a0 = p * ep.inv_freq[i];
    in.a1 = p * ep.inv_freq[i + 1];
  }
  return in;
}

// Columns n .. n + 3 of row m (lane half h): v = the raw products.
template <int EPI, int OUT, int NPL>
__device__ __forceinline__ void fs_epilogue(const FsArgs& a, const EpiArgs& ep, int slice, int m,
                                            int n, int h, floatx4 v, const FsEpiIn& in) {
  if constexpr (OUT == FS_OUT_PARTIAL) {
    *reinterpret_cast<floatx4*>(a.Y + slice * a.slice_stride + (long)m * a.ldy + n) = v;
    return;
  }
  floatx4 o = {v[0] + in.b.x, v[1] + in.b.y, v[2] + in.b.z, v[3] + in.b.w};
  if constexpr (EPI == LX_EPI_SWIGLU_PAIRED) {
    // two outputs; lanes l and l + 32 hold neighbouring pairs of the same row
    // (so they are active together), joined by the lower lane
    static_assert(OUT == FS_OUT_FRAG, "SwiGLU feeds the next projection");
    const float g0 = (o[0] / (1.0f + expf(-o[0]))) * o[1];
    const float g1 = (o[2] / (1.0f + expf(-o[2]))) * o[3];
    const float t0 = lane_xor32(g0), t1 = lane_xor32(g1);
    if (h == 0)
      frag_store4<NPL>(reinterpret_cast<__bf16*>(a.Y), m, n >> 1, a.N / 32,
                       floatx4{g0, g1, t0, t1});
    return;
  }
  if (EPI == LX_EPI_GELU_TANH)
#pragma unroll
    for (int e = 0; e < 4; ++e) o[e] = gelu_tanh(o[e]);
  if (EPI == LX_EPI_GATED_RESID)
    o = floatx4{in.y.x + o[0] * in.g.x, in.y.y + o[1] * in.g.y, in.y.z + o[2] * in.g.z,
                in.y.w + o[3] * in.g.w};
  if (EPI == LX_EPI_RESID)
    o = floatx4{in.y.x + o[0], in.y.y + o[1], in.y.z + o[2], in.y.w + o[3]};
  if (EPI == LX_EPI_ROPE_PARTIAL && n < ep.sections * ep.section &&
      n % ep.section < ep.rot_dim) {
    float x0 = o[0], x1 = o[1], x2 = o[2], x3 = o[3];
    rotate_pair(x0, x1, in.a0);
    rotate_pair(x2, x3, in.a1);
    o = floatx4{x0, x1, x2, x3};
  }
  if constexpr (OUT == FS_OUT_FRAG)
    frag_store4<NPL>(reinterpret_cast<__bf16*>(a.Y), m, n, a.N / 16, o);
  else if (OUT == FS_OUT_PACKED && n >= ep.pack_from)
    *reinterpret_cast<uintx4_t*>(a.Y + (long)m * a.ldy + n) = pack2_bf16(o);
  else
    *reinterpret_cast<floatx4*>(a.Y + (long)m * a.ldy + n) = o;
}

// The LM's q|k|v: channels c .. c + 3 (x0) and c + 32 .. (x1) of the head at
// column n0 of row m; bias, NEOX rotary, and q to Y, k / v to the caches.
struct FsNeoxIn {
  floatx4 b0, b1, co, si;
};
__device__ __forceinline__ FsNeoxIn fs_neox_load(const FsArgs& a, const EpiArgs& ep, int m, int n0,
                                                 int c) {
  FsNeoxIn in;
  const float* cs = a.rope_cs + (long)ep.pos[m] * 64 + c;
  in.b0 = *reinterpret_cast<const floatx4*>(a.bias + n0 + c);
  in.b1 = *reinterpret_cast<const floatx4*>(a.bias + n0 + 32 + c);
  in.co = *reinterpret_cast<const floatx4*>(cs);
  in.si = *reinterpret_cast<const floatx4*>(cs + 32);
  return in;
}
__device__ __forceinline__ void fs_neox(const FsArgs& a, int m, int n0, int c, floatx4 x0,
                                        floatx4 x1, const FsNeoxIn& in) {
  x0 += in.b0;
  x1 += in.b1;
  if (n0 / 64 < a.rope_heads) {
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      const float y0 = x0[e], y1 = x1[e];
      x0[e] = y0 * in.co[e] - y1 * in.si[e];
      x1[e] = y1 * in.co[e] + y0 * in.si[e];
    }
  }
  float* dst = n0 < a.q_cols ? a.Y + (long)m * a.ldy + n0
               : n0 < a.q_cols + a.kv_cols
                   ? a.k_cache + (long)m * a.kv_cols + (n0 - a.q_cols)
                   : a.v_cache + (long)m * a.kv_cols + (n0 - a.q_cols - a.kv_cols);
  *reinterpret_cast<floatx4*>(dst + c) = x0;
  *reinterpret_cast<floatx4*>(dst + 32 + c) = x1;
}

}  // namespace lx
