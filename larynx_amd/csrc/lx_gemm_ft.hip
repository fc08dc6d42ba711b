// Split-operand GEMM past the few-row kernel's tiles (lx_gemm_fs.hip): operands in
// MFMA fragment order, staged through LDS in large tiles.
//
// The arithmetic of gemm_bx_kernel with three products (two bf16 parts per operand,
// v_mfma_f32_32x32x16_bf16, fp32 accumulation), for activations written in fragment
// order by their producers (LX_ACT_FRAG2).  That kernel streams every wave's W columns
// from L2 once per 64-row tile.  Here 2 x 2 waves of (32 RB) x (32 CB) outputs share
// both operands in LDS, in tiles of 128 x 128, 128 x 64 or (the LM's q|k|v, a head per
// wave) 64 x 128, and 1 KB fragments go global -> registers -> LDS -> registers in lane
// order, with no address arithmetic, split or bank conflict on the way.  Two workgroups
// (64 KB of LDS each at most) share a CU and cover each other's barriers.  W is the
// MFMA's A operand: a lane's accumulator quad is four consecutive columns of one row,
// and the epilogue works on float4 straight from the accumulators.
//
// It runs the LM prefill's gate/up past 64 rows, down_proj past 128, q|k|v past 896 and
// o_proj past 1152, the estimator's q|k|v at 321-512 rows and FF0 of an MLP wider than
// 2048.  With cold weights: gate/up L = 256 31.4 -> 25.7 us, L = 1531 99.9 -> 96.0; down_proj
// L = 1531, three K slices, 63.7 -> 42.4.  Under counters the L = 1531 launches keep the
// matrix pipe 0.52-0.54 and the LDS 0.36 busy at a clock of 1.7 GHz; at L = 256 (152 tiles,
// one workgroup on 152 of 256 CUs) 0.24 and 0.17 at 2.0: a wave per SIMD waiting.
#include <algorithm>

#include "lx_common.hpp"
#include "lx_gemm_frag.hpp"
#include "lx_internal.hpp"

namespace lx {
namespace {

template <int EPI, int RB, int CB, int KSL, int OUT>
__global__ __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(2, 2))) void
gemm_ft_kernel(FsArgs a, EpiArgs ep) {
  constexpr int NP = 3, NPL = 2;
  constexpr int CA = 2 * RB * KSL * NPL, CW = 2 * CB * KSL * NPL;  // 1 KB chunks per slab
  constexpr int LA = CA / 4, LW = CW / 4;                          // per wave
  static_assert(LA * 4 == CA && LW * 4 == CW, "chunks split evenly over the waves");
  constexpr int SLAB = (CA + CW) * 64;  // 16-byte slots per LDS buffer
  extern __shared__ __attribute__((aligned(16))) uintx4_t sm4[];
  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int wm = wave & 1, wn = wave >> 1;
  const int r = lane & 31, h = lane >> 5;
  // each XCD (workgroups are dealt to them round-robin) takes a contiguous run of
  // (slice, N tile, M tile): its L2 keeps the W columns and meets each A tile once
  // per N tile
  int w = blockIdx.x;
  {
    const int full = gridDim.x / 8 * 8;
    if (w < full) w = (w % 8) * (full / 8) + w / 8;
  }
  const int mt = w % a.tiles_m, rest = w / a.tiles_m;
  const int nt = rest % a.tiles_n, slice = rest / a.tiles_n;
  const int nks = a.K / 16, nslab = nks / KSL;
  const int s0 = (int)((long)slice * nslab / a.slices);
  const int s1 = (int)((long)(slice + 1) * nslab / a.slices);
  const int nrb = (a.M + 31) / 32;
  const __amdgpu_buffer_rsrc_t ars = __builtin_amdgcn_make_buffer_rsrc(
      const_cast<void*>(a.A), (short)0, (int)a.a_bytes, 0x00020000);
  const __amdgpu_buffer_rsrc_t wrs = __builtin_amdgcn_make_buffer_rsrc(
      const_cast<void*>(a.Wf), (short)0, (int)a.w_bytes, 0x00020000);
  // This wave's chunks: A chunk c is (row block, k step, part), W chunk c likewise
  // with three parts per k step in memory.  Row blocks past the last repeat it.
  int ca[LA], cw[LW];
#pragma unroll
  for (int j = 0; j < LA; ++j) {
    const int c = wave * LA + j, rb = c / (KSL * NPL), kp = c % (KSL * NPL);
    ca[j] = (min(mt * 2 * RB + rb, nrb - 1) * nks * NPL + kp) * 1024;
  }
#pragma unroll
  for (int j = 0; j < LW; ++j) {
    const int c = wave * LW + j, cb = c / (KSL * NPL), kp = c % (KSL * NPL);
    cw[j] = ((nt * 2 * CB + cb) * nks * 3 + kp / NPL * 3 + kp % NPL) * 1024;
  }
  const int vl = lane * 16;
  auto load = [&](uintx4_t* ga, uintx4_t* gw, int s) {
#pragma unroll
    for (int j = 0; j < LA; ++j)
      ga[j] = __builtin_amdgcn_raw_buffer_load_b128(ars, vl, ca[j] + s * (KSL * NPL * 1024), 0);
#pragma unroll
    for (int j = 0; j < LW; ++j)
      gw[j] = __builtin_amdgcn_raw_buffer_load_b128(wrs, vl, cw[j] + s * (KSL * 3072), 0);
  };
  auto store = [&](const uintx4_t* ga, const uintx4_t* gw, int buf) {
    uintx4_t* d = sm4 + buf * SLAB + lane;
#pragma unroll
    for (int j = 0; j < LA; ++j) d[(wave * LA + j) * 64] = ga[j];
#pragma unroll
    for (int j = 0; j < LW; ++j) d[(CA + wave * LW + j) * 64] = gw[j];
  };
  constexpr int kPa[NP] = {1, 0, 0}, kPw[NP] = {0, 1, 0};
  floatx16 acc[RB][CB];
#pragma unroll
  for (int b = 0; b < RB; ++b)
#pragma unroll
    for (int c = 0; c < CB; ++c)
#pragma unroll
      for (int e = 0; e < 16; ++e) acc[b][c][e] = 0.0f;
  struct Frag {
    uintx4_t a[RB][NPL], w[CB][NPL];
  };
  auto read = [&](Frag& f, int b, int k) {
    const uintx4_t* base = sm4 + b * SLAB + lane;
#pragma unroll
    for (int c = 0; c < CB; ++c)
#pragma unroll
      for (int p = 0; p < NPL; ++p)
        f.w[c][p] = base[(CA + ((wn * CB + c) * KSL + k) * NPL + p) * 64];
#pragma unroll
    for (int i = 0; i < RB; ++i)
#pragma unroll
      for (int p = 0; p < NPL; ++p) f.a[i][p] = base[(((wm * RB + i) * KSL + k) * NPL + p) * 64];
  };
  auto mul = [&](const Frag& f) {
#pragma unroll
    for (int q = 0; q < NP; ++q)
#pragma unroll
      for (int i = 0; i < RB; ++i)
#pragma unroll
        for (int c = 0; c < CB; ++c)
          acc[i][c] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(
              frag_bf(f.w[c][kPw[q]]), frag_bf(f.a[i][kPa[q]]), acc[i][c], 0, 0, 0);
  };
  static_assert(KSL == 2, "two k steps per slab");
  constexpr int NM = NP * RB * CB, NR = NPL * (RB + CB), NL = LA + LW;
  constexpr int NST = 2;  // staging register sets: slab t in set t % NST
  const int last = s1 - 1;
  uintx4_t ga[NST][LA], gw[NST][LW];
  Frag f0, f1;
  load(ga[0], gw[0], s0);
  load(ga[1], gw[1], min(s0 + 1, last));
  store(ga[0], gw[0], 0);
  load(ga[0], gw[0], min(s0 + NST, last));
  __syncthreads();
  read(f0, 0, 0);
  // Slab s (LDS buffer b = s % 2).  First k step: its MFMAs, beside them the
  // fragment reads of the second and the staging of slab s + 1 into the other
  // buffer (every wave is past its reads of slab s - 1 there).  Barrier.  Second
  // k step: beside its MFMAs the first fragments of slab s + 1 and the request
  // of slab s + 1 + NST into the staging registers just stored.  (Loads past the range
  // repeat the last slab, stored to a buffer nobody reads.)
  auto body = [&](int s, int b) {
    read(f1, b, 1);
    store(ga[(b ^ 1) % NST], gw[(b ^ 1) % NST], b ^ 1);
    mul(f0);
#pragma unroll
    for (int k = 0; k < NR; ++k) {
      __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);  // MFMA
      __builtin_amdgcn_sched_group_barrier(0x100, 1, 0);  // DS read
      if (k < NL) __builtin_amdgcn_sched_group_barrier(0x200, 1, 0);  // DS write
    }
    if (NL > NR) __builtin_amdgcn_sched_group_barrier(0x200, NL - NR, 0);
    __builtin_amdgcn_sched_group_barrier(0x008, NM - NR, 0);
    __builtin_amdgcn_sched_barrier(0);
    __syncthreads();
    __builtin_amdgcn_sched_barrier(0);
    read(f0, b ^ 1, 0);
    load(ga[(b ^ 1) % NST], gw[(b ^ 1) % NST], min(s + 1 + NST, last));
    mul(f1);
#pragma unroll
    for (int k = 0; k < NR; ++k) {
      __builtin_amdgcn_sched_group_barrier(0x008, 1, 1);
      __builtin_amdgcn_sched_group_barrier(0x100, 1, 1);
      if (k < NL) __builtin_amdgcn_sched_group_barrier(0x020, 1, 1);  // VMEM read
    }
    if (NL > NR) __builtin_amdgcn_sched_group_barrier(0x020, NL - NR, 1);
    __builtin_amdgcn_sched_group_barrier(0x008, NM - NR, 1);
    __builtin_amdgcn_sched_barrier(0);
  };
  int s = s0;
  for (; s + 1 < s1; s += 2) {
    body(s, 0);
    body(s + 1, 1);
  }
  if (s < s1) body(s, 0);
  // element 4 q + e of lane l in block (i, c): row 32 i + l % 32, column
  // 32 c + 8 q + (l / 32) * 4 + e
  const int mb = (mt * 2 + wm) * RB * 32 + r, n0 = (nt * 2 + wn) * CB * 32;
  auto quad = [&](int i, int c, int q) {
    return floatx4{acc[i][c][4 * q], acc[i][c][4 * q + 1], acc[i][c][4 * q + 2],
                   acc[i][c][4 * q + 3]};
  };
#pragma unroll
  for (int i = 0; i < RB; ++i) {
    const int m = mb + i * 32;
    if (m >= a.M) continue;
    if constexpr (EPI == kEpiNeox) {
      static_assert(CB == 2, "a head per wave");
#pragma unroll
      for (int q = 0; q < 4; ++q)
        fs_neox(a, m, n0, q * 8 + h * 4, quad(i, 0, q), quad(i, CB - 1, q),
                fs_neox_load(a, ep, m, n0, q * 8 + h * 4));
    } else {
#pragma unroll
      for (int c = 0; c < CB; ++c)
#pragma unroll
        for (int q = 0; q < 4; ++q) {
          const int n = n0 + c * 32 + q * 8 + h * 4;
          fs_epilogue<EPI, OUT, NPL>(a, ep, slice, m, n, h, quad(i, c, q),
                                     fs_epi_load<EPI, OUT>(a, ep, m, n));
        }
    }
  }
}

template <int EPI, int RB, int CB, int KSL, int OUT>
int launch_ft(const FsArgs& a, const EpiArgs& ep, hipStream_t s) {
  auto kern = gemm_ft_kernel<EPI, RB, CB, KSL, OUT>;
  static LdsLimit once;
  const size_t lds = (size_t)2 * 2 * (RB + CB) * KSL * 2 * 1024;
  int rc = raise_lds_limit((const void*)kern, lds, once, "linear_ft");
  if (rc) return rc;
  hipLaunchKernelGGL(kern, dim3((unsigned)(a.tiles_m * a.tiles_n * a.slices)), dim3(256), lds, s,
                     a, ep);
  return check_launch("gemm_ft_kernel");
}

template <int RB, int CB>
int dispatch_ft(const FsArgs& a, int out, const EpiArgs& ep, hipStream_t s) {
  if (out == FS_OUT_PARTIAL) return launch_ft<LX_EPI_NONE, RB, CB, 2, FS_OUT_PARTIAL>(a, ep, s);
  if (out == FS_OUT_FRAG) {
    if (ep.kind == LX_EPI_GELU_TANH)
      return launch_ft<LX_EPI_GELU_TANH, RB, CB, 2, FS_OUT_FRAG>(a, ep, s);
    return launch_ft<LX_EPI_SWIGLU_PAIRED, RB, CB, 2, FS_OUT_FRAG>(a, ep, s);
  }
  if (ep.kind == LX_EPI_RESID) return launch_ft<LX_EPI_RESID, RB, CB, 2, FS_OUT_F32>(a, ep, s);
  set_error("linear_ft: epilogue kind %d not available", ep.kind);
  return LX_ERR_ARG;
}

}  // namespace

// Tiles of 128 x 128 or 128 x 64 (kFtWideTiles).  The LM's q|k|v takes 64 x 128, a head per
// wave; the estimator's rotary q|k|v 128 x 64 (at most 512 rows: 96 tiles of 128 x 128).
int linear_ft(FsArgs a, int out, const EpiArgs& ep, hipStream_t s) {
  auto tiles = [&](int rb, int cb) {
    a.tiles_m = (a.M + 64 * rb - 1) / (64 * rb);
    a.tiles_n = a.N / (64 * cb);
  };
  if (ep.kind == kEpiNeox) {
    tiles(1, 2);
    return launch_ft<kEpiNeox, 1, 2, 2, FS_OUT_F32>(a, ep, s);
  }
  if (ep.kind == LX_EPI_ROPE_PARTIAL) {
    tiles(2, 1);
    return launch_ft<LX_EPI_ROPE_PARTIAL, 2, 1, 2, FS_OUT_F32>(a, ep, s);
  }
  tiles(2, 2);
  if ((long)a.tiles_m * a.tiles_n * a.slices >= kFtWideTiles * device_cus() / 256)
    return dispatch_ft<2, 2>(a, out, ep, s);
  tiles(2, 1);
  return dispatch_ft<2, 1>(a, out, ep, s);
}

}  // namespace lx
