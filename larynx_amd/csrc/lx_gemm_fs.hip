// Split-operand GEMM for few rows: both operands streamed in MFMA fragment
// order, K split over the waves of a workgroup.
//
// The arithmetic of gemm_bx_kernel (operands as two or three bf16 parts, three
// or six products on v_mfma_f32_32x32x16_bf16, fp32 accumulation).  With few
// rows that kernel has too few tiles for the device (M = 148, N = 3072: 72
// workgroups) and each walks K behind a barrier per 32-wide slab, so a launch
// waits on memory latency.  Here a workgroup of KW waves owns a tile of RB x CB
// 32 x 32 blocks; wave w computes the whole tile over the w-th of KW K ranges.
// Activations (LX_ACT_FRAG*, or fp32 rows split in registers) and weights
// (wfrag_pack) both arrive as whole fragments by coalesced 16-byte loads, D k
// steps ahead in a register ring, with no LDS and no barrier in the K loop.  The
// KW partial tiles meet in LDS once and are summed in wave order, so a result
// does not depend on timing.  W is the MFMA's A operand: a lane's accumulator
// quad is four consecutive columns of one output row, so the epilogue works on
// float4 straight from the sum.
#include <algorithm>

#include "lx_gemm_frag.hpp"

namespace lx {
namespace {

constexpr unsigned kOob = 1u << 31;  // past every operand (all are below 2 GiB): loads give zero

// A operand: fp32 rows (split in registers), fragment order, two-part packed rows
// (three products).  The last two hold the same parts as the first splits into.
enum { kARows = 0, kAFrag = 1, kAPacked = 2 };

template <int RB, int CB, int NP>
constexpr int fs_depth() {
  constexpr int NPL = NP == 6 ? 3 : 2;
  constexpr int d = (208 - 16 * RB * CB) / (4 * NPL * (RB + CB));
  return d > 8 ? 8 : d;
}

// The bf16 parts of eight fp32 values, as fragments.
template <int NPL>
__device__ __forceinline__ void fs_split(uintx4_t lo, uintx4_t hi, uintx4_t* f) {
  floatx4 v[2] = {__builtin_bit_cast(floatx4, lo), __builtin_bit_cast(floatx4, hi)};
#pragma unroll
  for (int e = 0; e < 2; ++e) {
#pragma unroll
    for (int p = 0; p < NPL; ++p) {
      const bf16x4_t x = __builtin_convertvector(v[e], bf16x4_t);
      const uintx2_t u = __builtin_bit_cast(uintx2_t, x);
      f[p][2 * e] = u[0];
      f[p][2 * e + 1] = u[1];
      if (p + 1 < NPL) v[e] = v[e] - bf16x4_back(x);
    }
  }
}

template <int EPI, int RB, int CB, int KW, int OUT, int NP, int AF>
__global__ __launch_bounds__(64 * KW) __attribute__((amdgpu_waves_per_eu(2, 2))) void
gemm_fs_kernel(FsArgs a, EpiArgs ep) {
  constexpr int NPL = NP == 6 ? 3 : 2;
  constexpr int D = fs_depth<RB, CB, NP>();
  constexpr int AV = AF == kAFrag ? NPL : 2;  // 16-byte loads per A fragment set
  extern __shared__ __attribute__((aligned(16))) float red[];  // [KW][RB * CB * 4][64] float4
  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int r = lane & 31, h = lane >> 5;
  // the dispatcher deals workgroups round-robin over the 8 XCDs: a contiguous
  // run of (slice, N tile, M tile) each, so an XCD's L2 reads its W columns once
  int w = blockIdx.x;
  {
    const int full = gridDim.x / 8 * 8;
    if (w < full) w = (w % 8) * (full / 8) + w / 8;
  }
  const int mt = w % a.tiles_m, rest = w / a.tiles_m;
  const int nt = rest % a.tiles_n, slice = rest / a.tiles_n;
  const int nks = a.K / 16;
  const int parts = a.slices * KW, part = slice * KW + wave;
  const int k0 = (int)((long)part * nks / parts), k1 = (int)((long)(part + 1) * nks / parts);
  const int n = k1 - k0;
  const int rb0 = mt * RB, n0 = nt * CB * 32;

  const __amdgpu_buffer_rsrc_t ars = __builtin_amdgcn_make_buffer_rsrc(
      const_cast<void*>(a.A), (short)0, (int)a.a_bytes, 0x00020000);
  const __amdgpu_buffer_rsrc_t wrs = __builtin_amdgcn_make_buffer_rsrc(
      const_cast<void*>(a.Wf), (short)0, (int)a.w_bytes, 0x00020000);
  // lane offsets at k step 0; row blocks past the last read zeros
  unsigned oa[RB], ow[CB];
  const int nrb = (a.M + 31) / 32;
#pragma unroll
  for (int i = 0; i < RB; ++i) {
    if (AF == kAFrag)
      oa[i] = rb0 + i < nrb ? (unsigned)(rb0 + i) * nks * (NPL * 1024) + lane * 16 : kOob;
    else
      oa[i] = (unsigned)min((rb0 + i) * 32 + r, a.M - 1) * (unsigned)(a.lda * 4) + h * 32;
  }
#pragma unroll
  for (int c = 0; c < CB; ++c) ow[c] = (unsigned)(n0 / 32 + c) * nks * 3072 + lane * 16;

  uintx4_t fa[D][RB][AV], fw[D][CB][NPL];
  auto load = [&](int i, int s) {  // k step k0 + s into ring slot i; past the range: no access
    const unsigned past = s < n ? 0u : kOob;
    const int sa = (k0 + s) * (AF == kAFrag ? NPL * 1024 : 64), sw = (k0 + s) * 3072;
#pragma unroll
    for (int c = 0; c < CB; ++c)
#pragma unroll
      for (int p = 0; p < NPL; ++p)
        fw[i][c][p] =
            __builtin_amdgcn_raw_buffer_load_b128(wrs, (ow[c] + sw + p * 1024) | past, 0, 0);
#pragma unroll
    for (int b = 0; b < RB; ++b)
#pragma unroll
      for (int p = 0; p < AV; ++p)
        fa[i][b][p] = __builtin_amdgcn_raw_buffer_load_b128(
            ars, (oa[b] + sa + p * (AF == kAFrag ? 1024 : 16)) | past, 0, 0);
  };
  constexpr int kPa6[6] = {2, 1, 0, 1, 0, 0}, kPw6[6] = {0, 1, 2, 0, 1, 0};
  constexpr int kPa3[3] = {1, 0, 0}, kPw3[3] = {0, 1, 0};
  floatx16 acc[RB][CB];
#pragma unroll
  for (int b = 0; b < RB; ++b)
#pragma unroll
    for (int c = 0; c < CB; ++c)
#pragma unroll
      for (int e = 0; e < 16; ++e) acc[b][c][e] = 0.0f;
#pragma unroll
  for (int i = 0; i < D; ++i) load(i, i);
  // One epilogue quad per wave: its operands are requested behind the first
  // fragments, so the epilogue waits on no load of its own.
  constexpr int SL = RB * CB * 4;
  constexpr bool PRE = SL == KW && EPI != kEpiNeox;
  FsEpiIn pre;
  FsNeoxIn npre;
  if constexpr (EPI == kEpiNeox) {
    static_assert(RB * 4 == KW, "one quad per wave");
    npre = fs_neox_load(a, ep, min(rb0 * 32 + (wave >> 2) * 32 + r, a.M - 1), n0,
                        (wave & 3) * 8 + h * 4);
  }
  if constexpr (PRE)
    pre = fs_epi_load<EPI, OUT>(a, ep, min(rb0 * 32 + wave / (4 * CB) * 32 + r, a.M - 1),
                                n0 + wave % CB * 32 + (wave / CB & 3) * 8 + h * 4);
  for (int s = 0; s < n; s += D) {
#pragma unroll
    for (int i = 0; i < D; ++i) {  // (k steps past the range multiply zeros)
      uintx4_t f[RB][NPL];
#pragma unroll
      for (int b = 0; b < RB; ++b) {
        if (AF == kAFrag) {
#pragma unroll
          for (int p = 0; p < NPL; ++p) f[b][p] = fa[i][b][p];
        } else if (AF == kAPacked) {
#pragma unroll
          for (int p = 0; p < NPL; ++p) {
            const uintx4_t lo = fa[i][b][0], hi = fa[i][b][1];
            f[b][p] = uintx4_t{lo[2 * p], lo[2 * p + 1], hi[2 * p], hi[2 * p + 1]};
          }
        } else {
          fs_split<NPL>(fa[i][b][0], fa[i][b][1], f[b]);
        }
      }
#pragma unroll
      for (int q = 0; q < NP; ++q)
#pragma unroll
        for (int b = 0; b < RB; ++b)
#pragma unroll
          for (int c = 0; c < CB; ++c)
            acc[b][c] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(
                frag_bf(fw[i][c][NP == 6 ? kPw6[q] : kPw3[q]]),
                frag_bf(f[b][NP == 6 ? kPa6[q] : kPa3[q]]), acc[b][c], 0, 0, 0);
      load(i, s + i + D);
    }
  }
  // Partial tiles to LDS in accumulator order: element 4 q + e of lane l in block
  // (b, c) is row 32 b + l % 32, column 32 c + 8 q + (l / 32) * 4 + e.
  floatx4* part4 = reinterpret_cast<floatx4*>(red);
#pragma unroll
  for (int b = 0; b < RB; ++b)
#pragma unroll
    for (int c = 0; c < CB; ++c)
#pragma unroll
      for (int q = 0; q < 4; ++q)
        part4[(wave * SL + (b * 4 + q) * CB + c) * 64 + lane] =
            floatx4{acc[b][c][4 * q], acc[b][c][4 * q + 1], acc[b][c][4 * q + 2],
                    acc[b][c][4 * q + 3]};
  __syncthreads();
  auto total = [&](int slot) {
    floatx4 t = part4[slot * 64 + lane];
#pragma unroll
    for (int g = 1; g < KW; ++g) t += part4[(g * SL + slot) * 64 + lane];
    return t;
  };
  if constexpr (EPI == kEpiNeox) {
    // one head of 64 columns per tile: channels c and c + 32 are the two blocks'
    // elements of the same lane
    static_assert(CB == 2, "a head per tile");
    for (int u = wave; u < RB * 4; u += KW) {
      const floatx4 x0 = total(u * CB), x1 = total(u * CB + 1);
      const int m = rb0 * 32 + (u >> 2) * 32 + r;
      if (m < a.M) fs_neox(a, m, n0, (u & 3) * 8 + h * 4, x0, x1, npre);
    }
  } else {
    for (int slot = wave; slot < SL; slot += KW) {
      const floatx4 v = total(slot);
      const int m = rb0 * 32 + slot / (4 * CB) * 32 + r;
      const int nn = n0 + slot % CB * 32 + (slot / CB & 3) * 8 + h * 4;
      if (m >= a.M) continue;
      if constexpr (PRE)
        fs_epilogue<EPI, OUT, NPL>(a, ep, slice, m, nn, h, v, pre);
      else
        fs_epilogue<EPI, OUT, NPL>(a, ep, slice, m, nn, h, v,
                                   fs_epi_load<EPI, OUT>(a, ep, m, nn));
    }
  }
}

template <int EPI, int RB, int CB, int KW, int OUT, int NP, int AF>
int launch_fs(const FsArgs& a, const EpiArgs& ep, hipStream_t s) {
  auto kern = gemm_fs_kernel<EPI, RB, CB, KW, OUT, NP, AF>;
  static LdsLimit once;
  const size_t lds = (size_t)KW * RB * CB * 4096;
  int rc = raise_lds_limit((const void*)kern, lds, once, "linear_fs");
  if (rc) return rc;
  hipLaunchKernelGGL(kern, dim3((unsigned)(a.tiles_m * a.tiles_n * a.slices)), dim3(64 * KW), lds,
                     s, a, ep);
  return check_launch("gemm_fs_kernel");
}

// The modulated LayerNorm of the block input inside the projection that reads it, for
// launches of at most one workgroup per CU (three products, rows of 1024): a launch of
// its own costs 4.5 us at these sizes, nearly all of it latency.  Eight waves own a
// 32 x 64 tile, an eighth of K each.  Every workgroup normalises its 32 rows itself
// (four rows per wave, the arithmetic of adaln_kernel), splits them into fragments in LDS
// (128 KB; the 16-byte slots of a 32-row fragment are XOR-swizzled by k step and half, so
// that a row's 8-byte stores fall on all banks) and multiplies from there, while its
// first W fragments are on their way.  The partial tiles then reuse the LDS.  One
// evaluation at B = 2, T = 50 1406 -> 1299 us, T = 74 1468 -> 1303, T = 128 1785 -> 1434 (FF0's
// alone there).
constexpr int kLnK = 1024;

template <int EPI, int OUT>
__global__ __launch_bounds__(512) __attribute__((amdgpu_waves_per_eu(2, 2))) void
gemm_fs_ln_kernel(FsArgs a, EpiArgs ep, FsLn ln) {
  constexpr int KW = 8, CB = 2, NPL = 2, D = 4, NKS = kLnK / 16, NW = NKS / KW, NV = kLnK / 256;
  extern __shared__ __attribute__((aligned(16))) float red[];
  char* fl = reinterpret_cast<char*>(red);  // [NKS][NPL][64] 16-byte slots
  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int r = lane & 31, h = lane >> 5;
  int w = blockIdx.x;
  {
    const int full = gridDim.x / 8 * 8;
    if (w < full) w = (w % 8) * (full / 8) + w / 8;
  }
  const int mt = w % a.tiles_m, nt = w / a.tiles_m;
  const int m0 = mt * 32, n0 = nt * 64;
  // rows and the first row's modulation ahead of the weights (loads retire in order)
  floatx4 x[4][NV];
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    const floatx4* src = reinterpret_cast<const floatx4*>(
        ln.x + (long)min(m0 + wave + 8 * i, a.M - 1) * kLnK);
#pragma unroll
    for (int j = 0; j < NV; ++j) x[i][j] = src[lane + 64 * j];
  }
  int batch = min(m0 + wave, a.M - 1) / ln.T;
  floatx4 sc[NV], sh[NV];
  auto mods = [&](int b) {
#pragma unroll
    for (int j = 0; j < NV; ++j) {
      sc[j] = reinterpret_cast<const floatx4*>(ln.scale + b * ln.mod_stride)[lane + 64 * j];
      sh[j] = reinterpret_cast<const floatx4*>(ln.shift + b * ln.mod_stride)[lane + 64 * j];
    }
  };
  mods(batch);
  const __amdgpu_buffer_rsrc_t wrs = __builtin_amdgcn_make_buffer_rsrc(
      const_cast<void*>(a.Wf), (short)0, (int)a.w_bytes, 0x00020000);
  unsigned ow[CB];
#pragma unroll
  for (int c = 0; c < CB; ++c)
    ow[c] = (unsigned)((n0 / 32 + c) * NKS + wave * NW) * 3072 + lane * 16;
  uintx4_t fw[D][CB][NPL];
  auto load = [&](int i, int s) {
#pragma unroll
    for (int c = 0; c < CB; ++c)
#pragma unroll
      for (int p = 0; p < NPL; ++p)
        fw[i][c][p] =
            __builtin_amdgcn_raw_buffer_load_b128(wrs, ow[c] + s * 3072 + p * 1024, 0, 0);
  };
#pragma unroll
  for (int i = 0; i < D; ++i) load(i, i);
  // one epilogue quad per wave
  constexpr int SL = CB * 4;
  static_assert(SL == KW, "one quad per wave");
  const int em = m0 + r, en = n0 + wave % CB * 32 + (wave / CB & 3) * 8 + h * 4;
  const FsEpiIn pre = fs_epi_load<EPI, OUT>(a, ep, min(em, a.M - 1), en);
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    const int lr = wave + 8 * i, m = min(m0 + lr, a.M - 1);
    if (m / ln.T != batch) {  // wave-uniform
      batch = m / ln.T;
      mods(batch);
    }
    float sm = 0.0f;
#pragma unroll
    for (int j = 0; j < NV; ++j) sm += (x[i][j][0] + x[i][j][1]) + (x[i][j][2] + x[i][j][3]);
    const float mean = wave_sum(sm) / (float)kLnK;
    float q = 0.0f;
#pragma unroll
    for (int j = 0; j < NV; ++j) {
      const floatx4 d = x[i][j] - mean;
      q += (d[0] * d[0] + d[1] * d[1]) + (d[2] * d[2] + d[3] * d[3]);
    }
    const float rstd = 1.0f / sqrtf(wave_sum(q) / (float)kLnK + ln.eps);
#pragma unroll
    for (int j = 0; j < NV; ++j) {
      const floatx4 o = ((x[i][j] - mean) * rstd) * (1.0f + sc[j]) + sh[j];
      const int k4 = lane + 64 * j, ks = k4 >> 2, hh = (k4 >> 1) & 1;
      char* d = fl + ((ks * NPL) * 64 + hh * 32 + (lr ^ ((2 * ks + hh) & 31))) * 16 + (k4 & 1) * 8;
      const uintx4_t pk = pack2_bf16(o);
      *reinterpret_cast<uintx2_t*>(d) = uintx2_t{pk[0], pk[1]};
      *reinterpret_cast<uintx2_t*>(d + 1024) = uintx2_t{pk[2], pk[3]};
    }
  }
  __syncthreads();
  floatx16 acc[CB];
#pragma unroll
  for (int c = 0; c < CB; ++c)
#pragma unroll
    for (int e = 0; e < 16; ++e) acc[c][e] = 0.0f;
#pragma unroll
  for (int s = 0; s < NW; ++s) {
    const int ks = wave * NW + s;
    const char* src = fl + (ks * NPL * 64 + h * 32 + (r ^ ((2 * ks + h) & 31))) * 16;
    uintx4_t f[NPL];
#pragma unroll
    for (int p = 0; p < NPL; ++p) f[p] = *reinterpret_cast<const uintx4_t*>(src + p * 1024);
    constexpr int kPa[3] = {1, 0, 0}, kPw[3] = {0, 1, 0};
#pragma unroll
    for (int q = 0; q < 3; ++q)
#pragma unroll
      for (int c = 0; c < CB; ++c)
        acc[c] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(frag_bf(fw[s % D][c][kPw[q]]),
                                                         frag_bf(f[kPa[q]]), acc[c], 0, 0, 0);
    if (s + D < NW) load(s % D, s + D);
  }
  __syncthreads();  // every wave is past its fragments
  floatx4* part4 = reinterpret_cast<floatx4*>(red);
#pragma unroll
  for (int c = 0; c < CB; ++c)
#pragma unroll
    for (int q = 0; q < 4; ++q)
      part4[(wave * SL + q * CB + c) * 64 + lane] =
          floatx4{acc[c][4 * q], acc[c][4 * q + 1], acc[c][4 * q + 2], acc[c][4 * q + 3]};
  __syncthreads();
  floatx4 t = part4[wave * 64 + lane];
#pragma unroll
  for (int g = 1; g < KW; ++g) t += part4[(g * SL + wave) * 64 + lane];
  if (em < a.M) fs_epilogue<EPI, OUT, NPL>(a, ep, 0, em, en, h, t, pre);
}

template <int EPI, int OUT>
int launch_fs_ln(const FsArgs& a, const EpiArgs& ep, const FsLn& ln, hipStream_t s) {
  auto kern = gemm_fs_ln_kernel<EPI, OUT>;
  static LdsLimit once;
  constexpr size_t lds = (size_t)32 * kLnK * 4;
  const int rc = raise_lds_limit((const void*)kern, lds, once, "linear_fs_ln");
  if (rc) return rc;
  hipLaunchKernelGGL(kern, dim3((unsigned)(a.tiles_m * a.tiles_n)), dim3(512), lds, s, a, ep, ln);
  return check_launch("gemm_fs_ln_kernel");
}

template <int RB, int CB, int KW, int NP, int AF>
int dispatch_fs(FsArgs a, int out, const EpiArgs& ep, hipStream_t s) {
  a.tiles_m = (a.M + 32 * RB - 1) / (32 * RB);
  a.tiles_n = a.N / (32 * CB);
  // 64 x 64 tiles of fragment-order operands: no gated residual and, with six products,
  // no residual or partials (pick_fs)
  constexpr bool GATED = AF != kAFrag || RB == 1, RESID = GATED || NP == 3;
  if constexpr (AF == kAFrag) {
    if constexpr (RESID)
      if (out == FS_OUT_PARTIAL)
        return launch_fs<LX_EPI_NONE, RB, CB, KW, FS_OUT_PARTIAL, NP, AF>(a, ep, s);
    if (out == FS_OUT_FRAG) {
      if (ep.kind == LX_EPI_GELU_TANH)
        return launch_fs<LX_EPI_GELU_TANH, RB, CB, KW, FS_OUT_FRAG, NP, AF>(a, ep, s);
      return launch_fs<LX_EPI_SWIGLU_PAIRED, RB, CB, KW, FS_OUT_FRAG, NP, AF>(a, ep, s);
    }
  }
  if constexpr (AF != kAFrag) {
    if constexpr (NP == 3)
      if (out == FS_OUT_PACKED) {
        if (ep.kind == LX_EPI_ROPE_PARTIAL)
          return launch_fs<LX_EPI_ROPE_PARTIAL, RB, CB, KW, FS_OUT_PACKED, NP, AF>(a, ep, s);
        if (ep.kind == LX_EPI_GELU_TANH)
          return launch_fs<LX_EPI_GELU_TANH, RB, CB, KW, FS_OUT_PACKED, NP, AF>(a, ep, s);
        return launch_fs<LX_EPI_NONE, RB, CB, KW, FS_OUT_PACKED, NP, AF>(a, ep, s);
      }
    if (ep.kind == LX_EPI_NONE)
      return launch_fs<LX_EPI_NONE, RB, CB, KW, FS_OUT_F32, NP, AF>(a, ep, s);
    if (ep.kind == LX_EPI_GELU_TANH)
      return launch_fs<LX_EPI_GELU_TANH, RB, CB, KW, FS_OUT_F32, NP, AF>(a, ep, s);
  }
  switch (ep.kind) {
    case LX_EPI_ROPE_PARTIAL:
      return launch_fs<LX_EPI_ROPE_PARTIAL, RB, CB, KW, FS_OUT_F32, NP, AF>(a, ep, s);
    case LX_EPI_GATED_RESID:
      if constexpr (GATED)
        return launch_fs<LX_EPI_GATED_RESID, RB, CB, KW, FS_OUT_F32, NP, AF>(a, ep, s);
      break;
    case LX_EPI_RESID:
      if constexpr (RESID)
        return launch_fs<LX_EPI_RESID, RB, CB, KW, FS_OUT_F32, NP, AF>(a, ep, s);
      break;
    default: break;
  }
  set_error("linear_fs: epilogue kind %d not available", ep.kind);
  return LX_ERR_ARG;
}

// 32 x 32 tiles while they number at most two per CU, 64 x 64 tiles up to one per
// CU; past that (false) the tiled kernel, whose wide tiles re-read W less often.
// With cold weights, M = 148, N = 3072, K = 1024 (480 tiles) 12.7 us against 16.0 on
// gemm_bx_kernel; M = 300, N = 3072 (240 of 64 x 64) 14.9 against 17.6; M = 1000, N =
// 3072 (768 of 64 x 64) 32.1 against 27.8 on the tiled kernel.  Six products come with few
// rows only and stay here at any tile count (FF0 of F = 8192, 150 rows, 384 tiles: an
// evaluation of four blocks 604 -> 592 us against 128 x 64 tiled ones).  The gated residual
// (N = 1024, at most 512 rows: two 32 x 32 tiles per CU) and, with six products, the residual
// and the partials (the LM's o_proj and down_proj of at most 64 rows) keep 32 x 32 tiles.
template <int NP>
bool pick_fs(const FsArgs& a, int out, const EpiArgs& ep, hipStream_t s, int* rc) {
  const long nrb = (a.M + 31) / 32, cus = device_cus();
  if (ep.kind == kEpiNeox) {
    if (NP == 3 && nrb * (a.N / 64) > 2 * cus) return false;
    FsArgs b = a;
    b.tiles_m = (int)nrb;
    b.tiles_n = a.N / 64;
    *rc = launch_fs<kEpiNeox, 1, 2, 4, FS_OUT_F32, NP, 1>(b, ep, s);
    return true;
  }
  const bool fine = ep.kind == LX_EPI_GATED_RESID ||
                    (NP == 6 && (out == FS_OUT_PARTIAL || ep.kind == LX_EPI_RESID));
  if (fine || nrb * (a.N / 32) * a.slices <= 2 * cus)
    *rc = dispatch_fs<1, 1, 4, NP, 1>(a, out, ep, s);
  else if (NP == 6 || (nrb + 1) / 2 * (a.N / 64) * a.slices <= cus)
    *rc = dispatch_fs<2, 2, 4, NP, 1>(a, out, ep, s);
  else
    return false;
  return true;
}

// fp32 or packed rows: one 32 x 32 tile per CU at most, else one 32 x 64.  N = K = 1024:
// 148 rows 14.3 -> 8.0 us, 512 rows 14.7 -> 12.3; N = 3072: 148 rows 19.4 -> 14.3, 200 rows
// (336 tiles) 19.3 -> 20.6 and left alone.  Six products N = 1024, K = 2048: 148 rows 32.1 ->
// 12.8 us; past one per CU they lose too (N = 896, K = 4864, 768 rows, 336 tiles: 70.1 us on
// gemm_bx_kernel, 76.9 here; N = 9728, K = 896, 48 rows, 304 tiles: 17.1 / 18.6; N = 3072, K =
// 1024, 200 rows, 336 tiles: 18.9 / 18.7).
template <int NP, int AF>
bool pick_fs_rows(const FsArgs& a, int out, const EpiArgs& ep, hipStream_t s, int* rc) {
  const long nrb = (a.M + 31) / 32, cus = device_cus();
  if (nrb * (a.N / 32) <= cus)
    *rc = dispatch_fs<1, 1, 4, NP, AF>(a, out, ep, s);
  else if (nrb * (a.N / 64) <= cus)
    *rc = dispatch_fs<1, 2, 4, NP, AF>(a, out, ep, s);
  else
    return false;
  return true;
}

}  // namespace

bool linear_fs_rows(const lx_linear_bx& g, const EpiArgs& ep, hipStream_t stream, int* rc) {
  const size_t ab = ((size_t)(g.M - 1) * g.lda + g.K) * 4, wb = (size_t)g.N * g.K * 6;
  if (ep.kind == LX_EPI_SWIGLU_PAIRED || ab >= (1ull << 31) || wb >= (1ull << 31)) return false;
  FsArgs a{};
  a.A = g.A;
  a.lda = g.lda;
  a.a_bytes = (unsigned)ab;
  a.Wf = g.Wf;
  a.w_bytes = (unsigned)wb;
  a.bias = g.bias;
  a.Y = g.Y;
  a.ldy = g.ldy;
  a.M = g.M;
  a.N = g.N;
  a.K = g.K;
  a.slices = 1;
  const int out = g.out == LX_BX_OUT_PACKED ? FS_OUT_PACKED : FS_OUT_F32;
  if (g.a_packed) return pick_fs_rows<3, kAPacked>(a, out, ep, stream, rc);
  return g.products == 3 ? pick_fs_rows<3, kARows>(a, out, ep, stream, rc)
                         : pick_fs_rows<6, kARows>(a, out, ep, stream, rc);
}

// From 65 rows (two row blocks leave the 32 x 64 tiles at 96 workgroups for q|k|v: T =
// 24 1313 against 1296 us an evaluation) to one workgroup per CU.
bool fs_takes_ln(int M, int N, int K, int products) {
  return products == 3 && K == kLnK && N % 64 == 0 && M > 64 &&
         (long)((M + 31) / 32) * (N / 64) <= device_cus();
}

int linear_fs_ln(const FsLinear& g, const FsLn& ln, hipStream_t stream) {
  const size_t wb = (size_t)g.N * g.K * 6;
  LX_REQUIRE(ln.x && ln.shift && ln.scale && ln.T > 0 && g.Wf && g.Y && g.M > 0 &&
                 fs_takes_ln(g.M, g.N, g.K, g.products) && wb < (1ull << 31) && g.epi &&
                 (g.epi->kind == LX_EPI_ROPE_PARTIAL || g.epi->kind == LX_EPI_GELU_TANH),
             "linear_fs_ln: bad arguments (M=%d N=%d K=%d)", g.M, g.N, g.K);
  FsArgs a{};
  a.Wf = g.Wf;
  a.w_bytes = (unsigned)wb;
  a.bias = g.bias;
  a.Y = g.Y;
  a.ldy = g.ldy;
  a.M = g.M;
  a.N = g.N;
  a.K = g.K;
  a.slices = 1;
  a.tiles_m = (g.M + 31) / 32;
  a.tiles_n = g.N / 64;
  EpiArgs ep;
  LX_TRY(make_epi(g.epi, g.N, &ep));
  if (g.epi->kind == LX_EPI_GELU_TANH) {
    LX_REQUIRE(g.out == FS_OUT_FRAG, "linear_fs_ln: GELU is written in fragment order");
    return launch_fs_ln<LX_EPI_GELU_TANH, FS_OUT_FRAG>(a, ep, ln, stream);
  }
  LX_REQUIRE(g.out == FS_OUT_F32, "linear_fs_ln: rotary rows are fp32");
  return launch_fs_ln<LX_EPI_ROPE_PARTIAL, FS_OUT_F32>(a, ep, ln, stream);
}

int linear_fs(const FsLinear& g, hipStream_t stream) {
  const int npl = g.products == 6 ? 3 : 2;
  LX_REQUIRE(g.A && g.Wf && g.Y, "linear_fs: null operand");
  LX_REQUIRE(g.products == 3 || g.products == 6, "linear_fs: %d products (3 or 6)", g.products);
  LX_REQUIRE(g.M > 0 && g.N > 0 && g.K > 0 && g.N % 128 == 0 && g.K % 32 == 0 && g.slices >= 1 &&
                 g.slices <= g.K / 32 && (g.slices == 1 || g.out == FS_OUT_PARTIAL),
             "linear_fs: bad shape M=%d N=%d K=%d slices=%d", g.M, g.N, g.K, g.slices);
  const size_t ab = (size_t)((g.M + 31) / 32) * (g.K / 16) * npl * 1024;
  const size_t wb = (size_t)g.N * g.K * 6;
  LX_REQUIRE(ab < (1ull << 31) && wb < (1ull << 31) && (size_t)g.M * g.ldy < (1ull << 40),
             "linear_fs: operands must stay below 2 GiB");
  const int kind = g.epi ? g.epi->kind : LX_EPI_NONE;
  LX_REQUIRE(g.neox_pos || g.out == FS_OUT_PARTIAL ||
                 (g.out == FS_OUT_FRAG
                      ? kind == LX_EPI_GELU_TANH || kind == LX_EPI_SWIGLU_PAIRED
                      : g.out == FS_OUT_F32 &&
                            (kind == LX_EPI_RESID || kind == LX_EPI_GATED_RESID ||
                             kind == LX_EPI_ROPE_PARTIAL)),
             "linear_fs: epilogue %d with output %d", kind, g.out);
  FsArgs a{};
  a.A = g.A;
  a.a_bytes = (unsigned)ab;
  a.Wf = g.Wf;
  a.w_bytes = (unsigned)wb;
  a.bias = g.bias;
  a.Y = g.Y;
  a.ldy = g.ldy;
  a.slice_stride = g.slice_stride;
  a.M = g.M;
  a.N = g.N;
  a.K = g.K;
  a.slices = g.slices;
  EpiArgs ep;
  LX_TRY(make_epi(g.epi, g.N, &ep));
  if (g.neox_pos) {
    LX_REQUIRE(g.bias && g.rope_cs && g.k_cache && g.v_cache && g.out == FS_OUT_F32 &&
                   g.q_cols % 64 == 0 && g.kv_cols % 64 == 0 && g.q_cols + 2 * g.kv_cols == g.N,
               "linear_fs: bad q|k|v arguments");
    ep.kind = kEpiNeox;
    ep.pos = g.neox_pos;
    a.q_cols = g.q_cols;
    a.kv_cols = g.kv_cols;
    a.rope_heads = g.rope_heads;
    a.rope_cs = g.rope_cs;
    a.k_cache = g.k_cache;
    a.v_cache = g.v_cache;
  }
  int rc = LX_OK;
  if (g.products == 3 ? pick_fs<3>(a, g.out, ep, stream, &rc) : pick_fs<6>(a, g.out, ep, stream, &rc))
    return rc;
  return linear_ft(a, g.out, ep, stream);
}

}  // namespace lx
