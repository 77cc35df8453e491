// Grouped GEMMs between the weight streams of decode steps and the large
// prefill tiles: a few dozen to a few hundred rows per group, where neither
// the weights nor the matrix pipe alone sets the time, and the fp8 / int4
// GEMMs of any row count that have no tile copy (int4: with at most
// kMidScaleMax scale groups along K).
#include "smoe_common.hpp"
#include "smoe_gemm.hpp"
#include "smoe_internal.hpp"

namespace smoe {

int device_cus();

namespace {

template <int FMT>
constexpr int mid_wb() {  // bytes of one channel's 64-k slice
  return FMT == SMOE_BF16 ? 128 : (FMT == SMOE_FP8_E4M3 ? 64 : 32);
}
// int4 scale groups along K: the [groups, 128] table of a tile is 16 KB of LDS
// beside the ring (three workgroups of 2 stages per CU).  Wider tables, e.g. the
// 44 groups of U 2816 in groups of 64, leave that GEMM on the general kernel:
// 777 tokens, H 1024, 16 int4 experts 1224 us in groups of 64, 774 in groups of 128.
constexpr int kMidScaleMax = 32;

// The tile of workgroup bid: tiles go group by group, within a group strip by
// strip and the strip's row tiles next to each other, so that a weight strip
// is fetched once for all rows of its group; workgroup ids are dealt to the 8
// XCDs round robin and each XCD takes one contiguous part of the order, so a
// group's rows stay in one L2.
template <int BM, int BN>
__device__ __forceinline__ bool mid_tile(const GemmArgs& p, int bid, int& g, int& m0, int& mrows,
                                         int& n0) {
  const int strips = (p.N_out + BN - 1) / BN;
  const int T = count_tiles(p, BM) * strips;
  if (bid >= T) return false;
  const int x = bid & 7, base = T >> 3, rem = T & 7;
  const int logical = x * base + min(x, rem) + (bid >> 3);
  int lo = 0, hi = p.single_rows, in = logical;
  g = 0;
  if (p.G > 0) {
    int acc = 0;
    for (int b = 0; b < p.G; b += 64) {
      int l, h, t;
      group_chunk(p, BM, b, l, h, t);
      const int incl = wave_incl_scan(t) * strips + acc;
      const uint64_t m = __ballot(logical < incl);
      if (m) {
        const int f = __builtin_ctzll(m);
        g = b + f;
        in = logical - __builtin_amdgcn_readlane(incl - t * strips, f);
        lo = __builtin_amdgcn_readlane(l, f);
        hi = __builtin_amdgcn_readlane(h, f);
        break;
      }
      acc = __builtin_amdgcn_readlane(incl, 63);
    }
  }
  const int tm = (hi - lo + BM - 1) / BM;
  m0 = lo + (in % tm) * BM;
  mrows = min(BM, hi - m0);
  n0 = (in / tm) * BN;
  return true;
}

// BM x BN tile, WM x WN waves, K in 64-wide stages that go global -> LDS by
// DMA (weights in their storage format, widened as the fragments are read)
// through an NS-stage ring, NS - 1 stages in flight while one computes.  A
// stage's two MFMAs take its lower and its upper 32 k, the order of the other
// large-tile kernels, or with PAIRS the low and the high 8 of the 16 k at
// 16 q of lane quarter q, the order of k_gemm_stream4 (fp8: one 16-byte
// fragment read then holds both).  LDS rows are swizzled as sw_chunk
// says.
//
// Bound: the operand stream into the CUs and its latency (with the MFMAs and
// fragment reads taken out a launch keeps 85-95% of its time; fragments read
// a stage ahead into a second register set, or 32-k stages twice as deep,
// changed nothing or lost 10-20%), so what counts is the number of
// workgroups that wait at the same time and that their last round is full:
// small rings and two or three workgroups per CU beat one deep ring (H 1024
// -> 2816 GELU, 16 groups of 250 rows: 128 x 128 tiles, 2 stages, 2
// workgroups per CU 51 us; 4 stages, 8 waves, 1 per CU 71 us).
template <int FMT, int EPI, int BM, int BN, int WM, int WN, int NS, int OCC, bool PAIRS>
__global__ __launch_bounds__(WM* WN * 64, OCC) void k_gemm_mid(const GemmArgs p) {
  constexpr int NW = WM * WN, TM = BM / WM, TN = BN / WN, FM = TM / 16, FN = TN / 16;
  constexpr int WB = mid_wb<FMT>(), CPR = WB / 16;
  constexpr int A_BYTES = BM * 128, STAGE = A_BYTES + BN * WB;
  constexpr int A_LD = A_BYTES / 1024 / NW, W_LD = BN * WB / 1024 / NW, LD = A_LD + W_LD;
  constexpr int ESZ2 = FMT == SMOE_BF16 ? 4 : (FMT == SMOE_FP8_E4M3 ? 2 : 1);  // 2 x bytes/elt
  constexpr int SCALES = FMT == SMOE_INT4 ? kMidScaleMax * BN * 4 : 0;
  static_assert(A_LD * NW * 1024 == A_BYTES && W_LD * NW * 1024 == BN * WB, "whole DMA instructions");
  static_assert(EPI != EPI_SWIGLU || TN % 64 == 0, "SwiGLU pairs channel c with c + 32");
  static_assert(NS * STAGE >= BM * BN * 2, "the output tile is staged in the ring");
  static_assert(!PAIRS || FMT != SMOE_INT4, "int4 at these row counts: k_gemm_stream4");
  __shared__ __attribute__((aligned(1024))) uint8_t ring[NS * STAGE + SCALES];
  int g, m0, mrows, n0;
  if (!mid_tile<BM, BN>(p, blockIdx.x, g, m0, mrows, n0)) return;  // uniform
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const int q = lane >> 4, l16 = lane & 15;
  const int wm = wave / WN, wn = wave % WN;

  const uint16_t* asrc[A_LD];
  const uint8_t* wsrc[W_LD];
#pragma unroll
  for (int j = 0; j < A_LD; ++j) {
    const int r = 8 * (NW * j + wave) + (lane >> 3);
    const int pr = m0 + (r < mrows ? r : 0);  // rows past the group's end: a valid row, never stored
    const int ar = p.a_rows ? p.a_rows[pr] : pr;
    asrc[j] = reinterpret_cast<const uint16_t*>(p.A) + static_cast<int64_t>(ar) * p.lda +
              8 * sw_chunk<8>(r, lane & 7);
  }
#pragma unroll
  for (int j = 0; j < W_LD; ++j) {
    const int b = (NW * j + wave) * 1024 + 16 * lane;
    const int row = b / WB, pc = (b % WB) >> 4;
    const int n = min(n0 + row, p.N_out - 1);  // channels past N_out: loaded, never stored
    wsrc[j] = reinterpret_cast<const uint8_t*>(p.W) +
              (g * p.w_gstride + static_cast<int64_t>(n) * p.ldw) * ESZ2 / 2 +
              sw_chunk<CPR>(row, pc) * 16;
  }
  float* stab = reinterpret_cast<float*>(ring + NS * STAGE);  // int4: [K / gs, BN] group scales
  int gs_shift = 0;
  if constexpr (FMT == SMOE_INT4) {
    gs_shift = 31 - __builtin_clz(p.group_size);
    const int ng = p.K >> gs_shift;
    for (int i = threadIdx.x; i < ng * BN; i += NW * 64) {
      const int n = min(n0 + i % BN, p.N_out - 1);
      stab[i] = load_scale(p.S, g * p.s_gstride + static_cast<int64_t>(n) * ng + i / BN, p.s_f16);
    }
  }
  auto issue = [&](int kc) {  // DMA of stage kc into ring slot kc % NS
    uint8_t* base = ring + (kc % NS) * STAGE;
#pragma unroll
    for (int j = 0; j < W_LD; ++j)
      __builtin_amdgcn_global_load_lds((gbl_vptr)(wsrc[j] + static_cast<int64_t>(kc) * WB),
                                       (lds_vptr)(base + A_BYTES + (NW * j + wave) * 1024), 16, 0, 0);
#pragma unroll
    for (int j = 0; j < A_LD; ++j)
      __builtin_amdgcn_global_load_lds((gbl_vptr)(asrc[j] + kc * 64),
                                       (lds_vptr)(base + (NW * j + wave) * 1024), 16, 0, 0);
  };
  f32x4 acc[FN][FM];
#pragma unroll
  for (int j = 0; j < FN; ++j)
#pragma unroll
    for (int i = 0; i < FM; ++i) acc[j][i] = f32x4{0.f, 0.f, 0.f, 0.f};

  const int KC = p.K / 64;
#pragma unroll
  for (int st = 0; st < NS - 1; ++st)
    if (st < KC) issue(st);
  const bool live = wm * TM < mrows;  // this wave has rows
  auto k8 = [&](int h) { return PAIRS ? 2 * q + h : 4 * h + q; };  // the 8 k of MFMA h, in eights
  for (int kc = 0; kc < KC; ++kc) {
    // own part of stage kc landed (later ones may fly); after the barrier
    // everybody's, and nobody reads stage kc - 1 any more
    if (kc + NS - 2 < KC) wait_vmcnt<(NS - 2) * LD>();
    else wait_vmcnt<0>();
    wait_lgkm0();
    __builtin_amdgcn_s_barrier();
    if (kc + NS - 1 < KC) issue(kc + NS - 1);  // into the slot of stage kc - 1
    if (!live) continue;
    const uint8_t* sa = ring + (kc % NS) * STAGE;
    const uint8_t* sw = sa + A_BYTES;
    bf16x8 wf[2][FN];
#pragma unroll
    for (int t = 0; t < FN; ++t) {
      const int row = wn * TN + t * 16 + l16;
      const uint8_t* wr = sw + row * WB;
      float scale = 0.f;
      if constexpr (FMT == SMOE_INT4) scale = stab[((kc * 64) >> gs_shift) * BN + row];
      u32x4 both = {0u, 0u, 0u, 0u};
      if constexpr (FMT == SMOE_FP8_E4M3 && PAIRS)
        both = *reinterpret_cast<const u32x4*>(wr + (sw_chunk<CPR>(row, q) << 4));
#pragma unroll
      for (int h = 0; h < 2; ++h) {
        u32x4 v;
        if constexpr (FMT == SMOE_BF16) {
          v = *reinterpret_cast<const u32x4*>(wr + (sw_chunk<CPR>(row, k8(h)) << 4));
        } else if constexpr (FMT == SMOE_FP8_E4M3) {
          u32x2 r;
          if constexpr (PAIRS) r = u32x2{both[2 * h], both[2 * h + 1]};
          else r = *reinterpret_cast<const u32x2*>(wr + (sw_chunk<CPR>(row, k8(h) >> 1) << 4) + 8 * (q & 1));
          const u32x2 lo = fp8x4_to_bf16x4(r.x), hi = fp8x4_to_bf16x4(r.y);
          v = u32x4{lo.x, lo.y, hi.x, hi.y};
        } else {
          v = int4x8_to_bf16x8(
              *reinterpret_cast<const uint32_t*>(wr + (sw_chunk<CPR>(row, h) << 4) + 4 * q), scale);
        }
        wf[h][t] = __builtin_bit_cast(bf16x8, v);
      }
    }
#pragma unroll
    for (int i = 0; i < FM; ++i) {
      const int r = wm * TM + i * 16 + l16;
      bf16x8 af[2];
#pragma unroll
      for (int h = 0; h < 2; ++h)
        af[h] = *reinterpret_cast<const bf16x8*>(sa + r * 128 + (sw_chunk<8>(r, k8(h)) << 4));
#pragma unroll
      for (int t = 0; t < FN; ++t)
#pragma unroll
        for (int h = 0; h < 2; ++h)
          acc[t][i] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(wf[h][t], af[h], acc[t][i], 0, 0, 0);
    }
  }
  if constexpr (EPI != EPI_F32_BIAS) {
    if (p.out_dtype == SMOE_BF16 && p.N_out % 8 == 0 && p.ldo % 8 == 0) {  // 16-byte stores
      tile_epilogue<BM, BN, TM, TN, NW * 64, EPI, FMT == SMOE_FP8_E4M3 ? SMOE_FP8_E4M3 : SMOE_BF16>(
          p, acc, g, m0, 0, mrows, n0, wm, wn, ring);
      return;
    }
  }
  if constexpr (EPI != EPI_SWIGLU) {
#pragma unroll
    for (int i = 0; i < FM; ++i) {
      const int r = wm * TM + i * 16 + l16;
      if (r >= mrows) continue;
#pragma unroll
      for (int j = 0; j < FN; ++j) {
        const int c = n0 + wn * TN + j * 16 + 4 * q;
        if (c < p.N_out) store4<EPI>(p, FMT, g, m0 + r, c, acc[j][i]);
      }
    }
  }
}

// The order of the sums, by rows per group: up to 128 that of k_gemm_stream4,
// which keeps the int4 groups of that size, so that the formats agree and a
// model's results at these sizes are those it has given before; past it that
// of the general and the prefill tiles, for the same reason.  Neither is
// faster.
bool k_pairs(const GemmArgs& a) {
  return a.G > 0 && a.max_rows / a.G <= 128 && a.fmt != SMOE_INT4;
}

template <int FMT, int EPI, int BM, int BN, int WM, int WN, int NS, int OCC>
int launch_tiles(const GemmArgs& a, hipStream_t s) {
  const int64_t rows = a.G == 0 ? a.single_rows : a.max_rows;
  const int64_t wgs = ((rows + BM - 1) / BM + a.G) * ((a.N_out + BN - 1) / BN);
  if (wgs > 0x7fffffff) return SMOE_EINVAL;
  if (wgs == 0) return SMOE_OK;
  const dim3 grid(static_cast<unsigned>(wgs)), block(WM * WN * 64);
  if constexpr (FMT != SMOE_INT4) {
    if (k_pairs(a)) {
      SMOE_LAUNCH((k_gemm_mid<FMT, EPI, BM, BN, WM, WN, NS, OCC, true>), grid, block, 0, s, a);
      return hipGetLastError() == hipSuccess ? SMOE_OK : SMOE_EHIP;
    }
  }
  SMOE_LAUNCH((k_gemm_mid<FMT, EPI, BM, BN, WM, WN, NS, OCC, false>), grid, block, 0, s, a);
  return hipGetLastError() == hipSuccess ? SMOE_OK : SMOE_EHIP;
}

// The tile, by the number of 64 x 128 tiles the rows make (us per launch, in
// brackets the kernel these shapes ran on before):
//   fewer than CUs: 64 x 64, so that more CUs take part (bf16 1024 -> 1024, 16
//     groups of 45 rows: 9.9 against 11.7 with 64 x 128 [19.4]; fp8 2816 ->
//     1024, one group of 1000 rows: 23.8 against 28.3 [92.4])
//   64 x 128 otherwise.  3 stages and 2 workgroups per CU where the tiles are
//     all resident at once (bf16 2816 -> 1024, 16 groups of 97 rows: 27.5
//     against 39.5 with 2 stages [79.6]; int4 2816 -> 1024, 16 of 200: 40.0
//     against 43.5 [118]) or bf16 weights are most of the traffic (2048 ->
//     2048, 64 groups of 56 rows: 120 against 136 [177]); else 2 stages and 3
//     workgroups (bf16 1024 -> 2816, 16 of 250: 53.6 against 58.0 [106]; int4
//     1024 -> 1408, 32 of 512: 91.6 against 95.6 [218]).  fp8 stages are
//     smaller and 3 workgroups better throughout (2816 -> 1024, 16 of 130:
//     30.7 against 32.5 [99.8]; 1408 -> 2048, 8192 rows: 76 against 82 [116]).
// SwiGLU pairs channels 32 apart, so a wave takes 64 of them: 128 x 128 in a 2 x
// 2 grid of waves (bf16 1024 -> 5632, 16 groups of 97 rows: 48.8 [79.6]; fp8,
// 130 rows: 47.6 [138]), or 64 rows where groups have no more (35 rows: bf16
// 35.8 against 46.9 [43.1], fp8 24.5 against 26.6 [27.8]).
template <int FMT, int EPI>
int launch_mid(const GemmArgs& a, hipStream_t s) {
  const int64_t rows = a.G == 0 ? a.single_rows : a.max_rows, groups = a.G == 0 ? 1 : a.G;
  if constexpr (EPI == EPI_SWIGLU) {
    if (rows / groups > 64) return launch_tiles<FMT, EPI, 128, 128, 2, 2, 2, 2>(a, s);
    if constexpr (FMT == SMOE_BF16) return launch_tiles<FMT, EPI, 64, 128, 2, 2, 3, 2>(a, s);
    return launch_tiles<FMT, EPI, 64, 128, 2, 2, 2, 3>(a, s);
  } else {
    const int64_t cus = device_cus() > 0 ? device_cus() : 256;
    // every group's last tile is half full on average
    const int64_t tiles = (rows / 64 + (groups + 1) / 2) * ((a.N_out + 127) / 128);
    if constexpr (FMT != SMOE_INT4)
      if (tiles < cus) return launch_tiles<FMT, EPI, 64, 64, 2, 2, 3, 3>(a, s);
    if constexpr (FMT != SMOE_FP8_E4M3)
      if (tiles <= 2 * cus || (FMT == SMOE_BF16 && rows / groups <= 128))
        return launch_tiles<FMT, EPI, 64, 128, 1, 4, 3, 2>(a, s);
    return launch_tiles<FMT, EPI, 64, 128, 1, 4, 2, 3>(a, s);
  }
}

template <int FMT>
int launch_mid_fmt(const GemmArgs& a, hipStream_t s) {
  switch (a.epi) {
    case EPI_F32_BIAS: return launch_mid<FMT, EPI_F32_BIAS>(a, s);
    case EPI_ROWSCALE:  // the edge projection: bf16 weights
      if constexpr (FMT == SMOE_BF16) return launch_mid<FMT, EPI_ROWSCALE>(a, s);
      return SMOE_EUNSUPPORTED;
    case EPI_GELU: return launch_mid<FMT, EPI_GELU>(a, s);
    case EPI_SWIGLU: return launch_mid<FMT, EPI_SWIGLU>(a, s);
    case EPI_DOWN: return launch_mid<FMT, EPI_DOWN>(a, s);
    default: return SMOE_EINVAL;
  }
}

}  // namespace

bool gemm_mid_fits(const GemmArgs& a) {
  const auto odd = [](const void* q) { return reinterpret_cast<uintptr_t>(q) % 16 != 0; };
  if (a.K % 64 || a.lda % 8 || a.N_out < 128 || !a.A || odd(a.A) || odd(a.W) || odd(a.out)) return false;
  const int walign = a.fmt == SMOE_BF16 ? 8 : (a.fmt == SMOE_FP8_E4M3 ? 16 : 32);  // 16-byte loads
  if (a.ldw % walign || a.w_gstride % walign) return false;
  if (a.fmt == SMOE_INT4 && (a.group_size % 64 || (a.group_size & (a.group_size - 1)) ||
                             a.K % a.group_size || a.K / a.group_size > kMidScaleMax))
    return false;
  if (a.fmt != SMOE_BF16 && a.epi == EPI_ROWSCALE) return false;
  if (a.epi == EPI_SWIGLU) return a.out_dtype == SMOE_BF16 && a.N_out % 128 == 0 && a.ldo % 8 == 0;
  // stores of four channels: f32 results, and bf16 rows of an odd number of
  // 8-byte pieces up to 128 rows per group (16 groups of 50 rows, 1024 -> 1004:
  // 11.0 us, 30.7 on the general kernel); otherwise of eight
  const bool four = a.epi == EPI_F32_BIAS || a.out_dtype == SMOE_F32 || k_pairs(a);
  return four ? a.N_out % 4 == 0 && a.ldo % 4 == 0 : a.N_out % 8 == 0 && a.ldo % 8 == 0;
}

int launch_gemm_mid(const GemmArgs& a, hipStream_t s) {
  switch (a.fmt) {
    case SMOE_BF16: return launch_mid_fmt<SMOE_BF16>(a, s);
    case SMOE_FP8_E4M3: return launch_mid_fmt<SMOE_FP8_E4M3>(a, s);
    case SMOE_INT4: return launch_mid_fmt<SMOE_INT4>(a, s);
    default: return SMOE_EUNSUPPORTED;
  }
}

}  // namespace smoe
