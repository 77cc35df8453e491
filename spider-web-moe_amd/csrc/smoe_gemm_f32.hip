// Grouped GEMMs of fp32 models on the fp32 matrix instruction
// (v_mfma_f32_16x16x4_f32, f32 products and f32 accumulation).
//
// k index of a lane: both operands of the four MFMAs that cover a 16-k block
// come from one 16-byte load, lane quarter q holding k = 4q .. 4q+3; MFMA e
// multiplies the e-th of each, i.e. k in {e, 4+e, 8+e, 12+e}.  The order of
// k is the same for both operands, and every k is taken once.
#include "smoe_common.hpp"
#include "smoe_gemm.hpp"
#include "smoe_internal.hpp"

namespace smoe {

int device_cus();

namespace {

// Four consecutive channels of one row; a partial last quad (N_out % 4) and
// rows that are not 16-byte aligned go element by element.
template <int EPI>
__device__ __forceinline__ void put_quad(const GemmArgs& p, bool vec, int g, int row, int c, f32x4 v) {
  if (vec) {
    if (c < p.N_out) store4<EPI>(p, SMOE_F32, g, row, c, v);
    return;
  }
#pragma unroll
  for (int i = 0; i < 4; ++i)
    if (c + i < p.N_out) epi_one<EPI>(p, SMOE_F32, g, row, c + i, v[i]);
}

__device__ __forceinline__ bool vec_out(const GemmArgs& p) {
  return p.N_out % 4 == 0 && p.ldo % 4 == 0 && reinterpret_cast<uintptr_t>(p.out) % 16 == 0;
}

// BM x BN tile, 4 waves in a 2 x 2 grid, K in 32-wide stages (128-byte rows)
// that go global -> LDS by DMA through a 3-stage ring, two stages in flight
// while one computes.  Bound: the fp32 matrix pipe (256 flop per clock and
// CU); a wave of a 64 x 64 tile reads 4 KB of fragments per 16-k block for 16
// MFMAs (512 cycles of its SIMD's pipe), the workgroup 16 KB in that time, a
// quarter of what LDS delivers, and 48 KB of LDS let three workgroups share a
// CU and hide each other's waits.  Against
// the VALU tile kernel (scalar loads, one barrier pair per 16 k): H 256, U
// 512, E 8, 2048 tokens (about 512 rows per expert, 1200 per destination),
// us per launch: up 63 -> 21.5, down 98.5 -> 22.9, edge projection 61.7 ->
// 20.4 (63 TFLOP/s, a launch's own ~4 us included).
template <int BM, int BN, int EPI>
__global__ __launch_bounds__(256) void k_gemm_f32(const GemmArgs p) {
  constexpr int TM = BM / 2, TN = BN / 2, FM = TM / 16, FN = TN / 16;
  constexpr int NS = 3, A_BYTES = BM * 128, STAGE = A_BYTES + BN * 128;
  constexpr int A_LD = BM / 32, B_LD = BN / 32, LD = A_LD + B_LD;  // DMA instructions per wave
  __shared__ __attribute__((aligned(1024))) uint8_t ring[NS * STAGE];
  int g, m0, mrows;
  if (!find_tile(p, BM, blockIdx.x, g, m0, mrows)) return;  // uniform, before any barrier
  const int n0 = blockIdx.y * BN;
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const int q = lane >> 4, l16 = lane & 15;
  const int wm = wave >> 1, wn = wave & 1;

  // DMA instruction j of this wave covers rows 8 (4 j + wave) .. + 7, lane l
  // row l / 8 and physical 16-byte chunk l % 8
  const float* asrc[A_LD];
  const float* bsrc[B_LD];
#pragma unroll
  for (int j = 0; j < A_LD; ++j) {
    const int r = 8 * (4 * j + wave) + (lane >> 3);
    const int pr = m0 + (r < mrows ? r : 0);  // rows past the group's end: a valid row, never stored
    const int ar = p.a_rows ? p.a_rows[pr] : pr;
    asrc[j] = reinterpret_cast<const float*>(p.A) + static_cast<int64_t>(ar) * p.lda +
              4 * sw_chunk<8>(r, lane & 7);
  }
#pragma unroll
  for (int j = 0; j < B_LD; ++j) {
    const int r = 8 * (4 * j + wave) + (lane >> 3);
    const int n = min(n0 + r, p.N_out - 1);  // channels past N_out: loaded, never stored
    bsrc[j] = reinterpret_cast<const float*>(p.W) + g * p.w_gstride +
              static_cast<int64_t>(n) * p.ldw + 4 * sw_chunk<8>(r, lane & 7);
  }
  auto issue = [&](int st) {  // DMA of stage st into ring slot st % NS
    uint8_t* base = ring + (st % NS) * STAGE;
#pragma unroll
    for (int j = 0; j < A_LD; ++j)
      __builtin_amdgcn_global_load_lds((gbl_vptr)(asrc[j] + st * 32),
                                       (lds_vptr)(base + (4 * j + wave) * 1024), 16, 0, 0);
#pragma unroll
    for (int j = 0; j < B_LD; ++j)
      __builtin_amdgcn_global_load_lds((gbl_vptr)(bsrc[j] + st * 32),
                                       (lds_vptr)(base + A_BYTES + (4 * j + wave) * 1024), 16, 0, 0);
  };

  f32x4 acc[FN][FM];
#pragma unroll
  for (int j = 0; j < FN; ++j)
#pragma unroll
    for (int i = 0; i < FM; ++i) acc[j][i] = f32x4{0.f, 0.f, 0.f, 0.f};

  const int KT = p.K / 32;
#pragma unroll
  for (int st = 0; st < NS - 1; ++st)
    if (st < KT) issue(st);
  for (int st = 0; st < KT; ++st) {
    // own part of stage st landed (a later one may fly); after the barrier
    // everybody's, and nobody reads stage st - 1 any more
    if (st + NS - 2 < KT) wait_vmcnt<(NS - 2) * LD>();
    else wait_vmcnt<0>();
    wait_lgkm0();
    __builtin_amdgcn_s_barrier();
    if (st + NS - 1 < KT) issue(st + NS - 1);  // into the slot of stage st - 1
    const uint8_t* sa = ring + (st % NS) * STAGE;
    const uint8_t* sb = sa + A_BYTES;
#pragma unroll
    for (int b = 0; b < 2; ++b) {
      f32x4 af[FM], wf[FN];
#pragma unroll
      for (int i = 0; i < FM; ++i) {
        const int r = wm * TM + i * 16 + l16;
        af[i] = *reinterpret_cast<const f32x4*>(sa + r * 128 + 16 * sw_chunk<8>(r, 4 * b + q));
      }
#pragma unroll
      for (int j = 0; j < FN; ++j) {
        const int r = wn * TN + j * 16 + l16;
        wf[j] = *reinterpret_cast<const f32x4*>(sb + r * 128 + 16 * sw_chunk<8>(r, 4 * b + q));
      }
#pragma unroll
      for (int e = 0; e < 4; ++e)
#pragma unroll
        for (int j = 0; j < FN; ++j)
#pragma unroll
          for (int i = 0; i < FM; ++i)
            acc[j][i] = __builtin_amdgcn_mfma_f32_16x16x4f32(wf[j][e], af[i][e], acc[j][i], 0, 0, 0);
    }
  }
  const bool vec = vec_out(p);
#pragma unroll
  for (int i = 0; i < FM; ++i) {
    const int r = wm * TM + i * 16 + l16;
    if (r >= mrows) continue;
#pragma unroll
    for (int j = 0; j < FN; ++j)
      put_quad<EPI>(p, vec, g, m0 + r, n0 + wn * TN + j * 16 + 4 * q, acc[j][i]);
  }
}

// 16 rows x 16 TN channels, K split over the 4 waves, operands straight from
// memory to registers (U 16-k blocks requested at once), partial sums added
// through LDS in wave order.  For the few rows of a decode step and the
// narrow outputs (router / edge logits), where a launch is one or two memory
// round trips long and the number of workgroups counts (2048 x 256 -> 8
// logits: 30 -> 4.8 us against 64-row VALU tiles on 32 workgroups).
template <int EPI, int TN>
__global__ __launch_bounds__(256) void k_gemm_f32_skinny(const GemmArgs p) {
  constexpr int U = 4;
  __shared__ f32x4 red[4][TN][64];
  int g, m0, mrows;
  if (!find_tile(p, 16, blockIdx.x, g, m0, mrows)) return;  // uniform, before any barrier
  const int n0 = blockIdx.y * 16 * TN;
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const int q = lane >> 4, l16 = lane & 15;
  const int pr = m0 + (l16 < mrows ? l16 : 0);  // rows past the group's end: a valid row, never stored
  const int ar = p.a_rows ? p.a_rows[pr] : pr;
  const float* arow = reinterpret_cast<const float*>(p.A) + static_cast<int64_t>(ar) * p.lda + 4 * q;
  const float* wrow[TN];
#pragma unroll
  for (int t = 0; t < TN; ++t) {
    const int n = min(n0 + 16 * t + l16, p.N_out - 1);
    wrow[t] = (p.W2 && n >= p.n_split)
                  ? reinterpret_cast<const float*>(p.W2) + static_cast<int64_t>(n - p.n_split) * p.ldw2 + 4 * q
                  : reinterpret_cast<const float*>(p.W) + g * p.w_gstride +
                        static_cast<int64_t>(n) * p.ldw + 4 * q;
  }
  f32x4 acc[TN];
#pragma unroll
  for (int t = 0; t < TN; ++t) acc[t] = f32x4{0.f, 0.f, 0.f, 0.f};
  const int nb = p.K / 16, b_end = (wave + 1) * nb / 4;
  for (int b0 = wave * nb / 4; b0 < b_end; b0 += U) {
    f32x4 av[U], wv[U][TN];
#pragma unroll
    for (int u = 0; u < U; ++u) {  // blocks past the end: the last one again (multiplied as zeros)
      const int k = 16 * min(b0 + u, b_end - 1);
      av[u] = *reinterpret_cast<const f32x4*>(arow + k);
#pragma unroll
      for (int t = 0; t < TN; ++t) wv[u][t] = *reinterpret_cast<const f32x4*>(wrow[t] + k);
    }
#pragma unroll
    for (int u = 0; u < U; ++u) {
      const bool live = b0 + u < b_end;
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        const float a = live ? av[u][e] : 0.f;
#pragma unroll
        for (int t = 0; t < TN; ++t)
          acc[t] = __builtin_amdgcn_mfma_f32_16x16x4f32(live ? wv[u][t][e] : 0.f, a, acc[t], 0, 0, 0);
      }
    }
  }
#pragma unroll
  for (int t = 0; t < TN; ++t) red[wave][t][lane] = acc[t];
  __syncthreads();
  if (wave >= TN || l16 >= mrows) return;
  f32x4 v = red[0][wave][lane];
#pragma unroll
  for (int w = 1; w < 4; ++w) v += red[w][wave][lane];
  put_quad<EPI>(p, vec_out(p), g, m0 + l16, n0 + 16 * wave + 4 * q, v);
}

int tiles_of(const GemmArgs& a, int bm) {
  if (a.G == 0) return (a.single_rows + bm - 1) / bm;
  return (a.max_rows + bm - 1) / bm + a.G;
}

template <int EPI>
int launch_epi(const GemmArgs& a, hipStream_t s) {
  const int rpg = a.G == 0 ? a.single_rows : a.max_rows / a.G;
  if (a.N_out <= 32 || rpg <= 16) {
    const int tiles = tiles_of(a, 16);
    if (tiles == 0) return SMOE_OK;
    if (a.N_out <= 16)
      SMOE_LAUNCH((k_gemm_f32_skinny<EPI, 1>), dim3(tiles), dim3(256), 0, s, a);
    else
      SMOE_LAUNCH((k_gemm_f32_skinny<EPI, 2>), dim3(tiles, (a.N_out + 31) / 32), dim3(256), 0, s, a);
  } else {
    // 64 x 64 tiles, or 32 x 64 where those would leave CUs without one
    const int strips = (a.N_out + 63) / 64;
    const int cus = device_cus();
    if (static_cast<int64_t>(tiles_of(a, 64)) * strips >= (cus > 0 ? cus : 256))
      SMOE_LAUNCH((k_gemm_f32<64, 64, EPI>), dim3(tiles_of(a, 64), strips), dim3(256), 0, s, a);
    else
      SMOE_LAUNCH((k_gemm_f32<32, 64, EPI>), dim3(tiles_of(a, 32), strips), dim3(256), 0, s, a);
  }
  return hipGetLastError() == hipSuccess ? SMOE_OK : SMOE_EHIP;
}

}  // namespace

bool gemm_f32_fits(const GemmArgs& a) {
  const auto odd = [](const void* q) { return reinterpret_cast<uintptr_t>(q) % 16 != 0; };
  return a.fmt == SMOE_F32 && a.epi != EPI_SWIGLU && a.K % 32 == 0 && a.lda % 4 == 0 &&
         a.ldw % 4 == 0 && a.w_gstride % 4 == 0 && !odd(a.A) && !odd(a.W);
}

// The logits of [router | edge generator] rows (two weight segments): the
// kernel the separate stages' logits (N_out = E <= 16) run on, which sums
// every output in the same order whatever its strip.
int launch_gemm_f32_front(const GemmArgs& a, hipStream_t s) {
  if (!gemm_f32_fits(a) || a.ldw2 % 4 || reinterpret_cast<uintptr_t>(a.W2) % 16 ||
      reinterpret_cast<uintptr_t>(a.out) % 16)
    return SMOE_EINVAL;
  SMOE_LAUNCH((k_gemm_f32_skinny<EPI_F32_BIAS, 1>),
              dim3((a.single_rows + 15) / 16, (a.N_out + 15) / 16), dim3(256), 0, s, a);
  return hipGetLastError() == hipSuccess ? SMOE_OK : SMOE_EHIP;
}

int launch_gemm_f32(const GemmArgs& a, hipStream_t s) {
  switch (a.epi) {
    case EPI_F32_BIAS: return launch_epi<EPI_F32_BIAS>(a, s);
    case EPI_ROWSCALE: return launch_epi<EPI_ROWSCALE>(a, s);
    case EPI_GELU: return launch_epi<EPI_GELU>(a, s);
    case EPI_DOWN: return launch_epi<EPI_DOWN>(a, s);
    default: return SMOE_EINVAL;
  }
}

}  // namespace smoe
