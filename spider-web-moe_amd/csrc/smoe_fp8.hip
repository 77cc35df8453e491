// fp8 x fp8 path of the Forge GEMM (forge/gemm/fp8.py:22-76 with
// quantize_input=True): activations quantized per tensor to e4m3 on the
// device, then a GEMM whose both operands are e4m3 codes, on gfx950's
// v_mfma_f32_16x16x128_f8f6f4, the two per-tensor scales applied in the
// epilogue.  The instruction multiplies the codes exactly but sums each
// block of 128 products below f32 precision (measured: within 2^-14 of the
// block's largest product); the blocks accumulate in f32.
#include "smoe_common.hpp"
#include "smoe_internal.hpp"

namespace smoe {
namespace {

typedef int i32x8 __attribute__((ext_vector_type(8)));

constexpr float kE4m3Max = 448.0f;
constexpr int kAmaxParts = 1024;  // workgroups (and partials) of the amax pass

// max that keeps a NaN once seen (torch's amax propagates NaN)
__device__ __forceinline__ float nan_max(float m, float a) { return (a > m || a != a) ? a : m; }

__device__ __forceinline__ float wave_nan_max(float v) {
#pragma unroll
  for (int o = 32; o >= 1; o >>= 1) v = nan_max(v, __shfl_xor(v, o));
  return v;
}

// float -> OCP e4m3fn code, round to nearest even, not saturating: the cast
// torch.Tensor.to(torch.float8_e4m3fn) performs (|v| > 464 and NaN -> the
// NaN code S.1111.111; 464 itself ties to 448).
__device__ __forceinline__ uint32_t f32_to_e4m3(float v) {
  const uint32_t b = __float_as_uint(v);
  const uint32_t sign = (b >> 24) & 0x80u;
  const uint32_t a = b & 0x7fffffffu;
  if (a > 0x7f800000u) return sign | 0x7fu;              // NaN
  const float av = __uint_as_float(a);
  if (av < 0.015625f) {                                  // below 2^-6: subnormal codes m * 2^-9
    const float q = __builtin_rintf(av * 512.0f);        // exact scaling, RNE to 0 .. 8
    return sign | static_cast<uint32_t>(q);              // 8 reads as the smallest normal
  }
  int e = static_cast<int>(a >> 23) - 127;               // >= -6
  uint32_t m = (a >> 20) & 7u;
  const uint32_t rem = a & 0xfffffu;
  if (rem > 0x80000u || (rem == 0x80000u && (m & 1u))) ++m;
  if (m == 8u) {
    m = 0;
    ++e;
  }
  if (e > 8 || (e == 8 && m == 7u)) return sign | 0x7fu;  // above 464: NaN (inf too)
  return sign | (static_cast<uint32_t>(e + 7) << 3) | m;
}

template <int XDT>
__device__ __forceinline__ float load_x(const void* x, int64_t i) {
  if constexpr (XDT == SMOE_F32) return reinterpret_cast<const float*>(x)[i];
  else if constexpr (XDT == SMOE_BF16) return bf2f(reinterpret_cast<const uint16_t*>(x)[i]);
  else return static_cast<float>(reinterpret_cast<const _Float16*>(x)[i]);
}

// Whether eight consecutive elements load as 16-byte vectors.
template <int XDT>
__device__ __forceinline__ bool vec8(const void* x) {
  return reinterpret_cast<uintptr_t>(x) % 16 == 0;
}

// Elements i .. i + 7 (i a multiple of 8, x as vec8 asks).
template <int XDT>
__device__ __forceinline__ void load_x8(const void* x, int64_t i, float (&v)[8]) {
  if constexpr (XDT == SMOE_F32) {
    const f32x4* p = reinterpret_cast<const f32x4*>(reinterpret_cast<const float*>(x) + i);
    const f32x4 a = p[0], b = p[1];
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      v[j] = a[j];
      v[4 + j] = b[j];
    }
  } else {
    const u32x4 a = *reinterpret_cast<const u32x4*>(reinterpret_cast<const uint16_t*>(x) + i);
#pragma unroll
    for (int j = 0; j < 8; ++j) {
      const uint16_t h = static_cast<uint16_t>(a[j >> 1] >> (16 * (j & 1)));
      v[j] = XDT == SMOE_BF16 ? bf2f(h) : static_cast<float>(__builtin_bit_cast(_Float16, h));
    }
  }
}

// Partial amax |x| of each workgroup's grid-stride share: 8 elements a lane
// and load, the rest one by one (n % 8, unaligned x).
template <int XDT>
__global__ __launch_bounds__(256) void k_amax_partial(const void* __restrict__ x, int64_t n,
                                                      float* __restrict__ partial) {
  __shared__ float red[4];
  float m = 0.f;
  const int64_t t = static_cast<int64_t>(blockIdx.x) * 256 + threadIdx.x;
  const int64_t stride = static_cast<int64_t>(gridDim.x) * 256;
  const int64_t octs = vec8<XDT>(x) ? n >> 3 : 0;
  for (int64_t o = t; o < octs; o += stride) {
    float v[8];
    load_x8<XDT>(x, 8 * o, v);
#pragma unroll
    for (int j = 0; j < 8; ++j) m = nan_max(m, fabsf(v[j]));
  }
  for (int64_t i = 8 * octs + t; i < n; i += stride) m = nan_max(m, fabsf(load_x<XDT>(x, i)));
  m = wave_nan_max(m);
  if ((threadIdx.x & 63) == 0) red[threadIdx.x >> 6] = m;
  __syncthreads();
  if (threadIdx.x == 0)
    partial[blockIdx.x] = nan_max(nan_max(red[0], red[1]), nan_max(red[2], red[3]));
}

// scale = max(amax / 448, 1e-12) (quant.py:30-33), codes = e4m3(x / scale)
// (quant.py:52), 8 codes per thread (4 where rows are not whole 16-byte
// vectors); columns cols .. ld_out-1 of each row are written as code 0 (value
// 0: the GEMM's K padding).  Every workgroup reduces the partials itself, its
// 256 threads loading them at once; one wave in a loop of 16 dependent loads
// was half the launch (4096 x 1024 bf16: 15.6 -> 9.0 us with the wider
// accesses, the amax pass 6.3 -> 4.1; both launches back to back with rows of
// 1004, four codes at a time: 20.5 -> 12.4, and 13.3 with twice the workgroups).
template <int XDT>
__global__ __launch_bounds__(256) void k_quant_fp8(const void* __restrict__ x, int rows, int cols,
                                                   int ld_out, const float* __restrict__ partial,
                                                   int nparts, uint8_t* __restrict__ codes,
                                                   float* __restrict__ scale_out) {
  __shared__ float red[4];
  {
    float v[kAmaxParts / 256];
#pragma unroll
    for (int i = 0; i < kAmaxParts / 256; ++i)  // unconditional loads at clamped indices
      v[i] = partial[min(static_cast<int>(threadIdx.x) + 256 * i, nparts - 1)];
    float m = 0.f;
#pragma unroll
    for (int i = 0; i < kAmaxParts / 256; ++i) m = nan_max(m, v[i]);
    m = wave_nan_max(m);
    if ((threadIdx.x & 63) == 0) red[threadIdx.x >> 6] = m;
  }
  __syncthreads();
  float sc = __fdiv_rn(nan_max(nan_max(red[0], red[1]), nan_max(red[2], red[3])), kE4m3Max);
  sc = sc < 1e-12f ? 1e-12f : sc;  // clamp_min (a NaN scale stays NaN)
  if (blockIdx.x == 0 && threadIdx.x == 0) *scale_out = sc;
  const int64_t t = static_cast<int64_t>(blockIdx.x) * 256 + threadIdx.x;
  const int64_t stride = static_cast<int64_t>(gridDim.x) * 256;
  if (vec8<XDT>(x) && cols % 8 == 0 && ld_out % 8 == 0 && reinterpret_cast<uintptr_t>(codes) % 8 == 0) {
    const int octs = ld_out >> 3;
    const int64_t total = static_cast<int64_t>(rows) * octs;
    for (int64_t o = t; o < total; o += stride) {
      const int r = static_cast<int>(o / octs);
      const int c = static_cast<int>(o - static_cast<int64_t>(r) * octs) * 8;
      u32x2 w = {0u, 0u};
      if (c < cols) {
        float v[8];
        load_x8<XDT>(x, static_cast<int64_t>(r) * cols + c, v);
#pragma unroll
        for (int j = 0; j < 8; ++j) w[j >> 2] |= f32_to_e4m3(__fdiv_rn(v[j], sc)) << (8 * (j & 3));
      }
      *reinterpret_cast<u32x2*>(codes + static_cast<int64_t>(r) * ld_out + c) = w;
    }
    return;
  }
  const int quads = ld_out >> 2;
  const int64_t total = static_cast<int64_t>(rows) * quads;
  for (int64_t q = t; q < total; q += stride) {
    const int r = static_cast<int>(q / quads);
    const int c0 = static_cast<int>(q - static_cast<int64_t>(r) * quads) * 4;
    uint32_t word = 0;
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const int c = c0 + i;
      if (c < cols) {
        const float v = load_x<XDT>(x, static_cast<int64_t>(r) * cols + c);
        word |= f32_to_e4m3(__fdiv_rn(v, sc)) << (8 * i);
      }
    }
    *reinterpret_cast<uint32_t*>(codes + static_cast<int64_t>(r) * ld_out + c0) = word;
  }
}

// Per-row scales (quant.py:146-169 with a per-row amax, the block's fp8
// expert format): one wave per row, scale[r] = max(amax_r / 448, 1e-12),
// codes = e4m3(x / scale[r]); columns cols .. ld_out-1 get code 0.
template <int XDT>
__global__ __launch_bounds__(256) void k_quant_fp8_rows(const void* __restrict__ x, int rows,
                                                        int cols, int ld_out,
                                                        uint8_t* __restrict__ codes,
                                                        float* __restrict__ scale) {
  const int lane = threadIdx.x & 63;
  const int r = blockIdx.x * 4 + (threadIdx.x >> 6);
  if (r >= rows) return;  // wave-uniform
  const int64_t rb = static_cast<int64_t>(r) * cols;
  float m = 0.f;
  for (int c = lane; c < cols; c += 64) m = nan_max(m, fabsf(load_x<XDT>(x, rb + c)));
  m = wave_nan_max(m);
  float sc = __fdiv_rn(m, kE4m3Max);
  sc = sc < 1e-12f ? 1e-12f : sc;
  if (lane == 0) scale[r] = sc;
  for (int q = lane; q < (ld_out >> 2); q += 64) {
    uint32_t word = 0;
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const int c = 4 * q + i;
      if (c < cols) word |= f32_to_e4m3(__fdiv_rn(load_x<XDT>(x, rb + c), sc)) << (8 * i);
    }
    *reinterpret_cast<uint32_t*>(codes + static_cast<int64_t>(r) * ld_out + 4 * q) = word;
  }
}

// out[m, n] = act(xs * ws * sum_k X[m, k] W[n, k] + bias[n]) over e4m3
// codes X [N, ldx], W [N_out, ldw] (K a multiple of 256, zero-padded: the row
// length packed weights are kept in by the entry point's contract; the loop
// itself needs 128).
//
// 128 x 128 block tile, 4 waves in a 2 x 2 grid (wave tile 64 x 64), K
// advancing 128 per stage (128-byte rows, swizzled as sw_chunk says) through a
// 2-stage LDS ring (32 KB a stage) fed by global_load_lds_dwordx4; a lane's
// 32-byte MFMA fragment (row l % 16, k bytes 32 (l / 16) ..) is two
// ds_read_b128.  Both operands use the same lane -> k assignment, so every lane
// group multiplies matching k.  A launch is a few stages long (K 1024: 8) and
// waits for memory in every one, so two workgroups share a CU.  1024 -> 2816,
// 4096 rows, bf16 out: 44.5 -> 27 us (875 TFLOP/s) against one workgroup with
// a 3-stage ring of 64-byte rows, fragments a stage ahead in registers and
// 8-byte stores.  Workgroup ids are dealt to the 8 XCDs round robin and each
// XCD takes one contiguous part of the tiles, row tile by row tile, so its
// rows and the weights stay in its L2.
template <int EPI, int ODT>
__global__ __launch_bounds__(256, 2) void k_gemm_f8f8(const uint8_t* __restrict__ X, int ldx,
                                                      const uint8_t* __restrict__ W, int ldw,
                                                      const float* __restrict__ xs,
                                                      const float* __restrict__ ws,
                                                      const float* __restrict__ bias, int N, int K,
                                                      int N_out, void* __restrict__ out, int ldo,
                                                      int tiles_n) {
  constexpr int BM = 128, BN = 128, NS = 2, OPB = 128 * 128, STAGE = 2 * OPB, LD = 8;
  __shared__ __attribute__((aligned(1024))) uint8_t ring[NS * STAGE];
  const int T = gridDim.x, x = blockIdx.x & 7, rem = T & 7;
  const int logical = x * (T >> 3) + min(x, rem) + (blockIdx.x >> 3);
  const int m0 = logical / tiles_n * BM, n0 = logical % tiles_n * BN;
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const int wm = wave >> 1, wn = wave & 1;

  // DMA: instruction j of this wave covers rows 8 (4 (j % 4) + wave) .. of
  // operand j / 4 (X, W); lane i: row i / 8, physical chunk i % 8, loading the
  // logical chunk the swizzle puts there
  const uint8_t* src[LD];
#pragma unroll
  for (int j = 0; j < LD; ++j) {
    const int r = 8 * (4 * (j & 3) + wave) + (lane >> 3), c = 16 * sw_chunk<8>(r, lane & 7);
    // rows past the end: valid data, never stored
    src[j] = j < 4 ? X + static_cast<int64_t>(min(m0 + r, N - 1)) * ldx + c
                   : W + static_cast<int64_t>(min(n0 + r, N_out - 1)) * ldw + c;
  }
  auto issue = [&](int stage) {
    uint8_t* base = ring + (stage % NS) * STAGE;
#pragma unroll
    for (int j = 0; j < LD; ++j)
      __builtin_amdgcn_global_load_lds((gbl_vptr)(src[j] + static_cast<int64_t>(stage) * 128),
                                       (lds_vptr)(base + (j >> 2) * OPB + (4 * (j & 3) + wave) * 1024),
                                       16, 0, 0);
  };
  const int fr = lane & 15, g = lane >> 4;
  auto frag = [&](const uint8_t* op, int r) {
    const u32x4 lo = *reinterpret_cast<const u32x4*>(op + r * 128 + (sw_chunk<8>(r, 2 * g) << 4));
    const u32x4 hi = *reinterpret_cast<const u32x4*>(op + r * 128 + (sw_chunk<8>(r, 2 * g + 1) << 4));
    return __builtin_bit_cast(i32x8, (uint32_t __attribute__((ext_vector_type(8)))){
                                         lo.x, lo.y, lo.z, lo.w, hi.x, hi.y, hi.z, hi.w});
  };

  f32x4 acc[4][4];
#pragma unroll
  for (int j = 0; j < 4; ++j)
#pragma unroll
    for (int i = 0; i < 4; ++i) acc[j][i] = f32x4{0.f, 0.f, 0.f, 0.f};

  const int KT = K / 128;
  issue(0);
  for (int s = 0; s < KT; ++s) {
    // own part of stage s landed; after the barrier everybody's, and nobody
    // reads stage s - 1 any more
    wait_vmcnt<0>();
    wait_lgkm0();
    __builtin_amdgcn_s_barrier();
    if (s + 1 < KT) issue(s + 1);  // into the slot of stage s - 1
    const uint8_t* sx = ring + (s % NS) * STAGE;
    i32x8 xf[4], wf[4];
#pragma unroll
    for (int i = 0; i < 4; ++i) xf[i] = frag(sx, wm * 64 + i * 16 + fr);
#pragma unroll
    for (int j = 0; j < 4; ++j) wf[j] = frag(sx + OPB, wn * 64 + j * 16 + fr);
#pragma unroll
    for (int j = 0; j < 4; ++j)
#pragma unroll
      for (int i = 0; i < 4; ++i)
        acc[j][i] = __builtin_amdgcn_mfma_scale_f32_16x16x128_f8f6f4(wf[j], xf[i], acc[j][i], 0, 0, 0,
                                                                     0, 0, 0);
  }

  // epilogue: lane holds channels n .. n+3 (4 (l / 16) + v) of row m (l % 16)
  const float sc = xs[0] * ws[0];
  float b4[4][4];
#pragma unroll
  for (int j = 0; j < 4; ++j) {
    const int n = n0 + wn * 64 + j * 16 + 4 * g;
#pragma unroll
    for (int v = 0; v < 4; ++v) b4[j][v] = (bias && n + v < N_out) ? bias[n + v] : 0.f;
  }
  auto value = [&](int i, int j, int v) {
    const float y = acc[j][i][v] * sc + b4[j][v];
    return EPI == 1 ? gelu_erf(y) : y;
  };
  if constexpr (ODT == SMOE_BF16) {
    // whole 16-byte chunks: the tile is staged in the ring (chunk c of row r
    // at c ^ (r & 15)) and leaves in rows of 256 bytes
    if (N_out % 8 == 0 && ldo % 8 == 0 && reinterpret_cast<uintptr_t>(out) % 16 == 0) {
      uint16_t* stg = reinterpret_cast<uint16_t*>(ring);
      auto at = [&](int r, int c) { return stg + r * BN + ((((c >> 3) ^ (r & 15)) << 3) | (c & 7)); };
      __syncthreads();  // every wave is done with the ring
#pragma unroll
      for (int j = 0; j < 4; ++j)
#pragma unroll
        for (int i = 0; i < 4; ++i)
          *reinterpret_cast<u32x2*>(at(wm * 64 + i * 16 + fr, wn * 64 + j * 16 + 4 * g)) =
              u32x2{pack_bf2(value(i, j, 0), value(i, j, 1)), pack_bf2(value(i, j, 2), value(i, j, 3))};
      __syncthreads();
      for (int q = tid; q < BM * (BN / 8); q += 256) {
        const int r = q / (BN / 8), c = q % (BN / 8) * 8;
        if (m0 + r < N && n0 + c < N_out)
          *reinterpret_cast<u32x4*>(reinterpret_cast<uint16_t*>(out) +
                                    static_cast<int64_t>(m0 + r) * ldo + n0 + c) =
              *reinterpret_cast<const u32x4*>(at(r, c));
      }
      return;
    }
  }
#pragma unroll
  for (int j = 0; j < 4; ++j) {
    const int n = n0 + wn * 64 + j * 16 + 4 * g;
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const int m = m0 + wm * 64 + i * 16 + fr;
      if (m >= N) continue;
      float o[4];
#pragma unroll
      for (int v = 0; v < 4; ++v) o[v] = value(i, j, v);
      const int64_t base = static_cast<int64_t>(m) * ldo + n;
      if (ODT == SMOE_F32) {
        float* po = reinterpret_cast<float*>(out) + base;
        if (n + 3 < N_out && (base & 3) == 0) {
          *reinterpret_cast<f32x4*>(po) = f32x4{o[0], o[1], o[2], o[3]};
        } else {
#pragma unroll
          for (int v = 0; v < 4; ++v)
            if (n + v < N_out) po[v] = o[v];
        }
      } else {
        uint16_t* po = reinterpret_cast<uint16_t*>(out) + base;
        if (n + 3 < N_out && (base & 3) == 0) {
          *reinterpret_cast<u32x2*>(po) = u32x2{pack_bf2(o[0], o[1]), pack_bf2(o[2], o[3])};
        } else {
#pragma unroll
          for (int v = 0; v < 4; ++v)
            if (n + v < N_out) po[v] = f2bf(o[v]);
        }
      }
    }
  }
}

int rc() { return hipGetLastError() == hipSuccess ? SMOE_OK : SMOE_EHIP; }

}  // namespace

size_t quantize_fp8_workspace_bytes() { return kAmaxParts * sizeof(float); }

int launch_quantize_fp8(const void* x, int xdt, int rows, int cols, int ld_out, int per_row,
                        uint8_t* codes, float* scale, void* workspace, hipStream_t s) {
  if (rows < 1 || cols < 1 || ld_out < cols || ld_out % 4) return SMOE_EINVAL;
  if (per_row) {
    auto go = [&](auto xd) {
      hipLaunchKernelGGL((k_quant_fp8_rows<decltype(xd)::value>), dim3((rows + 3) / 4), dim3(256),
                         0, s, x, rows, cols, ld_out, codes, scale);
      return rc();
    };
    switch (xdt) {
      case SMOE_F32: return go(std::integral_constant<int, SMOE_F32>{});
      case SMOE_BF16: return go(std::integral_constant<int, SMOE_BF16>{});
      case SMOE_F16: return go(std::integral_constant<int, SMOE_F16>{});
      default: return SMOE_EUNSUPPORTED;
    }
  }
  const int64_t n = static_cast<int64_t>(rows) * cols;
  const int parts = static_cast<int>(std::min<int64_t>(kAmaxParts, (n + 4095) / 4096));
  float* partial = static_cast<float*>(workspace);
  const int64_t quads = static_cast<int64_t>(rows) * (ld_out / 4);
  const int qblocks = static_cast<int>(std::min<int64_t>(2048, (quads + 511) / 512));
  auto run = [&](auto xd) {
    constexpr int XD = decltype(xd)::value;
    hipLaunchKernelGGL((k_amax_partial<XD>), dim3(parts), dim3(256), 0, s, x, n, partial);
    hipLaunchKernelGGL((k_quant_fp8<XD>), dim3(qblocks), dim3(256), 0, s, x, rows, cols, ld_out,
                       partial, parts, codes, scale);
    return rc();
  };
  switch (xdt) {
    case SMOE_F32: return run(std::integral_constant<int, SMOE_F32>{});
    case SMOE_BF16: return run(std::integral_constant<int, SMOE_BF16>{});
    case SMOE_F16: return run(std::integral_constant<int, SMOE_F16>{});
    default: return SMOE_EUNSUPPORTED;
  }
}

int launch_gemm_f8f8(const uint8_t* xq, int ldx, const float* xs, const uint8_t* wq, int ldw,
                     const float* ws, const float* bias, int N, int K, int N_out, int gelu,
                     void* out, int odt, int ldo, hipStream_t s) {
  if (N < 0 || K <= 0 || K % 256 || N_out <= 0 || ldx < K || ldw < K || ldx % 16 || ldw % 16 ||
      ldo < N_out)
    return SMOE_EINVAL;
  if (N == 0) return SMOE_OK;
  const int tiles_m = (N + 127) / 128, tiles_n = (N_out + 127) / 128;
  if (static_cast<int64_t>(tiles_m) * tiles_n > 0x7fffffff) return SMOE_EINVAL;
  const dim3 grid(tiles_m * tiles_n), block(256);
  auto go = [&](auto epi, auto od) {
    SMOE_LAUNCH((k_gemm_f8f8<decltype(epi)::value, decltype(od)::value>), grid, block, 0, s, xq,
                ldx, wq, ldw, xs, ws, bias, N, K, N_out, out, ldo, tiles_n);
    return rc();
  };
  using I0 = std::integral_constant<int, 0>;
  using I1 = std::integral_constant<int, 1>;
  using OF = std::integral_constant<int, SMOE_F32>;
  using OB = std::integral_constant<int, SMOE_BF16>;
  if (odt == SMOE_F32) return gelu ? go(I1{}, OF{}) : go(I0{}, OF{});
  if (odt == SMOE_BF16) return gelu ? go(I1{}, OB{}) : go(I0{}, OB{});
  return SMOE_EUNSUPPORTED;
}

}  // namespace smoe
