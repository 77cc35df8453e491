// Device helpers shared by the grouped GEMM kernels: the tile lookup over a
// plan's groups and the per-element epilogues.
#pragma once
#include "smoe_common.hpp"
#include "smoe_internal.hpp"

namespace smoe {

// Tile lookups over the plan's groups, wave-parallel: lane i holds group
// b + i of a 64-group chunk (offsets by one clamped load per lane), the
// per-group tile counts are prefix-summed by DPP, and the group holding a
// tile is the first lane whose inclusive count exceeds it (a ballot).  A
// serial loop over the groups would wait on one scalar load per group at the
// start of every workgroup.  Every lane of the wave must be active; the
// results are wave-uniform.
__device__ __forceinline__ void group_chunk(const GemmArgs& p, int BM, int b, int& lo, int& hi,
                                            int& t) {
  const int i = b + static_cast<int>(threadIdx.x & 63);
  const int ic = i < p.G ? i : p.G - 1;
  lo = p.grp_off[ic];
  hi = p.grp_off[ic + 1];
  t = i < p.G ? (hi - lo + BM - 1) / BM : 0;
}

// Number of BM-row tiles over all groups.
__device__ __forceinline__ int count_tiles(const GemmArgs& p, int BM) {
  if (p.G == 0) return (p.single_rows + BM - 1) / BM;
  int total = 0;
  for (int b = 0; b < p.G; b += 64) {
    int lo, hi, t;
    group_chunk(p, BM, b, lo, hi, t);
    total += __builtin_amdgcn_readlane(wave_incl_scan(t), 63);
  }
  return total;
}

// The tile-th BM-row tile in group order: group, first row, rows.  skip:
// the first `skip` tiles of every group are left out of the count (their
// workgroups find them directly).
__device__ __forceinline__ bool find_tile(const GemmArgs& p, int BM, int tile, int& g, int& m0,
                                          int& mrows, int skip = 0) {
  if (p.G == 0) {
    const int t = (p.single_rows + BM - 1) / BM;
    if (tile >= t) return false;
    g = 0;
    m0 = tile * BM;
    mrows = min(BM, p.single_rows - m0);
    return true;
  }
  int acc = 0;
  for (int b = 0; b < p.G; b += 64) {
    int lo, hi, t;
    group_chunk(p, BM, b, lo, hi, t);
    t = max(t - skip, 0);
    const int incl = wave_incl_scan(t) + acc;
    const uint64_t m = __ballot(tile < incl);  // empty groups never come first
    if (m) {
      const int f = __builtin_ctzll(m);
      g = b + f;
      const int excl = __builtin_amdgcn_readlane(incl - t, f);
      const int glo = __builtin_amdgcn_readlane(lo, f), ghi = __builtin_amdgcn_readlane(hi, f);
      m0 = glo + (tile - excl + skip) * BM;
      mrows = min(BM, ghi - m0);
      return true;
    }
    acc = __builtin_amdgcn_readlane(incl, 63);
  }
  return false;
}

__device__ __forceinline__ void store_out(void* out, int dtype, int64_t idx, float v) {
  if (dtype == SMOE_F32)
    reinterpret_cast<float*>(out)[idx] = v;
  else
    reinterpret_cast<uint16_t*>(out)[idx] = f2bf(v);
}

__device__ __forceinline__ float col_scale(const GemmArgs& p, int fmt, int g, int n) {
  if (fmt == SMOE_FP8_E4M3) return reinterpret_cast<const float*>(p.S)[g * p.s_gstride + n];
  return 1.0f;
}

__device__ __forceinline__ float bias_at(const GemmArgs& p, int g, int n) {
  return p.bias ? p.bias[g * p.bias_gstride + n] : 0.0f;
}

// Single-element epilogue (all but SwiGLU).
template <int EPI>
__device__ __forceinline__ void epi_one(const GemmArgs& p, int fmt, int g, int row, int n,
                                        float acc) {
  const int64_t o = static_cast<int64_t>(row) * p.ldo + n;
  if constexpr (EPI == EPI_F32_BIAS) {
    reinterpret_cast<float*>(p.out)[o] = acc * col_scale(p, fmt, g, n) + bias_at(p, g, n);
  } else if constexpr (EPI == EPI_ROWSCALE) {
    store_out(p.out, p.out_dtype, o, acc * p.row_scale[row]);
  } else if constexpr (EPI == EPI_GELU) {
    store_out(p.out, p.out_dtype, o, gelu_erf(acc * col_scale(p, fmt, g, n) + bias_at(p, g, n)));
  } else if constexpr (EPI == EPI_DOWN) {
    store_out(p.out, p.out_dtype, o,
              (acc * col_scale(p, fmt, g, n) + bias_at(p, g, n)) * p.row_scale[row]);
  }
}

// SwiGLU pair: interleaved column c (gate, c % 64 < 32) and c + 32 (up).
__device__ __forceinline__ void epi_swiglu(const GemmArgs& p, int fmt, int g, int row, int c,
                                           float gate, float up) {
  const int u = (c >> 6) * 32 + (c & 31);
  const float gs = gate * col_scale(p, fmt, g, c);
  const float us = up * col_scale(p, fmt, g, c + 32) + bias_at(p, g, u);
  store_out(p.out, p.out_dtype, static_cast<int64_t>(row) * p.ldo + u, silu(gs) * us);
}

template <int EPI>
__device__ __forceinline__ void store4(const GemmArgs& p, int fmt, int g, int row, int n, f32x4 v) {
  // 4 consecutive channels n..n+3 of one row
  const int64_t o = static_cast<int64_t>(row) * p.ldo + n;
  float r[4];
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    const float a = v[i] * col_scale(p, fmt, g, n + i);
    if constexpr (EPI == EPI_F32_BIAS)
      r[i] = a + ((p.W2 && n >= p.n_split) ? (p.bias2 ? p.bias2[n - p.n_split + i] : 0.f)
                                            : bias_at(p, g, n + i));
    else if constexpr (EPI == EPI_ROWSCALE) r[i] = v[i] * p.row_scale[row];
    else if constexpr (EPI == EPI_GELU) r[i] = gelu_erf(a + bias_at(p, g, n + i));
    else r[i] = (a + bias_at(p, g, n + i)) * p.row_scale[row];  // EPI_DOWN
  }
  if (EPI == EPI_F32_BIAS || p.out_dtype == SMOE_F32) {
    *reinterpret_cast<f32x4*>(reinterpret_cast<float*>(p.out) + o) = f32x4{r[0], r[1], r[2], r[3]};
  } else {
    *reinterpret_cast<u32x2*>(reinterpret_cast<uint16_t*>(p.out) + o) =
        u32x2{pack_bf2(r[0], r[1]), pack_bf2(r[2], r[3])};
  }
}

}  // namespace smoe
