// Device helpers shared by the grouped GEMM kernels: the tile lookup over a
// plan's groups, the tile order, the weight widening and the epilogues.
#pragma once
#include <type_traits>

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

// A lane's raw 16 consecutive k of one weight row, in its storage format
// (only what the format needs stays in registers).
template <int FMT> struct WRaw;
template <> struct WRaw<SMOE_BF16> { u32x4 a, b; };
template <> struct WRaw<SMOE_FP8_E4M3> { u32x4 a; };
template <> struct WRaw<SMOE_INT4> { u32x2 a; float s; };  // 16 nibbles + their group scale

// The raw 16 k of a lane -> the bf16 A operands of the step's two MFMAs.
template <int FMT>
__device__ __forceinline__ void skinny_wconv(const WRaw<FMT>& r, bf16x8& lo, bf16x8& hi) {
  u32x4 l, h;
  if constexpr (FMT == SMOE_BF16) {
    l = r.a;
    h = r.b;
  } else if constexpr (FMT == SMOE_FP8_E4M3) {
    const u32x2 a0 = fp8x4_to_bf16x4(r.a.x), a1 = fp8x4_to_bf16x4(r.a.y);
    const u32x2 b0 = fp8x4_to_bf16x4(r.a.z), b1 = fp8x4_to_bf16x4(r.a.w);
    l = u32x4{a0.x, a0.y, a1.x, a1.y};
    h = u32x4{b0.x, b0.y, b1.x, b1.y};
  } else {
    l = int4x8_to_bf16x8(r.a.x, r.s);
    h = int4x8_to_bf16x8(r.a.y, r.s);
  }
  lo = __builtin_bit_cast(bf16x8, l);
  hi = __builtin_bit_cast(bf16x8, h);
}

// ------------------------------------------------ tile order, 4-wide out ----
// Tile order of the large-tile kernels: the tile grid (real count, from the
// plan) is split into 8 contiguous ranges, one per XCD (workgroup ids are
// dealt to XCDs round robin), and each range is walked in super-rows of GM
// m-tiles x all n-tiles so the super-row's A tiles stay in that XCD's L2
// while weight tiles stream.
template <int BM>
__device__ __forceinline__ int count_m_tiles(const GemmArgs& p) {
  return count_tiles(p, BM);
}

// Row tiles on 16-row bands (an operand or the output in the row-tile
// layout): group g's tiles start at its first row rounded down to a multiple
// of 16, BM rows apart; a tile's live rows are the group's, [rlo, rhi) in
// tile rows.  A band shared by two groups is computed by a tile of each, and
// each stores only its own rows.
__device__ __forceinline__ void band_chunk(const GemmArgs& p, int BM, int b, int& lo, int& hi,
                                           int& t) {
  const int i = b + static_cast<int>(threadIdx.x & 63);
  const int ic = i < p.G ? i : p.G - 1;
  lo = p.grp_off[ic];
  hi = p.grp_off[ic + 1];
  t = (i < p.G && hi > lo) ? (hi - (lo & ~15) + BM - 1) / BM : 0;
}

__device__ __forceinline__ int count_band_tiles(const GemmArgs& p, int BM) {
  if (p.G == 0) return (p.single_rows + BM - 1) / BM;
  int total = 0;
  for (int b = 0; b < p.G; b += 64) {
    int lo, hi, t;
    band_chunk(p, BM, b, lo, hi, t);
    total += __builtin_amdgcn_readlane(wave_incl_scan(t), 63);
  }
  return total;
}

__device__ __forceinline__ bool find_band_tile(const GemmArgs& p, int BM, int tile, int& g, int& m0,
                                               int& rlo, int& rhi) {
  if (p.G == 0) {
    int mrows;
    if (!find_tile(p, BM, tile, g, m0, mrows)) return false;
    rlo = 0;
    rhi = mrows;
    return true;
  }
  int acc = 0;
  for (int b = 0; b < p.G; b += 64) {
    int lo, hi, t;
    band_chunk(p, BM, b, lo, hi, t);
    const int incl = wave_incl_scan(t) + acc;
    const uint64_t m = __ballot(tile < incl);
    if (m) {
      const int f = __builtin_ctzll(m);
      g = b + f;
      const int excl = __builtin_amdgcn_readlane(incl - t, f);
      const int glo = __builtin_amdgcn_readlane(lo, f), ghi = __builtin_amdgcn_readlane(hi, f);
      m0 = (glo & ~15) + (tile - excl) * BM;
      rlo = max(glo - m0, 0);
      rhi = min(ghi - m0, BM);
      return true;
    }
    acc = __builtin_amdgcn_readlane(incl, 63);
  }
  return false;
}

__device__ __forceinline__ bool row_tiles(const GemmArgs& p) { return p.At != nullptr || p.out_tiles; }

// The tile of workgroup bid: group, first row m0, live rows
// [rlo, rhi) in tile rows (rlo > 0 only for band-aligned tiles), first
// output channel.  Workgroup ids are dealt to the 8 XCDs round robin
// (bid & 7 is the XCD).
template <int BM, int BN, int GM>
__device__ __forceinline__ bool big_tile(const GemmArgs& p, int bid, int& g, int& m0, int& rlo,
                                         int& rhi, int& n0) {
  const bool bands = row_tiles(p);
  const int tn_count = (p.N_out + BN - 1) / BN;
  const int tm_count = bands ? count_band_tiles(p, BM) : count_m_tiles<BM>(p);
  const int T = tm_count * tn_count;
  if (bid >= T) return false;
  const int x = bid & 7, local = bid >> 3;
  const int base = T >> 3, rem = T & 7;
  const int logical = x * base + min(x, rem) + local;
  const int grp = logical / (GM * tn_count);
  const int first_m = grp * GM;
  const int gsize = min(GM, tm_count - first_m);
  const int in = logical - grp * GM * tn_count;
  const int tm = first_m + in % gsize;
  n0 = (in / gsize) * BN;
  if (bands) return find_band_tile(p, BM, tm, g, m0, rlo, rhi);
  int mrows;
  if (!find_tile(p, BM, tm, g, m0, mrows)) return false;
  rlo = 0;
  rhi = mrows;
  return true;
}

// Epilogue of an LDS-staged tile: math in registers, the bf16 tile staged
// in the (idle) LDS ring, then coalesced 16-byte stores.  Staging layout:
// row r, 16-byte chunk c at chunk c ^ (r & 15) (rows of OW bf16, no padding;
// r & 7 for 8-chunk rows).  Only the live rows [rlo, rhi) are stored, and
// 16-row strips without any are skipped.  With p.out_tiles the stores follow
// the row-tile layout (m0 a multiple of 16): 64 consecutive threads write
// one 1 KB block (16 rows x 32 columns).
//
// The lane's bias values (4 channels of each fragment column; SwiGLU: of its
// up columns) and the row scales of its strips are loaded before any math
// (one memory round trip for the whole epilogue).  The costly activations
// (SwiGLU; GELU of small wave tiles) are computed into packed registers
// before the workgroup barrier that frees the ring (the caller need not
// synchronise), so one wave row's math overlaps the other's last MFMAs; the
// others are computed as they are staged (a packed tile of 4 channels per
// fragment column would not fit beside the accumulators).
// Without a bias (the SwiGLU experts) its loads and adds are compiled out.
// fp8 weights (WF): each channel's scale multiplies its accumulator first.
template <int BM, int BN, int TM, int TN, int NT, int EPI, int WF = SMOE_BF16>
__device__ __forceinline__ void tile_epilogue(const GemmArgs& p, const f32x4 (&acc)[TN / 16][TM / 16],
                                              int g, int m0, int rlo, int rhi, int n0, int wm,
                                              int wn, uint8_t* ring) {
  constexpr int FM = TM / 16, FN = TN / 16;
  constexpr int OW = (EPI == EPI_SWIGLU) ? BN / 2 : BN;  // output columns of the tile
  constexpr int SWM = (OW / 8 >= 16 ? 16 : OW / 8) - 1;  // chunk swizzle mask
  constexpr bool HAS_BIAS = EPI != EPI_ROWSCALE;
  constexpr bool HAS_RS = EPI == EPI_ROWSCALE || EPI == EPI_DOWN;
  constexpr int NJ = (EPI == EPI_SWIGLU) ? FN / 2 : FN;  // output fragment columns
  constexpr bool EARLY = EPI == EPI_SWIGLU || (EPI == EPI_GELU && FM * NJ <= 16);
  const int tid = threadIdx.x, lane = tid & 63;
  const int fr = lane & 15, fc = lane >> 4;
  uint16_t* stg = reinterpret_cast<uint16_t*>(ring);
  auto stg_at = [&](int r, int col) {  // staging row r, col: multiple of 4
    return stg + r * OW + ((((col >> 3) ^ (r & SWM)) << 3) | (col & 7));
  };
  const int ncol0 = (EPI == EPI_SWIGLU) ? (n0 >> 1) : n0;
  const int ncols = (EPI == EPI_SWIGLU) ? (p.N_out >> 1) : p.N_out;  // a last tile may be partial
  auto live = [&](int i) {  // strip i holds a live row (wave-uniform)
    const int tr0 = wm * TM + i * 16;
    return tr0 < rhi && tr0 + 16 > rlo;
  };
  constexpr bool F8 = WF == SMOE_FP8_E4M3;
  auto body = [&](auto with_bias) {
    constexpr bool WB = HAS_BIAS && decltype(with_bias)::value;
    float bq[WB ? NJ : 1][4];
    float rsv[HAS_RS ? FM : 1];
    // fp8 channel scales: [fragment column][channel] (SwiGLU: gate, then up 32 on)
    float sc[F8 ? FN : 1][4];
    if constexpr (F8) {
#pragma unroll
      for (int j = 0; j < FN; ++j) {
        const int c = n0 + wn * TN + j * 16 + fc * 4;
#pragma unroll
        for (int q = 0; q < 4; ++q)
          sc[j][q] = c + q < p.N_out
                         ? reinterpret_cast<const float*>(p.S)[g * p.s_gstride + c + q]
                         : 0.f;
      }
    }
    if constexpr (WB) {
#pragma unroll
      for (int j = 0, b = 0; j < FN; ++j) {
        if (EPI == EPI_SWIGLU && (j & 3) >= 2) continue;
        const int cl = wn * TN + j * 16 + fc * 4;
        const int c = (EPI == EPI_SWIGLU) ? (n0 >> 1) + (cl >> 6) * 32 + (cl & 31) : n0 + cl;
#pragma unroll
        for (int q = 0; q < 4; ++q) bq[b][q] = c + q < ncols ? bias_at(p, g, c + q) : 0.f;
        ++b;
      }
    }
    if constexpr (HAS_RS) {
#pragma unroll
      for (int i = 0; i < FM; ++i) {
        const int lr = wm * TM + i * 16 + fr;
        rsv[i] = lr >= rlo && lr < rhi ? p.row_scale[m0 + lr] : 0.f;
      }
    }
    // the packed outputs of strip i, fragment column j (bias slot b)
    auto value = [&](int i, int j, int b) {
      float r[4];
#pragma unroll
      for (int q = 0; q < 4; ++q) {
        if constexpr (EPI == EPI_SWIGLU) {
          const float gate = F8 ? acc[j][i][q] * sc[F8 ? j : 0][q] : acc[j][i][q];
          const float up = F8 ? acc[j + 2][i][q] * sc[F8 ? j + 2 : 0][q] : acc[j + 2][i][q];
          r[q] = silu(gate) * (WB ? up + bq[WB ? b : 0][q] : up);
        } else {
          const float v = F8 ? acc[j][i][q] * sc[F8 ? j : 0][q] : acc[j][i][q];
          const float a = WB ? v + bq[WB ? b : 0][q] : v;
          if constexpr (HAS_RS) r[q] = a * rsv[HAS_RS ? i : 0];
          else if constexpr (EPI == EPI_GELU) r[q] = gelu_erf(a);
          else r[q] = a;
        }
      }
      return u32x2{pack_bf2(r[0], r[1]), pack_bf2(r[2], r[3])};
    };
    u32x2 pk[EARLY ? FM : 1][NJ];
    if constexpr (EARLY) {
#pragma unroll
      for (int i = 0; i < FM; ++i) {
        if (!live(i)) continue;
#pragma unroll
        for (int j = 0, b = 0; j < FN; ++j) {
          if (EPI == EPI_SWIGLU && (j & 3) >= 2) continue;
          pk[i][b] = value(i, j, b);
          ++b;
        }
      }
    }
    __syncthreads();  // every wave is done with the ring: it becomes the staging buffer
#pragma unroll
    for (int i = 0; i < FM; ++i) {
      if (!live(i)) continue;
      const int sr = wm * TM + i * 16 + fr;  // staging row = tile row
#pragma unroll
      for (int j = 0, b = 0; j < FN; ++j) {
        if (EPI == EPI_SWIGLU && (j & 3) >= 2) continue;
        const int cl = wn * TN + j * 16 + fc * 4;  // channel within the tile
        const int col = (EPI == EPI_SWIGLU) ? (cl >> 6) * 32 + (cl & 31) : cl;
        *reinterpret_cast<u32x2*>(stg_at(sr, col)) = EARLY ? pk[EARLY ? i : 0][b] : value(i, j, b);
        ++b;
      }
    }
  };
  if (!HAS_BIAS || p.bias) body(std::true_type{});
  else body(std::false_type{});
  __syncthreads();
  uint16_t* out = reinterpret_cast<uint16_t*>(p.out);
  if (p.out_tiles) {
    constexpr int KB = OW / 32;  // 32-column blocks per tile row band
    const int ldb = p.ldo >> 5;  // blocks per band of the whole output
    for (int q = tid; q < BM / 16 * KB * 64; q += NT) {
      const int blk = q >> 6, l = q & 63;
      const int r = (blk / KB) * 16 + (l & 15), cc = (blk % KB) * 32 + (l >> 4) * 8;
      if (r >= rlo && r < rhi && ncol0 + cc < ncols)
        __builtin_nontemporal_store(
            *reinterpret_cast<const u32x4*>(stg_at(r, cc)),
            reinterpret_cast<u32x4*>(out + ((static_cast<int64_t>((m0 + r) >> 4) * ldb +
                                             ((ncol0 + cc) >> 5)) << 9) + 8 * l));
    }
    return;
  }
  constexpr int CPR_OUT = OW / 8;  // 16-byte chunks per output row
  for (int q = tid; q < BM * CPR_OUT; q += NT) {
    const int r = q / CPR_OUT, cc = (q % CPR_OUT) * 8;
    // non-temporal: every CU stores its tile at about the same time, and
    // the burst streams past the caches (the next kernel reads it once).
    // With the epilogue loads hoisted: C1's up GEMM 2.20 -> 2.15 ms per
    // step, C3's step 3.66 -> 3.49 ms.
    if (r >= rlo && r < rhi && ncol0 + cc < ncols)
      __builtin_nontemporal_store(
          *reinterpret_cast<const u32x4*>(stg_at(r, cc)),
          reinterpret_cast<u32x4*>(out + static_cast<int64_t>(m0 + r) * p.ldo + ncol0 + cc));
  }
}

}  // namespace smoe
