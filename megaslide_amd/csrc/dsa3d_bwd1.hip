// First kernel of the matrix-core attention backward for gfx950 (bf16 or fp32
// storage, head_dim 32, 64, 96 or 128): one workgroup per (batch, head, frame,
// tile of 16 queries), over the same whole-box tables as the forward
// (dsa3d_box.h).  It rebuilds S = q K^T, takes every tap's value and coordinate
// derivatives from it, then does the same with dP = dO V^T in the same LDS, and
// writes the offset gradients and, for the second kernel, p times its dropout
// factor and ds * softmax_scale of every tap (fp32 storage: two fp32 arrays
// [token][head][tap]; bf16: one word of two fp16, p * factor and ds * scale / l1,
// with l1 = sum over the query's taps of |ds * scale| per token and head).
//
// Bound: like the forward, waiting for the K and V rows' loads (0.53 of a wave's life,
// 0.73 of all requests hit the L2) and VALU issue (2,379 instructions a wave, 50 %);
// then the per-tap results (26 bytes a tap in bf16 with records).  Against tables
// of one plane at a time, two of them (S and dP) double-buffered: 4.37 -> 4.05 ms
// at 65,536 tokens, 16 x 64, bf16; 6.84 -> 6.40 ms at 46,800 tokens, 16 x 96,
// offsets biased by up to 4 units; 16.3 -> 16.1 ms at 131,072 tokens, 24 x 128;
// 1.90 -> 1.75 ms at 32,768 tokens, 8 x 64, fp32; 120 -> 74 us at 2,048 tokens,
// 16 x 64, window 3x5x5.
#include <algorithm>
#include <type_traits>

#include "dsa3d_box.h"
#include "dsa3d_bwd1.h"

namespace msd {

namespace {

using namespace tiled;

// A tap's interpolated value and its derivatives with respect to the sampling
// coordinates, from a table (EDGE: see box_gather; the derivative along an axis with
// upper weight 1 is masked, the position is on the volume's last voxel).
struct TapGrad {
  float v, dx, dy, dz;
};
template <bool EDGE>
__device__ __forceinline__ TapGrad box_gather_grad(const float* table, const BoxTap& t, int dx,
                                                   int dy, int dz) {
  const float* const p = &table[t.at];
  const float* const pz = p + dz;
  auto plane = [&](const float* q) {
    float t0 = q[0], t1 = q[dx], b0 = q[dy], b1 = q[dy + dx];
    if (EDGE && t.fx == 1.0f) {
      t0 = t1;
      b0 = b1;
    }
    if (EDGE && t.fy == 1.0f) {
      t0 = b0;
      t1 = b1;
    }
    return bilerp(t.fx, t.fy, t0, t1, b0, b1);
  };
  Bilerp lo = plane(p);
  if (EDGE && dz == 0) return TapGrad{lo.val, lo.dx, lo.dy, 0.0f};  // one frame (uniform)
  const Bilerp hi = plane(pz);
  if (EDGE && t.fz == 1.0f) lo = hi;
  const float gz = 1.0f - t.fz;
  TapGrad r;
  r.v = __builtin_fmaf(t.fz, hi.val, gz * lo.val);
  r.dx = __builtin_fmaf(t.fz, hi.dx, gz * lo.dx);
  r.dy = __builtin_fmaf(t.fz, hi.dy, gz * lo.dy);
  r.dz = hi.val - lo.val;
  return r;
}

// AE: bytes of one dK / dV accumulator element (4 = fp32 rows, 2 = scaled fp16).
// REC: also write the tap records, tile header and transposed q / dO of the
// column-streaming kernel (bf16 storage).  SPLIT: the scores' sums in short chains
// (padded head sizes, box_scores_split), and
// rc.collist set where a tap's gradient is not finite.
template <int HD, typename E, int AE, bool REC, bool DROP, bool SPLIT>
__global__ __launch_bounds__(kThreads, 4) void dsa3d_bwd_p1_kernel(
    Args a, const E* __restrict__ dout, const float* __restrict__ lse,
    const float* __restrict__ dlse, E* __restrict__ doff, float* __restrict__ p_ws,
    float* __restrict__ b_ws, void* __restrict__ dk_acc, void* __restrict__ dv_acc, int64_t acc_ks,
    int64_t acc_vs, RecArgs rc) {
  static_assert(!REC || sizeof(E) == 2, "the records carry bf16 storage's fp16 pairs");
  __shared__ __attribute__((aligned(16))) float s_tab[kTQ * kBoxRow];
  __shared__ uint32_t s_row[kBoxCap];
  __shared__ int s_box[8];
  __shared__ int s_bin[REC ? 2 * kRecBins : 1];  // record bins: counts, then starts
  __shared__ float s_l1[REC ? kTQ : 1];
  const int unit = box_unit(a);
  if (unit < 0) return;  // the grid is rounded up to the 8 XCDs
  const Tile tl = box_tile(a, unit, threadIdx.x);
  const int D = a.nh * HD;
  BoxTaps<kSlots> tp;
  BoxPieces bx;
  op_t<E> x[HD / 32];
  {
    RawOffsets<E, kSlots> raw;
    box_load_offsets<E, kSlots>(a, tl, raw);
    box_tile_rows<HD, E, E, false>(a, tl, static_cast<const E*>(a.q), a.qs, HD, x);
    box_init(s_box);
    if (REC && threadIdx.x < kRecBins) s_bin[threadIdx.x] = 0;
    __syncthreads();
    box_setup<E, kSlots, true, DROP, false>(a, tl, raw, tp, bx, s_box);
  }
  {
    // The second kernel adds dK and dV into accumulator rows (the fp32 outputs
    // for fp32 storage, fp32 or scaled fp16 rows for bf16): zero this tile's
    // rows of the head first (the tiles of a launch partition the (token, head)
    // pairs, and the second kernel starts after this one ends), 16 bytes a thread.
    constexpr int CPR = HD * AE / 16;
    for (int e = threadIdx.x; e < 2 * kTQ * CPR; e += kThreads) {
      const int t = e / (kTQ * CPR), m = (e / CPR) % kTQ, ch = (e % CPR) * (16 / AE);
      const int64_t row = tile_row(a, tl, m);
      if (row < 0) continue;
      const int64_t el = row * (t == 0 ? acc_ks : acc_vs) + tl.head * HD + ch;
      char* dst = static_cast<char*>(t == 0 ? dk_acc : dv_acc) + el * AE;
      *reinterpret_cast<uint4*>(dst) = uint4{0u, 0u, 0u, 0u};
    }
  }

  // ---- per tap: the interpolated S, then dP, and their derivatives ------------
  constexpr int NB = box_score_blocks<HD, E>() > 4 ? 4 : box_score_blocks<HD, E>();
  TapGrad ts[kSlots], td[kSlots];
#pragma unroll
  for (int i = 0; i < kSlots; ++i) ts[i] = td[i] = TapGrad{0.0f, 0.0f, 0.0f, 0.0f};
  auto sweep = [&](const void* base, int64_t stride, bool keep_rows, TapGrad (&tg)[kSlots]) {
    const E* const p = static_cast<const E*>(base) + tl.sample0 * stride + tl.head * HD;
    const __amdgpu_buffer_rsrc_t rows =
        box_rows(p, ((a.N - 1) * stride + HD) * static_cast<int64_t>(sizeof(E)));
    auto row_off = [&](int v) { return s_row[v]; };
    auto piece = [&](int s, auto only) __attribute__((always_inline)) {  // `only`: of one
      constexpr bool kOnly = decltype(only)::value;
      const BoxSeg g = box_seg(bx, s);
      if (!kOnly || !keep_rows)
        box_row_offsets(a, tl, bx, g, static_cast<uint32_t>(stride * sizeof(E)), s_row);
      if constexpr (SPLIT) box_scores_split<HD, E, false>(tl, rows, row_off, bx.nv, HD, x, s_tab);
      else box_scores<HD, E, E, false, NB>(tl, rows, row_off, bx.nv, HD, x, s_tab);
      __syncthreads();
      auto gather = [&](auto edge) __attribute__((always_inline)) {
#pragma unroll
        for (int i = 0; i < kSlots; ++i) {
          if (kSubs * i >= a.K) continue;
          BoxTap t = box_tap(tp, i);
          if (!kOnly && !box_in(g, tl.q, t)) continue;
          tg[i] = box_gather_grad<decltype(edge)::value>(s_tab, t, kOnly ? 1 : bx.dx, bx.dy, bx.dz);
        }
      };
      if (kOnly && !bx.edge) gather(std::false_type{});
      else gather(std::true_type{});
      __syncthreads();  // the next table takes this one's place
    };
    if (bx.n == 1) {
      piece(0, std::true_type{});
    } else {
#pragma nounroll
      for (int s = 0; s < bx.n; ++s) piece(s, std::false_type{});
    }
  };
  sweep(a.k, a.ks, false, ts);
  box_tile_rows<HD, E, E, false>(a, tl, dout, D, HD, x);
  sweep(a.v, a.vs, a.vs == a.ks, td);

  // Delta = dO . O - dlse.  dO . O = sum_k p_k f_k dP_k over the query's taps
  // plus, with extra keys, the same sum over the keys (formed by their kernel
  // before this one): neither sees the rounding of the stored output (bf16
  // storage), which a peaked softmax would otherwise turn into ds errors as large
  // as ds itself.
  float delta = 0.0f, lse_q = 0.0f;
  if (tl.q_ok) {
    if (a.G > 0) delta = a.dlt[tl.qn * a.nh + tl.head];
    lse_q = lse[tl.qn * a.nh + tl.head];
    if (dlse != nullptr) delta -= dlse[tl.qn * a.nh + tl.head];
  }
  auto has_tap = [&](int i) { return tl.q_ok && tl.sub + kSubs * i < a.K; };
  auto drop_factor = [&](int i) {
    return !DROP ? 1.0f : ((tp.flags >> (4 * i)) & 8u) ? 0.0f : a.drop.scale;
  };
  // p = exp(scale * s - lse) in place of s.  Dropout: o sums pd * v_s with pd =
  // p * factor, so dp and the V-side coordinate gradient see the factor.
  float pdp = 0.0f;  // sum_k p_k f_k dP_k over this lane's taps
#pragma unroll
  for (int i = 0; i < kSlots; ++i) {
    ts[i].v = has_tap(i) ? __expf(ts[i].v * a.softmax_scale - lse_q) : 0.0f;
    pdp = __builtin_fmaf(ts[i].v * drop_factor(i), td[i].v, pdp);
  }
  delta += half_reduce<false>(pdp);
  // the whole Delta for the extra keys' kernel that runs next (each query's
  // entry is read above and written here by this workgroup only)
  if (a.G > 0 && tl.sub == 0 && tl.q_ok) a.dlt[tl.qn * a.nh + tl.head] = delta;
  // p * factor in place of p, ds * scale = p (f dP - Delta) scale in place of dP
  float l1 = 0.0f;
#pragma unroll
  for (int i = 0; i < kSlots; ++i) {
    const float f = drop_factor(i);
    // (a lane without a tap holds a copy of another's, with p = 0)
    td[i].v = has_tap(i) ? ts[i].v * (f * td[i].v - delta) * a.softmax_scale : 0.0f;
    ts[i].v *= f;
    l1 += fabsf(td[i].v);
  }
  if constexpr (SPLIT) {  // l1 is a sum of absolute values: none cancels
    if (__builtin_amdgcn_ballot_w64(!__builtin_isfinite(l1)) != 0 && (threadIdx.x & 63) == 0)
      atomicOr(rc.collist, 1);
  }
  // bf16 storage: normalised ds lie in [-1, 1], where fp16 keeps 11 bits
  float rl1 = 1.0f;
  if constexpr (sizeof(E) == 2) {
    l1 = half_reduce<false>(l1);
    rl1 = l1 > 1e-30f ? 1.0f / l1 : 0.0f;
    if (tl.sub == 0 && tl.q_ok) b_ws[tl.qn * a.nh + tl.head] = l1;
  }

  // ---- records for the column-streaming kernel, counting-sorted by z0: the
  // bins' counts by LDS atomics (their return values place each record in its
  // bin), then one wave's prefix sum.  Within a bin the order is the atomics'
  // order, which no result depends on (the consumer sums integers).
  const bool rec_wide = REC && bx.zhi - bx.zlo + 1 > kRecBins;
  const int64_t trec =
      REC ? static_cast<int64_t>(tl.head) * rc.tiles +
                rec_tile(a, tl.b, tl.t0, tl.h0 / kTileH, tl.w0 / kTileW)
          : 0;
  // lower corner of tap i, from its word
  const int layer = bx.cm * bx.cn;
  const uint32_t m_col = REC && bx.n > 1 ? 0xffffffffu / static_cast<uint32_t>(bx.len * layer) : 0;
  const uint32_t m_layer = REC && bx.n > 1 ? 0xffffffffu / static_cast<uint32_t>(layer) : 0;
  auto corner = [&](int i, int& z, int& y, int& xx) {
    int col = 0, r, va;
    if (bx.n > 1) {
      col = bx.n > bx.slabs ? box_div(tp.at[i], bx.len * layer, m_col) : 0;
      r = tp.at[i] - col * (bx.len * layer);
      va = box_div(r, layer, m_layer);
    } else {
      r = tp.at[i] - tl.q * kBoxRow;
      va = static_cast<int>((static_cast<float>(r) + 0.5f) * bx.rlayer);
    }
    r -= va * layer;
    int vm = static_cast<int>((static_cast<float>(r) + 0.5f) * bx.rrow);
    int vl = r - vm * bx.cn;
    if (bx.n > bx.slabs) {
      const int q = col / bx.pn;
      vm += q * (bx.cm - 1);
      vl += (col - q * bx.pn) * (bx.cn - 1);
    }
    // (a position on the last voxel is that voxel's, with weight 0 above it)
    z = bx.zlo + (bx.axis == 2 ? va : vm) + (tp.fz[i] == 1.0f);
    y = bx.ylo + (bx.axis == 2 ? vm : bx.axis == 1 ? va : vl) + (tp.fy[i] == 1.0f);
    xx = bx.xlo + (bx.axis == 0 ? va : vl) + (tp.fx[i] == 1.0f);
  };
  int pos[kSlots];
  if constexpr (REC) {
    // the column list's count and, after the list, the 8 work counters of the
    // column-streaming kernel
    if (unit == 0 && threadIdx.x < 9)
      rc.collist[threadIdx.x == 0 ? 0 : a.nh * a.B * a.tiles_h * a.tiles_w + threadIdx.x] = 0;
    if (tl.sub == 0) s_l1[tl.q] = l1;
#pragma unroll
    for (int i = 0; i < kSlots; ++i) {
      pos[i] = 0;
      if (kSubs * i >= a.K || rec_wide || !has_tap(i)) continue;
      int z, y, xx;
      corner(i, z, y, xx);
      pos[i] = atomicAdd(&s_bin[z - bx.zlo], 1);
    }
    // q and dO rows of the tile, [tensor][query][channel], in the table's memory
    uint16_t* const sx = reinterpret_cast<uint16_t*>(s_tab);
    constexpr int XR = HD + 16, CPR = HD / 8;
    for (int e = threadIdx.x; e < 2 * kTQ * CPR; e += kThreads) {
      const int t = e / (kTQ * CPR), m = (e / CPR) % kTQ, ch = (e % CPR) * 8;
      const int64_t row = tile_row(a, tl, m);
      u32x4_t w = {0u, 0u, 0u, 0u};
      if (row >= 0)
        w = load16((t == 0 ? static_cast<const E*>(a.q) + row * a.qs : dout + row * D) +
                   tl.head * HD + ch);
      __builtin_memcpy(&sx[(t * kTQ + m) * XR + ch], &w, sizeof(w));
    }
    __syncthreads();
    // exclusive prefix of the 16 counts in wave 0 (lane bb holds bin bb)
    if (threadIdx.x < 64) {
      const int bb = threadIdx.x & (kRecBins - 1);
      const int cnt = threadIdx.x < kRecBins ? s_bin[bb] : 0;
      int inc = cnt;
#pragma unroll
      for (int m = 1; m < kRecBins; m <<= 1) {
        const int o = __shfl_up(inc, m, kRecBins);
        if (bb >= m) inc += o;
      }
      int* const hdr = rc.hdr + trec * kRecHdr;
      if (threadIdx.x < kRecBins) {
        s_bin[kRecBins + bb] = inc - cnt;
        hdr[8 + bb] = inc - cnt;
        if (bb == kRecBins - 1) hdr[8 + kRecBins] = inc;
      }
      if (threadIdx.x == 0) {
        hdr[0] = bx.zlo;
        hdr[1] = bx.zhi;
        hdr[2] = bx.ylo;
        hdr[3] = bx.yhi;
        hdr[4] = bx.xlo;
        hdr[5] = bx.xhi;
        hdr[6] = rec_wide ? -1 : bx.zhi - bx.zlo + 1;
      }
    }
    __syncthreads();
    // q and dO transposed, with the fixed-point scales of the B (l1 / 2^30, per
    // query) and A (1 / fix_a) tables: item e = (tensor, channel, query half)
    // writes 8 queries (16 bytes)
    E* const qt = static_cast<E*>(rc.qt) + trec * (2 * HD * kTQ);
    for (int e = threadIdx.x; e < 2 * HD * 2; e += kThreads) {
      const int t = e / (2 * HD), chn = (e / 2) % HD, h8 = 8 * (e & 1);
      uint16_t v8[8];
#pragma unroll
      for (int j = 0; j < 8; ++j) {
        const int m = h8 + j;
        const float sc = t == 0 ? s_l1[m] * kFixAInv : a.fix_a_inv;
        const uint16_t raw = sx[(t * kTQ + m) * XR + chn];
        v8[j] = from_f32<E>(__uint_as_float(static_cast<uint32_t>(raw) << 16) * sc).bits;
      }
      __builtin_memcpy(&qt[(t * HD + chn) * kTQ + h8], v8, sizeof(v8));
    }
  }

  // ---- per-tap results.  The coordinate gradient of a tap is ds*scale*dS/du +
  // p*dP/du; chain it through the clamp mask, the unnormalisation (S/2), the slot
  // divisor and offset_scale into d offsets.
  const int64_t tap0 = (tl.qn * a.nh + tl.head) * a.K;
  u32x4_t* const rec = REC ? rc.rec + trec * (static_cast<int64_t>(a.K) * kTQ) : nullptr;
#pragma unroll
  for (int i = 0; i < kSlots; ++i) {
    if (kSubs * i >= a.K || !has_tap(i)) continue;
    const float pd = ts[i].v, dss = td[i].v;
    const int kap = tl.sub + kSubs * i;
    uint32_t pair = 0;
    if constexpr (sizeof(E) == 4) {
      p_ws[tap0 + kap] = pd;
      b_ws[tap0 + kap] = dss;
    } else {
      pair = pack_h2(pd, dss * rl1);
      reinterpret_cast<uint32_t*>(p_ws)[tap0 + kap] = pair;
    }
    E* const dp = doff + tl.qn * a.C + (static_cast<int64_t>(tl.head) * a.K + kap) * 3;
    const uint32_t m = tp.flags >> (4 * i);
    dp[0] = from_f32<E>((m & 1) ? (dss * ts[i].dx + pd * td[i].dx) * a.gsx : 0.0f);
    dp[1] = from_f32<E>((m & 2) ? (dss * ts[i].dy + pd * td[i].dy) * a.gsy : 0.0f);
    dp[2] = from_f32<E>((m & 4) ? (dss * ts[i].dz + pd * td[i].dz) * a.gsz : 0.0f);
    if constexpr (REC) {
      if (rec_wide) continue;
      int z, y, xx;
      corner(i, z, y, xx);
      auto upper = [](float f) { return f == 1.0f ? 0.0f : f; };
      const uint32_t ux = min(65535u, static_cast<uint32_t>(upper(tp.fx[i]) * 65536.0f + 0.5f));
      const uint32_t uy = min(65535u, static_cast<uint32_t>(upper(tp.fy[i]) * 65536.0f + 0.5f));
      u32x4_t r;
      r[0] = static_cast<uint32_t>(y) | (static_cast<uint32_t>(xx) << 14) |
             (static_cast<uint32_t>(tl.q) << 28);
      r[1] = ux | (uy << 16);
      r[2] = __float_as_uint(upper(tp.fz[i]));
      r[3] = pair;
      rec[s_bin[kRecBins + z - bx.zlo] + pos[i]] = r;
    }
  }
}

}  // namespace

template <int HD, typename E, int AE, bool REC, bool SPLIT>
void launch_bwd_p1(const Args& a, const E* dout, const float* lse, const float* dlse, E* doff,
                   float* p_ws, float* b_ws, void* dk_acc, void* dv_acc, int64_t acc_ks,
                   int64_t acc_vs, const RecArgs& rc, hipStream_t s) {
  const dim3 grid = box_grid(a.B, a.T, a.H, a.W, a.nh), block(kThreads);
  if (a.drop.threshold != 0)
    hipLaunchKernelGGL((dsa3d_bwd_p1_kernel<HD, E, AE, REC, true, SPLIT>), grid, block, 0, s, a, dout,
                       lse, dlse, doff, p_ws, b_ws, dk_acc, dv_acc, acc_ks, acc_vs, rc);
  else
    hipLaunchKernelGGL((dsa3d_bwd_p1_kernel<HD, E, AE, REC, false, SPLIT>), grid, block, 0, s, a,
                       dout, lse, dlse, doff, p_ws, b_ws, dk_acc, dv_acc, acc_ks, acc_vs, rc);
}

#define MSD_P1(HD, E, AE, REC, SPLIT)                                                             \
  template void launch_bwd_p1<HD, E, AE, REC, SPLIT>(                                             \
      const Args&, const E*, const float*, const float*, E*, float*, float*, void*, void*,        \
      int64_t, int64_t, const RecArgs&, hipStream_t);
#define MSD_P1_HD(HD)                \
  MSD_P1(HD, float, 4, false, false) \
  MSD_P1(HD, float, 4, false, true)  \
  MSD_P1(HD, bf16, 4, false, false)  \
  MSD_P1(HD, bf16, 4, true, false)   \
  MSD_P1(HD, bf16, 2, false, false)
MSD_P1_HD(32)
MSD_P1_HD(64)
MSD_P1_HD(96)
MSD_P1_HD(128)

}  // namespace msd
