// Matrix-core 3D-DSA forward for gfx950: bf16 or fp32 storage, fp32 accumulation.
//
// One workgroup = one (batch, head, frame, tile of 16 queries).  Instead of
// gathering the 8 corner rows of K and V for each of a query's taps, it builds
// dense tables on the matrix cores over the box of voxels that the tile's taps
// reach (dsa3d_box.h: the whole box at once, or pieces of it):
//   S[q][v] = q . K[v]  (MFMA, fp32 in LDS)  ->  per tap s = scale * sum_c w_c S[q][c]
//   softmax over each query's taps in registers (wave reductions)
//   A[q][v] = sum over taps/corners landing on v of p * w  (LDS integer adds)
//   O[q] += A[q] . V  (MFMA, V transposed on the matrix cores)
// This equals the reference's grid_sample + matmul + softmax + matmul
// (infinity/video/attention.py:106-186) because trilinear sampling is linear in
// the sampled rows.  Coordinates and corner choice round exactly as the fp32
// reference does (div_rn, dsa3d_coords.h).
//
// Bound: waiting (0.54 of a wave's life at 65,536 tokens, 16 x 64, bf16), for the K
// and V rows' loads above all (the box of a tile is about 900 rows of each; 0.83 of
// all requests hit the L2), and VALU issue (1,591 instructions a wave, 46 % of the
// time).  Tables of the whole box against tables of one plane at a time (tested by
// every tap on every plane, two or three barriers each): 3.21 -> 2.87 ms there; 5.9 ->
// 5.2 ms at 46,800 tokens, 16 x 96, offsets biased by up to 4 units; 11.4 -> 11.1 ms at
// 131,072 tokens, 24 x 128; 2.04 -> 1.53 ms at 32,768 tokens, 8 x 64, fp32; 41 -> 30 us
// at 2,048 tokens, 4 x 64, fp32.  Slower where two frames stretch the box over the
// volume's width (offsets of x count T - 1 to the axis): 0.205 -> 0.211 ms at 2 x 60 x
// 90, 4 x 64, 0.275 -> 0.302 biased.  Tried and slower: a persistent grid with the next
// tile's offsets loaded ahead (registers spill), 8 or 10 blocks of K rows in flight per
// wave instead of 6.
#pragma once

#include <algorithm>
#include <type_traits>

#include "dsa3d_box.h"

namespace msd {

namespace {

using namespace tiled;

// Waves per SIMD: 4 (two workgroups per CU, 128 registers) except where the
// fp32 operands of a wide head need more registers.
template <int HD, typename E>
constexpr int fwd_min_waves() {
  return sizeof(E) == 4 && HD > 64 ? 2 : 4;
}

// S: storage, E: element type of the products.  EPL: extra keys a lane holds (0: none).
// RG: head_dim hd below HD (a multiple of 8), channels past it read as zero.
// SAFE: the weighted sum by plain arithmetic.
// Returns whether a sum (RG: or a score) was not finite.
template <int HD, typename S, typename E, int EPL, bool RG, bool DROP, bool SAFE>
__device__ __forceinline__ bool fwd_tile(const Args& a, S* __restrict__ out,
                                         float* __restrict__ lse, int hd_arg, unsigned tid,
                                         int* s_tab, uint32_t* s_row, int* s_box,
                                         float* s_qnan) {
  constexpr bool XK = EPL > 0;
  float* const s_val = reinterpret_cast<float*>(s_tab);
  const int hd = RG ? hd_arg : HD;

  const Tile tl = box_tile(a, box_unit(a), tid);
  RawOffsets<S, kSlots> raw;
  box_load_offsets<S, kSlots>(a, tl, raw);
  box_init(s_box);
  __syncthreads();
  // the tile's q rows load while the taps are set up
  op_t<E> qx[HD / 32];
  box_tile_rows<HD, S, E, RG>(a, tl, static_cast<const S*>(a.q), a.qs, hd, qx);
  // (a score below the type's limit whose terms are beyond it: q times a power of two)
  constexpr float kDown = SAFE && RG ? 0x1p-16f : 1.0f;
  if constexpr (SAFE && RG) {
#pragma unroll
    for (int c = 0; c < HD / 32; ++c) qx[c] *= kDown;
  }
  const float scale = a.softmax_scale * (1.0f / kDown);
  BoxTaps<kSlots> tp;
  BoxPieces bx;
  box_setup<S, kSlots, false, DROP, RG>(a, tl, raw, tp, bx, s_box);

  auto rows_of = [&](const void* base, int64_t stride) {
    const S* p = static_cast<const S*>(base) + tl.sample0 * stride + static_cast<int64_t>(tl.head) * hd;
    return box_rows(p, ((a.N - 1) * stride + hd) * static_cast<int64_t>(sizeof(S)));
  };
  auto set_rows = [&](const BoxSeg& g, int64_t stride) {
    box_row_offsets(a, tl, bx, g, static_cast<uint32_t>(stride * sizeof(S)), s_row);
  };
  auto row_off = [&](int v) { return s_row[v]; };
  // extra keys: row g of the sample
  const int G = XK ? a.G : 0, Gp = (G + 31) & ~31;
  const int64_t D = static_cast<int64_t>(a.nh) * hd;
  auto extra_rows = [&](const void* base) {
    const S* p = static_cast<const S*>(base) + tl.b * static_cast<int64_t>(G) * D +
                 static_cast<int64_t>(tl.head) * hd;
    return box_rows(p, ((G - 1) * D + hd) * static_cast<int64_t>(sizeof(S)));
  };
  auto extra_off = [&](int g) {
    return g < G ? static_cast<uint32_t>(g * static_cast<int>(D * sizeof(S))) : kNoRow;
  };
  constexpr int NB = SAFE ? 2 : box_score_blocks<HD, E>();
  auto scores = [&](__amdgpu_buffer_rsrc_t r, const auto& off, int n) {
    if constexpr (RG) box_scores_split<HD, S, RG>(tl, r, off, n, hd, qx, s_val);
    else box_scores<HD, S, E, RG, NB>(tl, r, off, n, hd, qx, s_val);
  };

  // ---- scores ---------------------------------------------------------------
  float sc[kSlots];
#pragma unroll
  for (int i = 0; i < kSlots; ++i) sc[i] = 0.0f;
  {
    const __amdgpu_buffer_rsrc_t kr = rows_of(a.k, a.ks);
    auto piece = [&](int s, auto only) __attribute__((always_inline)) {  // `only`: of one
      constexpr bool kOnly = decltype(only)::value;
      const BoxSeg g = box_seg(bx, s);
      set_rows(g, a.ks);
      scores(kr, row_off, bx.nv);
      __syncthreads();
      auto gather = [&](auto edge, auto dx, auto dy) __attribute__((always_inline)) {
#pragma unroll
        for (int i = 0; i < kSlots; ++i) {
          if (kSubs * i >= a.K) continue;
          BoxTap t = box_tap(tp, i);
          if (!kOnly && !box_in(g, tl.q, t)) continue;
          if constexpr (SAFE && RG)
            sc[i] = box_gather_safe(s_val, t.at, dx, dy, bx.dz, t.fx, t.fy, t.fz);
          else
            sc[i] = box_gather<decltype(edge)::value>(s_val, t.at, dx, dy, bx.dz, t.fx, t.fy, t.fz);
        }
      };
      // neighbours at distance 1 along x, or along y in slabs along x, come in one read
      constexpr std::integral_constant<int, 1> kNext{};
      if constexpr (SAFE) {
        gather(std::true_type{}, bx.dx, bx.dy);
      } else if (kOnly || bx.axis != 0) {
        if (bx.edge) gather(std::true_type{}, kNext, bx.dy);
        else gather(std::false_type{}, kNext, bx.dy);
      } else if (bx.edge || a.H == 1) {
        gather(std::true_type{}, bx.dx, bx.dy);
      } else {
        gather(std::false_type{}, bx.dx, kNext);
      }
      __syncthreads();  // the next piece, the extra keys or the weights take the table
    };
    if (bx.n == 1) {
      piece(0, std::true_type{});
    } else {
#pragma nounroll
      for (int s = 0; s < bx.n; ++s) piece(s, std::false_type{});
    }
  }

  // ---- extra keys (attention.py:160-173): lane `sub` of a query takes keys
  // sub + 32 j ------------------------------------------------------------------
  float se[XK ? EPL : 1];
  if constexpr (XK) {
    scores(extra_rows(a.ek), extra_off, Gp);
    __syncthreads();
#pragma unroll
    for (int j = 0; j < EPL; ++j) {
      const int g = tl.sub + kSubs * j;
      se[j] = g < G ? s_val[tl.q * kBoxRow + g] * scale : -INFINITY;
    }
    __syncthreads();  // the weights take the table
  }

  // ---- softmax over each query's taps (32 lanes x kSlots) and extra keys ----
  auto has_tap = [&](int i) { return tl.q_ok && tl.sub + kSubs * i < a.K; };
  float mx = -INFINITY;
#pragma unroll
  for (int i = 0; i < kSlots; ++i) {
    sc[i] = has_tap(i) ? sc[i] * scale : -INFINITY;
    mx = fmaxf(mx, sc[i]);
  }
  if constexpr (XK) {
#pragma unroll
    for (int j = 0; j < EPL; ++j) mx = fmaxf(mx, se[j]);
  }
  mx = half_reduce<true>(mx);
  float den = 0.0f;
#pragma unroll
  for (int i = 0; i < kSlots; ++i) {
    sc[i] = has_tap(i) ? __expf(sc[i] - mx) : 0.0f;
    den += sc[i];
  }
  if constexpr (XK) {
#pragma unroll
    for (int j = 0; j < EPL; ++j) {
      se[j] = tl.sub + kSubs * j < G ? __expf(se[j] - mx) : 0.0f;
      den += se[j];
    }
  }
  den = half_reduce<false>(den);
  const float inv_den = 1.0f / den;
  // a query past the grid's edge weighs nothing (its lanes hold copies of the tile's taps),
  // nor does one with a score that is not finite (its output is NaN: s_qnan)
  const bool weighs = tl.q_ok && den == den;
#pragma unroll
  for (int i = 0; i < kSlots; ++i) {
    // p times its dropout factor, in fixed-point units
    const float f = !DROP ? 1.0f : ((tp.flags >> (4 * i)) & 8u) ? 0.0f : a.drop.scale;
    sc[i] = weighs ? sc[i] * (inv_den * f * a.fix_a) : 0.0f;
  }
  if (tl.sub == 0) {
    s_qnan[tl.q] = den == den ? 1.0f : __builtin_nanf("");
    if (lse != nullptr && tl.q_ok) lse[tl.qn * a.nh + tl.head] = mx + logf(den);
  }
  if constexpr (XK) {
    // the keys' weights, in the units of the taps'
#pragma unroll
    for (int j = 0; j < EPL; ++j) {
      const int g = tl.sub + kSubs * j;
      const float f = DROP ? dropout_factor(a.drop, tl.qn, tl.head, a.K + g) : 1.0f;
      se[j] = g < G && weighs ? se[j] * inv_den * a.fix_a * f : 0.0f;
    }
  }

  // ---- weighted sum: the waves split the voxels, and their partial sums meet in
  // the table's memory at the end ------------------------------------------------
  const __amdgpu_buffer_rsrc_t vr = rows_of(a.v, a.vs);
  f32x4_t acc[HD / 16];
#pragma unroll
  for (int t = 0; t < HD / 16; ++t) acc[t] = f32x4_t{0.0f, 0.0f, 0.0f, 0.0f};
  // begin: loads of the first rows; fill: what the table still needs, barriers included.
  // taps: whether the caller keeps its taps over the call
  auto weighted = [&](auto floats, auto taps, __amdgpu_buffer_rsrc_t r, const auto& off, int n,
                      const auto& fill) __attribute__((always_inline)) {
    constexpr bool FT = decltype(floats)::value;
    constexpr int NC = HD / 32;
    constexpr int C = sizeof(E) == 2 ? box_groups<HD, decltype(taps)::value, XK>() : NC;
    if constexpr (SAFE) {
      fill();
      box_weighted_safe<HD, S, E, RG, FT>(tl, r, off, n, hd, s_tab, a.fix_a_inv, acc);
    } else {
      auto pass = [&](auto first) __attribute__((always_inline)) {
        constexpr int C0 = decltype(first)::value, C1 = C0 + C < NC ? C0 + C : NC;
        if constexpr (C0 < NC) {
          BoxAhead<C1 - C0, E> ah;
          box_weighted_begin<C1 - C0, S, E>(tl, r, off, n, C0, ah);
          if (C0 == 0) fill();
          box_weighted<HD, S, E, RG, FT, C0, C1>(tl, r, off, n, hd, s_tab, ah, acc);
        }
      };
      pass(std::integral_constant<int, 0>{});
      pass(std::integral_constant<int, C>{});
      pass(std::integral_constant<int, 2 * C>{});
      pass(std::integral_constant<int, 3 * C>{});
    }
  };
  auto piece = [&](int s, auto only) __attribute__((always_inline)) {
    constexpr bool kOnly = decltype(only)::value;
    const BoxSeg g = box_seg(bx, s);
    if (!kOnly || a.vs != a.ks) set_rows(g, a.vs);  // else as the scores left them
    weighted(std::false_type{}, std::bool_constant<!kOnly || XK>{}, vr, row_off, bx.nv, [&] {
      box_zero(s_tab, ((bx.nv + 31) & ~31) >> 2);
      __syncthreads();
#pragma unroll
      for (int i = 0; i < kSlots; ++i) {
        if (kSubs * i >= a.K) continue;
        if (SAFE && !has_tap(i)) continue;  // (a copy of another lane's tap)
        const BoxTap t = box_tap(tp, i);
        if constexpr (kOnly) box_scatter<SAFE>(s_tab, bx, t, sc[i]);
        else box_scatter<SAFE>(s_tab, bx, g, tl.q, t, sc[i]);
      }
      __syncthreads();
    });
    __syncthreads();  // the products have read the table
  };
  if (bx.n == 1) {  // the usual case apart: no tap stays live through its products
    piece(0, std::true_type{});
  } else {
#pragma nounroll
    for (int s = 0; s < bx.n; ++s) piece(s, std::false_type{});
  }
  if constexpr (XK) {
    // (after the taps, which are not kept over these products then)  The weights as they
    // are, in the units of the taps' (a key's is one number, not a sum of corners); SAFE:
    // the smallest above 0 marks a key of weight 0
#pragma unroll
    for (int j = 0; j < EPL; ++j)
      if (tl.sub + kSubs * j < Gp)
        s_val[tl.q * kBoxRow + tl.sub + kSubs * j] =
            SAFE && tl.sub + kSubs * j < G ? fmaxf(se[j], 1e-30f) : se[j];
    __syncthreads();
    weighted(std::true_type{}, std::false_type{}, extra_rows(a.ev), extra_off, Gp, [] {});
    __syncthreads();
  }
  // partial O of wave w: [w][query][channel]
  static_assert(kWaves * kTQ * HD <= kTQ * kBoxRow, "the partial sums fit the table");
#pragma unroll
  for (int t = 0; t < HD / 16; ++t)
#pragma unroll
    for (int r = 0; r < 4; ++r)
      s_val[(tl.wave * kTQ + 4 * (tl.lane >> 4) + r) * HD +
            box_channel<HD, E>(t, tl.lane & 15)] = acc[t][r];
  __syncthreads();
  bool bad = RG && tl.q_ok && !(den == den);
#pragma unroll
  for (int e0 = 0; e0 < kTQ * HD; e0 += kThreads) {
    const int e = e0 + static_cast<int>(tid);
    float o = 0.0f;
#pragma unroll
    for (int w = 0; w < kWaves; ++w) o += s_val[w * kTQ * HD + e];
    bad |= !__builtin_isfinite(o);
    const int m = e / HD, ch = e - m * HD;
    const int64_t n = tile_row(a, tl, m);
    if (n >= 0 && (!RG || ch < hd))
      out[n * D + tl.head * hd + ch] = from_f32<S>(SAFE ? o * s_qnan[m] : o * a.fix_a_inv * s_qnan[m]);
  }
  return bad;
}

// A non-finite sum means that a V row of the tile's box holds a non-finite value,
// which the products spread: to queries of the tile that do not sample the row
// and (bf16) over its channels.  The tile is then done again with the sum by
// plain arithmetic over what each query samples (from the start, so that nothing
// is kept live for it).  Padded head sizes, which the general kernels took before, do so
// for scores that are not finite too, and gather them as these do.  Whole-head fp32
// products (32, 64, 96, 128) go without.
template <int HD, typename S, typename E, int EPL, bool RG, bool DROP>
__global__ __launch_bounds__(kThreads, (fwd_min_waves<HD, E>())) void dsa3d_fwd_box_kernel(
    Args a, S* __restrict__ out, float* __restrict__ lse, int hd) {
  __shared__ __attribute__((aligned(16))) int s_tab[kTQ * kBoxRow];
  __shared__ uint32_t s_row[kBoxCap];
  __shared__ int s_box[8];
  __shared__ int s_bad;
  // per query: 1, or NaN when a score is not finite (its output is NaN then, as
  // softmax makes it in the reference; the fixed-point weights alone would drop it)
  __shared__ float s_qnan[kTQ];
  if (box_unit(a) < 0) return;  // the grid is rounded up to the 8 XCDs
  constexpr bool kCheck = sizeof(E) == 2 || RG;
  if (kCheck && threadIdx.x == 0) s_bad = 0;
  const bool bad = fwd_tile<HD, S, E, EPL, RG, DROP, false>(a, out, lse, hd, threadIdx.x, s_tab,
                                                            s_row, s_box, s_qnan);
  if constexpr (kCheck) {
    if (__builtin_amdgcn_ballot_w64(bad) != 0 && (threadIdx.x & 63) == 0) s_bad = 1;
    __syncthreads();
    if (s_bad == 0) return;
    // nothing of the first pass is kept for the second, the arguments included
    struct KernArgs {
      Args a;
      S* out;
      float* lse;
      int hd;
    };
    unsigned tid = threadIdx.x;
    auto kp = __builtin_amdgcn_kernarg_segment_ptr();
    asm volatile("" : "+v"(tid), "+s"(kp));
    KernArgs k;
    __builtin_memcpy(&k, (const void*)kp, sizeof(k));
    fwd_tile<HD, S, E, EPL, RG, DROP, true>(k.a, k.out, k.lse, k.hd, tid, s_tab, s_row, s_box,
                                           s_qnan);
  }
}

template <typename S, typename E, bool RG>
hipError_t fwd_typed(const msd_dsa3d_desc& d, const Args& a, void* out, float* lse, hipStream_t s) {
  const dim3 grid = box_grid(d.B, d.T, d.H, d.W, d.num_heads);
  const dim3 block(kThreads);
  S* const o = static_cast<S*>(out);
  auto go = [&]<int HD>() {
    auto run = [&]<int EPL, bool DROP>() {
      hipLaunchKernelGGL((dsa3d_fwd_box_kernel<HD, S, E, EPL, RG, DROP>), grid, block, 0, s, a, o,
                         lse, d.head_dim);
    };
    const bool drop = a.drop.threshold != 0;
    // lanes hold the keys' weights in registers: half as many for up to 128 keys
    constexpr int kMost = kMaxExtra / kSubs;
    auto keys = [&]<int EPL>() {
      drop ? run.template operator()<EPL, true>() : run.template operator()<EPL, false>();
    };
    if (a.G == 0) keys.template operator()<0>();
    else if (a.G <= kSubs * kMost / 2) keys.template operator()<kMost / 2>();
    else keys.template operator()<kMost>();
  };
  if (d.head_dim <= 32) go.template operator()<32>();
  else if (d.head_dim <= 64) go.template operator()<64>();
  else if (d.head_dim <= 96) go.template operator()<96>();
  else go.template operator()<128>();
  return hipGetLastError();
}

}  // namespace

}  // namespace msd
