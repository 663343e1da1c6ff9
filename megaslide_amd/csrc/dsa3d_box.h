// Whole-box tables of the matrix-core 3D-DSA kernels.
//
// A workgroup of 8 waves owns the 16 queries of one (batch, head, frame, 4 x 4
// tile).  All corners of the tile's taps lie in a small box of voxels (about
// 7 x 12 x 12 at the usual windows and offsets), and the table of one value per
// (query, voxel of the whole box) fits the LDS: 16 x 1,184 words, 76 KB, two
// workgroups per CU.  A tap then reads (or adds to) its eight corners in one
// visit, where a table of one plane at a time has every tap tested on every
// plane of the box and costs two or three barriers per plane.
//
// A box of more than kBoxCap voxels is cut along its longest axis into equal slabs
// that overlap by one voxel, so that the 2 x 2 x 2 footprint of every tap lies in
// exactly one; they are taken in turn.  (A box of more than 296 voxels per layer
// is first cut into such columns across that axis.)  The weighted sum gives the
// layer that two slabs share to the later one, so that a voxel's weight is
// rounded to the products' element type once, as in a box of one piece.
//
// The box ends at the volume.  A position on the last voxel of an axis is taken as the
// voxel before it with all weight on the upper corner (the reference samples the last
// alone: what reads a table leaves the lower corner out, box_gather), so that the
// corners of every tap sit at constant distances from its first.  An axis of one voxel
// has distance 0 (x: a column of zeros past it, rows that read past the end).
#pragma once

#include "dsa3d_tiled_common.h"

namespace msd {
namespace tiled {

constexpr int kBoxCap = 1184;  // voxels of a table: a multiple of 32
// Row stride (words) of a table: a multiple of 4 (16-byte accesses) whose
// quarter is odd, so that the 16 rows of a 16-byte access fall on 16 distinct
// windows of 4 banks.
constexpr int kBoxRow = 1188;
static_assert(kBoxCap % 32 == 0 && kBoxRow >= kBoxCap + 2 && (kBoxRow / 4) % 2 == 1);

// A tile's box and its pieces: slabs along `axis` of columns that the other two
// axes are cut into, a piece at every (extent - 1)-th voxel of the box.  A voxel's
// index in a table row counts along `axis` slowest, then along the middle axis (y
// where axis is z, else z), then along the last (y where axis is x, else x).
struct BoxPieces {
  int zlo, ylo, xlo;     // the box's first voxel
  int zhi, yhi, xhi;     // its last voxel inside the volume
  int n;                 // pieces; 1: the whole box, axis z
  int axis;              // 0 x, 1 y, 2 z
  int len, slabs;        // the box's layers along the axis; slabs of a column
  int pn;                // columns along the last axis
  int ca, cm, cn;        // voxels of a piece along the axis, the middle and the last
  int dz, dy, dx;        // distances of neighbours in a table row
  int nv;                // voxels of a piece
  float rlayer, rrow;    // 1 / (cm cn), 1 / cn for division-free voxel coordinates
  bool edge;             // taps may have weight 1 on a last voxel, or there is one frame
};

// One piece: its first voxel; the taps' words (BoxTaps) count from `base` there,
// words from `taps` on are of other pieces, and so are voxels from `own` on (the
// layer shared with the next slab).
struct BoxSeg {
  int z0, y0, x0, base, taps, own;
};

// Piece sizes for a box of na x nm x nn voxels, na the largest: columns are halved
// until slabs of 4 layers (of which 3 are new) fit the table.
__device__ __forceinline__ void box_cut(int na, int nm, int nn, int& ca, int& cm, int& cn) {
  cm = nm;
  cn = nn;
#pragma nounroll
  while (cm * cn * 4 > kBoxCap) {
    if (cm > cn) cm = cm / 2 + 1;
    else cn = cn / 2 + 1;
  }
  ca = min(kBoxCap / (cm * cn), na);
  const int p = (na - 2) / (ca - 1) + 1;  // ceil((na - 1) / (ca - 1))
  ca = (na - 2) / p + 2;                  // ceil((na - 1) / p) + 1
}

// Geometry of this lane's taps: corner weights, and the word index of the
// first corner in the query's table row (row offset included), or, where there
// are several pieces, (column * len + layer) * (cm cn) + index within the
// column's layer.  (A sample has less than 2^25 voxels, a box at W = 1 twice its
// voxels of the sample, and columns share at most 37 % more: less than 2^27.)
template <int SLOTS>
struct BoxTaps {
  float fx[SLOTS], fy[SLOTS], fz[SLOTS];
  int at[SLOTS];
  uint32_t flags;   // per tap, 4 bits: clamp-gradient mask x, y, z; dropped by dropout
};

// Wave minimum, on lane 63 (DPP row operations, no LDS).
__device__ __forceinline__ int wave_min63(int v) {
  constexpr int kMax = 0x7fffffff;
  auto step = [&](auto ctrl) {
    v = min(v, __builtin_amdgcn_update_dpp(kMax, v, decltype(ctrl)::value, 0xf, 0xf, true));
  };
  step(std::integral_constant<int, 0xB1>{});   // quad 1,0,3,2
  step(std::integral_constant<int, 0x4E>{});   // quad 2,3,0,1
  step(std::integral_constant<int, 0x141>{});  // half-row mirror
  step(std::integral_constant<int, 0x140>{});  // row mirror
  v = min(v, __builtin_amdgcn_update_dpp(kMax, v, 0x142, 0xa, 0xf, false));  // row 0 -> 1, 2 -> 3
  v = min(v, __builtin_amdgcn_update_dpp(kMax, v, 0x143, 0xc, 0xf, false));  // row 1 -> 2, 3
  return v;
}

// Sum (or maximum) over the 32 lanes of a half-wave, on all of them.
template <bool MAX>
__device__ __forceinline__ float half_reduce(float v) {
  auto op = [](float x, float y) { return MAX ? fmaxf(x, y) : x + y; };
  auto step = [&](auto ctrl) {
    v = op(v, __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(v),
                                                         decltype(ctrl)::value, 0xf, 0xf, true)));
  };
  step(std::integral_constant<int, 0xB1>{});
  step(std::integral_constant<int, 0x4E>{});
  step(std::integral_constant<int, 0x141>{});
  step(std::integral_constant<int, 0x140>{});
  return op(v, __shfl_xor(v, 16));
}

// One axis of a tap's sampling position: lower corner (at most `last` = max(S - 2, 0)),
// upper weight, and whether the position lies strictly inside the volume.  The operations and their
// rounding are those of base_coord_rn / grid_coord_rn / axis_sample: the tap
// index enters as an exact small float, and the halving of ((g + 1) S - 1) / 2 is
// taken into S and 1 (a power of two, which rounding commutes with).  `o` is 0
// and div = rdiv = 0 for a dropped slot (0 is then added to the base).
struct AxisTap {
  int lo;
  float f;
  bool in;
};
__device__ __forceinline__ AxisTap axis_tap(float pos2, float o, float bdiv, float rbdiv,
                                            float div, float rdiv, float S, float last) {
#pragma clang fp contract(off)
  const float g = (div_rn(pos2, bdiv, rbdiv) - 1.0f) + div_rn(o, div, rdiv);
  const float u = (g + 1.0f) * (0.5f * S) - 0.5f;
  // (a NaN position samples voxel 0, as fmaxf / fminf leave it)
  const float c = __builtin_amdgcn_fmed3f(u, 0.0f, S - 1.0f);
  const float fl = fminf(floorf(c), last);
  AxisTap r;
  r.lo = static_cast<int>(fl);
  r.f = c - fl;
  r.in = u > 0.0f && u < S - 1.0f;
  return r;
}

// One workgroup per unit (head, tile).  Workgroups are dispatched round-robin
// over the 8 XCDs; each XCD has a contiguous run of units, so that neighbouring
// tiles (frames vary fastest: they read nearly the same K/V planes) share its L2.
// A launch takes at most 2^32 - 1 threads along x, which 2^23 workgroups reach: more
// of them go on along y.
inline dim3 box_grid(int B, int T, int H, int W, int heads) {
  constexpr int64_t kMaxX = 1 << 22;
  const int64_t units = tile_count<1>(B, T, H, W) * heads;
  if (units <= kMaxX) return dim3(static_cast<unsigned>((units + 7) / 8 * 8));
  return dim3(static_cast<unsigned>(kMaxX), static_cast<unsigned>((units + kMaxX - 1) / kMaxX));
}
// This workgroup's unit, -1 past the last.
__device__ __forceinline__ int box_unit(const Args& a) {
  const unsigned i = blockIdx.y * gridDim.x + blockIdx.x;  // x is a multiple of 8
  const unsigned u = (i & 7) * ((gridDim.x >> 3) * gridDim.y) + (i >> 3);
  const unsigned n = static_cast<unsigned>(a.nh * a.B * a.T) * (a.tiles_h * a.tiles_w);
  return u < n ? static_cast<int>(u) : -1;
}
// a / d for 0 <= a < 2^31, m = floor(2^32 / d): scalar instructions only.
__device__ __forceinline__ int box_div(int a, int d, uint32_t m) {
  const int q = static_cast<int>(__umulhi(static_cast<uint32_t>(a), m));
  return a - q * d >= d ? q + 1 : q;
}

// Tile of unit u: frame fastest, then column, row, sample, head.
__device__ __forceinline__ Tile box_tile(const Args& a, int u, unsigned tid) {
  Tile t;
  int r = box_div(u, a.T, a.m_t);
  t.t0 = t.t = u - r * a.T;
  int c = box_div(r, a.tiles_w, a.m_tw);
  t.w0 = (r - c * a.tiles_w) * kTileW;
  r = box_div(c, a.tiles_h, a.m_th);
  t.h0 = (c - r * a.tiles_h) * kTileH;
  t.head = box_div(r, a.B, a.m_b);
  t.b = r - t.head * a.B;
  t.sample0 = static_cast<int64_t>(t.b) * a.N;
  t.wave = tid >> 6;
  t.lane = tid & 63;
  t.q = tid / kSubs;
  t.sub = tid % kSubs;
  const int s = t.q % kTQ;
  t.qh = t.h0 + s / kTileW;
  t.qw = t.w0 + s % kTileW;
  t.q_ok = t.qh < a.H && t.qw < a.W;
  t.qn = t.sample0 + (static_cast<int64_t>(t.t) * a.H + t.qh) * a.W + t.qw;
  return t;
}

// The offsets of this lane's taps as loaded (bf16: 6 bytes per tap, 2-byte
// aligned).  Lanes without a tap of
// their own (kap >= K, or a query past the grid's edge) load one of the tile's.
template <typename S, int SLOTS>
struct RawOffsets {
  uint32_t w[SLOTS][sizeof(S) == 2 ? 2 : 3];
};
template <typename S, int SLOTS>
__device__ __forceinline__ void box_load_offsets(const Args& a, const Tile& tl,
                                                 RawOffsets<S, SLOTS>& r) {
  const int qh = min(tl.qh, a.H - 1), qw = min(tl.qw, a.W - 1);
  const int64_t qn = tl.sample0 + (static_cast<int64_t>(tl.t) * a.H + qh) * a.W + qw;
  const S* const op = static_cast<const S*>(a.off) + qn * a.C + static_cast<int64_t>(tl.head) * a.K * 3;
#pragma unroll
  for (int i = 0; i < SLOTS; ++i) {
    if (kSubs * i >= a.K) {  // uniform; not left as it was, which would stay live
      for (auto& w : r.w[i]) w = 0;
      continue;
    }
    const S* const p = op + 3 * min(tl.sub + kSubs * i, a.K - 1);
    if constexpr (sizeof(S) == 2) {
      __builtin_memcpy(&r.w[i][0], p, 4);
      r.w[i][1] = p[2].bits;
    } else {
      __builtin_memcpy(r.w[i], p, 12);
    }
  }
}
template <typename S, int SLOTS>
__device__ __forceinline__ float raw_offset(const RawOffsets<S, SLOTS>& r, int i, int j,
                                            uint32_t keep) {
  if constexpr (sizeof(S) == 2) {
    const uint32_t b = j == 0 ? r.w[i][0] << 16 : j == 1 ? r.w[i][0] & 0xffff0000u : r.w[i][1] << 16;
    return __uint_as_float(b & keep);
  } else {
    return __uint_as_float(r.w[i][j] & keep);
  }
}

// Tap geometry of this lane and the pieces of the tile's box.  s_box: 8 words
// of LDS that box_init has set before the last barrier.  Weights of lanes without
// a tap of their own must be zeroed by the caller.  Contains one barrier.
__device__ __forceinline__ void box_init(int* s_box) {
  if (threadIdx.x < 8) s_box[threadIdx.x] = 0x7fffffff;
}

// CLAMP: an infinite offset samples the volume's face (div_rn makes it NaN, which
// samples voxel 0), as any offset beyond 10^30 does.
template <typename S, int SLOTS, bool MASK, bool DROP, bool CLAMP>
__device__ __forceinline__ void box_setup(const Args& a, const Tile& tl,
                                          const RawOffsets<S, SLOTS>& raw, BoxTaps<SLOTS>& tp,
                                          BoxPieces& bx, int* s_box) {
  const int qh = min(tl.qh, a.H - 1), qw = min(tl.qw, a.W - 1);
  const int64_t qn = tl.sample0 + (static_cast<int64_t>(tl.t) * a.H + qh) * a.W + qw;
  const float khkw = static_cast<float>(a.kh * a.kw), kw = static_cast<float>(a.kw);
  const float h1 = 0.5f * a.r_khkw, h2 = 0.5f * a.r_kw;
  // 2 (position + tap offset) per axis is 2 tap + these (exact small integers)
  const float px2 = static_cast<float>(2 * (qw - a.kw / 2));
  const float py2 = static_cast<float>(2 * (qh - a.kh / 2));
  const float pz2 = static_cast<float>(2 * (tl.t - a.kt / 2));
  const float Wf = static_cast<float>(a.W), Hf = static_cast<float>(a.H),
              Tf = static_cast<float>(a.T);
  const float Wl = static_cast<float>(max(a.W - 2, 0)), Hl = static_cast<float>(max(a.H - 2, 0)),
              Tl = static_cast<float>(max(a.T - 2, 0));
  int zl[SLOTS], yl[SLOTS], xl[SLOTS];
  // a slot whose axis has one voxel is dropped (attention.py:118-127)
  const uint32_t kx = a.div_x > 0.0f ? ~0u : 0u, ky = a.div_y > 0.0f ? ~0u : 0u,
                 kz = a.div_z > 0.0f ? ~0u : 0u;
  tp.flags = 0;
  constexpr int kMax = 0x7fffffff;
  int zn = kMax, zx = kMax, yn = kMax, yx = kMax, xn = kMax, xx = kMax;  // minima of v and -v
#pragma unroll
  for (int i = 0; i < SLOTS; ++i) {
    tp.fx[i] = tp.fy[i] = tp.fz[i] = 0.0f;
    tp.at[i] = 0;
    zl[i] = yl[i] = xl[i] = 0;
    if (kSubs * i >= a.K) continue;
    const int kap = min(tl.sub + kSubs * i, a.K - 1);
    const float kf = static_cast<float>(kap);
    // kap = (ci kh + cj) kw + ck; (kap + 0.5) RN(1/d) truncates exactly for kap < 2^16
    const float ci = floorf(__builtin_fmaf(kf, a.r_khkw, h1));
    const float rem = __builtin_fmaf(-khkw, ci, kf);
    const float cj = floorf(__builtin_fmaf(rem, a.r_kw, h2));
    const float ck = __builtin_fmaf(-kw, cj, rem);
    auto offset = [&](int j, uint32_t keep) {
      const float o = raw_offset(raw, i, j, keep) * a.offset_scale;
      return CLAMP ? __builtin_amdgcn_fmed3f(o, -1e30f, 1e30f) : o;
    };
    const AxisTap ax = axis_tap(__builtin_fmaf(2.0f, ck, px2), offset(0, kx), a.bdiv_x, a.rbdiv_x,
                                a.div_x, a.rdiv_x, Wf, Wl);
    const AxisTap ay = axis_tap(__builtin_fmaf(2.0f, cj, py2), offset(1, ky), a.bdiv_y, a.rbdiv_y,
                                a.div_y, a.rdiv_y, Hf, Hl);
    const AxisTap az = axis_tap(__builtin_fmaf(2.0f, ci, pz2), offset(2, kz), a.bdiv_z, a.rbdiv_z,
                                a.div_z, a.rdiv_z, Tf, Tl);
    tp.fx[i] = ax.f;
    tp.fy[i] = ay.f;
    tp.fz[i] = az.f;
    xl[i] = ax.lo;
    yl[i] = ay.lo;
    zl[i] = az.lo;
    if constexpr (MASK)
      tp.flags |= ((ax.in ? 1u : 0u) | (ay.in ? 2u : 0u) | (az.in ? 4u : 0u)) << (4 * i);
    if (DROP && dropout_factor(a.drop, qn, tl.head, kap) == 0.0f)
      tp.flags |= 8u << (4 * i);
    zn = min(zn, az.lo);
    zx = min(zx, -az.lo);
    yn = min(yn, ay.lo);
    yx = min(yx, -ay.lo);
    xn = min(xn, ax.lo);
    xx = min(xx, -ax.lo);
  }
  zn = wave_min63(zn);
  zx = wave_min63(zx);
  yn = wave_min63(yn);
  yx = wave_min63(yx);
  xn = wave_min63(xn);
  xx = wave_min63(xx);
  {
    // lanes 0..5 take one bound each
    auto top = [](int v) { return __builtin_amdgcn_readlane(v, 63); };
    const int z0 = top(zn), z1 = top(zx), y0 = top(yn), y1 = top(yx), x0 = top(xn), x1 = top(xx);
    const int l = tl.lane;
    const int v = l == 0 ? z0 : l == 1 ? z1 : l == 2 ? y0 : l == 3 ? y1 : l == 4 ? x0 : x1;
    if (l < 6) atomicMin(&s_box[l], v);
  }
  __syncthreads();
  // the same for every lane: kept in scalar registers
  bx.zlo = __builtin_amdgcn_readfirstlane(s_box[0]);
  const int zh = -__builtin_amdgcn_readfirstlane(s_box[1]);
  bx.ylo = __builtin_amdgcn_readfirstlane(s_box[2]);
  const int yh = -__builtin_amdgcn_readfirstlane(s_box[3]);
  bx.xlo = __builtin_amdgcn_readfirstlane(s_box[4]);
  const int xh = -__builtin_amdgcn_readfirstlane(s_box[5]);
  const int nz = zh - bx.zlo + (a.T > 1 ? 2 : 1), ny = yh - bx.ylo + (a.H > 1 ? 2 : 1);
  const int nx = xh - bx.xlo + 2;
  bx.edge = zh == a.T - 2 || yh == a.H - 2 || xh == a.W - 2 || a.T == 1;
  bx.zhi = min(zh + 1, a.T - 1);
  bx.yhi = min(yh + 1, a.H - 1);
  bx.xhi = min(xh + 1, a.W - 1);
  bx.n = bx.slabs = bx.pn = 1;
  bx.axis = 2;
  bx.ca = bx.len = nz;
  bx.cm = ny;
  bx.cn = nx;
  if (nz * ny * nx <= kBoxCap) {
    const int layer = nx * ny;
    bx.dx = 1;
    bx.dy = a.H > 1 ? nx : 0;
    bx.dz = a.T > 1 ? layer : 0;
    const int base = tl.q * kBoxRow - (bx.zlo * layer + bx.ylo * nx + bx.xlo);
#pragma unroll
    for (int i = 0; i < SLOTS; ++i)
      tp.at[i] = static_cast<int>(__umul24(zl[i], layer) + __umul24(yl[i], nx)) + xl[i] + base;
  } else {
    const bool isx = nx >= ny && nx >= nz, isy = !isx && ny >= nz;
    bx.axis = isx ? 0 : isy ? 1 : 2;
    bx.len = isx ? nx : isy ? ny : nz;
    const int nm = isx || isy ? nz : ny, nn = isx ? ny : nx;
    box_cut(bx.len, nm, nn, bx.ca, bx.cm, bx.cn);
    bx.ca = __builtin_amdgcn_readfirstlane(bx.ca);
    bx.cm = __builtin_amdgcn_readfirstlane(bx.cm);
    bx.cn = __builtin_amdgcn_readfirstlane(bx.cn);
    bx.slabs = __builtin_amdgcn_readfirstlane((bx.len - 2) / (bx.ca - 1) + 1);
    // (an axis of one voxel is a column of its own)
    auto columns = [](int n, int c) { return n < 2 ? 1 : (n - 2) / (c - 1) + 1; };
    const int pm = columns(nm, bx.cm);
    bx.pn = __builtin_amdgcn_readfirstlane(columns(nn, bx.cn));
    bx.n = __builtin_amdgcn_readfirstlane(bx.slabs * pm * bx.pn);
    const int layer = bx.cm * bx.cn;
    bx.dx = isx ? layer : 1;
    bx.dy = a.H == 1 ? 0 : isx ? 1 : isy ? layer : bx.cn;
    bx.dz = a.T == 1 ? 0 : isx || isy ? bx.cn : layer;
    // column of a corner v along an axis: floor(v / (c - 1)); (v + 0.5) / d is at least
    // 0.5 / d from an integer, far above the rounding for v < 2^15
    const float rm = 1.0f / static_cast<float>(bx.cm - 1), rn = 1.0f / static_cast<float>(bx.cn - 1);
    auto div = [](int v, float r) { return static_cast<int>((static_cast<float>(v) + 0.5f) * r); };
#pragma unroll
    for (int i = 0; i < SLOTS; ++i) {
      if (kSubs * i >= a.K) continue;
      const int z = zl[i] - bx.zlo, y = yl[i] - bx.ylo, x = xl[i] - bx.xlo;
      const int la = isx ? x : isy ? y : z;
      int m = isx || isy ? z : y, l = isx ? y : x, col = 0;
      if (bx.n > bx.slabs) {
        const int cm = pm > 1 ? div(m, rm) : 0, cn = bx.pn > 1 ? div(l, rn) : 0;
        col = cm * bx.pn + cn;
        m -= cm * (bx.cm - 1);
        l -= cn * (bx.cn - 1);
      }
      tp.at[i] = (col * bx.len + la) * layer + m * bx.cn + l;
    }
  }
  bx.nv = bx.ca * bx.cm * bx.cn;
  // hardware reciprocals (1 ulp): (v + 0.5) / d truncates exactly for v < kBoxCap
  bx.rrow = __builtin_amdgcn_rcpf(static_cast<float>(bx.cn));
  bx.rlayer = __builtin_amdgcn_rcpf(static_cast<float>(bx.cm * bx.cn));
}

__device__ __forceinline__ BoxSeg box_seg(const BoxPieces& bx, int s) {
  BoxSeg g{bx.zlo, bx.ylo, bx.xlo, 0, 0, 0};
  if (bx.n == 1) return g;
  const int col = s / bx.slabs, a0 = (s - col * bx.slabs) * (bx.ca - 1);
  const int m0 = col / bx.pn * (bx.cm - 1), l0 = col % bx.pn * (bx.cn - 1);
  const int layer = bx.cm * bx.cn;
  g.z0 = __builtin_amdgcn_readfirstlane(bx.zlo + (bx.axis == 2 ? a0 : m0));
  g.y0 = __builtin_amdgcn_readfirstlane(bx.ylo + (bx.axis == 2 ? m0 : bx.axis == 1 ? a0 : l0));
  g.x0 = __builtin_amdgcn_readfirstlane(bx.xlo + (bx.axis == 0 ? a0 : l0));
  g.base = __builtin_amdgcn_readfirstlane((col * bx.len + a0) * layer);
  // the box's last layer is no tap's first, and its last slab may reach past it
  const int left = bx.len - a0;
  g.taps = __builtin_amdgcn_readfirstlane((min(bx.ca, left) - 1) * layer);
  g.own = __builtin_amdgcn_readfirstlane((left > bx.ca ? bx.ca - 1 : left) * layer);
  return g;
}

// Rows of one sample and head behind a buffer resource: 32-bit byte offsets,
// rows outside the volume or the box at an offset past the end read as zero.
constexpr int kBufWord3 = 0x00020000;  // raw 32-bit dwords, no swizzle (gfx9)
__device__ __forceinline__ __amdgpu_buffer_rsrc_t box_rows(const void* base, int64_t bytes) {
  // wave-uniform by construction; said so, the resource stays in scalar registers
  const uint64_t p = reinterpret_cast<uint64_t>(base);
  const uint32_t lo = __builtin_amdgcn_readfirstlane(static_cast<uint32_t>(p));
  const uint32_t hi = __builtin_amdgcn_readfirstlane(static_cast<uint32_t>(p >> 32));
  const uint32_t n = __builtin_amdgcn_readfirstlane(
      static_cast<uint32_t>(bytes < static_cast<int64_t>(kNoRow) ? bytes : kNoRow));
  return __builtin_amdgcn_make_buffer_rsrc(
      reinterpret_cast<void*>(static_cast<uint64_t>(hi) << 32 | lo), 0, static_cast<int>(n),
      kBufWord3);
}

// The blocks of 16 voxels of a piece are dealt to the waves in pairs, wave w
// taking pairs w, w + 8, ...: in the score tables' build and in the weighted
// sums alike.  Byte offsets of the wave's own voxel rows of a piece (kNoRow where
// the piece reaches past the box or the volume), in LDS: written by the wave for
// itself (no barrier), once per piece, where a lane would otherwise derive ~16 of
// them, ~30 instructions each, four lanes of a wave the same.
__device__ __forceinline__ void box_row_offsets(const Args& a, const Tile& tl, const BoxPieces& bx,
                                                const BoxSeg& g, uint32_t stride, uint32_t* rows) {
  // the wave's voxels in order: e = 32 (pair / 8) + voxel of the pair
  const int np = (bx.nv + 31) >> 5;
#pragma nounroll
  for (int p = tl.wave + kWaves * (tl.lane >> 5); p < np; p += 2 * kWaves) {
    const int vi = 32 * p + (tl.lane & 31);
    const int va = static_cast<int>((static_cast<float>(vi) + 0.5f) * bx.rlayer);
    const int r = vi - va * (bx.cm * bx.cn);
    const int vm = static_cast<int>((static_cast<float>(r) + 0.5f) * bx.rrow);
    const int vl = r - vm * bx.cn;
    const int z = g.z0 + (bx.axis == 2 ? va : vm);
    const int y = g.y0 + (bx.axis == 2 ? vm : bx.axis == 1 ? va : vl);
    const int x = g.x0 + (bx.axis == 0 ? va : vl);
    const bool ok = vi < bx.nv && z <= bx.zhi && y <= bx.yhi && x <= bx.xhi;
    const uint32_t row = (static_cast<uint32_t>(z) * a.H + y) * static_cast<uint32_t>(a.W) + x;
    rows[vi] = ok ? row * stride : kNoRow;
  }
}

// 8 channels from byte offset `off` + `imm` of a row, as a matrix-core operand
// of element type E from storage type S.
template <typename S, typename E>
__device__ __forceinline__ op_t<E> buf_op(__amdgpu_buffer_rsrc_t r, uint32_t off, int imm) {
  if constexpr (sizeof(E) == 2) {
    return __builtin_bit_cast(bf16x8_t, __builtin_amdgcn_raw_buffer_load_b128(r, off, imm, 0));
  } else if constexpr (sizeof(S) == 4) {
    const u32x4_t x = __builtin_bit_cast(u32x4_t, __builtin_amdgcn_raw_buffer_load_b128(r, off, imm, 0));
    const u32x4_t y =
        __builtin_bit_cast(u32x4_t, __builtin_amdgcn_raw_buffer_load_b128(r, off, imm + 16, 0));
    f32x8_t o;
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      o[i] = __uint_as_float(x[i]);
      o[4 + i] = __uint_as_float(y[i]);
    }
    return o;
  } else {
    const u32x4_t x = __builtin_bit_cast(u32x4_t, __builtin_amdgcn_raw_buffer_load_b128(r, off, imm, 0));
    f32x8_t o;
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      o[2 * i] = __uint_as_float(x[i] << 16);
      o[2 * i + 1] = __uint_as_float(x[i] & 0xffff0000u);
    }
    return o;
  }
}

// N consecutive channels (2 or 4) as floats, from storage type S.
template <typename S, int N>
__device__ __forceinline__ void buf_f32(__amdgpu_buffer_rsrc_t r, uint32_t off, int imm,
                                        float (&o)[N]) {
  if constexpr (sizeof(S) == 4 && N == 4) {
    const u32x4_t x = __builtin_bit_cast(u32x4_t, __builtin_amdgcn_raw_buffer_load_b128(r, off, imm, 0));
#pragma unroll
    for (int i = 0; i < 4; ++i) o[i] = __uint_as_float(x[i]);
  } else if constexpr (sizeof(S) == 4 || N == 4) {
    typedef __attribute__((ext_vector_type(2))) unsigned int u32x2_t;
    const u32x2_t x = __builtin_bit_cast(u32x2_t, __builtin_amdgcn_raw_buffer_load_b64(r, off, imm, 0));
    if constexpr (sizeof(S) == 4) {
      o[0] = __uint_as_float(x[0]);
      o[1] = __uint_as_float(x[1]);
    } else {
#pragma unroll
      for (int i = 0; i < 2; ++i) {
        o[2 * i] = __uint_as_float(x[i] << 16);
        o[2 * i + 1] = __uint_as_float(x[i] & 0xffff0000u);
      }
    }
  } else {
    const uint32_t x = static_cast<uint32_t>(__builtin_amdgcn_raw_buffer_load_b32(r, off, imm, 0));
    o[0] = __uint_as_float(x << 16);
    o[1] = __uint_as_float(x & 0xffff0000u);
  }
}

// The tile's rows (queries lane % 16) as matrix-core operands: x[c] holds
// channels 32 c + 8 (lane / 16) + [0, 8); zero past hd and for queries outside.
template <int HD, typename S, typename E, bool RG>
__device__ __forceinline__ void box_tile_rows(const Args& a, const Tile& tl, const S* base,
                                              int64_t stride, int hd, op_t<E> (&x)[HD / 32]) {
  const int64_t row = tile_row(a, tl, tl.lane & 15);
  const int c0 = 8 * (tl.lane >> 4);
#pragma unroll
  for (int c = 0; c < HD / 32; ++c) {
    x[c] = zero_op<E>();
    if (row < 0 || (RG && c0 + 32 * c >= hd)) continue;
    const S* p = base + row * stride + static_cast<int64_t>(tl.head) * hd + c0 + 32 * c;
    if constexpr (sizeof(S) == sizeof(E)) {
      x[c] = load_op<E>(p);
    } else {
      const u32x4_t w = load16(p);
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        x[c][2 * i] = __uint_as_float(w[i] << 16);
        x[c][2 * i + 1] = __uint_as_float(w[i] & 0xffff0000u);
      }
    }
  }
}

// table[m][v] = x[m] . Y[v] for the n voxels (or extra keys) v, whose row
// offsets are off(v): NB blocks of loads in flight per wave.  The rows are the A
// operand, so a lane holds 4 consecutive voxels of one query and stores 16 bytes.
template <int HD, typename S, typename E, bool RG, int NB, typename Off>
__device__ __forceinline__ void box_scores(const Tile& tl, __amdgpu_buffer_rsrc_t rows,
                                           const Off& off, int n, int hd,
                                           const op_t<E> (&x)[HD / 32], float* table) {
  static_assert(NB % 2 == 0, "whole pairs of blocks");
  const int np = (n + 31) >> 5;
  const int c0 = 8 * (tl.lane >> 4);
  const uint32_t cb = static_cast<uint32_t>(c0) * sizeof(S);
  float* const trow = &table[(tl.lane & 15) * kBoxRow + 4 * (tl.lane >> 4)];
#pragma nounroll
  for (int p0 = tl.wave; p0 < np; p0 += kWaves * (NB / 2)) {
    op_t<E> y[NB][HD / 32];
#pragma unroll
    for (int j = 0; j < NB; ++j) {
      const int p = p0 + kWaves * (j / 2);
      if (p >= np) break;
      const uint32_t o = off(32 * p + 16 * (j & 1) + (tl.lane & 15)) + cb;
#pragma unroll
      for (int c = 0; c < HD / 32; ++c)
        y[j][c] = buf_op<S, E>(rows, RG && c0 + 32 * c >= hd ? kNoRow : o,
                               32 * c * static_cast<int>(sizeof(S)));
    }
#pragma unroll
    for (int j = 0; j < NB; ++j) {
      const int p = p0 + kWaves * (j / 2);
      if (p >= np) break;
      f32x4_t acc = {0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
      for (int c = 0; c < HD / 32; ++c) acc = mma16(y[j][c], x[c], acc);
      __builtin_memcpy(trow + 32 * p + 16 * (j & 1), &acc, sizeof(acc));
    }
  }
}

// box_scores for padded head sizes (fp32 products): the products of a score in chains of
// 16, whose sums are then added up.  The general kernels, which these sizes took before,
// sum in 16 short chains; one chain over the head (box_scores) put the offsets' gradients
// 28 % further from 64 bits than theirs at 112 channels, these are 4 % nearer.  The rows'
// next 32 channels load during a step's products.
template <int HD, typename S, bool RG, typename Off>
__device__ __forceinline__ void box_scores_split(const Tile& tl, __amdgpu_buffer_rsrc_t rows,
                                                 const Off& off, int n, int hd,
                                                 const f32x8_t (&x)[HD / 32], float* table) {
  const int np = (n + 31) >> 5;
  const int c0 = 8 * (tl.lane >> 4);
  const uint32_t cb = static_cast<uint32_t>(c0) * sizeof(S);
  float* const trow = &table[(tl.lane & 15) * kBoxRow + 4 * (tl.lane >> 4)];
  // blocks of 16 voxels in the wave's order: 2 pair, 2 pair + 1 of its pairs
  const int nb = 2 * np;
  f32x8_t y;
  uint32_t o;
  auto begin = [&](int b) {
    o = off(16 * b + (tl.lane & 15)) + cb;
    y = buf_op<S, float>(rows, RG && c0 >= hd ? kNoRow : o, 0);
  };
  if (2 * tl.wave < nb) begin(2 * tl.wave);
#pragma nounroll
  for (int b = 2 * tl.wave; b < nb;) {
    const int bn = b + ((b & 1) ? 2 * kWaves - 1 : 1);
    f32x4_t acc = {0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
    for (int c = 0; c < HD / 32; ++c) {
      const f32x8_t z = y;
      if (c + 1 < HD / 32)
        y = buf_op<S, float>(rows, RG && c0 + 32 * (c + 1) >= hd ? kNoRow : o,
                             32 * (c + 1) * static_cast<int>(sizeof(S)));
      else if (bn < nb)
        begin(bn);
      acc = mma16_add(z, x[c], acc);
      __builtin_amdgcn_sched_barrier(0);  // keeps the later steps' loads from moving up
    }
    __builtin_memcpy(trow + 16 * b, &acc, sizeof(acc));
    b = bn;
  }
}

// Blocks of rows whose loads a wave keeps in flight in box_scores.
template <int HD, typename E>
constexpr int box_score_blocks() {
  constexpr int regs = HD / 32 * (sizeof(E) == 2 ? 4 : 8);  // per block
  return regs > 8 ? 2 : sizeof(E) == 4 ? 4 : 6;
}

// Channel of accumulator tile t, column n (lane % 16), of box_weighted.
template <int HD, typename E>
__device__ __forceinline__ int box_channel(int t, int n) {
  if constexpr (sizeof(E) == 2) return 16 * t + n;
  // fp32: 64 channels as 4 consecutive ones per lane, a rest of 32 as 2
  if (t / 4 < HD / 64) return 64 * (t / 4) + 4 * n + t % 4;
  return 64 * (HD / 64) + 2 * n + t % 4;
}

// acc[t] += sum over this wave's voxels v of table[q][v] * Y[v][channels], the
// table in fixed point, or (FT) floats; blocks of 32 voxels over the waves (bf16), of 16
// (fp32).  acc[t] register r: query 4 (lane / 16) + r, channel box_channel(t).
//
// bf16: the product contracts over voxels, so its B operand needs 8 voxels of
// one channel per lane, while a row load gives 8 channels of one voxel.  The
// matrix cores transpose: rows as the A operand times a 32 x 16 selection of
// the identity leaves 4 voxels of one channel per lane, exact in fp32 (one
// product is the value, the rest are zeros), and truncates back to bf16 without
// rounding.  Two blocks' results make one B operand, with the table's voxels in
// the same order.  No LDS staging, no barrier.  (A row with a non-finite value
// spoils all its channels this way: the caller tests the result and takes
// box_weighted_safe then.)
// fp32: a 16x16x4 product takes one voxel per lane group, so rows are loaded in
// the B operand's layout directly.
// The rows of the wave's first pair of blocks are loaded by
// box_weighted_begin, ahead of the table's last updates and barrier.
// bf16: over the groups C0 .. C1 - 1 of 32 channels.  A caller that keeps its taps over
// the call (KEEP) takes fewer groups at a time: registers beside the accumulators (HD / 4)
// are 8 a group for the rows in flight, ~50 for the transposition, the table's operand and
// addresses, and ~30 for the taps (and extra keys, XK), of 128.
template <int HD, bool KEEP, bool XK>
constexpr int box_groups() {
  return !KEEP || HD == 32 ? HD / 32 : XK ? 1 : 2;
}
template <int N, typename E>
struct BoxAhead {
  bf16x8_t y[sizeof(E) == 4 ? 1 : N][2];
};
template <int N, typename S, typename E, typename Off>
__device__ __forceinline__ void box_weighted_begin(const Tile& tl, __amdgpu_buffer_rsrc_t rows,
                                                   const Off& off, int n, int c0,
                                                   BoxAhead<N, E>& ah) {
  if constexpr (sizeof(E) == 2) {
    if (tl.wave >= (n + 31) >> 5) return;
    const uint32_t cb = static_cast<uint32_t>(8 * (tl.lane >> 4) + 32 * c0) * sizeof(S);
    const int v = 32 * tl.wave + (tl.lane & 15);
    const uint32_t o0 = off(v) + cb, o1 = off(v + 16) + cb;
#pragma unroll
    for (int c = 0; c < N; ++c) {
      ah.y[c][0] = buf_op<S, E>(rows, o0, 64 * c);
      ah.y[c][1] = buf_op<S, E>(rows, o1, 64 * c);
    }
  }
}
// 8 words of a table as a bf16 operand.
template <bool FT>
__device__ __forceinline__ bf16x8_t table_op(const int (&w)[8]) {
  if constexpr (!FT) return fix_to_op<bf16>(w);
  u32x4_t r;
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    const f32x2_t f = {__int_as_float(w[2 * i]), __int_as_float(w[2 * i + 1])};
    r[i] = __builtin_bit_cast(uint32_t, __builtin_convertvector(f, bf16x2_t));
  }
  return __builtin_bit_cast(bf16x8_t, r);
}
template <int HD, typename S, typename E, bool RG, bool FT, int C0, int C1, typename Off>
__device__ __forceinline__ void box_weighted(const Tile& tl, __amdgpu_buffer_rsrc_t rows,
                                             const Off& off, int n, int hd, const int* table,
                                             BoxAhead<C1 - C0, E>& ah, f32x4_t (&acc)[HD / 16]) {
  const int m = tl.lane & 15, g = tl.lane >> 4;
  if constexpr (sizeof(E) == 2) {
    static_assert(!RG, "bf16 products take whole 32-channel groups");
    // selection operands: lane (n, g) holds rows k = 8 g + [0, 8) of column n,
    // one where k = n (first 16 channels) or n + 16 (second)
    bf16x8_t sel[2];
#pragma unroll
    for (int h = 0; h < 2; ++h) {
      u32x4_t w;
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        const int k = 8 * g + 2 * i - 16 * h;  // of the word's low half
        w[i] = k == m ? 0x3f80u : k + 1 == m ? 0x3f800000u : 0u;
      }
      sel[h] = __builtin_bit_cast(bf16x8_t, w);
    }
    const uint32_t cb = static_cast<uint32_t>(8 * g + 32 * C0) * sizeof(S);
    const int np = (n + 31) >> 5;
    const f32x4_t zero = {0.0f, 0.0f, 0.0f, 0.0f};
    auto& y = ah.y;
#pragma nounroll
    for (int p = tl.wave; p < np; p += kWaves) {
      const int* const tr = &table[m * kBoxRow + 32 * p + 4 * g];
      int w[8];
      __builtin_memcpy(&w[0], tr, 16);
      __builtin_memcpy(&w[4], tr + 16, 16);
      const int pn = p + kWaves;
      const bool more = pn < np;
      uint32_t o0 = kNoRow, o1 = kNoRow;
      if (more) {
        o0 = off(32 * pn + m) + cb;
        o1 = off(32 * pn + 16 + m) + cb;
      }
      const bf16x8_t av = table_op<FT>(w);
#pragma unroll
      for (int c = 0; c < C1 - C0; ++c) {
        f32x4_t d[2][2];
        auto transpose = [&](int h) {
          d[h][0] = mma16(y[c][0], sel[h], zero);
          d[h][1] = mma16(y[c][1], sel[h], zero);
        };
        auto product = [&](int h) {
          u32x4_t b;
#pragma unroll
          for (int j = 0; j < 2; ++j) {
            b[2 * j] = __builtin_amdgcn_perm(__float_as_uint(d[h][j][1]),
                                             __float_as_uint(d[h][j][0]), 0x07060302u);
            b[2 * j + 1] = __builtin_amdgcn_perm(__float_as_uint(d[h][j][3]),
                                                 __float_as_uint(d[h][j][2]), 0x07060302u);
          }
          const bf16x8_t bo = __builtin_bit_cast(bf16x8_t, b);
          acc[2 * (C0 + c) + h] = mma16(av, bo, acc[2 * (C0 + c) + h]);
        };
        transpose(0);
        if (C1 - C0 < HD / 32) product(0);  // (with the taps in registers)
        transpose(1);
        if (more) {  // later blocks' rows take these registers
          y[c][0] = buf_op<S, E>(rows, o0, 64 * c);
          y[c][1] = buf_op<S, E>(rows, o1, 64 * c);
        }
        if (C1 - C0 == HD / 32) product(0);
        product(1);
      }
    }
  } else {
    constexpr int N4 = HD / 64, N2 = (HD % 64) / 32;
    const int nblk = 2 * ((n + 31) >> 5);
#pragma nounroll
    for (int b = 2 * tl.wave; b < nblk; b += (b & 1) ? 2 * kWaves - 1 : 1) {
      const int blk = b;
      int w[4];
      __builtin_memcpy(w, &table[m * kBoxRow + 16 * blk + 4 * g], 16);
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        const uint32_t o = off(16 * blk + 4 * g + j);
        const float av = FT ? __int_as_float(w[j]) : static_cast<float>(w[j]);
#pragma unroll
        for (int c = 0; c < N4; ++c) {
          float y[4];
          const int ch = 64 * c + 4 * m;
          const bool none = RG && ch >= hd;
          buf_f32<S, 4>(rows, none ? kNoRow : o + 4 * m * static_cast<uint32_t>(sizeof(S)),
                        64 * c * static_cast<int>(sizeof(S)), y);
#pragma unroll
          for (int t = 0; t < 4; ++t)
            acc[4 * c + t] = __builtin_amdgcn_mfma_f32_16x16x4f32(av, y[t], acc[4 * c + t], 0, 0, 0);
        }
        if constexpr (N2 > 0) {
          float y[2];
          const int ch = 64 * N4 + 2 * m;
          const bool none = RG && ch >= hd;
          buf_f32<S, 2>(rows, none ? kNoRow : o + 2 * m * static_cast<uint32_t>(sizeof(S)),
                        64 * N4 * static_cast<int>(sizeof(S)), y);
#pragma unroll
          for (int t = 0; t < 2; ++t)
            acc[4 * N4 + t] =
                __builtin_amdgcn_mfma_f32_16x16x4f32(av, y[t], acc[4 * N4 + t], 0, 0, 0);
        }
      }
    }
  }
}

// box_weighted by plain arithmetic, one lane per output (register layout of
// acc), over the voxels a query's taps touch (a non-zero table entry: see
// box_scatter), as grid_sample reads them: taken after a non-finite result, where
// a product of a row's non-finite value and a zero weight would spoil queries
// that do not sample the row, and the transposition the row's other channels.  `unit`:
// the weights' unit (the products take it off the sum, where large values times 2^30
// overflow).
template <int HD, typename S, typename E, bool RG, bool FT, typename Off>
__device__ __forceinline__ void box_weighted_safe(const Tile& tl, __amdgpu_buffer_rsrc_t rows,
                                                  const Off& off, int n, int hd, const int* table,
                                                  float unit, f32x4_t (&acc)[HD / 16]) {
  const int m = tl.lane & 15, g = tl.lane >> 4;
#pragma nounroll
  for (int e = 0;; ++e) {  // the wave's voxels: pairs w, w + 8, ... of blocks
    const int v = 32 * (tl.wave + kWaves * (e >> 5)) + (e & 31);
    if (v >= n) break;
    const uint32_t o = off(v);
    if (o == kNoRow) continue;  // every lane: v is wave-uniform
    int w[4];
#pragma unroll
    for (int r = 0; r < 4; ++r) w[r] = table[(4 * g + r) * kBoxRow + v];
#pragma unroll
    for (int t = 0; t < HD / 16; ++t) {
      const int ch = box_channel<HD, E>(t, m);
      const uint32_t at = RG && ch >= hd ? kNoRow : o + static_cast<uint32_t>(ch * sizeof(S));
      float y;
      if constexpr (sizeof(S) == 2)
        y = __uint_as_float(
            static_cast<uint32_t>(__builtin_amdgcn_raw_buffer_load_b16(rows, at, 0, 0)) << 16);
      else
        y = __uint_as_float(
            static_cast<uint32_t>(__builtin_amdgcn_raw_buffer_load_b32(rows, at, 0, 0)));
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        float f = FT ? __int_as_float(w[r]) : static_cast<float>(w[r]);
        if constexpr (sizeof(E) == 2) f = to_f32(from_f32<bf16>(f));  // the products' operand
        f *= unit;
        if (w[r] != 0) acc[t][r] = __builtin_fmaf(f, y, acc[t][r]);
      }
      __builtin_amdgcn_sched_barrier(0);  // one load at a time: the caller keeps its taps
    }
  }
}

// Zeroes the first n4 * 4 words of every table row.
__device__ __forceinline__ void box_zero(int* table, int n4) {
  // thread: 32 lanes per row (16 rows, 512 threads)
  int* const row = &table[(threadIdx.x >> 5) * kBoxRow];
  const u32x4_t z = {0u, 0u, 0u, 0u};
#pragma nounroll
  for (int e = threadIdx.x & 31; e < n4; e += 32) __builtin_memcpy(&row[4 * e], &z, sizeof(z));
}

// The tap's value interpolated from a table: lo / hi planes combined with their
// weights (0 * value for the upper one where the position is on the plane).  EDGE:
// where an upper weight is 1 the lower corner, which the position does not sample, is
// replaced by the upper one (0 times a non-finite value is not 0).
template <bool EDGE>
__device__ __forceinline__ float box_gather(const float* table, int at, int dx, int dy, int dz,
                                            float fx, float fy, float fz) {
  const float* const p = &table[at];
  const float* const pz = p + dz;
  auto plane = [&](const float* q) {
    float t0 = q[0], t1 = q[dx], b0 = q[dy], b1 = q[dy + dx];
    if (EDGE && fx == 1.0f) {
      t0 = t1;
      b0 = b1;
    }
    float top = __builtin_fmaf(fx, t1 - t0, t0), bot = __builtin_fmaf(fx, b1 - b0, b0);
    if (EDGE && fy == 1.0f) top = bot;
    return __builtin_fmaf(fy, bot - top, top);
  };
  const float lo = plane(p);
  if (EDGE && dz == 0) return lo;  // one frame (uniform)
  const float hi = plane(pz);
  const float v = __builtin_fmaf(fz, hi, (1.0f - fz) * lo);
  return EDGE && fz == 1.0f ? hi : v;
}

// The same as the reference sums it, corner by corner of those it reads: a score that is
// infinite stays so (differences of table entries would make it NaN).
__device__ __forceinline__ float box_gather_safe(const float* table, int at, int dx, int dy, int dz,
                                                 float fx, float fy, float fz) {
  float s = 0.0f;
#pragma unroll
  for (int c = 0; c < 8; ++c) {
    const bool hx = c & 1, hy = c & 2, hz = c & 4;
    if (hz && dz == 0 || hy && dy == 0) continue;  // one frame, one row (uniform)
    const float w = (hz ? fz : 1.0f - fz) * (hy ? fy : 1.0f - fy) * (hx ? fx : 1.0f - fx);
    const bool read = (hx || fx != 1.0f) && (hy || fy != 1.0f) && (hz || fz != 1.0f);
    const float t = table[at + (hz ? dz : 0) + (hy ? dy : 0) + (hx ? dx : 0)];
    if (read) s = __builtin_fmaf(w, t, s);
  }
  return s;
}

// A tap's words as opaque values at this point: keeps the compiler from hoisting
// the corner weights and addresses it derives from them out of the loop over the
// pieces (registers are the limit).  Costs no instruction.
struct BoxTap {
  int at;
  float fx, fy, fz;
};
template <int SLOTS>
__device__ __forceinline__ BoxTap box_tap(const BoxTaps<SLOTS>& tp, int i) {
  BoxTap t{tp.at[i], tp.fx[i], tp.fy[i], tp.fz[i]};
  asm volatile("" : "+v"(t.at), "+v"(t.fx), "+v"(t.fy), "+v"(t.fz));
  return t;
}
// Whether piece g (of several) holds the tap's footprint; t.at becomes the word index
// of its first corner in the row of lane query q.
__device__ __forceinline__ bool box_in(const BoxSeg& g, int q, BoxTap& t) {
  const int r = t.at - g.base;
  t.at = q * kBoxRow + r;
  return static_cast<uint32_t>(r) < static_cast<uint32_t>(g.taps);
}

// Adds the tap's weight v (fixed-point units) to its eight corners.  TOUCH: at
// least one unit (2^-30) each, which marks the corners of zero weight too
// (grid_sample reads those as well: 0 times a non-finite value is not 0), but for
// the lower ones where the upper weight is 1.
template <bool TOUCH>
__device__ __forceinline__ void box_add4(int* q, int d0, int d1, float w, float f0, float f1) {
  const float w1 = w * f1, w0 = w * (1.0f - f1), g0 = 1.0f - f0;
  auto add = [](int* p, float x, bool read) {
    if (!TOUCH) atomicAdd(p, to_fix(x));
    else if (read) atomicAdd(p, max(to_fix(x), 1));
  };
  add(q, w0 * g0, f0 != 1.0f && f1 != 1.0f);
  add(q + d0, w0 * f0, f1 != 1.0f);
  add(q + d1, w1 * g0, f0 != 1.0f);
  add(q + d1 + d0, w1 * f0, true);
}
template <bool TOUCH>
__device__ __forceinline__ void box_scatter(int* table, const BoxPieces& bx, const BoxTap& t, float v) {
  int* const p = &table[t.at];
  if (!TOUCH || t.fz != 1.0f) box_add4<TOUCH>(p, 1, bx.dy, v * (1.0f - t.fz), t.fx, t.fy);
  if (bx.dz != 0) box_add4<TOUCH>(p + bx.dz, 1, bx.dy, v * t.fz, t.fx, t.fy);
}
// The same to the corners that piece g (of several) owns: those of the tap's two
// layers along the axis that lie in it.
template <bool TOUCH>
__device__ __forceinline__ void box_scatter(int* table, const BoxPieces& bx, const BoxSeg& g, int q,
                                            const BoxTap& t, float v) {
  const int r = t.at - g.base, layer = bx.cm * bx.cn;
  const bool lo = static_cast<uint32_t>(r) < static_cast<uint32_t>(g.own);
  const bool hi = static_cast<uint32_t>(r + layer) < static_cast<uint32_t>(g.own);
  if (!(lo | hi)) return;
  const float fx = t.fx, fy = t.fy, fz = t.fz;
  float fa = fz, fm = fy, fl = fx;  // along z
  int dm = bx.dy, dl = 1;
  if (bx.axis == 1) {
    fa = fy;
    fm = fz;
    dm = bx.dz;
  } else if (bx.axis == 0) {
    fa = fx;
    fm = fz;
    dm = bx.dz;
    fl = fy;
    dl = bx.dy;
  }
  int* const p = &table[q * kBoxRow + r];
  if (lo && (!TOUCH || fa != 1.0f)) box_add4<TOUCH>(p, dl, dm, v * (1.0f - fa), fl, fm);
  if (hi) box_add4<TOUCH>(p + layer, dl, dm, v * fa, fl, fm);
}

}  // namespace tiled
}  // namespace msd
