// The attention core for head sizes that are multiples of 8 below 128 other than
// 32, 64 and 96, on the matrix-core kernels of the next larger one of these.
//
// Products in fp32 for both storage types: the general kernels, which these
// calls took before, hold operands and weights in fp32, and bf16 operands of the
// weights would be less precise (2.9e-3 against 1.7e-3 relative error of dk in
// bf16).  The weights p w and ds w are summed in fixed point of 2^-30 of their
// query's total; every result is at least as near to 64 bits as the general
// kernels' (fp32, head sizes 8 to 120: 0.7 to 0.98 of their error).
//   forward   the forward kernel reads channels past head_dim as zero;
//   backward  the fp32 kernels run on fp32 copies padded with zero channels
//             (q, k, v, dout, and the offsets times offset_scale), whose gradients
//             are then packed into the outputs.  The copies cost ~7 % of the backward.
// 4,096 tokens, 16 x 80, window 3x5x5, bf16, forward and backward: 116 -> 1.7 ms.
//
// Non-finite values.  The general kernels gather what a query samples; products
// over whole boxes spread a non-finite row to other queries (0 * inf), and fixed
// point drops NaN.  The copies, the first kernel and the packing therefore test
// what they read and write, and where anything is not finite the general kernels
// do the whole backward again (they return at once otherwise).
#include "dsa3d_fwd.h"

namespace msd {

namespace {

// Matrix-core head size that holds hd channels (0: none).
int padded_head_dim(int hd) {
  if (hd % 8 != 0 || hd < 8 || hd > 128) return 0;
  return (hd + 31) / 32 * 32;
}

// The padded fp32 call over `heads` heads.
msd_dsa3d_desc padded_desc(const msd_dsa3d_desc& d, int heads) {
  msd_dsa3d_desc p = d;
  p.num_heads = heads;
  p.offset_scale = 1.0f;  // in the copies
  p.head_dim = padded_head_dim(d.head_dim);
  p.dtype = MSD_F32;
  p.dkv_accum = MSD_ACCUM_F32;
  p.q_stride = p.k_stride = p.v_stride = static_cast<int64_t>(heads) * p.head_dim;
  return p;
}

// Sets *flag where any lane of the wave saw a value that is not finite.
__device__ __forceinline__ void flag_if(bool bad, int* flag) {
  if (__builtin_amdgcn_ballot_w64(bad) != 0 && (threadIdx.x & 63) == 0) atomicOr(flag, 1);
}

// Up to four tensors of one shape (blockIdx.y).
struct Rows {
  const void* src[4];
  void* dst[4];
  int64_t stride[4];  // token stride of the packed side
};

// Heads h0 .. h0 + nh - 1 of rows of storage type S, hd channels a head -> fp32
// [rows, nh, hp], zero past hd.  A thread moves 8 channels.
template <typename S>
__global__ __launch_bounds__(256) void pad_rows_kernel(Rows t, int64_t rows, int h0, int nh, int hd,
                                                       int hp, int* __restrict__ flag) {
  const S* const src = static_cast<const S*>(t.src[blockIdx.y]) + static_cast<int64_t>(h0) * hd;
  float* const dst = static_cast<float*>(t.dst[blockIdx.y]);
  const int64_t stride = t.stride[blockIdx.y];
  const int64_t per = static_cast<int64_t>(nh) * (hp / 8), n = rows * per;
  bool bad = false;
  for (int64_t i = static_cast<int64_t>(blockIdx.x) * blockDim.x + threadIdx.x; i < n;
       i += static_cast<int64_t>(gridDim.x) * blockDim.x) {
    const int64_t r = i / per;
    const int e = static_cast<int>(i - r * per), h = e / (hp / 8), c = 8 * (e - h * (hp / 8));
    float v[8];
#pragma unroll
    for (int j = 0; j < 8; ++j) v[j] = 0.0f;
    if (c < hd) {
      S raw[8];
      __builtin_memcpy(raw, src + r * stride + h * hd + c, sizeof(raw));
#pragma unroll
      for (int j = 0; j < 8; ++j) {
        v[j] = to_f32(raw[j]);
        bad |= !__builtin_isfinite(v[j]);
      }
    }
    __builtin_memcpy(dst + 8 * i, v, sizeof(v));
  }
  flag_if(bad, flag);
}

// The reverse: fp32 [rows, nh, hp] -> heads h0 .. of rows of storage type S.
template <typename S>
__global__ __launch_bounds__(256) void unpad_rows_kernel(Rows t, int64_t rows, int h0, int nh,
                                                         int hd, int hp, int* __restrict__ flag) {
  const float* const src = static_cast<const float*>(t.src[blockIdx.y]);
  S* const dst = static_cast<S*>(t.dst[blockIdx.y]) + static_cast<int64_t>(h0) * hd;
  const int64_t stride = t.stride[blockIdx.y];
  const int64_t per = static_cast<int64_t>(nh) * (hd / 8), n = rows * per;
  bool bad = false;
  for (int64_t i = static_cast<int64_t>(blockIdx.x) * blockDim.x + threadIdx.x; i < n;
       i += static_cast<int64_t>(gridDim.x) * blockDim.x) {
    const int64_t r = i / per;
    const int e = static_cast<int>(i - r * per), h = e / (hd / 8), c = 8 * (e - h * (hd / 8));
    float v[8];
    __builtin_memcpy(v, src + (r * nh + h) * hp + c, sizeof(v));
    S o[8];
#pragma unroll
    for (int j = 0; j < 8; ++j) {
      bad |= !__builtin_isfinite(v[j]);
      o[j] = from_f32<S>(v[j]);
    }
    __builtin_memcpy(dst + r * stride + h * hd + c, o, sizeof(o));
  }
  flag_if(bad, flag);
}

// Offsets (or their gradients) between their tensor, rows of `row` elements of which
// `per` from element `first` on, and fp32 [rows, per]; times `scale`.  Offsets are
// limited to 10^30 (box_setup's CLAMP).  A thread moves 4 elements.
template <typename A, typename B, bool PACK>
__global__ __launch_bounds__(256) void offsets_kernel(const A* __restrict__ src,
                                                      B* __restrict__ dst, int64_t rows, int64_t row,
                                                      int64_t first, int64_t per, float scale,
                                                      int* __restrict__ flag) {
  const int64_t p4 = (per + 3) / 4, n = rows * p4;
  bool bad = false;
  auto one = [&](float x) {
    x *= scale;
    if (PACK) {
      bad |= !__builtin_isfinite(x);
      return x;
    }
    return __builtin_amdgcn_fmed3f(x, -1e30f, 1e30f);
  };
  for (int64_t i = static_cast<int64_t>(blockIdx.x) * blockDim.x + threadIdx.x; i < n;
       i += static_cast<int64_t>(gridDim.x) * blockDim.x) {
    const int64_t r = i / p4, e = 4 * (i - r * p4);
    const A* const s = src + (PACK ? r * per : r * row + first) + e;
    B* const d = dst + (PACK ? r * row + first : r * per) + e;
    if (e + 4 <= per) {
      A a[4];
      B b[4];
      __builtin_memcpy(a, s, sizeof(a));
#pragma unroll
      for (int j = 0; j < 4; ++j) b[j] = from_f32<B>(one(to_f32(a[j])));
      __builtin_memcpy(d, b, sizeof(b));
    } else {
      for (int j = 0; e + j < per; ++j) d[j] = from_f32<B>(one(to_f32(s[j])));
    }
  }
  flag_if(bad, flag);
}

// lse and dlse (may be null) [rows, all] -> heads h0 .. of each, [rows, nh].
__global__ __launch_bounds__(256) void lse_kernel(const float* __restrict__ lse,
                                                  const float* __restrict__ dlse, int64_t rows,
                                                  int all, int h0, int nh, float* __restrict__ l,
                                                  float* __restrict__ dl, int* __restrict__ flag) {
  bool bad = false;
  for (int64_t i = static_cast<int64_t>(blockIdx.x) * blockDim.x + threadIdx.x; i < rows * nh;
       i += static_cast<int64_t>(gridDim.x) * blockDim.x) {
    const int64_t r = i / nh, at = r * all + h0 + (i - r * nh);
    l[i] = lse[at];
    bad |= !__builtin_isfinite(lse[at]);
    if (dlse != nullptr) {
      dl[i] = dlse[at];
      bad |= !__builtin_isfinite(dlse[at]);
    }
  }
  flag_if(bad, flag);
}

unsigned copy_blocks(int64_t items) {
  return static_cast<unsigned>(std::min<int64_t>(std::max<int64_t>((items + 255) / 256, 1), 65536));
}

// Workspace (byte offsets) of a group of heads: padded q, k, v, dout, dq, dk, dv; padded
// extra keys, values and their gradients; fp32 offsets and their gradients; lse, dlse; the
// padded call's own workspace.  Before the flag, which follows, room for the general
// kernels' workspace in the same place.
struct RaggedWs {
  int heads;  // of a group
  size_t row[7], extra[4], off[2], lse[2], inner, flag, bytes;
};
RaggedWs ragged_group_ws(const msd_dsa3d_desc& d, int heads) {
  const msd_dsa3d_desc p = padded_desc(d, heads);
  const size_t rows = static_cast<size_t>(d.B) * d.T * d.H * d.W;
  const size_t D = static_cast<size_t>(heads) * p.head_dim;
  auto up = [](size_t x) { return (x + 255) / 256 * 256; };
  RaggedWs w;
  w.heads = heads;
  size_t at = 0;
  for (size_t& r : w.row) {
    r = at;
    at = up(at + rows * D * 4);
  }
  for (size_t& r : w.extra) {
    r = at;
    at = up(at + static_cast<size_t>(d.B) * d.extra_g * D * 4);
  }
  for (size_t& r : w.off) {
    r = at;
    at = up(at + rows * heads * d.kt * d.kh * d.kw * 3 * 4);
  }
  for (size_t& r : w.lse) {
    r = at;
    at = up(at + rows * heads * 4);
  }
  w.inner = at;
  w.flag = up(std::max(at + dsa3d_tiled_bwd_ws_bytes(p), dsa3d_bwd_ws_bytes(d)));
  w.bytes = w.flag + 256;
  return w;
}
// A call takes its heads in groups whose copies fit 1 GiB, or what the general kernels
// need where that is more (65,536 tokens, 16 x 80, window 3x7x7, bf16: 1.0 GB against
// 7.8 GB for all heads at once and 0.7 GB of the general kernels).
RaggedWs ragged_ws(const msd_dsa3d_desc& d) {
  const size_t most = std::max(size_t{1} << 30, dsa3d_bwd_ws_bytes(d));
  RaggedWs w = ragged_group_ws(d, d.num_heads);
  for (int groups = 2; w.flag > most && w.heads > 1; ++groups)
    w = ragged_group_ws(d, (d.num_heads + groups - 1) / groups);
  return w;
}

template <typename S>
hipError_t bwd_typed(const msd_dsa3d_desc& d, const void* q, const void* k, const void* v,
                     const void* off, const void* ek, const void* ev, const void* out,
                     const void* dout, const float* lse, const float* dlse, void* dq, void* dk,
                     void* dv, void* doff, void* dek, void* dev, char* ws, hipStream_t s) {
  const RaggedWs L = ragged_ws(d);
  const int hd = d.head_dim;
  const int64_t rows = static_cast<int64_t>(d.B) * d.T * d.H * d.W;
  const int64_t D = int64_t{d.num_heads} * hd, erows = static_cast<int64_t>(d.B) * d.extra_g;
  const int64_t K3 = int64_t{d.kt} * d.kh * d.kw * 3, C = d.num_heads * K3;
  int* const flag = reinterpret_cast<int*>(ws + L.flag);
  auto f32 = [&](size_t at) { return reinterpret_cast<float*>(ws + at); };
  hipLaunchKernelGGL(fill_zero_f32, dim3(1), dim3(64), 0, s, f32(L.flag), int64_t{1});
  for (int h0 = 0; h0 < d.num_heads; h0 += L.heads) {
    const int nh = std::min(L.heads, d.num_heads - h0);
    const msd_dsa3d_desc p = padded_desc(d, nh);
    const int hp = p.head_dim;
    auto pad = [&](std::initializer_list<const void*> src, std::initializer_list<int64_t> stride,
                   const size_t* at, int64_t n) {
      Rows t{};
      int i = 0;
      for (const void* x : src) t.src[i++] = x;
      i = 0;
      for (int64_t x : stride) t.stride[i++] = x;
      for (int j = 0; j < i; ++j) t.dst[j] = f32(at[j]);
      hipLaunchKernelGGL((pad_rows_kernel<S>), dim3(copy_blocks(n * nh * (hp / 8)), i), dim3(256), 0,
                         s, t, n, h0, nh, hd, hp, flag);
    };
    auto unpad = [&](std::initializer_list<void*> dst, std::initializer_list<int64_t> stride,
                     const size_t* at, int64_t n) {
      Rows t{};
      int i = 0;
      for (void* x : dst) t.dst[i++] = x;
      i = 0;
      for (int64_t x : stride) t.stride[i++] = x;
      for (int j = 0; j < i; ++j) t.src[j] = f32(at[j]);
      hipLaunchKernelGGL((unpad_rows_kernel<S>), dim3(copy_blocks(n * nh * (hd / 8)), i), dim3(256),
                         0, s, t, n, h0, nh, hd, hp, flag);
    };
    pad({q, k, v, dout}, {d.q_stride, d.k_stride, d.v_stride, D}, L.row, rows);
    if (erows > 0) pad({ek, ev}, {D, D}, L.extra, erows);
    const dim3 ogrid(copy_blocks(rows * ((nh * K3 + 3) / 4)));
    hipLaunchKernelGGL((offsets_kernel<S, float, false>), ogrid, dim3(256), 0, s,
                       static_cast<const S*>(off), f32(L.off[0]), rows, C, h0 * K3, nh * K3,
                       d.offset_scale, flag);
    hipLaunchKernelGGL(lse_kernel, dim3(copy_blocks(rows * nh)), dim3(256), 0, s, lse, dlse, rows,
                       d.num_heads, h0, nh, f32(L.lse[0]), f32(L.lse[1]), flag);
    auto extra = [&](int i) { return erows > 0 ? f32(L.extra[i]) : nullptr; };
    const PaddedBwd padded{h0, flag};
    const hipError_t e = launch_dsa3d_bwd_tiled(
        p, f32(L.row[0]), f32(L.row[1]), f32(L.row[2]), f32(L.off[0]), extra(0), extra(1), nullptr,
        f32(L.row[3]), f32(L.lse[0]), dlse != nullptr ? f32(L.lse[1]) : nullptr, f32(L.row[4]),
        f32(L.row[5]), f32(L.row[6]), f32(L.off[1]), extra(2), extra(3), ws + L.inner, s, &padded);
    if (e != hipSuccess) return e;
    unpad({dq, dk, dv}, {d.q_stride, d.k_stride, d.v_stride}, L.row + 4, rows);
    if (erows > 0) unpad({dek, dev}, {D, D}, L.extra + 2, erows);
    hipLaunchKernelGGL((offsets_kernel<float, S, true>), ogrid, dim3(256), 0, s, f32(L.off[1]),
                       static_cast<S*>(doff), rows, C, h0 * K3, nh * K3, d.offset_scale, flag);
  }
  return launch_dsa3d_bwd_direct(d, q, k, v, off, ek, ev, out, dout, lse, dlse, dq, dk, dv, doff,
                                 dek, dev, ws, s, flag);
}

}  // namespace

// Calls of MSD_ALGO_AUTO that the matrix-core kernels take at a padded head size:
// what they take themselves (windows, extra keys, sizes, alignment) but for the
// head size, within the padded fp32 call's limits.
bool dsa3d_ragged_supported(const msd_dsa3d_desc& d, const void* q, const void* k, const void* v) {
  if (d.algo != MSD_ALGO_AUTO || padded_head_dim(d.head_dim) == 0 || d.head_dim % 32 == 0)
    return false;
  if ((d.q_stride % 8) || (d.k_stride % 8) || (d.v_stride % 8)) return false;
  for (const void* p : {q, k, v})
    if (reinterpret_cast<uintptr_t>(p) % 16) return false;
  // the forward addresses the sample's own rows with 32-bit byte offsets, and its taps'
  // words hold a sample of less than 2^25 voxels
  if (static_cast<int64_t>(d.T) * d.H * d.W >= int64_t{1} << 25 || !rows_below_limit(d))
    return false;
  return dsa3d_tiled_supported(padded_desc(d, d.num_heads), nullptr, nullptr, nullptr);
}

hipError_t launch_dsa3d_fwd_ragged(const msd_dsa3d_desc& d, const void* q, const void* k,
                                   const void* v, const void* off, const void* ek, const void* ev,
                                   void* out, float* lse, hipStream_t s) {
  const Args a = make_tiled_args(d, q, k, v, off, tile_count<1>(d.B, d.T, d.H, d.W), ek, ev);
  if (d.dtype == MSD_BF16) return fwd_typed<bf16, float, true>(d, a, out, lse, s);
  return fwd_typed<float, float, true>(d, a, out, lse, s);
}

size_t dsa3d_ragged_bwd_ws_bytes(const msd_dsa3d_desc& d) { return ragged_ws(d).bytes; }

hipError_t launch_dsa3d_bwd_ragged(const msd_dsa3d_desc& d, const void* q, const void* k,
                                   const void* v, const void* off, const void* ek, const void* ev,
                                   const void* out, const void* dout, const float* lse,
                                   const float* dlse, void* dq, void* dk, void* dv, void* doff,
                                   void* dek, void* dev, void* ws, hipStream_t s) {
  auto* const w = static_cast<char*>(ws);
  if (d.dtype == MSD_BF16)
    return bwd_typed<bf16>(d, q, k, v, off, ek, ev, out, dout, lse, dlse, dq, dk, dv, doff, dek, dev,
                           w, s);
  return bwd_typed<float>(d, q, k, v, off, ek, ev, out, dout, lse, dlse, dq, dk, dv, doff, dek, dev,
                          w, s);
}

}  // namespace msd
