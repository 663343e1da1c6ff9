// The attention core for head sizes that are multiples of 8 below 128 other than
// 32, 64 and 96, on the matrix-core kernels of the next larger one of these.
//
// Products in fp32 for both storage types: the general kernels, which these
// calls took before, round nothing but the results, and bf16 operands of the
// weights would (2.9e-3 against 1.7e-3 relative error of dk in bf16).
//   forward   the forward kernel reads channels past head_dim as zero;
//   backward  the fp32 kernels run on fp32 copies padded with zero channels
//             (q, k, v, dout, and for bf16 the offsets), whose gradients are then
//             packed into the outputs.  The copies cost ~1 % of the backward.
// At 4,096 tokens, 16 x 80, window 3x5x5, bf16: see launch_dsa3d_bwd_ragged.
#include "dsa3d_fwd.h"

namespace msd {

namespace {

// Matrix-core head size that holds hd channels (0: none).
int padded_head_dim(int hd) {
  if (hd % 8 != 0 || hd < 8 || hd > 128) return 0;
  return (hd + 31) / 32 * 32;
}

// The padded fp32 call.
msd_dsa3d_desc padded_desc(const msd_dsa3d_desc& d) {
  msd_dsa3d_desc p = d;
  p.head_dim = padded_head_dim(d.head_dim);
  p.dtype = MSD_F32;
  p.dkv_accum = MSD_ACCUM_F32;
  p.q_stride = p.k_stride = p.v_stride = static_cast<int64_t>(d.num_heads) * p.head_dim;
  return p;
}

// [rows, nh, hd] of storage type S (token stride `stride`) -> fp32 [rows, nh, hp],
// zero past hd.  A thread moves 8 channels.
template <typename S>
__global__ __launch_bounds__(256) void pad_rows_kernel(const S* __restrict__ src, int64_t stride,
                                                       int64_t rows, int nh, int hd, int hp,
                                                       float* __restrict__ dst) {
  const int64_t per = static_cast<int64_t>(nh) * (hp / 8), n = rows * per;
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
      for (int j = 0; j < 8; ++j) v[j] = to_f32(raw[j]);
    }
    __builtin_memcpy(dst + 8 * i, v, sizeof(v));
  }
}

// fp32 [rows, nh, hp] -> storage type S [rows, nh, hd], token stride `stride`.
template <typename S>
__global__ __launch_bounds__(256) void unpad_rows_kernel(const float* __restrict__ src,
                                                         int64_t rows, int nh, int hd, int hp,
                                                         S* __restrict__ dst, int64_t stride) {
  const int64_t per = static_cast<int64_t>(nh) * (hd / 8), n = rows * per;
  for (int64_t i = static_cast<int64_t>(blockIdx.x) * blockDim.x + threadIdx.x; i < n;
       i += static_cast<int64_t>(gridDim.x) * blockDim.x) {
    const int64_t r = i / per;
    const int e = static_cast<int>(i - r * per), h = e / (hd / 8), c = 8 * (e - h * (hd / 8));
    float v[8];
    __builtin_memcpy(v, src + (r * nh + h) * hp + c, sizeof(v));
    S o[8];
#pragma unroll
    for (int j = 0; j < 8; ++j) o[j] = from_f32<S>(v[j]);
    __builtin_memcpy(dst + r * stride + h * hd + c, o, sizeof(o));
  }
}

// n elements between bf16 and fp32, 4 a thread.
template <typename A, typename B>
__global__ __launch_bounds__(256) void convert_kernel(const A* __restrict__ src,
                                                      B* __restrict__ dst, int64_t n) {
  for (int64_t i = 4 * (static_cast<int64_t>(blockIdx.x) * blockDim.x + threadIdx.x); i < n;
       i += 4 * static_cast<int64_t>(gridDim.x) * blockDim.x) {
    if (i + 4 <= n) {
      A a[4];
      B b[4];
      __builtin_memcpy(a, src + i, sizeof(a));
#pragma unroll
      for (int j = 0; j < 4; ++j) b[j] = from_f32<B>(to_f32(a[j]));
      __builtin_memcpy(dst + i, b, sizeof(b));
    } else {
      for (int64_t j = i; j < n; ++j) dst[j] = from_f32<B>(to_f32(src[j]));
    }
  }
}

unsigned copy_blocks(int64_t items) {
  return static_cast<unsigned>(std::min<int64_t>(std::max<int64_t>((items + 255) / 256, 1), 65536));
}

// Workspace (byte offsets): padded q, k, v, dout, dq, dk, dv; padded extra keys,
// values and their gradients; for bf16 fp32 offsets and their gradient; the
// padded call's own workspace.
struct RaggedWs {
  size_t row[7], extra[4], off[2], inner, bytes;
};
RaggedWs ragged_ws(const msd_dsa3d_desc& d) {
  const msd_dsa3d_desc p = padded_desc(d);
  const size_t rows = static_cast<size_t>(d.B) * d.T * d.H * d.W;
  const size_t D = static_cast<size_t>(d.num_heads) * p.head_dim;
  const size_t taps = rows * d.num_heads * d.kt * d.kh * d.kw * 3;
  auto up = [](size_t x) { return (x + 255) / 256 * 256; };
  RaggedWs w;
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
    if (d.dtype == MSD_BF16) at = up(at + taps * 4);
  }
  w.inner = at;
  w.bytes = at + dsa3d_tiled_bwd_ws_bytes(p);
  return w;
}

template <typename S>
hipError_t bwd_typed(const msd_dsa3d_desc& d, const void* q, const void* k, const void* v,
                     const void* off, const void* ek, const void* ev, const void* dout,
                     const float* lse, const float* dlse, void* dq, void* dk, void* dv, void* doff,
                     void* dek, void* dev, char* ws, hipStream_t s) {
  const msd_dsa3d_desc p = padded_desc(d);
  const RaggedWs L = ragged_ws(d);
  const int nh = d.num_heads, hd = d.head_dim, hp = p.head_dim;
  const int64_t rows = static_cast<int64_t>(d.B) * d.T * d.H * d.W, D = int64_t{nh} * hd;
  const int64_t erows = static_cast<int64_t>(d.B) * d.extra_g;
  const int64_t noff = rows * nh * d.kt * d.kh * d.kw * 3;
  auto f32 = [&](size_t at) { return reinterpret_cast<float*>(ws + at); };
  auto pad = [&](const void* src, int64_t stride, int64_t n, size_t at) {
    hipLaunchKernelGGL((pad_rows_kernel<S>), dim3(copy_blocks(n * nh * (hp / 8))), dim3(256), 0, s,
                       static_cast<const S*>(src), stride, n, nh, hd, hp, f32(at));
  };
  auto unpad = [&](size_t at, int64_t n, void* dst, int64_t stride) {
    hipLaunchKernelGGL((unpad_rows_kernel<S>), dim3(copy_blocks(n * nh * (hd / 8))), dim3(256), 0,
                       s, f32(at), n, nh, hd, hp, static_cast<S*>(dst), stride);
  };
  pad(q, d.q_stride, rows, L.row[0]);
  pad(k, d.k_stride, rows, L.row[1]);
  pad(v, d.v_stride, rows, L.row[2]);
  pad(dout, D, rows, L.row[3]);
  if (erows > 0) {
    pad(ek, D, erows, L.extra[0]);
    pad(ev, D, erows, L.extra[1]);
  }
  const void* off32 = off;
  void* doff32 = doff;
  if constexpr (sizeof(S) == 2) {
    hipLaunchKernelGGL((convert_kernel<bf16, float>), dim3(copy_blocks((noff + 3) / 4)), dim3(256),
                       0, s, static_cast<const bf16*>(off), f32(L.off[0]), noff);
    off32 = f32(L.off[0]);
    doff32 = f32(L.off[1]);
  }
  auto extra = [&](int i) { return erows > 0 ? f32(L.extra[i]) : nullptr; };
  const hipError_t e = launch_dsa3d_bwd_tiled(
      p, f32(L.row[0]), f32(L.row[1]), f32(L.row[2]), off32, extra(0), extra(1), nullptr,
      f32(L.row[3]), lse, dlse, f32(L.row[4]), f32(L.row[5]), f32(L.row[6]), doff32, extra(2),
      extra(3), ws + L.inner, s, true);
  if (e != hipSuccess) return e;
  unpad(L.row[4], rows, dq, d.q_stride);
  unpad(L.row[5], rows, dk, d.k_stride);
  unpad(L.row[6], rows, dv, d.v_stride);
  if (erows > 0) {
    unpad(L.extra[2], erows, dek, D);
    unpad(L.extra[3], erows, dev, D);
  }
  if constexpr (sizeof(S) == 2)
    hipLaunchKernelGGL((convert_kernel<float, bf16>), dim3(copy_blocks((noff + 3) / 4)), dim3(256),
                       0, s, f32(L.off[1]), static_cast<bf16*>(doff), noff);
  return hipGetLastError();
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
  // the forward addresses a sample's rows with 32-bit byte offsets, and packs a
  // tap's piece of a cut box into 17 bits (a sample of less than 2^25 voxels)
  const msd_dsa3d_desc p = padded_desc(d);
  if (static_cast<int64_t>(d.T) * d.H * d.W >= int64_t{1} << 25 || !rows_below_limit(d) ||
      !rows_below_limit(p))
    return false;
  return dsa3d_tiled_supported(p, nullptr, nullptr, nullptr);
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
                                   const void* dout, const float* lse, const float* dlse, void* dq,
                                   void* dk, void* dv, void* doff, void* dek, void* dev, void* ws,
                                   hipStream_t s) {
  auto* const w = static_cast<char*>(ws);
  if (d.dtype == MSD_BF16)
    return bwd_typed<bf16>(d, q, k, v, off, ek, ev, dout, lse, dlse, dq, dk, dv, doff, dek, dev, w, s);
  return bwd_typed<float>(d, q, k, v, off, ek, ev, dout, lse, dlse, dq, dk, dv, doff, dek, dev, w, s);
}

}  // namespace msd
