// The small data movements of the action head around the MSAT blocks, one launch
// where the eager chain has several.  Each torch launch there runs 4-5 us of a
// captured graph on a few KB to a few hundred KB: latency, not bandwidth, so the win is
// the number of launches: an action of 4 steps at the release shape took 4.740 ms with
// the 14 index_selects, 12 copies and 12 modulation launches they replace, 4.64 ms now,
// with the same bits: everything here copies, or rounds where the eager chain does.
// A workgroup copies 16 KB of rows or slabs (4 loads of 16 bytes in flight per thread):
// 37 workgroups for a step's inputs, about 1250 for an embodiment's weights.
//   * copy_rows_many: up to 4 strided row blocks (time token, SA and VL inputs of a
//     denoising step into the chain's buffers);
//   * gather_slabs: slab idx[b] of up to 16 stacked parameters (the embodiment's
//     encoder / decoder weights) into per-robot buffers;
//   * modulate_pack: the output modulation LN(x) (1 + scale) + shift of normalised rows
//     and their packing for the output projection.  (The LayerNorm stays torch's: one
//     in this kernel adds in another order, and a value that rounds the other way in an
//     early denoising step shows in the action.)
#include "rldx_amd.h"
#include "rldx_common.h"

namespace rldx {
namespace {

typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));

constexpr int kMaxCopies = 4, kMaxSlabs = 16;
constexpr int kPiece = 1024;  // 16-byte units per workgroup (256 threads x 4)

bool a16(const void* p) { return (reinterpret_cast<uintptr_t>(p) & 15u) == 0; }

struct CopyArgs {
  const char* src[kMaxCopies];
  char* dst[kMaxCopies];
  int64_t src_row[kMaxCopies], src_batch[kMaxCopies], dst_row[kMaxCopies], dst_batch[kMaxCopies];
  int units[kMaxCopies];          // 16-byte units per row
  int total[kMaxCopies];          // rows x units
  int begin[kMaxCopies + 1];      // first workgroup
  int count;
};

__global__ __launch_bounds__(256) void copy_rows_kernel(CopyArgs a) {
  int i = 0;
#pragma unroll
  for (int c = 1; c < kMaxCopies; ++c)
    if (c < a.count && static_cast<int>(blockIdx.x) >= a.begin[c]) i = c;
  const int64_t b = blockIdx.y;
  const int base = (static_cast<int>(blockIdx.x) - a.begin[i]) * kPiece + static_cast<int>(threadIdx.x);
  const int units = a.units[i], total = a.total[i];
  u32x4 v[4];
#pragma unroll
  for (int j = 0; j < 4; ++j) {
    const int u = min(base + 256 * j, total - 1), r = u / units;
    v[j] = *reinterpret_cast<const u32x4*>(a.src[i] + b * a.src_batch[i] + r * a.src_row[i] + (u - r * units) * 16LL);
  }
#pragma unroll
  for (int j = 0; j < 4; ++j) {
    const int u = base + 256 * j, r = u / units;
    if (u < total)
      *reinterpret_cast<u32x4*>(a.dst[i] + b * a.dst_batch[i] + r * a.dst_row[i] + (u - r * units) * 16LL) = v[j];
  }
}

struct SlabArgs {
  const char* src[kMaxSlabs];
  char* dst[kMaxSlabs];
  int64_t units[kMaxSlabs];  // units per slab
  int begin[kMaxSlabs + 1];
  uint32_t narrow;           // bit i: units of 2 bytes (a bias of 7 actions: 14), else of 16
  const int64_t* idx;
  int64_t num;
  int count;
};

// piece `piece` of slab e of src -> slab b of dst; e < 0: bytes 0xff, NaN in every floating-point type
template <class T>
__device__ __forceinline__ void gather_piece(const char* src, char* dst, int64_t units, int64_t e, int64_t b, int piece,
                                             T nan) {
  const T* s = reinterpret_cast<const T*>(src) + e * units;
  T* d = reinterpret_cast<T*>(dst) + b * units;
  const int64_t base = static_cast<int64_t>(piece) * kPiece + threadIdx.x;
  T v[4];
#pragma unroll
  for (int j = 0; j < 4; ++j) {
    const int64_t u = base + 256 * j;
    v[j] = nan;
    if (e >= 0) v[j] = s[u < units ? u : units - 1];
  }
#pragma unroll
  for (int j = 0; j < 4; ++j)
    if (base + 256 * j < units) d[base + 256 * j] = v[j];
}

__global__ __launch_bounds__(256) void gather_slabs_kernel(SlabArgs a) {
  int i = 0;
  for (int c = 1; c < a.count; ++c)
    if (static_cast<int>(blockIdx.x) >= a.begin[c]) i = c;
  const int64_t b = blockIdx.y;
  int64_t e = a.idx[b];
  // (a bad id reads nothing, and the robot's weights become NaN: the previous robot's would pass for its own)
  if (e < 0 || e >= a.num) e = -1;
  const int piece = static_cast<int>(blockIdx.x) - a.begin[i];
  if (a.narrow >> i & 1u)
    gather_piece<uint16_t>(a.src[i], a.dst[i], a.units[i], e, b, piece, 0xffff);
  else
    gather_piece<u32x4>(a.src[i], a.dst[i], a.units[i], e, b, piece, u32x4{~0u, ~0u, ~0u, ~0u});
}

// One thread per 8 columns: bf16(1 + scale), the product and the sum, each rounded, as the eager chain.
struct ModulateArgs {
  const uint16_t* x;
  const uint16_t *shift, *scale;
  uint16_t* out;
  int64_t x_row, x_batch, mod_batch;
  int rows, total, d;  // total: 8-column pieces
};

__global__ __launch_bounds__(256) void modulate_pack_kernel(ModulateArgs a) {
#pragma clang fp contract(off)
  const int p = static_cast<int>(blockIdx.x) * 256 + static_cast<int>(threadIdx.x);
  if (p >= a.total) return;
  const int per = a.d / 8, t = p / per, col = (p - t * per) * 8;  // t: row of the packed output
  const int b = t / a.rows, r = t - b * a.rows;
  const u32x4 x = *reinterpret_cast<const u32x4*>(a.x + b * a.x_batch + r * a.x_row + col);
  const u32x4 sh = *reinterpret_cast<const u32x4*>(a.shift + b * a.mod_batch + col);
  const u32x4 sc = *reinterpret_cast<const u32x4*>(a.scale + b * a.mod_batch + col);
  u32x4 o;
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    const uint32_t s1 = pack_bf16x2(1.0f + bf16x2_lo(sc[i]), 1.0f + bf16x2_hi(sc[i]));
    const uint32_t m = pack_bf16x2(bf16x2_lo(x[i]) * bf16x2_lo(s1), bf16x2_hi(x[i]) * bf16x2_hi(s1));
    o[i] = pack_bf16x2(bf16x2_lo(m) + bf16x2_lo(sh[i]), bf16x2_hi(m) + bf16x2_hi(sh[i]));
  }
  *reinterpret_cast<u32x4*>(a.out + packed_act_offset(t, col, a.d)) = o;
}

}  // namespace
}  // namespace rldx

using namespace rldx;

extern "C" hipError_t rldx_copy_rows_many(const rldx_copy_rows_t* copies, int32_t count, int64_t batch,
                                          hipStream_t stream) {
  if (!copies || count < 1 || count > kMaxCopies || batch < 0 || batch > 65535) return hipErrorInvalidValue;
  CopyArgs a{};
  int n = 0;
  int64_t blocks = 0;
  for (int i = 0; i < count; ++i) {
    const rldx_copy_rows_t& c = copies[i];
    if (c.rows < 0 || c.row_bytes < 0 || c.row_bytes % 16) return hipErrorInvalidValue;
    if (c.rows == 0 || c.row_bytes == 0) continue;
    if (!c.src || !c.dst || !a16(c.src) || !a16(c.dst) || c.src_row_stride % 16 || c.src_batch_stride % 16 ||
        c.dst_row_stride % 16 || c.dst_batch_stride % 16)
      return hipErrorInvalidValue;
    const int64_t units = c.row_bytes / 16;
    if (c.rows > (1 << 24) || units > (1 << 24) || c.rows * units > (1 << 30)) return hipErrorInvalidValue;
    a.src[n] = static_cast<const char*>(c.src);
    a.dst[n] = static_cast<char*>(c.dst);
    a.src_row[n] = c.src_row_stride;
    a.src_batch[n] = c.src_batch_stride;
    a.dst_row[n] = c.dst_row_stride;
    a.dst_batch[n] = c.dst_batch_stride;
    a.units[n] = static_cast<int>(units);
    a.total[n] = static_cast<int>(c.rows * units);
    a.begin[n] = static_cast<int>(blocks);
    blocks += (c.rows * units + kPiece - 1) / kPiece;
    ++n;
  }
  if (n == 0 || batch == 0) return hipSuccess;
  a.count = n;
  hipLaunchKernelGGL(copy_rows_kernel, dim3(static_cast<unsigned>(blocks), static_cast<unsigned>(batch)), dim3(256), 0,
                     stream, a);
  return hipGetLastError();
}

extern "C" hipError_t rldx_gather_slabs(const void* const* src, void* const* dst, const int64_t* slab_bytes,
                                        int32_t count, const int64_t* idx, int64_t batch, int64_t num_slabs,
                                        hipStream_t stream) {
  if (!src || !dst || !slab_bytes || count < 1 || count > kMaxSlabs || batch < 0 || batch > 65535 || num_slabs < 0)
    return hipErrorInvalidValue;
  SlabArgs a{};
  int n = 0;
  int64_t blocks = 0;
  for (int i = 0; i < count; ++i) {
    if (slab_bytes[i] < 0 || slab_bytes[i] % 2) return hipErrorInvalidValue;
    if (slab_bytes[i] == 0) continue;
    if (!src[i] || !dst[i] || reinterpret_cast<uintptr_t>(src[i]) % 2 || reinterpret_cast<uintptr_t>(dst[i]) % 2)
      return hipErrorInvalidValue;
    const bool wide = slab_bytes[i] % 16 == 0 && a16(src[i]) && a16(dst[i]);
    a.src[n] = static_cast<const char*>(src[i]);
    a.dst[n] = static_cast<char*>(dst[i]);
    a.units[n] = slab_bytes[i] / (wide ? 16 : 2);
    if (!wide) a.narrow |= 1u << n;
    a.begin[n] = static_cast<int>(blocks);
    blocks += (a.units[n] + kPiece - 1) / kPiece;
    if (blocks > (1 << 30)) return hipErrorInvalidValue;
    ++n;
  }
  if (n == 0 || batch == 0) return hipSuccess;
  if (!idx || reinterpret_cast<uintptr_t>(idx) % 8) return hipErrorInvalidValue;
  a.idx = idx;
  a.num = num_slabs;
  a.count = n;
  hipLaunchKernelGGL(gather_slabs_kernel, dim3(static_cast<unsigned>(blocks), static_cast<unsigned>(batch)), dim3(256),
                     0, stream, a);
  return hipGetLastError();
}

extern "C" hipError_t rldx_modulate_pack_bf16(const void* x, int64_t x_row_stride, int64_t x_batch_stride, int64_t rows,
                                              int64_t batch, const void* shift, const void* scale,
                                              int64_t mod_batch_stride, int64_t d, void* packed, hipStream_t stream) {
  if (rows < 0 || batch < 0 || d < 0) return hipErrorInvalidValue;
  if (rows == 0 || batch == 0 || d == 0) return hipSuccess;
  if (!x || !shift || !scale || !packed || !a16(x) || !a16(shift) || !a16(scale) || !a16(packed) || x_row_stride % 8 ||
      x_batch_stride % 8 || mod_batch_stride % 8 || d % 16 || d > (1 << 24) || rows > (1 << 24) || batch > (1 << 24) ||
      rows * batch > (1 << 28) || rows * batch * (d / 8) > (1 << 30))
    return hipErrorInvalidValue;
  const ModulateArgs a{static_cast<const uint16_t*>(x),
                       static_cast<const uint16_t*>(shift),
                       static_cast<const uint16_t*>(scale),
                       static_cast<uint16_t*>(packed),
                       x_row_stride,
                       x_batch_stride,
                       mod_batch_stride,
                       static_cast<int>(rows),
                       static_cast<int>(rows * batch * (d / 8)),
                       static_cast<int>(d)};
  hipLaunchKernelGGL(modulate_pack_kernel, dim3(static_cast<unsigned>((a.total + 255) / 256)), dim3(256), 0, stream, a);
  return hipGetLastError();
}
