// Python module `sparse_attn_cuda`: a thin pybind11 shim over the C ABI of libsma_hip.so.
//
// It keeps the module name and the two Python-visible signatures of the reference binding
// (csrc/binding.cpp:9-18 `forward`, csrc/binding.cpp:49 `pack_mask`, registered at
// csrc/binding.cpp:68-71) so that python/sparse_attention.py can stay as it is:
//
//   forward(q, k, v, mask_packed, out, lse, scale, is_training, tile_map=None) -> None
//   pack_mask(mask) -> int32 Tensor [B, H, N, ceil(N/32)]
//   tile_map(mask_packed) -> int32 Tensor [B, H, ceil(N/64), 2, ceil(ceil(N/64)/32)]   (not in the
//       reference: which 64 x 64 blocks of the mask hold a set bit / nothing but set bits; passed to
//       `forward` as tile_map, key tiles without a set bit are neither loaded nor computed)
//   backward(dout, q, k, v, out, lse, mask_packed, dq, dk, dv, scale, tile_map=None) -> None   (called by the
//       reference's Python API, python/sparse_attention.py:91-94, but absent from its binding)
//   forward_bool_mask(q, k, v, mask, out, lse, scale, is_training, packed_out=None, map_out=None) -> None   (not in
//       the reference: `forward` with the boolean mask itself in place of the packed one, one launch
//       instead of pack_mask + forward; `packed_out`, if given, receives what pack_mask would
//       return and `map_out` what tile_map would return for it; `bool_mask_supported(q, k, v, mask)`
//       says whether it applies)
//   attention(q, k, v, mask, mask_packed, tile_map, autograd) -> Tensor or None   (not in the reference:
//       everything python/sparse_attention.py does for one call - conversions, padding, allocation,
//       launches and the autograd node - without returning to Python in between; None when an
//       argument is not what the Python layer's own checks demand, which then say what is wrong)
//   attention_function(q, k, v, mask_packed, mask, scale, tile_map) -> Tensor   (SparseAttentionFunction.apply: the same
//       with the scale given; wrong arguments raise)
//   addressable(t) -> bool   (whether the kernels take a tensor as it is)
//
// Differences, all on the safe side: `lse` may be None (the reference's own inference wrapper
// passes None, python/sparse_attention.py:170-171); every tensor argument is checked (device,
// dtype, shape, layout, head_dim 32, 64 or 128, or any up to 128 in `attention` and
// `attention_function`) instead of only `q`; launches go to the current HIP stream of q's device
// under a device guard; a failed launch raises RuntimeError.
// q, k, v, out and the gradients need not be contiguous: any view whose last dimension is
// contiguous and whose other strides are multiples of 8 elements is passed on with its strides
// (the reference reserves such strides, csrc/sparse_attention.h:30-33, and ignores them), and
// mask_packed may be [1|B, 1|H, N, ceil(N/32)]: a size of 1 shares the mask between batch
// entries / heads.
// This file is host-only C++ (compiled by g++); all GPU code lives behind include/sma.h.
#include <torch/extension.h>
#include <ATen/EmptyTensor.h>
#include <ATen/hip/impl/HIPCachingAllocatorMasqueradingAsCUDA.h>
#include <c10/core/DeviceGuard.h>
#include <c10/hip/HIPStream.h>
#include <torch/csrc/autograd/functions/utils.h>
#include <torch/csrc/autograd/python_cpp_function.h>
#include <torch/csrc/autograd/saved_variable.h>
#include <torch/csrc/jit/frontend/tracer.h>

#include <cmath>
#include <mutex>

#include "sma.h"

namespace {

void check_status(int st, const char *what)
{
    TORCH_CHECK(st == SMA_OK, what, " failed: ", sma_strerror(st), " (code ", st, ")");
}

// Uninitialised tensors straight from PyTorch's caching allocator of the current device (the callers
// hold the device guard), without the dispatcher in between.
torch::Tensor empty_rows(c10::IntArrayRef sizes, c10::IntArrayRef strides, at::ScalarType dtype)
{
    static c10::Allocator *const allocator = c10::hip::HIPCachingAllocatorMasqueradingAsCUDA::get();
    return torch::Tensor(at::detail::empty_strided_generic(sizes, strides, allocator, c10::DispatchKeySet(c10::DispatchKey::CUDA), dtype));
}

torch::Tensor empty_dense(c10::IntArrayRef sizes, at::ScalarType dtype)
{
    static c10::Allocator *const allocator = c10::hip::HIPCachingAllocatorMasqueradingAsCUDA::get();
    return torch::Tensor(at::detail::empty_generic(sizes, allocator, c10::DispatchKeySet(c10::DispatchKey::CUDA), dtype, c10::nullopt));
}

// Descriptor of a [B,H,N,D] tensor for the strided C entry points.  Extents of size 1 get stride 0
// (PyTorch leaves their strides arbitrary).
sma_tensor rows_of(const torch::Tensor &t, const char *name)
{
    if (t.numel() == 0) return sma_tensor{t.data_ptr(), 0, 0, 0};     // nothing will be read or written
    TORCH_CHECK(t.stride(3) == 1 || t.size(3) == 1, name, ": the last dimension must be contiguous");
    sma_tensor d;
    d.data = t.data_ptr();
    d.stride_b = t.size(0) == 1 ? 0 : t.stride(0);
    d.stride_h = t.size(1) == 1 ? 0 : t.stride(1);
    d.stride_n = t.size(2) == 1 ? 0 : t.stride(2);
    TORCH_CHECK(((d.stride_b | d.stride_h | d.stride_n) & 7) == 0 && d.stride_b >= 0 && d.stride_h >= 0 &&
                    d.stride_n >= 0,
                name, ": strides must be non-negative multiples of 8 elements (call .contiguous())");
    return d;
}

// Checks mask_packed ([1|B, 1|H, N, nw] int32, contiguous) and returns its word strides (0 = shared).
void mask_strides(const torch::Tensor &mp, const torch::Tensor &q, int64_t *sb, int64_t *sh)
{
    const int64_t B = q.size(0), H = q.size(1), N = q.size(2), nw = (N + 31) / 32;
    TORCH_CHECK(mp.device() == q.device(), "mask_packed must be on q's device");
    TORCH_CHECK(mp.scalar_type() == at::kInt, "mask_packed must be int32");
    TORCH_CHECK(mp.dim() == 4 && (mp.size(0) == B || mp.size(0) == 1) && (mp.size(1) == H || mp.size(1) == 1) &&
                    mp.size(2) == N && mp.size(3) == nw,
                "mask_packed must be [B or 1, H or 1, N, ceil(N/32)]");
    TORCH_CHECK(mp.is_contiguous(), "mask_packed must be contiguous");
    *sb = mp.size(0) == 1 ? 0 : mp.size(1) * N * nw;
    *sh = mp.size(1) == 1 ? 0 : N * nw;
}

// The optional tile map of mask_packed ([Bm, Hm, T, 2, ceil(T/32)] int32, T = ceil(N/64)), checked; nullptr if absent.
const uint32_t *map_pointer(const c10::optional<torch::Tensor> &tile_map, const torch::Tensor &mask_packed,
                            const torch::Tensor &q)
{
    if (!tile_map.has_value() || !tile_map->defined()) return nullptr;
    const torch::Tensor &m = *tile_map;
    const int64_t T = (q.size(2) + 63) / 64;
    TORCH_CHECK(m.device() == q.device() && m.scalar_type() == at::kInt && m.dim() == 5 &&
                    m.size(0) == mask_packed.size(0) && m.size(1) == mask_packed.size(1) && m.size(2) == T &&
                    m.size(3) == 2 && m.size(4) == (T + 31) / 32 && m.is_contiguous(),
                "tile_map must be the contiguous int32 result of tile_map(mask_packed)");
    return reinterpret_cast<const uint32_t *>(m.data_ptr<int32_t>());
}

void forward(const torch::Tensor &q, const torch::Tensor &k, const torch::Tensor &v,
             const torch::Tensor &mask_packed, torch::Tensor out,
             const c10::optional<torch::Tensor> &lse, double scale, bool is_training,
             const c10::optional<torch::Tensor> &tile_map)
{
    TORCH_CHECK(q.is_cuda(), "q must be a GPU tensor");
    TORCH_CHECK(q.dim() == 4, "q must be 4D [B, H, N, D]");
    const auto dt = q.scalar_type();
    TORCH_CHECK(dt == at::kHalf || dt == at::kBFloat16, "Unsupported dtype, need BF16 or FP16");
    const int64_t B = q.size(0), H = q.size(1), N = q.size(2), D = q.size(3);
    TORCH_CHECK(D == 32 || D == 64 || D == 128, "head_dim must be 32, 64 or 128, got ", D);
    for (const torch::Tensor *t : {&k, &v, static_cast<const torch::Tensor *>(&out)}) {
        TORCH_CHECK(t->device() == q.device(), "q, k, v, out must be on the same device");
        TORCH_CHECK(t->scalar_type() == dt, "q, k, v, out must have the same dtype");
        TORCH_CHECK(t->sizes() == q.sizes(), "q, k, v, out must have the same shape");
    }
    const sma_tensor tq = rows_of(q, "q"), tk = rows_of(k, "k"), tv = rows_of(v, "v"), to = rows_of(out, "out");
    int64_t msb = 0, msh = 0;
    mask_strides(mask_packed, q, &msb, &msh);
    float *lse_ptr = nullptr;
    if (is_training) {
        TORCH_CHECK(lse.has_value() && lse->defined(), "is_training=True needs an lse tensor");
        TORCH_CHECK(lse->device() == q.device() && lse->scalar_type() == at::kFloat &&
                        lse->dim() == 3 && lse->size(0) == B && lse->size(1) == H &&
                        lse->size(2) == N && lse->is_contiguous(),
                    "lse must be a contiguous float32 [B, H, N] tensor on q's device");
        lse_ptr = lse->data_ptr<float>();
    }
    TORCH_CHECK(B <= INT32_MAX && H <= INT32_MAX && N <= INT32_MAX, "extent too large");
    const uint32_t *map_ptr = map_pointer(tile_map, mask_packed, q);

    const c10::DeviceGuard guard(q.device());
    hipStream_t stream = c10::hip::getCurrentHIPStream(q.device().index()).stream();
    const int st = sma_attn_fwd_map_strided(&tq, &tk, &tv,
                                            reinterpret_cast<const uint32_t *>(mask_packed.data_ptr<int32_t>()),
                                            msb, msh, map_ptr, &to, lse_ptr, (int)B, (int)H, (int)N, (int)D,
                                            (float)scale, dt == at::kBFloat16 ? SMA_DTYPE_BF16 : SMA_DTYPE_F16,
                                            stream);
    check_status(st, "sma_attn_fwd_map_strided");
}

// Whether the kernels can address t as it is: contiguous last dimension, the strides of the others
// non-negative multiples of 8 elements, 16-byte aligned storage.
bool addressable(const torch::Tensor &t)
{
    if (t.dim() != 4) return false;
    if (t.stride(3) != 1 && t.size(3) != 1) return false;
    if (reinterpret_cast<uintptr_t>(t.data_ptr()) % 16 != 0) return false;
    for (int d = 0; d < 3; ++d)
        if (t.size(d) > 1 && (t.stride(d) < 0 || t.stride(d) % 8 != 0)) return false;
    return true;
}

// Limits of sma_attn_fwd_bool_mask, so that callers can choose between it and pack_mask + forward
// without provoking an error: q, k, v with contiguous rows and strides that are multiples of 8
// elements, head dim 32, 64 or 128, 16 <= N < 46341, a contiguous bool mask [1|B, 1|H, N, N].
bool bool_mask_supported(const torch::Tensor &q, const torch::Tensor &k, const torch::Tensor &v,
                         const torch::Tensor &mask)
{
    if (!q.is_cuda() || q.dim() != 4 || mask.dim() != 4) return false;
    const int64_t B = q.size(0), H = q.size(1), N = q.size(2), D = q.size(3);
    if (!(D == 32 || D == 64 || D == 128) || N < 16 || N * N >= (int64_t(1) << 31)) return false;
    for (const torch::Tensor *t : {&q, &k, &v})
        if (t->sizes() != q.sizes() || !addressable(*t)) return false;
    if (mask.scalar_type() != at::kBool || !mask.is_contiguous() || mask.device() != q.device()) return false;
    if (!((mask.size(0) == B || mask.size(0) == 1) && (mask.size(1) == H || mask.size(1) == 1) &&
          mask.size(2) == N && mask.size(3) == N))
        return false;
    // the kernel copies mask rows from whatever byte address they start at: the library checks once
    // per device that such copies are served (always, under ROCm); where not, pack_mask + forward
    const c10::DeviceGuard guard(q.device());
    return sma_device_check(c10::hip::getCurrentHIPStream(q.device().index()).stream()) == SMA_OK;
}

void forward_bool_mask(const torch::Tensor &q, const torch::Tensor &k, const torch::Tensor &v,
                       const torch::Tensor &mask, torch::Tensor out,
                       const c10::optional<torch::Tensor> &lse, double scale, bool is_training,
                       const c10::optional<torch::Tensor> &packed_out,
                       const c10::optional<torch::Tensor> &map_out)
{
    TORCH_CHECK(q.is_cuda(), "q must be a GPU tensor");
    TORCH_CHECK(q.dim() == 4, "q must be 4D [B, H, N, D]");
    const auto dt = q.scalar_type();
    TORCH_CHECK(dt == at::kHalf || dt == at::kBFloat16, "Unsupported dtype, need BF16 or FP16");
    TORCH_CHECK(bool_mask_supported(q, k, v, mask),
                "forward_bool_mask needs q, k, v with contiguous rows (strides multiples of 8 elements), head_dim "
                "32, 64 or 128, N >= 16 and a contiguous bool mask [B or 1, H or 1, N, N]; use pack_mask + forward otherwise");
    const int64_t B = q.size(0), H = q.size(1), N = q.size(2), D = q.size(3);
    for (const torch::Tensor *t : {&k, &v, static_cast<const torch::Tensor *>(&out)}) {
        TORCH_CHECK(t->device() == q.device(), "q, k, v, out must be on the same device");
        TORCH_CHECK(t->scalar_type() == dt, "q, k, v, out must have the same dtype");
        TORCH_CHECK(t->sizes() == q.sizes(), "q, k, v, out must have the same shape");
    }
    const sma_tensor tq = rows_of(q, "q"), tk = rows_of(k, "k"), tv = rows_of(v, "v"), to = rows_of(out, "out");
    float *lse_ptr = nullptr;
    if (is_training) {
        TORCH_CHECK(lse.has_value() && lse->defined(), "is_training=True needs an lse tensor");
        TORCH_CHECK(lse->device() == q.device() && lse->scalar_type() == at::kFloat &&
                        lse->dim() == 3 && lse->size(0) == B && lse->size(1) == H &&
                        lse->size(2) == N && lse->is_contiguous(),
                    "lse must be a contiguous float32 [B, H, N] tensor on q's device");
        lse_ptr = lse->data_ptr<float>();
    }
    uint32_t *packed_ptr = nullptr;
    if (packed_out.has_value() && packed_out->defined()) {
        const torch::Tensor &p = *packed_out;
        TORCH_CHECK(p.device() == q.device() && p.scalar_type() == at::kInt && p.dim() == 4 &&
                        p.size(0) == mask.size(0) && p.size(1) == mask.size(1) && p.size(2) == N &&
                        p.size(3) == (N + 31) / 32 && p.is_contiguous(),
                    "packed_out must be a contiguous int32 [mask.size(0), mask.size(1), N, ceil(N/32)] tensor on q's device");
        packed_ptr = reinterpret_cast<uint32_t *>(p.data_ptr<int32_t>());
    }
    uint32_t *map_ptr = nullptr;
    if (map_out.has_value() && map_out->defined()) {
        const torch::Tensor &m = *map_out;
        const int64_t T = (N + 63) / 64;
        TORCH_CHECK(m.device() == q.device() && m.scalar_type() == at::kInt && m.dim() == 5 &&
                        m.size(0) == mask.size(0) && m.size(1) == mask.size(1) && m.size(2) == T &&
                        m.size(3) == 2 && m.size(4) == (T + 31) / 32 && m.is_contiguous(),
                    "map_out must be a contiguous int32 [mask.size(0), mask.size(1), T, 2, ceil(T/32)] tensor "
                    "on q's device, T = ceil(N/64)");
        map_ptr = reinterpret_cast<uint32_t *>(m.data_ptr<int32_t>());
    }
    const int64_t msb = mask.size(0) == 1 ? 0 : mask.size(1) * N * N;
    const int64_t msh = mask.size(1) == 1 ? 0 : N * N;
    const c10::DeviceGuard guard(q.device());
    hipStream_t stream = c10::hip::getCurrentHIPStream(q.device().index()).stream();
    const int st = sma_attn_fwd_bool_mask_strided(&tq, &tk, &tv,
                                                  reinterpret_cast<const uint8_t *>(mask.data_ptr<bool>()), msb, msh,
                                                  &to, lse_ptr, packed_ptr, map_ptr, (int)B, (int)H, (int)N,
                                                  (int)D, (float)scale,
                                                  dt == at::kBFloat16 ? SMA_DTYPE_BF16 : SMA_DTYPE_F16, stream);
    check_status(st, "sma_attn_fwd_bool_mask_strided");
}

// backward(dout, q, k, v, out, lse, mask_packed, dq, dk, dv, scale) -> None, the call the
// reference's autograd function makes (python/sparse_attention.py:91-94) to a function its
// binding never had.  dq, dk, dv are overwritten (not accumulated into).
void backward(const torch::Tensor &dout, const torch::Tensor &q, const torch::Tensor &k,
              const torch::Tensor &v, const torch::Tensor &out, const torch::Tensor &lse,
              const torch::Tensor &mask_packed, torch::Tensor dq, torch::Tensor dk,
              torch::Tensor dv, double scale, const c10::optional<torch::Tensor> &tile_map)
{
    TORCH_CHECK(q.is_cuda(), "q must be a GPU tensor");
    TORCH_CHECK(q.dim() == 4, "q must be 4D [B, H, N, D]");
    const auto dt = q.scalar_type();
    TORCH_CHECK(dt == at::kHalf || dt == at::kBFloat16, "Unsupported dtype, need BF16 or FP16");
    const int64_t B = q.size(0), H = q.size(1), N = q.size(2), D = q.size(3);
    TORCH_CHECK(D == 32 || D == 64 || D == 128, "head_dim must be 32, 64 or 128, got ", D);
    const torch::Tensor *all[8] = {&dout, &q, &k, &v, &out, &dq, &dk, &dv};
    const char *names[8] = {"dout", "q", "k", "v", "out", "dq", "dk", "dv"};
    sma_tensor d[8];
    for (int i = 0; i < 8; ++i) {
        const torch::Tensor *t = all[i];
        TORCH_CHECK(t->device() == q.device(), "dout, q, k, v, out, dq, dk, dv must be on the same device");
        TORCH_CHECK(t->scalar_type() == dt, "dout, q, k, v, out, dq, dk, dv must have the same dtype");
        TORCH_CHECK(t->sizes() == q.sizes(), "dout, q, k, v, out, dq, dk, dv must have the same shape");
        d[i] = rows_of(*t, names[i]);
    }
    int64_t msb = 0, msh = 0;
    mask_strides(mask_packed, q, &msb, &msh);
    TORCH_CHECK(lse.device() == q.device() && lse.scalar_type() == at::kFloat && lse.dim() == 3 &&
                    lse.size(0) == B && lse.size(1) == H && lse.size(2) == N && lse.is_contiguous(),
                "lse must be a contiguous float32 [B, H, N] tensor on q's device");
    TORCH_CHECK(B <= INT32_MAX && H <= INT32_MAX && N <= INT32_MAX, "extent too large");

    const uint32_t *map_ptr = map_pointer(tile_map, mask_packed, q);

    const c10::DeviceGuard guard(q.device());
    torch::Tensor delta = empty_dense({B, H, N}, at::kFloat);      // workspace of the C entry point
    hipStream_t stream = c10::hip::getCurrentHIPStream(q.device().index()).stream();
    const int st = sma_attn_bwd_map_strided(&d[0], &d[1], &d[2], &d[3], &d[4], lse.data_ptr<float>(),
                                            reinterpret_cast<const uint32_t *>(mask_packed.data_ptr<int32_t>()),
                                            msb, msh, map_ptr, &d[5], &d[6], &d[7], delta.data_ptr<float>(), (int)B,
                                            (int)H, (int)N, (int)D, (float)scale,
                                            dt == at::kBFloat16 ? SMA_DTYPE_BF16 : SMA_DTYPE_F16, stream);
    check_status(st, "sma_attn_bwd_map_strided");
}

torch::Tensor pack_mask(const torch::Tensor &mask)
{
    TORCH_CHECK(mask.is_cuda(), "mask must be a GPU tensor");
    TORCH_CHECK(mask.dim() == 4, "mask must be 4D [B, H, N, N]");
    TORCH_CHECK(mask.scalar_type() == at::kBool, "mask must be bool");
    TORCH_CHECK(mask.size(2) == mask.size(3), "mask must be [B, H, N, N]");
    // a mask shared between batch entries / heads is given as [1 or B, 1 or H, N, N] and packed as it is
    const torch::Tensor m = mask.contiguous();
    const int64_t B = m.size(0), H = m.size(1), N = m.size(2);
    TORCH_CHECK(B <= INT32_MAX && H <= INT32_MAX && N <= INT32_MAX, "extent too large");
    const c10::DeviceGuard guard(m.device());
    // Every word is written by the kernel, so no zero-fill is needed.
    torch::Tensor packed = empty_dense({B, H, N, (N + 31) / 32}, at::kInt);
    hipStream_t stream = c10::hip::getCurrentHIPStream(m.device().index()).stream();
    const int st = sma_pack_mask(reinterpret_cast<const uint8_t *>(m.data_ptr<bool>()),
                                 reinterpret_cast<uint32_t *>(packed.data_ptr<int32_t>()), (int)B,
                                 (int)H, (int)N, stream);
    check_status(st, "sma_pack_mask");
    return packed;
}

// Longest sequence that a tile map is made for (sma_tile_map, sma_pack_mask_map).
constexpr int64_t MAP_MAX_N = 131072;

// tile_map(mask_packed): [Bm, Hm, N, ceil(N/32)] int32 -> [Bm, Hm, T, 2, ceil(T/32)] int32, T = ceil(N/64).
torch::Tensor tile_map(const torch::Tensor &mask_packed)
{
    TORCH_CHECK(mask_packed.is_cuda(), "mask_packed must be a GPU tensor");
    TORCH_CHECK(mask_packed.scalar_type() == at::kInt && mask_packed.dim() == 4 && mask_packed.is_contiguous(),
                "mask_packed must be a contiguous int32 [B, H, N, ceil(N/32)] tensor");
    const int64_t B = mask_packed.size(0), H = mask_packed.size(1), N = mask_packed.size(2);
    TORCH_CHECK(mask_packed.size(3) == (N + 31) / 32, "mask_packed must be [B, H, N, ceil(N/32)]");
    TORCH_CHECK(B <= INT32_MAX && H <= INT32_MAX && N <= MAP_MAX_N, "extent too large");
    const int64_t T = (N + 63) / 64;
    const c10::DeviceGuard guard(mask_packed.device());
    torch::Tensor map = empty_dense({B, H, T, 2, (T + 31) / 32}, at::kInt);    // every word is written
    hipStream_t stream = c10::hip::getCurrentHIPStream(mask_packed.device().index()).stream();
    const int st = sma_tile_map(reinterpret_cast<const uint32_t *>(mask_packed.data_ptr<int32_t>()),
                                reinterpret_cast<uint32_t *>(map.data_ptr<int32_t>()), (int)B, (int)H, (int)N, stream);
    check_status(st, "sma_tile_map");
    return map;
}

// ---- one call of the Python layer, whole --------------------------------------------------------
//
// What bounds a small call is the host, not the GPU: the kernels of a 128-token request take 5 us,
// the same steps written in Python 11 us for the forward and 105 us for forward + backward (measured
// with 3 kernels of 10 us each in flight).  So the conversions, the allocations, the choice of the
// kernel and the autograd node live here; Python only calls `attention` and, when it declines,
// explains why.

using torch::Tensor;

// Head dim of the kernels' tensors for one of the caller's: the next multiple of 8 (16 bytes).
int64_t padded_head_dim(int64_t D) { return (D + 7) / 8 * 8; }

// q, k, v or a gradient as the kernels take them: 16-bit elements of type `dtype`, head dim Dk (zeros after the
// tensor's own), addressable.  fp32 tensors that leave no gaps, all of one size, are converted in one launch that
// keeps their layout; the caller holds the device guard.
template <size_t COUNT>
bool flat_f32(const Tensor *const (&from)[COUNT], int64_t Dk)
{
    bool flat = COUNT <= 3;
    for (const Tensor *t : from)
        flat = flat && t->scalar_type() == at::kFloat && t->size(3) == Dk && t->is_non_overlapping_and_dense() && t->stride(3) == 1 &&
               t->numel() == from[0]->numel() && reinterpret_cast<uintptr_t>(t->data_ptr()) % 16 == 0;
    return flat;
}
Tensor empty_flat(const Tensor &t, at::ScalarType dtype)
{
    return t.is_contiguous() ? empty_dense(t.sizes(), dtype) : empty_rows(t.sizes(), t.strides(), dtype);
}
template <size_t COUNT> void flat_rows(const Tensor *const (&from)[COUNT], Tensor *const (&to)[COUNT])
{
    const float *src[COUNT];
    uint16_t *dst[COUNT];
    for (size_t i = 0; i < COUNT; ++i) {
        *to[i] = empty_flat(*from[i], at::kBFloat16);
        src[i] = static_cast<const float *>(from[i]->data_ptr());
        dst[i] = static_cast<uint16_t *>(to[i]->data_ptr());
    }
    hipStream_t stream = c10::hip::getCurrentHIPStream(from[0]->device().index()).stream();
    check_status(sma_to_bf16(src, dst, (int)COUNT, from[0]->numel(), stream), "sma_to_bf16");
}
template <size_t COUNT>
void kernel_rows(const Tensor *const (&from)[COUNT], Tensor *const (&to)[COUNT], at::ScalarType dtype, int64_t Dk)
{
    if (dtype == at::kBFloat16 && flat_f32(from, Dk)) return flat_rows(from, to);
    for (size_t i = 0; i < COUNT; ++i) {
        Tensor r = from[i]->scalar_type() == dtype ? *from[i] : from[i]->to(dtype);
        if (r.size(3) != Dk) r = at::constant_pad_nd(r, {0, Dk - r.size(3)});
        *to[i] = addressable(r) ? r : r.contiguous();
    }
}

// An uninitialised tensor laid out like t, of another element type.
Tensor empty_like_rows(const Tensor &t, at::ScalarType dtype)
{
    if (t.is_contiguous()) return empty_dense(t.sizes(), dtype);
    if (t.is_non_overlapping_and_dense()) return empty_rows(t.sizes(), t.strides(), dtype);
    return at::empty_like(t.detach(), t.options().dtype(dtype));
}

// Whether the kernels reach every row of an fp32 tensor laid out like t (a kernel tensor, 16 bits): a lane's byte
// offset inside one (b, h) slab has 31 bits, half the rows of a 16-bit one.
bool reaches_f32(const Tensor &t)
{
    return t.numel() == 0 || (t.size(2) - 1) * t.stride(2) * 4 + t.size(3) * 4 < (int64_t(1) << 31);
}

// The mask with its expanded (stride 0) batch / head extents taken back to 1: it is then read once
// and shared.
Tensor unexpand(Tensor m)
{
    if (m.size(0) > 1 && m.stride(0) == 0) m = m.narrow(0, 0, 1);
    if (m.size(1) > 1 && m.stride(1) == 0) m = m.narrow(1, 0, 1);
    return m.is_contiguous() ? m : m.contiguous();
}

struct Call {                       // one problem as the kernels see it
    Tensor q, k, v;                 // kernel_rows of the caller's
    Tensor q32;                     // undefined, or the fp32 q that the kernel itself rounds (into q, if there is a backward; else q is q32)
    Tensor mask;                    // the boolean mask, unexpanded; undefined if only the packed one is there
    Tensor packed, map;             // packed mask and tile map, either may be undefined
    int64_t B, H, N, D;             // the caller's extents
    double scale;
};

// Whether a mask that several heads share is packed, with its tile map, before the attention instead of
// being read as bytes by every head.  The extra launch costs 4 us whatever the size; the attention
// then reads an eighth of the mask's bytes, visits no key tile in which the mask keeps nothing and needs
// no room for bytes in LDS.  Measured (4 x 32 heads, one mask for the heads of a batch entry or for all):
// N = 1000, random: 49.3 us either way; N = 2048, causal: 128 -> 111 us forward, 514 -> 458 us
// forward + backward; 8 x 16 heads, N = 512: 15 -> 19 us.  The line lies at 2^27 scores.
// A sequence too long for a map is packed without one, further down, like any whose bytes the kernel cannot address.
bool pack_first(const Call &c)
{
    const int64_t heads = c.B * c.H, masks = c.mask.size(0) * c.mask.size(1);
    return c.N <= MAP_MAX_N && heads >= 4 * masks && (double)heads * c.N * c.N >= (double)(1 << 27);
}

// Packed words and tile map of the boolean mask, in one launch.
void pack_with_map(Call &c)
{
    const int64_t Bm = c.mask.size(0), Hm = c.mask.size(1), T = (c.N + 63) / 64;
    c.packed = empty_dense({Bm, Hm, c.N, (c.N + 31) / 32}, at::kInt);
    c.map = empty_dense({Bm, Hm, T, 2, (T + 31) / 32}, at::kInt);
    hipStream_t stream = c10::hip::getCurrentHIPStream(c.mask.device().index()).stream();
    const int st = sma_pack_mask_map(reinterpret_cast<const uint8_t *>(c.mask.data_ptr<bool>()),
                                     reinterpret_cast<uint32_t *>(c.packed.data_ptr<int32_t>()),
                                     reinterpret_cast<uint32_t *>(c.map.data_ptr<int32_t>()), (int)Bm, (int)Hm,
                                     (int)c.N, stream);
    check_status(st, "sma_pack_mask_map");
}

// Whether the forward can read c's boolean mask as it is (c.mask is contiguous, q, k and v addressable).
bool reads_bytes(const Call &c)
{
    if (c.N < 16 || c.N * c.N >= (int64_t(1) << 31)) return false;
    // the kernel copies mask rows from whatever byte address they start at: the library checks once
    // per device that such copies are served (always, under ROCm); where not, the mask is packed
    return sma_device_check(c10::hip::getCurrentHIPStream(c.q.device().index()).stream()) == SMA_OK;
}

// Forward of `c` into `out` and / or its fp32 copy `out_f32`; with `lse` defined, the packed mask is left in
// c.packed and, if `want_map` or if one was made anyway, the tile map in c.map, for the backward.
void run_forward(Call &c, const Tensor &out, const Tensor &out_f32, const Tensor &lse, bool want_map)
{
    const bool training = lse.defined();
    const int64_t T = (c.N + 63) / 64;
    TORCH_CHECK(c.B <= INT32_MAX && c.H <= INT32_MAX && c.N <= INT32_MAX, "extent too large");
    sma_fwd_call f = {};
    if (!c.packed.defined() && c.q.numel() > 0) {
        if (pack_first(c) || (training && want_map && !reads_bytes(c))) {
            pack_with_map(c);
        } else if (reads_bytes(c)) {
            f.mask = reinterpret_cast<const uint8_t *>(c.mask.data_ptr<bool>());
            f.mask_stride_b = c.mask.size(0) == 1 ? 0 : c.mask.size(1) * c.N * c.N;
            f.mask_stride_h = c.mask.size(1) == 1 ? 0 : c.N * c.N;
            if (training) {
                c.packed = empty_dense({c.mask.size(0), c.mask.size(1), c.N, (c.N + 31) / 32}, at::kInt);
                f.packed_out = reinterpret_cast<uint32_t *>(c.packed.data_ptr<int32_t>());
            }
            if (training && want_map) {
                c.map = empty_dense({c.mask.size(0), c.mask.size(1), T, 2, (T + 31) / 32}, at::kInt);
                f.map_out = reinterpret_cast<uint32_t *>(c.map.data_ptr<int32_t>());
            }
        }
    }
    if (!f.mask) {
        if (!c.packed.defined()) c.packed = pack_mask(c.mask);
        mask_strides(c.packed, c.q, &f.mask_stride_b, &f.mask_stride_h);
        f.mask_packed = reinterpret_cast<const uint32_t *>(c.packed.data_ptr<int32_t>());
        f.tile_map = map_pointer(c.map.defined() ? c10::optional<Tensor>(c.map) : c10::nullopt, c.packed, c.q);
    }
    sma_tensor t[6] = {rows_of(c.q32.defined() ? c.q32 : c.q, "q"), rows_of(c.k, "k"), rows_of(c.v, "v")};
    f.q = &t[0], f.k = &t[1], f.v = &t[2];
    if (out.defined()) t[3] = rows_of(out, "out"), f.out = &t[3];
    if (out_f32.defined()) t[4] = rows_of(out_f32, "out"), f.out_f32 = &t[4];
    f.lse = training ? lse.data_ptr<float>() : nullptr;
    f.B = (int)c.B, f.H = (int)c.H, f.N = (int)c.N, f.D = (int)c.q.size(3);
    f.scale = (float)c.scale;
    f.dtype = c.q.scalar_type() == at::kHalf ? SMA_DTYPE_F16 : SMA_DTYPE_BF16;
    if (c.q32.defined()) {
        if (training) t[5] = rows_of(c.q, "q");
        check_status(sma_attn_fwd_call_q32(&f, training ? &t[5] : nullptr,
                                           c10::hip::getCurrentHIPStream(c.q.device().index()).stream()), "sma_attn_fwd_call_q32");
        return;
    }
    check_status(sma_attn_fwd_call(&f, c10::hip::getCurrentHIPStream(c.q.device().index()).stream()), "sma_attn_fwd_call");
}

// The autograd node of one training forward.
struct SparseAttentionBackward : public torch::autograd::Node {
    std::recursive_mutex mutex;     // (a saved-tensor hook that the backward calls may look at saved_tensors)
    torch::autograd::SavedVariable q, k, v, out, lse, packed;
    Tensor map;                     // undefined without a tile map
    bool map_shown = false;         // the caller gave the map or asked for it
    double scale = 1.0;
    at::ScalarType grad_dtype = at::kHalf;      // what the caller's q, k, v are made of ...
    int64_t grad_D = 0;                         // ... and their head dim
    bool out_is_output = false;     // `out` is the tensor handed to the caller (nothing was converted)

    std::string name() const override { return "SparseAttentionFunctionBackward"; }

    void release_variables() override
    {
        std::lock_guard<std::recursive_mutex> lock(mutex);
        for (torch::autograd::SavedVariable *s : {&q, &k, &v, &out, &lse, &packed}) s->reset_data();
        map.reset();
    }

    // Saved-tensor hooks give back what they like; the kernels address it by raw pointers.  (The packed mask and the map
    // are checked where their strides are taken.)
    void check_saved(const Tensor &grad, std::initializer_list<const Tensor *> rows, const Tensor &tlse) const
    {
        const at::ScalarType kdt = grad_dtype == at::kFloat ? at::kBFloat16 : grad_dtype;
        const int64_t B = grad.size(0), H = grad.size(1), N = grad.size(2);
        for (const Tensor *t : rows)
            TORCH_CHECK(t->device() == grad.device() && t->scalar_type() == kdt && t->dim() == 4 && t->size(0) == B && t->size(1) == H &&
                            t->size(2) == N && t->size(3) == padded_head_dim(grad_D),
                        "a saved tensor came back with another device, dtype or shape");
        TORCH_CHECK(tlse.device() == grad.device() && tlse.scalar_type() == at::kFloat && tlse.dim() == 3 && tlse.size(0) == B &&
                        tlse.size(1) == H && tlse.size(2) == N && tlse.is_contiguous(),
                    "the saved lse came back with another device, dtype, shape or layout");
    }

    torch::autograd::variable_list apply(torch::autograd::variable_list &&grads) override
    {
        if (!grads[0].defined()) return {Tensor(), Tensor(), Tensor()};
        std::lock_guard<std::recursive_mutex> lock(mutex);
        const Tensor tq = q.unpack(), tk = k.unpack(), tv = v.unpack();
        const Tensor tout = out.unpack(out_is_output ? shared_from_this() : nullptr);
        const Tensor tlse = lse.unpack(), tpacked = packed.unpack();
        at::NoGradGuard no_grad;
        check_saved(grads[0], {&tq, &tk, &tv, &tout}, tlse);
        const c10::DeviceGuard guard(tq.device());
        Tensor dout;
        kernel_rows<1>({&grads[0]}, {&dout}, tq.scalar_type(), tq.size(3));
        // the gradients in the caller's type and layout at once, unless its rows are no multiple of 16 bytes or too far apart
        const bool direct = grad_D == tq.size(3) &&
                            (grad_dtype == tq.scalar_type() || (reaches_f32(tq) && reaches_f32(tk) && reaches_f32(tv)));
        const at::ScalarType made = direct ? grad_dtype : tq.scalar_type();
        Tensor d[3] = {empty_like_rows(tq, made), empty_like_rows(tk, made), empty_like_rows(tv, made)};
        const int64_t B = tq.size(0), H = tq.size(1), N = tq.size(2);
        Tensor delta = empty_dense({B, H, N}, at::kFloat);             // workspace of the C entry point
        sma_tensor t[8] = {rows_of(dout, "dout"), rows_of(tq, "q"), rows_of(tk, "k"), rows_of(tv, "v"), rows_of(tout, "out"),
                           rows_of(d[0], "dq"), rows_of(d[1], "dk"), rows_of(d[2], "dv")};
        sma_bwd_call c = {};
        c.dout = &t[0], c.q = &t[1], c.k = &t[2], c.v = &t[3], c.out = &t[4], c.dq = &t[5], c.dk = &t[6], c.dv = &t[7];
        c.lse = tlse.data_ptr<float>();
        mask_strides(tpacked, tq, &c.mask_stride_b, &c.mask_stride_h);
        c.mask_packed = reinterpret_cast<const uint32_t *>(tpacked.data_ptr<int32_t>());
        c.tile_map = map_pointer(map.defined() ? c10::optional<Tensor>(map) : c10::nullopt, tpacked, tq);
        c.delta_ws = delta.data_ptr<float>();
        c.B = (int)B, c.H = (int)H, c.N = (int)N, c.D = (int)tq.size(3);
        c.scale = (float)scale;
        c.dtype = tq.scalar_type() == at::kBFloat16 ? SMA_DTYPE_BF16 : SMA_DTYPE_F16;
        c.grads_f32 = made == at::kFloat;
        check_status(sma_attn_bwd_call(&c, c10::hip::getCurrentHIPStream(tq.device().index()).stream()), "sma_attn_bwd_call");
        if (!direct)
            for (Tensor &g : d) {
                if (g.size(3) != grad_D) g = g.narrow(3, 0, grad_D);
                g = g.scalar_type() != grad_dtype ? g.to(grad_dtype) : g.contiguous();      // without the padding's gaps
            }
        return {d[0], d[1], d[2]};
    }
};

// Forward-mode AD has no formula here: a tangent is refused, not dropped.
void refuse_tangents(const Tensor &q, const Tensor &k, const Tensor &v)
{
    for (const Tensor *t : {&q, &k, &v})
        TORCH_CHECK_NOT_IMPLEMENTED(!t->_fw_grad(/*level=*/0).defined(), "sparse attention does not support forward mode AD");
}

// Whether the forward itself rounds q of fp32 callers: q is read once and can be rounded where it is read; k and v are read once per 128 query
// rows.  What it costs is a longer way to the first tile.  Conversion and forward, pass over all three -> this, in us (heads, N, D):
//   inference from 2^20 elements on -8 to +0.5 % (200 grids): 64, 256, 64 12.5 -> 11.7;  192, 512, 128 75.8 -> 69.8;  128, 1000, 32 51.0 -> 49.8.  0.8 to
//             1 million: -6 to +4 %, -1 to -3 on average;  around 0.72 million -1.4 % on average at head dim 64, +0.5 at 128.  Below: 64, 128, 64
//             9.2 -> 9.7;  128, 128, 32 9.3 -> 9.6;  64, 64, 128 9.4 -> 10.1
//   training  (from 2^20 elements on) it also writes the rounded rows.  Long sequences hide that: 160, 768, 128 113.5 -> 108.2;  200, 1024, 64 117 -> 112.  Short ones don't (512, 64, 128 24.6 -> 27.3;  192, 200, 128 33.5 -> 34.2), nor does head dim 32 (300, 512 42.3 -> 43.9), and where every head has a boolean mask of its own, whose bytes
//             bound it, nothing is gained (200, 600, 64 72.1 -> 77.1;  96, 1024, 64 69.0 -> 67.5)
//   with the kernels for 80, GPU time: inference 32, 512, 80 18.4 -> 17.0;  100, 256, 80 21.2 -> 19.1;  around the line 40, 256 12.4 -> 11.9;  below it 24, 256 10.4 -> 10.6;  12, 512
//             12.5 -> 12.7.  Whole training steps 96, 512, 80 88.5 -> 86.4;  300, 512 227 -> 222;  48, 2048 343 -> 339;  below 512 keys 200, 320 109 -> 111, packed 107 -> 104;  64, 448 59.7 -> 58.4
bool forward_rounds_q(const Call &c, const Tensor &q, bool training)
{
    if (!training) return q.numel() >= 11 * (int64_t(1) << 16);
    const bool own_bytes = !c.packed.defined() && c.mask.size(0) * c.mask.size(1) == c.B * c.H;
    return q.numel() >= (int64_t(1) << 20) && c.N >= 512 && c.D > 32 && !own_bytes;
}

// Output of one call: out, with its autograd node when q, k or v want gradients and `autograd`.
Tensor run_call(const Tensor &q, const Tensor &k, const Tensor &v, Call &c, bool want_map, bool autograd)
{
    const at::ScalarType dtype = q.scalar_type();
    const at::ScalarType kdt = dtype == at::kFloat ? at::kBFloat16 : dtype;
    const int64_t Dk = padded_head_dim(c.D);
    const bool map_shown = want_map || c.map.defined();
    const bool tracked = autograd && torch::autograd::compute_requires_grad(q, k, v);
    std::shared_ptr<SparseAttentionBackward> node;
    if (tracked) {
        refuse_tangents(q, k, v);
        // freed node by node like PyTorch's own, not by recursion along a chain of them
        node = std::shared_ptr<SparseAttentionBackward>(new SparseAttentionBackward(), torch::autograd::deleteNode);
        node->set_next_edges(torch::autograd::collect_next_edges(q, k, v));
    }
    const c10::DeviceGuard guard(q.device());
    at::AutoDispatchBelowADInplaceOrView below_autograd;
    if (dtype == at::kFloat && forward_rounds_q(c, q, tracked) && flat_f32<3>({&q, &k, &v}, Dk) && reaches_f32(q)) {
        flat_rows<2>({&k, &v}, {&c.k, &c.v});
        c.q32 = q;
        c.q = tracked ? empty_flat(q, kdt) : q;
    } else {
        kernel_rows<3>({&q, &k, &v}, {&c.q, &c.k, &c.v}, kdt, Dk);
    }
    // fp32 callers get their result from the kernel itself (unless its rows are too far apart); the 16-bit one is then made
    // for the backward only
    const bool wide = kdt != dtype && Dk == c.D && reaches_f32(c.q);
    Tensor out, result, lse;
    if (!wide || tracked) out = empty_like_rows(c.q, kdt);
    if (wide) result = empty_like_rows(c.q, dtype);
    if (tracked) lse = empty_dense({c.B, c.H, c.N}, at::kFloat);
    run_forward(c, out, result, lse, want_map);
    if (!wide) {
        result = out;
        if (Dk != c.D) {
            result = result.narrow(3, 0, c.D);
            // made below autograd, such a view counts versions of its own: with the count of the tensor that the
            // backward reads, a change of the result in place is noticed there
            if (tracked) torch::autograd::impl::set_version_counter(result, torch::autograd::impl::version_counter(out));
        }
        if (kdt != dtype) result = result.to(dtype);
    }
    if (!tracked) return result;
    torch::autograd::set_history(result, node);
    node->out_is_output = result.is_same(out);
    node->q = torch::autograd::SavedVariable(c.q, false);
    node->k = torch::autograd::SavedVariable(c.k, false);
    node->v = torch::autograd::SavedVariable(c.v, false);
    node->out = torch::autograd::SavedVariable(out, node->out_is_output);
    node->lse = torch::autograd::SavedVariable(lse, false);
    node->packed = torch::autograd::SavedVariable(c.packed, false);
    node->map = c.map;
    node->map_shown = map_shown;
    node->scale = c.scale;
    node->grad_dtype = dtype;
    node->grad_D = c.D;
    return result;
}

// What is wrong with the tensors of one call, or nullptr.  Everything below reaches them through raw pointers, with
// offsets computed from q's extents, so each entry point asks here first.
const char *refusal(const Tensor &q, const Tensor &k, const Tensor &v, const c10::optional<Tensor> &mask,
                    const c10::optional<Tensor> &mask_packed)
{
    if (!q.is_cuda()) return "q must be a GPU tensor";
    if (q.dim() != 4 || k.sizes() != q.sizes() || v.sizes() != q.sizes()) return "q, k, v must have the same 4D shape";
    if (k.device() != q.device() || v.device() != q.device()) return "q, k, v must be on the same device";
    const at::ScalarType dtype = q.scalar_type();
    if (dtype != at::kHalf && dtype != at::kBFloat16 && dtype != at::kFloat) return "Unsupported dtype, need BF16 or FP16 (or FP32)";
    if (dtype != at::kFloat && (k.scalar_type() != dtype || v.scalar_type() != dtype)) return "q, k, v must have the same dtype";
    const int64_t B = q.size(0), H = q.size(1), N = q.size(2), D = q.size(3);
    if (D < 1 || D > 128) return "head_dim must be at most 128";
    auto shared_or = [](int64_t have, int64_t want) { return have == 1 || have == want; };
    if (mask_packed.has_value() && mask_packed->defined()) {
        const Tensor &p = *mask_packed;
        if (p.device() != q.device()) return "mask_packed must be on q's device";
        if (p.scalar_type() != at::kInt || p.dim() != 4 || !shared_or(p.size(0), B) || !shared_or(p.size(1), H) || p.size(2) != N ||
            p.size(3) != (N + 31) / 32)
            return "mask_packed must be int32 [B or 1, H or 1, N, ceil(N/32)]";
        return nullptr;
    }
    if (!mask.has_value() || !mask->defined()) return "a mask or a packed mask is needed";
    const Tensor &m = *mask;
    if (m.device() != q.device()) return "mask must be on q's device";
    if (m.scalar_type() != at::kBool || m.dim() != 4 || !shared_or(m.size(0), B) || !shared_or(m.size(1), H) || m.size(2) != N ||
        m.size(3) != N)
        return "mask must be bool [B or 1, H or 1, N, N]";
    return nullptr;
}

// The problem of a call whose tensors have passed the checks above; `tile_map` is a tensor's Python object or nullptr.
Call problem(const Tensor &q, const c10::optional<Tensor> &mask, const c10::optional<Tensor> &mask_packed, const py::object *tile_map,
             double scale)
{
    Call c;
    c.B = q.size(0), c.H = q.size(1), c.N = q.size(2), c.D = q.size(3);
    if (mask_packed.has_value() && mask_packed->defined()) {
        c.packed = *mask_packed;
        if (tile_map) c.map = tile_map->cast<Tensor>();
    } else {
        c.mask = unexpand(*mask);
    }
    c.scale = scale;
    return c;
}

// sparse_attention / sparse_attention_func of the Python layer.  `tile_map` is None, True (leave a map
// behind for the backward) or a tensor.  None is returned, before anything has been done, for
// arguments that the Python layer refuses or has to prepare first (a boolean mask shorter than one
// 16-byte copy per row is packed there), and while torch.jit traces, which sees nothing of a native call.
c10::optional<Tensor> attention(const Tensor &q, const Tensor &k, const Tensor &v, const c10::optional<Tensor> &mask,
                                const c10::optional<Tensor> &mask_packed, const py::object &tile_map, bool autograd)
{
    if (refusal(q, k, v, mask, mask_packed) != nullptr || torch::jit::tracer::isTracing()) return c10::nullopt;
    const bool packed = mask_packed.has_value() && mask_packed->defined();
    const bool want_map = tile_map.ptr() == Py_True;
    const bool has_map = !want_map && !tile_map.is_none();
    if (packed ? want_map && autograd : has_map || (q.size(2) < 16 && q.numel() > 0)) return c10::nullopt;
    Call c = problem(q, mask, mask_packed, has_map ? &tile_map : nullptr, 1.0 / std::sqrt((double)q.size(3)));
    return run_call(q, k, v, c, want_map, autograd);
}

// SparseAttentionFunction.apply of the Python layer: the same with the scale given, for q, k and v of one type, whose
// wrong arguments are errors.  Without a packed mask, a tile map given as a tensor is not used.
Tensor attention_function(const Tensor &q, const Tensor &k, const Tensor &v, const c10::optional<Tensor> &mask_packed,
                          const c10::optional<Tensor> &mask, double scale, const py::object &tile_map)
{
    const char *const why = refusal(q, k, v, mask, mask_packed);
    TORCH_CHECK(why == nullptr, why);
    refuse_tangents(q, k, v);
    TORCH_CHECK(k.scalar_type() == q.scalar_type() && v.scalar_type() == q.scalar_type(), "q, k, v must have the same dtype");
    const bool packed = mask_packed.has_value() && mask_packed->defined();
    const bool want_map = tile_map.ptr() == Py_True;
    TORCH_CHECK(!(packed && want_map), "with mask_packed, pass the result of tile_map(mask_packed)");
    Call c = problem(q, mask, mask_packed, !want_map && !tile_map.is_none() ? &tile_map : nullptr, scale);
    return run_call(q, k, v, c, want_map, true);
}

// The Python type of the node, so that grad_fn shows what it carries.
PyObject *node_tile_map(PyObject *self, void *)
{
    const auto *node = static_cast<SparseAttentionBackward *>(reinterpret_cast<torch::autograd::THPCppFunction *>(self)->cdata.get());
    if (!node->map.defined() || !node->map_shown) Py_RETURN_NONE;
    return THPVariable_Wrap(node->map);
}

PyObject *node_scale(PyObject *self, void *)
{
    const auto *node = static_cast<SparseAttentionBackward *>(reinterpret_cast<torch::autograd::THPCppFunction *>(self)->cdata.get());
    return PyFloat_FromDouble(node->scale);
}

// What the backward will use: q, k, v, out, lse and the packed mask as the kernels take them, for as long as the
// backward can still run.  (Waiting for the lock and unpacking happen without the interpreter's lock: the backward holds the first
// while a saved-tensor hook may ask for the second.)
PyObject *node_saved_tensors(PyObject *self, void *)
{
    HANDLE_TH_ERRORS
    const std::shared_ptr<torch::autograd::Node> keep = reinterpret_cast<torch::autograd::THPCppFunction *>(self)->cdata;
    auto *node = static_cast<SparseAttentionBackward *>(keep.get());
    std::vector<Tensor> saved;
    {
        const py::gil_scoped_release no_gil;
        const std::lock_guard<std::recursive_mutex> lock(node->mutex);
        for (const torch::autograd::SavedVariable *s : {&node->q, &node->k, &node->v}) saved.push_back(s->unpack());
        saved.push_back(node->out.unpack(node->out_is_output ? keep : nullptr));
        for (const torch::autograd::SavedVariable *s : {&node->lse, &node->packed}) saved.push_back(s->unpack());
    }
    py::tuple result(saved.size());
    for (size_t i = 0; i < saved.size(); ++i) result[i] = py::reinterpret_steal<py::object>(THPVariable_Wrap(saved[i]));
    return result.release().ptr();
    END_HANDLE_TH_ERRORS
}

void register_node_type()
{
    using namespace torch::autograd;
    static PyTypeObject type;
    static PyGetSetDef properties[] = {THP_FUNCTION_DEFAULT_PROPERTIES,
                                       {"tile_map", node_tile_map, nullptr, nullptr, nullptr},
                                       {"scale", node_scale, nullptr, nullptr, nullptr},
                                       {"saved_tensors", node_saved_tensors, nullptr, nullptr, nullptr},
                                       {nullptr, nullptr, nullptr, nullptr, nullptr}};
    _initFunctionPyTypeObject(type, "SparseAttentionFunctionBackward", properties, nullptr);
    Py_INCREF(&type);
    registerCppFunction(typeid(SparseAttentionBackward), &type);
}

}  // namespace

PYBIND11_MODULE(sparse_attn_cuda, m)
{
    m.doc() = "sparse-mask attention for MI355X (gfx950): pybind shim over libsma_hip.so";
    m.def("forward", &forward, "Sparse-mask attention forward", py::arg("q"), py::arg("k"),
          py::arg("v"), py::arg("mask_packed"), py::arg("out"), py::arg("lse"), py::arg("scale"),
          py::arg("is_training"), py::arg("tile_map") = py::none());
    m.def("tile_map", &tile_map,
          "Which 64 x 64 blocks of a packed mask hold a set bit / only set bits (pass to forward as tile_map)",
          py::arg("mask_packed"));
    m.def("backward", &backward, "Sparse-mask attention backward (dq, dk, dv are overwritten)",
          py::arg("dout"), py::arg("q"), py::arg("k"), py::arg("v"), py::arg("out"), py::arg("lse"),
          py::arg("mask_packed"), py::arg("dq"), py::arg("dk"), py::arg("dv"), py::arg("scale"),
          py::arg("tile_map") = py::none());
    m.def("forward_bool_mask", &forward_bool_mask,
          "Sparse-mask attention forward straight from the bool mask (one launch; see bool_mask_supported)",
          py::arg("q"), py::arg("k"), py::arg("v"), py::arg("mask"), py::arg("out"), py::arg("lse"),
          py::arg("scale"), py::arg("is_training"), py::arg("packed_out") = py::none(),
          py::arg("map_out") = py::none());
    m.def("bool_mask_supported", &bool_mask_supported,
          "Whether forward_bool_mask applies to these tensors (else use pack_mask + forward)", py::arg("q"),
          py::arg("k"), py::arg("v"), py::arg("mask"));
    m.def("addressable", &addressable,
          "Whether the kernels take a [B, H, N, D] tensor as it is (else a contiguous copy of it)", py::arg("t"));
    m.def("pack_mask", &pack_mask, "Pack a bool mask into uint32 words (returned as int32)",
          py::arg("mask"));
    m.def("attention", &attention, "One call of the Python layer; None if its arguments need the checks made there",
          py::arg("q"), py::arg("k"), py::arg("v"), py::arg("mask"), py::arg("mask_packed"), py::arg("tile_map"),
          py::arg("autograd"));
    m.def("attention_function", &attention_function, "Forward with an autograd node, scale given", py::arg("q"),
          py::arg("k"), py::arg("v"), py::arg("mask_packed"), py::arg("mask"), py::arg("scale"), py::arg("tile_map"));
    register_node_type();
    m.def("version", []() { return sma_version(); });
}
