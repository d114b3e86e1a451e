// Shared device-side helpers of the attention kernels (gfx950): vector types, the fp16 / bf16
// element traits, cross-half lane exchanges, LDS reads (plain and transposing) and the asynchronous
// global -> LDS copies.  Included by attn_fwd.hip and attn_bwd.hip; everything has internal linkage.
#pragma once
#include "sma_internal.h"

namespace sma {
namespace {

typedef _Float16 f16x8 __attribute__((ext_vector_type(8)));
typedef _Float16 f16x2 __attribute__((ext_vector_type(2)));
typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef __bf16 bf16x2 __attribute__((ext_vector_type(2)));
typedef short i16x4 __attribute__((ext_vector_type(4)));
typedef float f32x2 __attribute__((ext_vector_type(2)));
typedef float f32x4 __attribute__((ext_vector_type(4)));
typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));
typedef uint32_t u32x2 __attribute__((ext_vector_type(2)));

// Which way a wave-uniform branch usually goes: the usual way falls through, the other is placed out of line.
#define LIKELY(c) __builtin_expect(c, 1)
#define UNLIKELY(c) __builtin_expect(c, 0)

#define LDS_PTR(T) __attribute__((address_space(3))) T *

// First element of the (b, h) slab of a strided tensor / of the packed mask.
__device__ __forceinline__ uint16_t *slab(const Rows &r, int b, int h) {
    return r.p + ((size_t)b * r.sb8 + (size_t)h * r.sh8) * 8;
}
__device__ __forceinline__ const uint32_t *slab(const PackedMask &m, int b, int h) { return m.p + b * m.sb + h * m.sh; }

template <bool BF16> struct Elem;

template <> struct Elem<false> {
    static constexpr uint32_t ONES = 0x3c003c00u;           // two fp16 1.0
    static __device__ __forceinline__ f32x4 mfma(u32x4 a, u32x4 b, f32x4 c) {
        return __builtin_amdgcn_mfma_f32_16x16x32_f16(__builtin_bit_cast(f16x8, a),
                                                      __builtin_bit_cast(f16x8, b), c, 0, 0, 0);
    }
    // Two probabilities -> one packed register with the cheapest conversion the format has (fp16:
    // v_cvt_pkrtz, round toward zero); the row sum is taken over the SAME rounded values, so
    // numerator and denominator stay consistent whatever the rounding.
    static __device__ __forceinline__ uint32_t pack2_prob(float a, float b) {
        return __builtin_bit_cast(uint32_t, __builtin_amdgcn_cvt_pkrtz(a, b));
    }
    static __device__ __forceinline__ uint32_t pack2_rne(float a, float b) {     // round to nearest even
        const f16x2 h = {(_Float16)a, (_Float16)b};
        return __builtin_bit_cast(uint32_t, h);
    }
    // acc and the sum of a pair; `ones` is ONES (from a scalar register half the code of a literal)
    static __device__ __forceinline__ float add2(uint32_t p, uint32_t ones, float acc) {
        return __builtin_amdgcn_fdot2(__builtin_bit_cast(f16x2, p), __builtin_bit_cast(f16x2, ones), acc, false);
    }
    static __device__ __forceinline__ uint16_t cvt1(float a) {          // round to nearest even
        return __builtin_bit_cast(uint16_t, (_Float16)a);
    }
    static __device__ __forceinline__ float up1(uint16_t h) {
        return (float)__builtin_bit_cast(_Float16, h);
    }
    static constexpr float TERM_MAX = 60000.0f;             // keep split terms finite in fp16
};

template <> struct Elem<true> {
    static constexpr uint32_t ONES = 0x3f803f80u;           // two bf16 1.0
    static __device__ __forceinline__ f32x4 mfma(u32x4 a, u32x4 b, f32x4 c) {
        return __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8, a),
                                                       __builtin_bit_cast(bf16x8, b), c, 0, 0, 0);
    }
    static __device__ __forceinline__ uint32_t pack2_prob(float a, float b) {
        // one v_cvt_pk_bf16_f32 (round to nearest even)
        const bf16x2 h = {(__bf16)a, (__bf16)b};
        return __builtin_bit_cast(uint32_t, h);
    }
    static __device__ __forceinline__ uint32_t pack2_rne(float a, float b) {
        const bf16x2 h = {(__bf16)a, (__bf16)b};
        return __builtin_bit_cast(uint32_t, h);
    }
    static __device__ __forceinline__ float add2(uint32_t p, uint32_t ones, float acc) {
        return __builtin_amdgcn_fdot2_f32_bf16(__builtin_bit_cast(bf16x2, p), __builtin_bit_cast(bf16x2, ones), acc, false);
    }
    static __device__ __forceinline__ uint16_t cvt1(float a) {
        return __builtin_bit_cast(uint16_t, (__bf16)a);
    }
    static __device__ __forceinline__ float up1(uint16_t h) {
        return __builtin_bit_cast(float, (uint32_t)h << 16);
    }
    static constexpr float TERM_MAX = 3.0e38f;
};

// Bit reversal of a 3-bit value: the chunk swizzle of tiles that are read both by rows and transposed.
__device__ __forceinline__ int bitrev3(int f) { return ((f & 1) << 2) | (f & 2) | (f >> 2); }

// XCD-aware renumbering of the work-groups.  They are handed to the 8 XCDs round-robin by linear
// id; the number returned gives each XCD (own L2) a contiguous range of (b,h) pairs, with the
// tiles of one (b,h) dispatched next to each other: the matrices of a head are then fetched into
// one L2 only.
__device__ __forceinline__ int renumber_block(int bid, int total)
{
    const int xcd = bid & 7, j = bid >> 3;
    const int base = total >> 3, rem = total & 7;
    return xcd * base + (xcd < rem ? xcd : rem) + j;
}
__device__ __forceinline__ int renumber_block() { return renumber_block((int)blockIdx.x, (int)gridDim.x); }

// max / sum of a value with its partner in the other lane half (lane l <-> lane l ^ 32).
// v_permlane32_swap(a, b) leaves {own a | partner's b, partner's a | own b} in lanes < 32 | >= 32.
__device__ __forceinline__ float xhalf_max(float x) {
    const uint32_t u = __builtin_bit_cast(uint32_t, x);
    const auto r = __builtin_amdgcn_permlane32_swap(u, u, false, false);
    return __builtin_fmaxf(__builtin_bit_cast(float, (uint32_t)r[0]), __builtin_bit_cast(float, (uint32_t)r[1]));
}
__device__ __forceinline__ float xhalf_sum(float x) {
    const uint32_t u = __builtin_bit_cast(uint32_t, x);
    const auto r = __builtin_amdgcn_permlane32_swap(u, u, false, false);
    return __builtin_bit_cast(float, (uint32_t)r[0]) + __builtin_bit_cast(float, (uint32_t)r[1]);
}
// Products of 16 x 16 leave a lane values of the two rows 16x + lane % 16, x = 0, 1.  From these the largest / the sum of row lane % 32, in both
// lane halves, and from something of row lane % 32 (in both halves) that of the lane's two.
// v_permlane16_swap(a, b) leaves {a's lanes of even | b's of even sixteens, a's of odd | b's of odd sixteens} in even | odd sixteens.
__device__ __forceinline__ float rows_max(float x0, float x1) {
    const auto r = __builtin_amdgcn_permlane16_swap(__builtin_bit_cast(uint32_t, x0), __builtin_bit_cast(uint32_t, x1), false, false);
    return xhalf_max(__builtin_fmaxf(__builtin_bit_cast(float, (uint32_t)r[0]), __builtin_bit_cast(float, (uint32_t)r[1])));
}
__device__ __forceinline__ float rows_sum(float x0, float x1) {
    const auto r = __builtin_amdgcn_permlane16_swap(__builtin_bit_cast(uint32_t, x0), __builtin_bit_cast(uint32_t, x1), false, false);
    return xhalf_sum(__builtin_bit_cast(float, (uint32_t)r[0]) + __builtin_bit_cast(float, (uint32_t)r[1]));
}
struct RowPair {
    uint32_t w[2];
};
__device__ __forceinline__ RowPair of_rows(uint32_t u) {
    const auto r = __builtin_amdgcn_permlane16_swap(u, u, false, false);
    return RowPair{{(uint32_t)r[0], (uint32_t)r[1]}};
}
// The sum of a value and its partner's in the neighbouring sixteen (lane l <-> lane l ^ 16).
__device__ __forceinline__ float xrow_sum(float x) {
    const uint32_t u = __builtin_bit_cast(uint32_t, x);
    const auto r = __builtin_amdgcn_permlane16_swap(u, u, false, false);
    return __builtin_bit_cast(float, (uint32_t)r[0]) + __builtin_bit_cast(float, (uint32_t)r[1]);
}

__device__ __forceinline__ u32x4 lds_read_b128(uint32_t addr) {
    return *(LDS_PTR(const u32x4))(uintptr_t)addr;
}
__device__ __forceinline__ u32x2 lds_read_b64(uint32_t addr) {
    return *(LDS_PTR(const u32x2))(uintptr_t)addr;
}
// Transposing LDS read: within each group of 16 lanes, lane i receives element (i % 4) of the
// 8-byte rows addressed by lanes i/4, 4 + i/4, 8 + i/4, 12 + i/4 of the group.
__device__ __forceinline__ u32x2 lds_read_tr16_b64(uint32_t addr) {
    const i16x4 v = __builtin_amdgcn_ds_read_tr16_b64_v4i16((LDS_PTR(i16x4))(uintptr_t)addr);
    return __builtin_bit_cast(u32x2, v);
}

// Asynchronous global -> LDS copies.  Lane i's 16 (4) bytes land at lds_base + 16 (4) * i; the
// global address is base + voff (bytes).  They are issued from inline assembly so that the
// compiler's own wait-count bookkeeping does not serialise them against unrelated LDS reads; the
// kernel waits for them explicitly with s_waitcnt vmcnt(n) (completion is in issue order).
__device__ __forceinline__ void async_copy_b128(uint32_t lds_base, const void *base, uint32_t voff) {
    asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %1, %2"
                 :: "s"(lds_base), "v"(voff), "s"(base) : "memory", "m0");
}
__device__ __forceinline__ void async_copy_b32(uint32_t lds_base, const void *base, uint32_t voff) {
    asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tglobal_load_lds_dword %1, %2"
                 :: "s"(lds_base), "v"(voff), "s"(base) : "memory", "m0");
}
// The same with the LDS address given as a scalar base plus a compile-time offset: a loop that
// copies to many fixed places then keeps one base in a scalar register instead of one per place.
template <int OFF>
__device__ __forceinline__ void async_copy_b128_at(uint32_t lds_base, const void *base, uint32_t voff) {
    asm volatile("s_add_u32 m0, %0, %3\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %1, %2"
                 :: "s"(lds_base), "v"(voff), "s"(base), "n"(OFF) : "memory", "scc", "m0");
}
// ... two of them, in one statement: between two statements the compiler puts a wait state of its own
template <int OFF, int OFF2>
__device__ __forceinline__ void async_copy2_b128_at(uint32_t lds_base, const void *base, uint32_t voff, uint32_t voff2) {
    asm volatile("s_add_u32 m0, %0, %4\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %1, %3\n\t"
                 "s_add_u32 m0, %0, %5\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %2, %3"
                 :: "s"(lds_base), "v"(voff), "v"(voff2), "s"(base), "n"(OFF), "n"(OFF2) : "memory", "scc", "m0");
}
template <int OFF>
__device__ __forceinline__ void async_copy_b32_at(uint32_t lds_base, const void *base, uint32_t voff) {
    asm volatile("s_add_u32 m0, %0, %3\n\ts_nop 0\n\tglobal_load_lds_dword %1, %2"
                 :: "s"(lds_base), "v"(voff), "s"(base), "n"(OFF) : "memory", "scc", "m0");
}
#define WAIT_VMCNT(n) asm volatile("s_waitcnt vmcnt(" #n ")" ::: "memory")


// Where a wavefront's 32 x COLS block of results goes: 16-bit rows, 32-bit rows (the rounded values
// widened), or both; a null pointer leaves one out.
struct BlockDst {
    uint16_t *h;            // first row, first of the COLS columns
    float *f;
    uint32_t h_sn, f_sn;    // row strides in elements
    int cols;               // columns of the tensor from there on: columns beyond are not stored
};
__device__ __forceinline__ BlockDst block_dst(const Rows &h, const Rows &f, int b, int hd, int row0, int D)
{
    BlockDst d;
    d.h = h.p != nullptr ? slab(h, b, hd) + (size_t)row0 * h.sn : nullptr;
    d.f = f.p != nullptr ? reinterpret_cast<float *>(f.p) + ((size_t)b * f.sb8 + (size_t)hd * f.sh8) * 8 + (size_t)row0 * f.sn
                         : nullptr;
    d.h_sn = h.sn;
    d.f_sn = f.sn;
    d.cols = D;
    return d;
}
__device__ __forceinline__ BlockDst columns_from(const BlockDst &d, int col)
{
    return BlockDst{d.h + col, d.f + col, d.h_sn, d.f_sn, d.cols - col};
}

// The second half of a transposed store: a 32 x COLS block of 16-bit results that lies in 4 KiB of wave-private LDS (row r at 128 r, its
// 16-byte chunks at their position ^ (r / 2) % 8) goes out as whole pieces of rows.  Non-temporal stores: what is written is not
// read again by the kernel and should not displace its inputs from the caches.
template <bool BF16, int COLS>
__device__ __forceinline__ void store_landed(uint32_t lds_wave, const BlockDst &dst, bool has_h, bool has_f, int row0, int N, int lane)
{
    using E = Elem<BF16>;
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
    constexpr int LPR = COLS / 8;                 // lanes (16-byte chunks) per row
    constexpr int STEPS = LPR / 2;
    const int pos = lane % LPR, row_in = lane / LPR;
    u32x4 v[STEPS];
#pragma unroll
    for (int j = 0; j < STEPS; ++j) {
        const int row = (64 / LPR) * j + row_in;
        v[j] = lds_read_b128(lds_wave + row * 128 + ((pos ^ ((row >> 1) & 7)) << 4));
    }
    // every branch on `has_h`, `has_f` and `whole` is wave-uniform and taken once, not per row: tested row by row
    // the stores of the two kernels of the backward cost 3 us of 110 (64 x 16 heads, N = 256)
    const bool whole = row0 + 32 <= N && dst.cols >= COLS;
    auto each = [&](auto store) __attribute__((always_inline)) {
        if (whole) {
#pragma unroll
            for (int j = 0; j < STEPS; ++j) store(j, (64 / LPR) * j + row_in);
        } else {
#pragma unroll
            for (int j = 0; j < STEPS; ++j) {
                const int row = (64 / LPR) * j + row_in;
                if (row0 + row < N && pos * 8 < dst.cols) store(j, row);
            }
        }
    };
    if (has_h)
        each([&](int j, int row) __attribute__((always_inline)) {
            __builtin_nontemporal_store(v[j], reinterpret_cast<u32x4 *>(dst.h + (size_t)row * dst.h_sn + pos * 8));
        });
    if (has_f)
        each([&](int j, int row) __attribute__((always_inline)) {
            f32x4 lo, hi;
#pragma unroll
            for (int i = 0; i < 2; ++i) {
                lo[2 * i] = E::up1((uint16_t)(v[j][i] & 0xffffu));
                lo[2 * i + 1] = E::up1((uint16_t)(v[j][i] >> 16));
                hi[2 * i] = E::up1((uint16_t)(v[j][2 + i] & 0xffffu));
                hi[2 * i + 1] = E::up1((uint16_t)(v[j][2 + i] >> 16));
            }
            f32x4 *f = reinterpret_cast<f32x4 *>(dst.f + (size_t)row * dst.f_sn + pos * 8);
            __builtin_nontemporal_store(lo, f);
            __builtin_nontemporal_store(hi, f + 1);
        });
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
}
// Transposed store of 32 rows from accumulators of 16 x 16 products, acc[rb][db][j] = value(row 16rb + lane % 16, column 16db + 4 (lane / 16) + j),
// times `mult` of the row's block: COLS columns from block DB0 on, through 4 KiB of wave-private LDS ...
template <bool BF16, int COLS, int DB0, int NB>
__device__ __forceinline__ void store_block(const f32x4 (&acc)[2][NB], const float (&mult)[2], uint32_t lds_wave,
                                              const BlockDst &dst, bool has_h, bool has_f, int row0, int N, int lane)
{
    using E = Elem<BF16>;
    const int l16 = lane & 15, q4 = lane >> 4;
    const uint32_t wrow = lds_wave + l16 * 128 + (q4 & 1) * 8;
    const int chunk = (q4 >> 1) ^ (l16 >> 1);
#pragma unroll
    for (int rb = 0; rb < 2; ++rb)
#pragma unroll
        for (int db = 0; db < COLS / 16; ++db) {
            const f32x4 x = acc[rb][DB0 + db] * mult[rb];
            const u32x2 o = {E::pack2_rne(x[0], x[1]), E::pack2_rne(x[2], x[3])};
            *(LDS_PTR(u32x2))(uintptr_t)(wrow + 2048 * rb + ((chunk ^ (2 * db)) << 4)) = o;
        }
    store_landed<BF16, COLS>(lds_wave, dst, has_h, has_f, row0, N, lane);
}
// ... and all columns, 64 at a time; `stride` LDS bytes between the areas of the two column halves (0: one after the other through
// the same 4 KiB)
template <bool BF16, int NB>
__device__ __forceinline__ void store_rows(const f32x4 (&acc)[2][NB], const float (&mult)[2], uint32_t lds_wave, uint32_t stride,
                                             const BlockDst &dst, bool has_h, bool has_f, int row0, int N, int lane)
{
    store_block<BF16, NB == 2 ? 32 : 64, 0>(acc, mult, lds_wave, dst, has_h, has_f, row0, N, lane);
    if constexpr (NB > 4)
        store_block<BF16, NB < 8 ? 16 * (NB - 4) : 64, 4>(acc, mult, lds_wave + stride, columns_from(dst, 64), has_h, has_f, row0, N, lane);
}

}  // namespace
}  // namespace sma
