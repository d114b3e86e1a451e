// Internal C++ interface between the C-ABI layer (capi.hip) and the kernel launchers.
// Not installed; the public interface is include/sma.h.
#pragma once

#include <hip/hip_runtime.h>
#include <stdint.h>

namespace sma {

// A [B, H, N, D] tensor of 16-bit elements (fp16 or bf16 bit patterns).  The D elements of a row
// are contiguous; the other extents have strides that are multiples of 8 elements (rows stay
// 16-byte aligned).  Byte offsets inside one (b, h) slab fit 31 bits (checked by the C-ABI layer).
// Kept small: kernel arguments are fetched by every work-group before it can request any data.
struct Rows {
    uint16_t *p;
    uint32_t sb8, sh8;              // batch and head strides in units of 8 elements (16 bytes)
    uint32_t sn;                    // row stride in elements
};

// The packed mask [Bm, Hm, N, nw] with Bm in {1, B}, Hm in {1, H}: rows are contiguous, a stride of
// 0 (in words) repeats the same mask for every batch entry / head.
struct PackedMask {
    const uint32_t *p;
    long long sb, sh;
};

// Division of a work-group number by a launch constant without the (long, VALU) division sequence:
// n / d == (n * mul) >> shift in 64-bit arithmetic for every 0 <= n < 2^31, with
// shift = 31 + ceil(log2 d) and mul = ceil(2^shift / d) < 2^32 (round-up method: mul * d exceeds
// 2^shift by at most 2^(shift - 31), which cannot carry into the quotient while n < 2^31).
struct FastDiv {
    uint32_t mul, shift;
};
inline FastDiv make_fastdiv(uint32_t d)
{
    uint32_t l = 0;
    while ((1ull << l) < d) ++l;
    const uint64_t p = 1ull << (31 + l);
    return FastDiv{(uint32_t)((p + d - 1) / d), 31 + l};
}
__host__ __device__ inline uint32_t fastdiv(uint32_t n, FastDiv f)
{
    return (uint32_t)(((uint64_t)n * f.mul) >> f.shift);
}

// How work-groups, each a tile of a head, are dealt out: `together` heads' tiles in turn, the first of all of them first.
struct Deal {
    int together;
    FastDiv div_heads, div_groups;  // by `together` and by the tiles of so many heads
};
// One head after the other, unless neighbours have the same mask and there is more than one round of work-groups
// (`resident` of them at once).  Then the tiles of the heads are alike, the longest come first (the last rows of a causal mask, its first
// keys), and an XCD that takes as many heads in turn as it holds at once ends its share with the short tiles of all heads instead of with the
// long and the short ones of the last.  The group is the largest divisor of the share (no group lies on two XCDs) that is not
// more than that, or the next one up to two thirds above where its K and V fit an XCD's L2 (an eighth more is no loss yet) or the other is half of what is held or
// less.  What an XCD holds at once reads about as much K and V as its L2 has room for (96 work-groups at head dim 64 3 MB, 64 at 128 4 MB); a much
// larger group sends every K and V out of it between the tiles of its head.
// bf16, in us, one head after the other, groups of (held at once):
//   forward, no map   D =  64  232 heads, N = 4096 causal 699, 29 (3) 1048, random 1042, 1086;  488, N = 2048 causal 387, 61 (6) 560;  1016, N = 512 causal
//                              70.3, 127 (24) 91.2, random 87.6, 92.7;  40, N = 4096 causal 140.4, 5 (3) 134.7, random 182.0, 183.4
//                     D = 128  104, N = 4096 causal 540, 13 (2) 807;  192, N = 512 random 31.3, 12 (16) 31.5, 24 32.6;  256, N = 512 random 41.0,
//                              16 (16) 39.5, 32 46.7;  192, N = 800 random 79.2, 8 (9) 79.8, 24 85.4;  192, N = 1024 random 101.6, 8 (8) 102.5, 24 112.7
//   forward, map      blocks, one mask a batch entry: D = 128  192 heads, N = 512, mean of 24 masks drawn 26.0, 8 26.0, 12 (16) 26.6, 24 27.3;  N = 1024 62.5, 8 (8) 57.5,
//                              24 69.0;  D = 64 35.1, 12 (12) 32.4, 24 34.7
//                     D =  64  128 heads, N = 4096 causal 329, 2 309, 4 (3) 298;  192, N = 640 causal 21.9, 12 19.0, 24 (19) 18.4, blocks 19.6, 18.7, 18.2;  N = 700
//                              causal 29.8, 12 25.1, 24 (16) 22.1, blocks 22.7, 22.8, 21.9, random without a map 34.9, 35.0, 35.2
//                     D = 128  104, N = 1024 causal 48.2, 13 (8) 38.4, random 64.6, 65.5;  24, N = 4096 causal 124.8, 3 (2) 106.9, random 189.8, 190.0
//   backward, no map  D = 128  104, N = 1024 causal 168.9, 13 (8) 141.4;  232, N = 2048 causal 1047, 29 (4) 1120, random 1519, 1587
// A causal mask with a map, whose far tiles are not visited, gains from the larger groups too (232 heads, N = 4096, D = 64: 597 -> 543), but nothing here
// tells it from the others.
// Neighbours with the same mask are enough: that a group reaches into another batch entry, with a mask of its own, costs nothing by itself (64 x 2 heads,
// N = 2048, D = 64, groups of 1, 2, 4: causal, map 100.9, 95.6, 87.7, blocks 69.4, 67.9, 67.0, random 147.6, 149.5, 147.9).
// Where two long heads in turn read more from memory than one after the other (4 x 32, N = 4096, D = 128, one mask a batch entry: forward 583 -> 773 MB, dQ
// 852 -> 1043), they take no longer: random, forward 987 -> 974, backward 3052 -> 3021, causal 682 -> 677, 2030 -> 1934.
// One head after the other -> groups, in us, bf16:
//   forward, map      causal  D = 64: 64 heads, N = 2048 56.2 -> 39.9;  192, N = 1024 49.8 -> 38.5;  32, N = 4096 98.3 -> 76.2;  128, N = 4096 308 ->
//                             289;  D = 128: 64, N = 2048 92.9 -> 75.8;  256, N = 1024 98.6 -> 84.2;  128, N = 4096 537 -> 528
//                     blocks  192 heads, N = 1024: D = 32 25.8 -> 24.3, 64 35.2 -> 32.4, 128 60.6 -> 57.2;  N = 512, D = 128: see above
//                     random  192 heads, N = 1024: 56.3 either way;  D = 128 97.5;  128, N = 4096, D = 64 527 -> 530
//   forward, no map   causal  192 heads, N = 1024: D = 32 37.6 -> 31.4, 64 53.2 -> 43.6, 96 73.3 -> 60.7, 128 83.3 -> 71.7;  32, N = 4096: 97.9 ->
//                             64.4, 106.8 -> 85.6, 139.0 -> 127.6, 163.9 -> 150.7;  128, N = 4096, D = 128 558.6 -> 547.9
//                     blocks  192 heads, N = 1024: D = 32 32.4 -> 30.8, 64 41.5 -> 39.1, 128 67.5 -> 63.6
//                     random  192 heads, N = 1024: D = 32 46.7 -> 47.7 (three tiles of a CU no longer read the same mask rows), 64 63.4 -> 63.9, 128
//                             105.6 -> 106.1;  64, N = 2048, D = 32 57.6 -> 58.6, 64 80.3 -> 80.9, 128 132.2 either way
//   backward, map     causal  192 heads, N = 1024: D = 32 95.4 -> 71.0, 64 130.0 -> 114.5, 128 257.5 -> 215.5;  64, N = 2048, D = 128 304 -> 223;  128, N =
//                             4096: D = 64 942 -> 912, 128 1814 -> 1686
//                     blocks  192 heads, N = 1024: D = 32 73.7 -> 66.3, 64 95.5 -> 88.8, 128 198.3 -> 192.1
//                     random  D = 64: 192, N = 1024 182.9 -> 182.7;  128 heads, N = 4096: D = 64 1681 -> 1674, 128 2934 -> 2971
//   backward, no map  causal  192 heads, N = 1024: D = 32 105 -> 83, 64 153 -> 132, 128 265 -> 229;  random, 128, N = 4096, D = 128 3021 -> 3017
// With a mask for every head there is nothing alike to sort (forward, blocks, 192 heads, N = 1024: D = 64 33.9 -> 35.2, 128 58.6 -> 60.0).
inline bool heads_alike(const PackedMask &mask, int H) { return (H > 1 ? mask.sh : mask.sb) == 0; }
constexpr long long L2_BYTES = 4ll << 20;         // of an XCD
// head_bytes: what the tiles of a head all read (K and V, or Q and dO)
inline Deal make_deal(bool alike, int heads, int tiles, long long resident, long long head_bytes)
{
    int g = 1;
    if (alike && heads % 8 == 0 && (long long)heads * tiles > resident) {
        const int share = heads / 8;
        const long long held = resident / 8;
        while (g < share && (long long)(g + 1) * tiles <= held) ++g;
        while (share % g != 0) --g;
        const int below = g;
        for (long long more = below + 1; more <= share && 3 * more * tiles <= 5 * held; ++more)
            if (share % more == 0) {
                if (2ll * below * tiles <= held || more * head_bytes <= L2_BYTES + L2_BYTES / 8) g = (int)more;
                break;
            }
    }
    return Deal{g, make_fastdiv((uint32_t)g), make_fastdiv((uint32_t)(g * tiles))};
}
// Head and tile of work-group n.
struct Dealt {
    int head, tile;
};
__host__ __device__ inline Dealt deal(const Deal &d, int tiles, int n)
{
    const int first = (int)fastdiv((uint32_t)n, d.div_groups) * d.together, i = n - first * tiles;
    const int tile = (int)fastdiv((uint32_t)i, d.div_heads);
    return Dealt{first + i - tile * d.together, tile};
}

// Arguments of the fused forward kernel, already validated by the C-ABI layer.
struct AttnArgs {
    Rows q, k, v;                   // inputs (never written)
    Rows q16;                       // with q_f32: where to leave q's rounded rows, p == nullptr: nowhere
    int q_f32;                      // q.p names floats (bf16 kernels)
    PackedMask mask;                // byte_mask != 0: p names boolean bytes [Bm, Hm, N, N], strides in bytes
    Rows out, out32;                // 16-bit output and its fp32 copy (p names floats); p == nullptr: not wanted
    float *lse;                     // [BH, N] contiguous, or nullptr
    int groups;                     // work-groups of the launch: filled in by the launcher (the grid's own size lies behind all of this)
    int H, N;
    int D;                          // head dim: a multiple of 8 up to 128
    int BH;
    int byte_mask;                  // the mask is the caller's boolean tensor, not packed words
    uint32_t *mask_out;             // byte_mask only: nullptr, or where to leave the packed words [Bm, Hm, N, nw]
    uint32_t *map_out;              // byte_mask only: nullptr, or where to leave the tile map (layout as tile_map below)
    long long map_slabs;            // (batch entry, head) pairs of the mask
    // packed mask only: nullptr, or the tile map [Bm, Hm, T, 2, ceil(T/32)] (T = ceil(N/64)): per block
    // of 64 query rows one bit per 64-key tile "some mask bit set", then one bit per key tile "all
    // mask bits set"; strides between batch entries / heads in words, 0 = shared
    const uint32_t *tile_map;
    long long map_sb, map_sh;
    int qtiles;                     // ceil(N / 128): query tiles (work-groups) per (b,h)
    FastDiv div_H;                  // filled in by the launcher ...
    Deal deal;                      // ... like this; with a boolean mask one head after the other
    // exp(scale * s) is evaluated as exp2(post_mul * (q_scale * q) . k): q is multiplied by
    // q_scale (sign of scale included, |q_scale| <= 1) when it is loaded, post_mul is a power of
    // two that is 1 unless |scale| * log2(e) > 1.
    float q_scale;
    float post_mul;
    uint32_t last_mask0, last_mask1;   // valid-bit masks of the two mask words of the last key tile
    // Work-groups with a linear id >= tail_start lower their waves' priority as they advance, so
    // that the (up to four) work-groups of a CU finish together instead of oldest first.  The
    // launcher sets 0 when the whole grid is resident at once, else the grid size (nobody yields).
    int tail_start;
};

// Arguments of the two backward kernels (dQ, then dK and dV), already validated.
struct AttnBwdArgs {
    Rows dout, q, k, v, out;                   // inputs (never written)
    const float *lse;                          // [BH, N] natural-log-sum-exp saved by the forward
    PackedMask mask;
    Rows dq, dk, dv;                           // outputs: 16-bit elements, or floats if grads_f32
    int grads_f32;
    float *delta;                              // [BH, N] workspace: sum_d dout * out per query row
    const uint32_t *tile_map;                  // nullptr, or the tile map of the mask (as in AttnArgs)
    long long map_sb, map_sh;
    int BH, H, N;
    int D;                                     // head dim: a multiple of 8 up to 128
    int qtiles;                                // ceil(N / 128)
    int ktiles;                                // key tiles (work-groups of the dK/dV kernel) per (b,h) ...
    FastDiv div_qtiles, div_H;                 // ... and these: filled in by the launcher
    Deal deal;                                 // of the kernel that is launched
    int whole_heads, whole_groups;             // head dim 128, eight wavefronts: the heads, and their work-groups, of 256 keys each
    float scale;                               // as given by the caller
    float q_scale, post_mul;                   // as in AttnArgs
    uint32_t last_mask0, last_mask1;
};

// The kernels exist for head dims of 32, 64, 80, 96 and 128; any multiple of 8 in between runs in the next larger
// one: the copies fill an LDS row beyond the tensor's with its last 16 bytes once more, the fragments that the
// wavefronts hold in registers are zero there, and results beyond it are not stored.
// 80 differs from 96 in what has the head dim as its result (O, dQ, dK, dV): five blocks of 16 columns instead of six, one product in 12 less in the
// forward, in 18 in dQ, in 12 in dK/dV, with the operands read for them; the contractions take three steps of 32 in either.  (The whole-head backward, up
// to 256 keys, has none of its own.)  The kernels for 96 -> this, us, D = 80: training 128 heads, N = 2048 838 -> 801, 64, N = 1500 258 -> 246, 4,
// N = 3000 121 -> 116, 192, N = 1024, blocks with a map 211 -> 202, 128, N = 700 151 -> 147;  forward 64, N = 1500 82.2 -> 79.6, 128, N = 2048, packed 214 -> 206,
// causal 132 -> 125, 1024, N = 64 12.5 -> 11.7, 2, N = 333 9.98 -> 9.28, 128, N = 700, bound by the mask's bytes, 41.9 either way.  D = 72 the same (512 heads,
// N = 300, training 144.7 -> 140.9).
inline int kernel_head_dim(int D) { return D <= 32 ? 32 : D <= 64 ? 64 : D <= 80 ? 80 : D <= 96 ? 96 : 128; }

// Number of compute units of the current device (asked for once).
int compute_units();

hipError_t launch_attn_fwd(const AttnArgs &a, bool bf16, hipStream_t stream);
hipError_t launch_attn_bwd(const AttnBwdArgs &a, bool bf16, hipStream_t stream);
// ... by the kernel that holds a whole head in one work-group, where that is the faster; false: nothing was launched
bool launch_attn_bwd_head(const AttnBwdArgs &a, bool bf16, hipStream_t stream);
// fp32 -> bf16 (round to nearest even), `count` (at most 3) arrays of n elements, n a multiple of 8
hipError_t launch_to_bf16(const float *const *src, uint16_t *const *dst, int count, long long n, hipStream_t stream);
hipError_t launch_pack_mask(const uint8_t *mask, uint32_t *packed, long long rows, int N,
                            hipStream_t stream);
// Whether the current device serves 8- and 16-byte loads from unaligned addresses (the row packers
// and the forward that reads the boolean mask depend on it): 1 yes, 0 no, -1 not known (the
// one-time check could not run because `stream` is being captured into a graph, or failed).  The
// first call per device launches a one-wavefront check on `stream` and waits for it.
int unaligned_access_state(hipStream_t stream);
// tile map [slabs, ceil(N/64), 2, ceil(ceil(N/64)/32)] of packed words [slabs, N, ceil(N/32)]
hipError_t launch_tile_map(const uint32_t *packed, uint32_t *map, long long slabs, int N, hipStream_t stream);

// a tile map from which bits are then taken and to which bits are added: nothing kept, everything kept
hipError_t launch_tile_map_start(uint32_t *map, long long slabs, int N, hipStream_t stream);
// both of the above in one pass over the mask
hipError_t launch_pack_mask_map(const uint8_t *mask, uint32_t *packed, uint32_t *map, long long slabs, int N,
                                hipStream_t stream);

}  // namespace sma
