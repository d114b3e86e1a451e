// Fused masked-attention forward for gfx950 (MI355X), head_dim 32, 64, 80, 96 or 128, fp16 / bf16, fp32 accumulate.
//
// Stands in for sparse_attn_wmma_full_fp16 (csrc/sparse_attention.cu:82-412 of the reference) and
// for its scalar bf16 kernel (csrc/sparse_attention.cu:418-543); the design below is specific to
// CDNA4 and shares nothing with either beyond the function computed.
//
// Work decomposition
//   work-group  = 4 wavefronts = 128 query rows of one (b,h); it walks the keys in tiles of 64.
//                 Three work-groups fit a CU (<= 168 VGPRs, ~34 KB LDS each): one wavefront of
//                 each per SIMD, so that the softmax VALU work of one overlaps the MFMAs of another.
//   wavefront   = 32 query rows.  It computes S^T = K_tile (64x64) * Q^T (64x32) with
//                 v_mfma_f32_16x16x32, so every lane owns two query rows (lane % 16 and 16 more) and 16 of the
//                 tile's 64 keys: the online softmax is a per-lane register loop, and what is looked at once
//                 a tile or less (maximum, reference point, total) is kept for row lane % 32 by two
//                 exchanges (v_permlane16_swap, v_permlane32_swap).  P^T is already in
//                 the B-operand layout of O^T += V^T * P^T: probabilities never leave registers.
//                 The long grids run at the clock that the matrix cores' power leaves, and 16 x 16 x 32 draws
//                 less than 32 x 32 x 16 (a stream on random operands, benchprobe/: 1968 TFLOP/s at 1.97 GHz, 1820 at 1.77).
//                 These products are short, so their operands are requested two or three steps of two
//                 products ahead (four or more of V while the exponentials run), in an order that scheduling barriers
//                 hold.  Forward, 32 x 32 x 16 with operands one step ahead -> this, in us:
//                   packed, 128 heads, N = 2048    D = 32 99 -> 96, 64 147 -> 138, 96 213 -> 200, 128 257 -> 239
//                   causal, 128 heads, N = 2000    D = 64 105 -> 102, 96 148 -> 144, 128 175 -> 167
//                   boolean, 128 heads, N = 1000   D = 64 49.5 -> 48.4, 128 76.9 -> 74.8;  1024 heads, N = 200: D = 64 30.0 -> 29.9
//                   packed, 192 heads, N = 1024    D = 64 59.3 -> 56.5 (blocks, map 37.3 -> 36.9), 128 106 -> 100 (62.2 -> 61.2)
//                 A call of one or two tiles takes the same cycles as before.
//   K/V tiles   = copied global -> LDS by global_load_lds_dwordx4 (no VGPR staging) into a ring of
//                 two stages, one tile ahead of the one being computed.  Rows are 128 B; the
//                 16-byte chunks of a row are XOR-swizzled (the permutation is applied to the
//                 global address of each lane; the LDS side of such a load is always linear) so
//                 that K's ds_read_b128 (16 consecutive rows x 64 B) and V's
//                 ds_read_b64_tr_b16 (transposing read, 16 consecutive rows x 32 B) are free of
//                 bank conflicts on the 64-bank LDS.
//   mask        = each wavefront copies the two packed words per query row of a tile into LDS with
//                 one global_load_lds_dword, one tile ahead.  A lane reads the two words of
//                 row lane % 32 and has those of its two rows by an exchange; each nibble selects one of 16 rows of a small LDS table of four floats that
//                 are 0 (keep) or -inf (drop); one ds_read_b128 of that row initialises four
//                 accumulator registers of the QK^T MFMA chain.  Masking costs no VALU work per score.
//   exponent    = q is multiplied by scale*log2(e) when it is loaded, and the reference point of
//                 the softmax (a per-row value r, see below) is subtracted INSIDE the MFMA chain by
//                 one extra MFMA whose B operand holds -r split into four 16-bit terms and whose
//                 A operand is all ones.  The accumulator then holds log2 of the unnormalised
//                 probability: the per-score VALU work is exp2, pack, row-sum and row-max only.
//   reference r = the online softmax does not track the running maximum.  r moves (and O, l are
//                 rescaled) only when a row's scores leave the window [r-8, r+8] upwards, or when its
//                 first kept score lies below the window.  The row maximum of a tile is not even
//                 computed unless a row meets its first kept key there or the sum of the tile's
//                 weights shows, afterwards, that a score has run away (then they are redone).
//   skipping    = with a tile map (one "some bit set" bit per 64 x 64 block of the mask, made by
//                 the packer) the work-group visits only the key tiles that hold a set bit for its
//                 rows: no copies, no barrier for the others.  Without a map every tile is
//                 copied.  Either way a wavefront whose own 32 x 64 block of mask bits is empty
//                 skips its GEMMs and its softmax for that tile.
//   head dim    = the description above is for 64.  128 runs the same code on two column halves of
//                 64 (see Cfg below): twice the MFMAs per tile for the same softmax work, a ring of
//                 two stages and two work-groups per CU.  32, 80 and 96 keep short rows (second_row).
#include <atomic>
#include <type_traits>

#include "attn_common.h"

namespace sma {
namespace {

constexpr int HD = 64;             // columns of one LDS tile: the head dim, or one half of a head dim of 128
constexpr int BM = 128;            // query rows per work-group
constexpr int BN = 64;             // keys per tile
constexpr int NTHREADS = 256;
constexpr int TILE_BYTES = BN * HD * 2;          // 8 KiB, rows of 128 B
constexpr float WINDOW_LOG2 = 8.0f;
constexpr float SUM_LIMIT = 16384.0f;     // a lane's 32 weights of a tile sum to more: some score is far above the window

// Head dims (HDIM) other than 64 reuse the 64-column LDS tile with its 128-byte rows, swizzles and
// read patterns:
//   128  two column halves (NH = 2): K and V tiles are kept in LDS as two 64-column tiles each, the
//        QK^T chain runs over both halves of K and q, and P multiplies each half of V into its own
//        pair of accumulators.  A stage is twice as large (32 KiB) and the kernel needs about 224
//        registers, so two work-groups share a CU.
//   32   half a tile: rows of 64 bytes (with SPLIT of 128, of which the copies fill the upper half with the row's last
//        16 bytes, which are never read); the QK^T chain has one step instead of two and P multiplies
//        two 16-column blocks of V.
//   96   128 with such a half tile as its second half: three steps, six blocks.  D = 80 and 96 ran in the
//        128 kernel before, through zero-padded copies (16 x 8 heads, N = 1088, D = 96: 156 -> 81 us)
//   80   as 96 with five blocks (what that gives stands at kernel_head_dim)
//
// BYTEMASK: the mask arrives as the caller's boolean bytes (one per score, 0 or 1) instead of packed
// words.  Each wavefront copies the 32 x 64 bytes of a tile for its rows into LDS and turns them
// into the two words per row itself (eight dot products with the weights 1, 2, 4 .. 128 per lane
// and one exchange between the lane halves): the separate packing pass, its launch and the
// round trip of the words through memory disappear for a mask that is used once.
// SECOND: bytes of a row in the second column half's tile (head dims beyond 64; at 32, but with SPLIT, all of the row: there is no first half).  At head dims 80 and 96, but with SPLIT, the rows there are only as long as
// what is used of them: 32 and 64 bytes, of which one request fills 32 or 16 rows.  A wavefront requests five or six pieces of K and V a tile instead of eight, and a stage is 20
// or 24 KiB instead of 32, which is what lets three work-groups share a CU (see three_on_a_cu).  Whole rows -> this with two on a CU all the same: D = 80, 512 heads, N = 320 33.7 ->
// 32.4 us, N = 512 67.1 -> 65.4; D = 96 36.4 -> 35.9, 69.9 -> 68.5.  64 bytes where by-products are asked for at 80 (two on a CU: 32, whose reads of K's last step
// meet in a bank, cost 64 heads, N = 1500 in training 281 -> 285 us, 64 282), and whole rows for fp32 queries at 96 (64, N = 1500 104.0 -> 109.5).
// Head dim 32, two requests a tile instead of four, stages of 8 KiB instead of 16, with which the boolean mask's bytes leave room for four work-groups on a CU instead of three (the packed words did already; with by-products
// 132 to 137 registers keep it at three, and in 128 of them 2 to 34 are spilled: the forward of a training step, 2048 heads, N = 100 19.0 -> 19.6 us, 256, N = 512 24.0 -> 22.5), whole rows -> this:
// boolean 2048 heads, N = 32 11.6 -> 9.8 us, N = 100 16.1 -> 14.5, N = 200 45.7 -> 42.3;  256, N = 1000 78.3 -> 73.4;  192, N = 1024 55.2 -> 52.6;  packed 2048, N = 200 33.2 -> 31.5, 128, N = 2048 96.4 -> 93.8,
// causal 60.5 -> 60.3;  2048, N = 128 boolean 18.2 -> 17.9.  Two packed tiles a head that are all but full, all bytes at 4.8 TB/s, win and lose by the number of work-groups on a CU, with inputs in the caches (from memory):
// N = 128, seven 12.8 -> 13.4 (13.6 -> 13.6), eight 14.5 -> 14.6 (15.3 -> 15.4), nine 15.7 -> 16.5 (17.3 -> 17.4), twelve 19.0 -> 19.2 (23.8 -> 22.6);  N = 120, 7 12.4 -> 12.7 (12.4 -> 12.7), 12 19.0 -> 18.6, 24 39.6 -> 38.8;
// an instance with whole rows for them gave as much back as it got.
constexpr int second_row(int hdim, bool split, bool byproducts, bool wide_q)
{
    return hdim == 32 ? (split ? 0 : 64) : hdim <= 64 ? 0 : split || hdim == 128 || (hdim == 96 && wide_q) ? 128 : hdim == 96 || byproducts ? 64 : 32;
}
template <int NH, bool BYTEMASK, bool SPLIT, int SECOND> struct Cfg {
    // SPLIT: one K and one V buffer for each of the four wavefronts, else a ring of two stages: copies run one tile ahead
    static constexpr int NSTAGE = SPLIT ? 4 : 2;
    static constexpr int MASK_COPIES = BYTEMASK ? 2 : 1;
    static constexpr int FIRST = NH == 1 && SECOND != 0 ? 0 : TILE_BYTES;                // the first half's tile: none at head dim 32, all of whose row is short
    static constexpr int KV_COPIES = (FIRST != 0 ? 4 : 0) + (SECOND == 32 ? 1 : SECOND / 32);
    static constexpr int COPIES = MASK_COPIES + KV_COPIES;          // async copies per wave and tile
    // LDS map (bytes), after the 256 of the table of the mask bias, which lies first: a read's immediate offset reaches 64 KiB
    static constexpr int OFF_V = FIRST + BN * SECOND;               // V inside a stage
    static constexpr int STAGE_BYTES = 2 * OFF_V;                   // K halves, then V halves
    // mask: packed words in NSTAGE slots of 4 waves x 64 words; bytes in slots of 4 waves x 2 KiB,
    // two of them for head dims up to 64 and, for want of LDS, ONE for 128: a wave has turned its
    // bytes into words before it requests the next tile's (see the main loop), so one slot is
    // enough, at the price of waiting for those reads before the requests (3 % on the headline
    // workload, which is why two are used where they fit)
    static constexpr int OFF_MASK = NSTAGE * STAGE_BYTES;
    static constexpr int BYTE_SLOTS = NH == 1 && !SPLIT ? 2 : 1;
    static constexpr int MASK_SLOT = BYTEMASK ? (BYTE_SLOTS - 1) * 8192 : 1024;     // distance between the slots
    // byte mask only: the tile-map bits the wavefronts collect, [4 waves][MAP_WORDS][some, hole],
    // and one arrival counter per pair of wavefronts (block of 64 rows)
    static constexpr int MAP_WORDS = 32;                            // 32 x 32 key tiles: N <= 65536
    // (SPLIT writes them to memory at once)
    static constexpr int OFF_MAP = OFF_MASK + (BYTEMASK ? BYTE_SLOTS * 8192 : SPLIT ? 1024 : NSTAGE * 1024);
    static constexpr int OFF_MAP_ARRIVED = OFF_MAP + 4 * MAP_WORDS * 8;
    static constexpr int LUT_BYTES = 256;                           // 16 x 16 B
    // head dim 32, packed words: the rows leave through 4 KiB a wavefront of their own (a stage is smaller than that)
    static constexpr int LDS_BYTES = LUT_BYTES + (BYTEMASK && !SPLIT ? OFF_MAP_ARRIVED + 16 : OFF_MAP + (FIRST == 0 ? 16384 : 0));
};

// Head dims beyond 64 of which three work-groups share a CU (but with SPLIT): where 168 registers hold the loop, with operands requested no further ahead
// than at head dim 64 (by-products: 34 spilled at 80;  fp32 queries at 96: 32), and the LDS three of them (the boolean mask's bytes at 96 do not fit).  A visit is bound by its chain of
// products, exponentials and products, which a third wavefront on the SIMD fills.  Two (with whole rows in the second half) -> three, us:
//   D = 80   packed 128 heads, N = 2048 206 -> 183, causal 125 -> 116;  192, N = 1024, blocks with a map 55.8 -> 49.0;  192, N = 512 27.1 -> 22.6;  512, N = 256 21.5 -> 19.2;
//            2048, N = 64 20.0 -> 17.2;  boolean 64, N = 1500 79.6 -> 73.0;  128, N = 700 41.9 -> 37.5;  fp32 64, N = 1500 99.6 -> 93.1
//   D = 96   packed 128, N = 2048 220 -> 202, causal 133 -> 125;  64, N = 1500 66.2 -> 58.0;  192, N = 1024, blocks with a map 58.1 -> 52.8;  192, N = 512 26.6 -> 23.2
// Work-groups of 64 rows (HALVES) have the registers anyway: 8 heads, N = 3000, boolean D = 80 50.8 -> 49.1, 96 56.4 -> 50.9.
constexpr bool three_on_a_cu(int hdim, bool bytemask, bool byproducts, bool wide_q)
{
    return !byproducts && (hdim == 80 || (hdim == 96 && !bytemask && !wide_q));
}

// The kernel's arguments where they lie.  What is read through this is requested no earlier than here: arguments are fetched from the host's
// memory, and a work-group can request no data before those that the compiler has moved to its start have arrived.
typedef const __attribute__((address_space(4))) AttnArgs *KernelArgs;
__device__ __forceinline__ KernelArgs kernel_args()
{
    auto p = (KernelArgs)__builtin_amdgcn_kernarg_segment_ptr();
    asm volatile("" : "+s"(p));
    return p;
}
__device__ __forceinline__ Rows rows_of(const __attribute__((address_space(4))) Rows &r) { return Rows{r.p, r.sb8, r.sh8, r.sn}; }

template <int N> __device__ __forceinline__ void wait_vmcnt() { asm volatile("s_waitcnt vmcnt(%0)" :: "n"(N) : "memory"); }

// PACKED_ROWS: the rows of q, k, v and out follow each other without gaps (row stride 64), as in
// contiguous tensors; the strides between heads and batch entries stay free.  A row stride known
// at compile time measured 0.25 us less fixed cost per launch than the same value read at run time.
// BYPRODUCTS (with BYTEMASK): the caller wants the packed words and / or the tile map of the mask
// left behind; a separate instantiation, so that the kernel of a caller who wants neither carries
// none of that code (it measured 1.5 % on the headline workload even when switched off at run time).
// PAIRS (FETCH != 0, with BYTEMASK, head dims up to 64): the mask bytes of
// TWO key tiles are requested at once, every second visit: 128 bytes per row, i.e. whole cache lines
// where one tile's 64 bytes are half of one.  The forward from the boolean mask measured 1 to 5 %
// faster this way on random masks of every length tried (128 to 2048) and 7 % on the
// block-structured workload -- except where the whole grid is one round of work-groups that run in
// step (the even-progress case of the launcher, e.g. the headline shape): there the first visit,
// which waits for twice the bytes, is not hidden behind other work-groups' work, it measured 1 to 4 %
// slower, and the launcher leaves it off.
// FETCH = 1: N a multiple of 128: no row and no pair ends within a request.  FETCH = 2: any N; the ends cost registers and 2 % (8 x 16
// heads, N = 1024: 55.9 -> 57.3 us), so the lengths that have none keep their own.  Against one tile's bytes requested two
// tiles ahead, which is what other lengths had before: 8 x 16 heads, bf16, N = 1000: 61.3 -> 59.0 us, 960: 57.1 -> 55.0; 4 x 16,
// N = 2000: 109 -> 105; D = 32, 16 x 16, N = 1000: 90.6 -> 86.3; up to 500 keys the same.
// SPLIT: for grids that leave most of the chip idle.  The four wavefronts of a work-group share 32 query
// rows and take every fourth key tile each, with a K and a V buffer of their own: no barriers, four times
// the work-groups, a quarter of the serial chain; what they found is combined through LDS at the end.
// K of the next tile is requested when the scores of this one are formed, V when its products are.
// Measured, D = 64, packed mask: 1 x 4 heads, N = 4096: 55 -> 31 us, 1 x 1: 55 -> 23 us; 2 x 8, N = 1024: 16.6
// -> 11.1 us; 4 x 8, N = 512: 10.1 -> 7.9 us.  A wavefront now copies 16 KB per tile instead of 4, and a tile takes
// 1.4 times as long.
template <bool BF16, bool POSTMUL, bool PACKED_ROWS, int HDIM, bool BYTEMASK = false, bool BYPRODUCTS = false,
          int FETCH = 0, bool SPLIT = false, bool WIDE_Q = false, bool HALVES = false>
__global__ __launch_bounds__(NTHREADS, SPLIT ? (HDIM > 64 ? 1 : 2) : HDIM > 64 ? (three_on_a_cu(HDIM, BYTEMASK, BYPRODUCTS, WIDE_Q) ? 3 : 2) : 3) void attn_fwd_kernel(const AttnArgs a)
{
    // HALVES: a work-group of 64 rows, two wavefronts to each 32 of them, which take 32 keys of every tile each and add their
    // sums at the end.  A visit's chain of products, exponentials and products is half as long, which is what bounds a grid whose work-groups of 128
    // rows are one or two to a CU.  Forward, before -> now, D = 128: 7 heads, N = 2048 46.1 -> 36.1 us (packed 42.5 -> 32.0); 16,
    // N = 1024 25.7 -> 21.0; 32, N = 512 15.6 -> 13.6; 32, N = 263 11.6 -> 10.7; D = 80: 5 heads, N = 3000 62.3 -> 52.3; 64, N = 192 8.7 -> 8.2.
    // D = 64: 24 heads, N = 2048 43.4 -> 35.1 us (packed 40.5 -> 32.8), 40, N = 1024 23.8 -> 19.3 (22.2 -> 17.7), 48, N = 990
    // 26.4 -> 21.6; on masks that nothing has touched before 45.2 -> 42.0, 25.5 -> 22.7, 28.9 -> 26.0.
    // The mask's bytes with HALVES: at head dims up to 64 always those of two tiles at once (FETCH != 0): each of the two wavefronts copies 16 of the 32
    // rows for both, into one of two slots, two visits before the first of them is looked at.  32 bytes of a row, what a wavefront needs
    // of a tile, copied by each for itself one or two visits ahead: on untouched masks 48 heads, N = 990 28.9 -> 30.4 us instead of 26.0.
    static_assert(!HALVES || (!SPLIT && (!BYTEMASK || (HDIM <= 64) == (FETCH != 0))), "HALVES: pairs of tiles up to head dim 64");
    static_assert(FETCH == 0 || (BYTEMASK && HDIM <= 64 && !SPLIT), "PAIRS: byte mask, two byte slots");
    constexpr bool PAIRS = FETCH != 0, WHOLE = FETCH == 1;
    // only the 32 keys of a tile that the wavefront takes: half the bytes to read from LDS and, without PAIRS, one copy instead of two.  (The
    // by-products are made of whole tiles.)
    constexpr bool HALF_BYTES = HALVES && BYTEMASK && !BYPRODUCTS;
    using E = Elem<BF16>;
    constexpr int NH = HDIM > 64 ? 2 : 1;         // 64-column tiles per matrix
    constexpr int KS = (HDIM + 31) / 32;          // MFMA steps of the QK^T chain
    constexpr int DB = HDIM / 16;                 // 16-column accumulator blocks of O
    constexpr bool THIRD = !SPLIT && !HALVES && three_on_a_cu(HDIM, BYTEMASK, BYPRODUCTS, WIDE_Q);
    constexpr int AHEAD = SPLIT ? 4 : HDIM <= 64 || THIRD ? 2 : 3;              // steps by which an operand is requested before its use: scores
    constexpr int V_AHEAD = SPLIT ? DB * 2 < 8 ? DB * 2 : 8 : HDIM <= 64 || THIRD ? 4 : 6;             // ... and values, when the scores' registers are free
    // second column half at a constant distance from the first in every row
    constexpr bool SAME_HALVES = HDIM == 128 && PACKED_ROWS;
    constexpr int SECOND = second_row(HDIM, SPLIT, BYPRODUCTS, WIDE_Q);
    constexpr bool NARROW = SECOND == 32 || SECOND == 64;
    using C = Cfg<NH, BYTEMASK, SPLIT, SECOND>;
    constexpr int FIRST = C::FIRST, SHORT_CHUNK = FIRST != 0 ? 8 : 0;        // (NARROW: where the short rows begin in LDS, and their first 16-byte chunk)
    constexpr int NSTAGE = C::NSTAGE, STAGE_BYTES = C::STAGE_BYTES, OFF_MASK = C::OFF_MASK;
    constexpr int MASK_SLOT = C::MASK_SLOT, COPIES = C::COPIES - (HALF_BYTES ? 1 : 0);
    const int D = PACKED_ROWS ? HDIM : a.D;
    const int last_chunk = (D >> 3) - 1;          // 16-byte chunks per global row, minus one
    __shared__ __attribute__((aligned(1024))) unsigned char smem[C::LDS_BYTES];
    const uint32_t lut_addr = (uint32_t)(uintptr_t)(LDS_PTR(unsigned char))smem, lds0 = lut_addr + C::LUT_BYTES;

    const int tid = threadIdx.x;
    const int lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int l32 = lane & 31, hh = lane >> 5;       // mask: a row and a half of its words
    const int l16 = lane & 15, q4 = lane >> 4;       // products: rows l16 and 16 + l16

    const int nid = SPLIT ? renumber_block() : renumber_block((int)blockIdx.x, a.groups);     // (SPLIT: 6.50 -> 6.37 us on 8 heads, N = 333, D = 32)
    // last rows first: where rows keep more keys the later they come (causal masks), the longest
    // work-groups of a head (of several heads: see make_deal) start first and the shortest fill the end of the launch
    int bh, qt;
    if constexpr (BYTEMASK) {
        bh = (int)fastdiv((uint32_t)nid, a.deal.div_groups);
        qt = a.qtiles - 1 - (nid - bh * a.qtiles);
    } else {
        const Dealt d = deal(a.deal, a.qtiles, nid);
        bh = d.head;
        qt = a.qtiles - 1 - d.tile;
    }
    const int half = HALVES ? wave >> 1 : 0;                             // which 32 keys of every tile
    const int row_base = SPLIT ? qt * 32 : HALVES ? qt * 64 + (wave & 1) * 32 : qt * BM + wave * 32;     // this wavefront's 32 query rows
    const int N = a.N, nw = (N + 31) >> 5;
    const int T = (N + BN - 1) / BN;
    const bool ragged = (N & (BN - 1)) != 0;
    const int cut_tile = ragged ? T - 1 : -1;                            // the tile that the keys end in
    const int odd_tile = (nw & 1) ? T - 1 : -1;                          // the tile of which there is one word: it is read twice
    const float pm = POSTMUL ? a.post_mul : 1.0f;

    const int bi = (int)fastdiv((uint32_t)bh, a.div_H), hi = bh - bi * a.H;
    // ---- tile map: which key tiles hold a set mask bit for this work-group's rows ("live"; the map
    // also says which hold nothing else, which this kernel does not use).  The map has one row of
    // bits (one per key tile, 32 per word) for every block of 64 query rows: this work-group ORs
    // the rows of its two blocks.  The first words are requested here with scalar loads and awaited
    // just before the first copies are issued; the address arithmetic in between covers the latency.
    const int TW = (T + 31) >> 5;
    const uint32_t *mapw = nullptr, *mapw2 = nullptr;       // the two 64-row blocks (the same one if the second does not exist)
    if constexpr (!BYTEMASK) {
        if (a.tile_map != nullptr) {
            mapw = a.tile_map + bi * a.map_sb + hi * a.map_sh + (size_t)(SPLIT ? qt >> 1 : HALVES ? qt : 2 * qt) * 2 * TW;
            mapw2 = (!SPLIT && !HALVES && 2 * qt + 1 < T) ? mapw + 2 * TW : mapw;
        }
    }
    // The first map words are read here, with ordinary (scalar) loads, long before they are needed:
    // the address arithmetic below covers their latency.
    // (Without a map they read the first word of q, which exists, and the result is dropped: no
    // branch, so the loads stay where they are written.  The words are combined only where the walk
    // starts; the compiler puts its wait there.)
    const bool has_map = mapw != nullptr;
    const uint32_t *mapa = has_map ? mapw : reinterpret_cast<const uint32_t *>(a.q.p);
    const uint32_t *mapb = has_map ? mapw2 : reinterpret_cast<const uint32_t *>(a.q.p);
    const uint32_t first_w = mapa[0], first_w2 = mapb[0];
    const uint16_t *qb = slab(a.q, bi, hi);
    const uint16_t *kb = slab(a.k, bi, hi);
    const uint16_t *vb = slab(a.v, bi, hi);
    // packed: words, strides in words; BYTEMASK: bytes, strides in bytes
    const uint32_t *mb = BYTEMASK ? reinterpret_cast<const uint32_t *>(reinterpret_cast<const uint8_t *>(a.mask.p) +
                                                                       bi * a.mask.sb + hi * a.mask.sh)
                                  : slab(a.mask, bi, hi);
    const uint32_t q_sn = PACKED_ROWS ? D : a.q.sn, k_sn = PACKED_ROWS ? D : a.k.sn;       // row strides, elements
    const uint32_t v_sn = PACKED_ROWS ? D : a.v.sn;
    const uint32_t q_rb = 2u * q_sn, k_rb = 2u * k_sn, v_rb = 2u * v_sn;                   // row pitch, bytes

    // ---- mask words: wave-private async copies, slot = tile % NSTAGE, lane i -> (row i/2, word i%2) ----
    // BYTEMASK (N >= 16): the wave's 32 x 64 bytes of a tile as two copies of 16 rows; lane i
    // fills (row 16j + i/4, position i%4) with the global 16-byte chunk position ^ ((row >> 2) & 3),
    // which makes the reads below (lane = row, two chunks each) free of bank conflicts.  The copies
    // take any byte address (rows of N bytes start anywhere; ROCm runs the memory pipeline in its
    // unaligned access mode, in which a 16-byte copy may start at any byte).  In a last tile of fewer than 64 keys
    // every chunk that would reach beyond the row's end is read from the 16 bytes before that end
    // instead, so that nothing after the mask's last byte is touched; the bits of the chunk that
    // holds the end are shifted to their places below, those of later chunks cleared as pad bits.
    const int mrow = BYTEMASK ? 0 : row_base + (lane >> 1);
    uint32_t m_voff = BYTEMASK ? 0u : (uint32_t)(((size_t)(mrow < N ? mrow : N - 1) * nw + (lane & 1)) * 4);
    uint32_t mb_voff[2] = {0u, 0u};
    auto mb_chunk = [&](int l) __attribute__((always_inline)) -> uint32_t {
        return HALF_BYTES ? 32 * half + (((l & 1) ^ ((l >> 4) & 1)) << 4) : ((l & 3) ^ ((l >> 4) & 3)) << 4;
    };
    if constexpr (BYTEMASK) {
#pragma unroll
        for (int j = 0; j < 2; ++j) {
            // (HALF_BYTES: row i/2, position i%2, of the wavefront's two chunks the one at position ^ ((row >> 3) & 1))
            const int row = HALF_BYTES ? lane >> 1 : 16 * j + (lane >> 2);
            const int grow = row_base + row;
            mb_voff[j] = (uint32_t)(grow < N ? grow : N - 1) * (uint32_t)N + mb_chunk(lane);
        }
    }
    const uint32_t mask_dst = lds0 + wave * (BYTEMASK ? 2048 : 256);
    auto issue_mask = [&](int x, auto slot_c) __attribute__((always_inline)) {
        constexpr int SLOT = decltype(slot_c)::value;
        if constexpr (BYTEMASK) {
            const uint8_t *src = reinterpret_cast<const uint8_t *>(mb) + (uint32_t)x * (uint32_t)BN;
            // a single slot is refilled: this wave's reads of the previous tile's bytes must be over
            if constexpr (C::BYTE_SLOTS == 1) asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
            if (UNLIKELY(x == cut_tile)) {        // (no tile follows it)
                const uint32_t row_end = (uint32_t)(N - x * BN);       // bytes of the row left in this tile
                // the lane offsets are unsigned: what is taken from them below is first taken from the
                // base (a tile that is not the first has 64 bytes of the row before it; in the first,
                // row_end = N >= 16 and nothing goes below zero)
                const uint32_t back = x > 0 ? 16u : 0u;
                src -= back;
                int l = lane;
                if constexpr (NARROW) asm volatile("" : "+v"(l));      // opaque: no register across the loop for what follows from it
                const uint32_t end = mb_chunk(l) + 16;
#pragma unroll
                for (int j = 0; j < 2; ++j) {
                    mb_voff[j] += back;
                    if (end > row_end) mb_voff[j] -= end - row_end;
                }
            }
            async_copy_b128_at<OFF_MASK + SLOT * MASK_SLOT>(mask_dst, src, mb_voff[0]);
            if constexpr (!HALF_BYTES) async_copy_b128_at<OFF_MASK + SLOT * MASK_SLOT + 1024>(mask_dst, src, mb_voff[1]);
        } else {
            if (UNLIKELY(x == odd_tile)) m_voff -= (lane & 1) * 4;      // the last tile: none follows it
            async_copy_b32_at<OFF_MASK + SLOT * MASK_SLOT>(mask_dst, mb + 2u * (uint32_t)x, m_voff);
        }
    };
    // PAIRS: four copies per wave and pair of tiles; lane i of copy j fills (row 8j + i/8, position i%8)
    // from the row's chunk (i%8) ^ ((row >> 1) & 7).  (row >> 1) & 7 is (i/8 >> 1) for j = 0, 2 and that
    // plus 4 for j = 1, 3.  In a pair that the row ends in, chunks move back as in issue_mask.
    uint32_t pair_voff = 0u;
    if constexpr (PAIRS) pair_voff = (uint32_t)(row_base + (lane >> 3)) * (uint32_t)N + (uint32_t)(((lane & 7) ^ (lane >> 4)) << 4);
    auto issue_mask_pair = [&](int p) __attribute__((always_inline)) {      // bytes of tiles 2p and 2p + 1
        const uint8_t *src = reinterpret_cast<const uint8_t *>(mb) + (size_t)p * (2 * BN);
        // HALVES: the two wavefronts of 32 rows copy 16 of them each, for both, into one of two slots
        const uint32_t dst = HALVES ? lds0 + (p & 1) * 8192 + (wave & 1) * 4096 + half * 2048 : lds0 + wave * 4096;
        if constexpr (WHOLE && HALVES) {
            src += (size_t)(16 * half) * N;
            async_copy_b128_at<OFF_MASK>(dst, src, pair_voff);
            async_copy_b128_at<OFF_MASK + 1024>(dst, src + (size_t)8 * N, pair_voff ^ 64u);
            return;
        }
        if constexpr (WHOLE) {                   // the low seven bits of the lane offset are the chunk alone
            async_copy_b128_at<OFF_MASK>(dst, src, pair_voff);
            async_copy_b128_at<OFF_MASK + 1024>(dst, src + (size_t)8 * N, pair_voff ^ 64u);
            async_copy_b128_at<OFF_MASK + 2048>(dst, src + (size_t)16 * N, pair_voff);
            async_copy_b128_at<OFF_MASK + 3072>(dst, src + (size_t)24 * N, pair_voff ^ 64u);
            return;
        }
        int ln = lane;
        asm volatile("" : "+v"(ln));             // opaque: what follows from it is made anew each time instead of kept in registers
        const uint32_t chunk = (uint32_t)(((ln & 7) ^ (ln >> 4)) << 4);
        uint32_t vo[4] = {pair_voff, pair_voff + 64u - 2u * (chunk & 64u), 0u, 0u};
        vo[2] = vo[0];
        vo[3] = vo[1];
        size_t step = (size_t)8 * N;                                         // eight rows
        if (row_base + 32 > N) {                                             // rows beyond N: copy row N - 1 instead
            step = 0;
#pragma unroll
            for (int j = 0; j < 4; ++j) {
                const int grow = row_base + 8 * j + (ln >> 3);
                vo[j] = (uint32_t)(grow < N ? grow : N - 1) * (uint32_t)N + (chunk ^ (64u * (j & 1)));
            }
        }
        const uint32_t row_end = (uint32_t)(N - p * (2 * BN));               // bytes of the row left
        if (row_end < 2u * BN) {
            const uint32_t back = p > 0 ? 16u : 0u;
            src -= back;
#pragma unroll
            for (int j = 0; j < 4; ++j) {
                const uint32_t end = (chunk ^ (64u * (j & 1))) + 16u;
                vo[j] += back;
                if (end > row_end) vo[j] -= end - row_end;
            }
        }
        if constexpr (HALVES) {
            src += 2 * half * step;
            async_copy_b128_at<OFF_MASK>(dst, src, half ? vo[2] : vo[0]);
            async_copy_b128_at<OFF_MASK + 1024>(dst, src + step, half ? vo[3] : vo[1]);
            return;
        }
        async_copy_b128_at<OFF_MASK>(dst, src, vo[0]);
        async_copy_b128_at<OFF_MASK + 1024>(dst, src + step, vo[1]);
        async_copy_b128_at<OFF_MASK + 2048>(dst, src + 2 * step, vo[2]);
        async_copy_b128_at<OFF_MASK + 3072>(dst, src + 3 * step, vo[3]);
    };
    // BYTEMASK: where this lane's row of packed words goes, if the caller wants them ([Bm, Hm, N, nw]
    // like the mask; a mask shared between batch entries / heads is written by the first of them)
    const int qrow = row_base + l32;
    uint32_t *words_out = nullptr;
    // ... and where the tile map of this work-group's two blocks of 64 rows goes ([Bm, Hm, T, 2, TW]).
    // Each wavefront notes per key tile whether its 32 rows hold a set bit and whether they hold a
    // clear one, 32 tiles to a pair of registers that goes to LDS when it is full.  After
    // its last tile a wavefront counts itself in; the second of a block's two to do so combines
    // both and writes the block's words, which then travel while the output is being stored.
    // (Per-lane bits ORed into LDS by all lanes at once, instead of the two ballots per tile,
    // measured 4 us slower on the headline workload: 64 atomics on one address.)
    uint32_t *map_dst = nullptr;
    uint32_t some_acc = 0u, hole_acc = 0u;
    u32x4 pend = {0u, 0u, 0u, 0u};        // packed words waiting to be stored, see mask_words
    if constexpr (BYPRODUCTS) {
        const bool writer = (a.mask.sb != 0 || bi == 0) && (a.mask.sh != 0 || hi == 0) && half == 0;
        const int Hm = a.mask.sh != 0 ? a.H : 1;
        const size_t slab_m = (size_t)((a.mask.sb != 0 ? bi : 0) * Hm + (a.mask.sh != 0 ? hi : 0));
        if (a.mask_out != nullptr && writer) words_out = a.mask_out + (slab_m * N + (qrow < N ? qrow : 0)) * nw;
        if (a.map_out != nullptr && writer) map_dst = a.map_out + (slab_m * T + (SPLIT ? qt >> 1 : HALVES ? qt : 2 * qt)) * 2 * TW;
    }
    const uint32_t map_lds = lds0 + C::OFF_MAP + wave * (C::MAP_WORDS * 8);
    if constexpr (BYPRODUCTS && !SPLIT) {     // ordered before any arrival by the barriers of the main loop (T >= 1)
        if (tid < 2) *(LDS_PTR(uint32_t))(uintptr_t)(lds0 + C::OFF_MAP_ARRIVED + 4 * tid) = 0u;
    }
    const uint32_t maddr = BYTEMASK ? lds0 + OFF_MASK + wave * 2048 + l32 * 64 : lds0 + OFF_MASK + wave * 256 + l32 * 8;
    const int msw = (l32 >> 2) & 3;
    // PAIRS: a wave's bytes of a pair of tiles are 32 rows of 128 bytes in the 4 KiB that its two byte
    // slots occupy otherwise; the 16-byte chunks of a row are swizzled like K's (position ^ ((row >> 1)
    // & 7), applied on the global side), which keeps the reads below free of bank conflicts.
    // `pair_half` (0 or 1) says which tile of the pair; -1: the ordinary slots.
    const uint32_t pair_base = lds0 + OFF_MASK + (HALVES ? wave & 1 : wave) * 4096 + l32 * 128;
    const int psw = (l32 >> 1) & 7;
    auto mask_words = [&](int x, int slot, int pair_half = -1) __attribute__((always_inline)) -> u32x2 {
        u32x2 w;
        // a byte counts as "attend" when it is non-zero, as in the packer: nz() leaves 0x80 in
        // every non-zero byte, the dot products weigh those with 1, 2, 4 .. 128 (times 128)
        auto nz = [](uint32_t x) -> uint32_t { return (((x & 0x7f7f7f7fu) + 0x7f7f7f7fu) | x) & 0x80808080u; };
        if constexpr (HALF_BYTES) {
            // this lane: 16 bytes of row l32, keys 32 half + 16hh .. + 15
            const u32x4 d = lds_read_b128(PAIRS ? pair_base + slot * 8192 + (((4 * pair_half + 2 * half + hh) ^ psw) << 4)
                                                : mask_dst + OFF_MASK + slot * MASK_SLOT + l32 * 32 + ((hh ^ ((l32 >> 3) & 1)) << 4));
            uint32_t mine;
            if (LIKELY(__builtin_amdgcn_ballot_w64(((d.x | d.y | d.z | d.w) & 0xfefefefeu) != 0u) == 0ull)) {
                uint32_t b0 = __builtin_amdgcn_udot4(d.x, 0x08040201u, 0u, false);
                uint32_t b1 = __builtin_amdgcn_udot4(d.z, 0x08040201u, 0u, false);
                b0 = __builtin_amdgcn_udot4(d.y, 0x80402010u, b0, false);
                b1 = __builtin_amdgcn_udot4(d.w, 0x80402010u, b1, false);
                mine = b0 | (b1 << 8);
            } else {
                uint32_t b0 = __builtin_amdgcn_udot4(nz(d.x), 0x08040201u, 0u, false);
                uint32_t b1 = __builtin_amdgcn_udot4(nz(d.z), 0x08040201u, 0u, false);
                b0 = __builtin_amdgcn_udot4(nz(d.y), 0x80402010u, b0, false);
                b1 = __builtin_amdgcn_udot4(nz(d.w), 0x80402010u, b1, false);
                mine = (b0 >> 7) | (b1 << 1);                        // each partial value is 128 x (8 bits): bits 7..14
            }
            const int row_end = N - x * BN;
            if (UNLIKELY(x == cut_tile) && (row_end >> 4) == 2 * half + hh) mine >>= (16 - (row_end & 15)) & 15;     // see below
            const auto r = __builtin_amdgcn_permlane32_swap(mine, mine, false, false);
            w.x = (uint32_t)r[0] | ((uint32_t)r[1] << 16);
            if (UNLIKELY(x == cut_tile)) w.x &= half ? a.last_mask1 : a.last_mask0;
            w.y = w.x;
        } else if constexpr (BYTEMASK) {
            // this lane: the 32 bytes of row l32 for keys 32hh .. 32hh+31 -> one word
            const uint32_t a0 = !PAIRS || pair_half < 0 ? maddr + slot * MASK_SLOT + (((2 * hh) ^ msw) << 4)
                                                        : pair_base + (HALVES ? slot * 8192 : 0) + (((4 * pair_half + 2 * hh) ^ psw) << 4);
            const uint32_t a1 = !PAIRS || pair_half < 0 ? maddr + slot * MASK_SLOT + (((2 * hh + 1) ^ msw) << 4)
                                                        : pair_base + (HALVES ? slot * 8192 : 0) + (((4 * pair_half + 2 * hh + 1) ^ psw) << 4);
            const u32x4 d0 = lds_read_b128(a0);
            const u32x4 d1 = lds_read_b128(a1);
            // nz() costs three instructions per four bytes.  Bytes that are all 0 or 1 (every
            // mask PyTorch itself made) need none of it: one look at the wavefront's 2 KiB decides.
            const uint32_t other = (d0.x | d0.y | d0.z | d0.w | d1.x | d1.y | d1.z | d1.w) & 0xfefefefeu;
            uint32_t mine;
            if (LIKELY(__builtin_amdgcn_ballot_w64(other != 0u) == 0ull)) {
                uint32_t b0 = __builtin_amdgcn_udot4(d0.x, 0x08040201u, 0u, false);
                uint32_t b1 = __builtin_amdgcn_udot4(d0.z, 0x08040201u, 0u, false);
                uint32_t b2 = __builtin_amdgcn_udot4(d1.x, 0x08040201u, 0u, false);
                uint32_t b3 = __builtin_amdgcn_udot4(d1.z, 0x08040201u, 0u, false);
                b0 = __builtin_amdgcn_udot4(d0.y, 0x80402010u, b0, false);
                b1 = __builtin_amdgcn_udot4(d0.w, 0x80402010u, b1, false);
                b2 = __builtin_amdgcn_udot4(d1.y, 0x80402010u, b2, false);
                b3 = __builtin_amdgcn_udot4(d1.w, 0x80402010u, b3, false);
                mine = b0 | (b1 << 8) | (b2 << 16) | (b3 << 24);
            } else {
                uint32_t b0 = __builtin_amdgcn_udot4(nz(d0.x), 0x08040201u, 0u, false);
                uint32_t b1 = __builtin_amdgcn_udot4(nz(d0.z), 0x08040201u, 0u, false);
                uint32_t b2 = __builtin_amdgcn_udot4(nz(d1.x), 0x08040201u, 0u, false);
                uint32_t b3 = __builtin_amdgcn_udot4(nz(d1.z), 0x08040201u, 0u, false);
                b0 = __builtin_amdgcn_udot4(nz(d0.y), 0x80402010u, b0, false);
                b1 = __builtin_amdgcn_udot4(nz(d0.w), 0x80402010u, b1, false);
                b2 = __builtin_amdgcn_udot4(nz(d1.y), 0x80402010u, b2, false);
                b3 = __builtin_amdgcn_udot4(nz(d1.w), 0x80402010u, b3, false);
                // each partial value is 128 x (8 bits): bits 7..14
                mine = (b0 >> 7) | (b1 << 1) | (b2 << 9) | (b3 << 17);
            }
            if (UNLIKELY(x == cut_tile)) {
                // the chunk that holds the row's end was copied from 16 bytes before that end: its
                // bits move down to their places (zeros follow them)
                const int row_end = N - x * BN, part = row_end >> 4, shift = (16 - (row_end & 15)) & 15;
                const uint32_t lo = (mine & 0xffffu) >> (part == 2 * hh ? shift : 0);
                const uint32_t hi = (mine >> 16) >> (part == 2 * hh + 1 ? shift : 0);
                mine = (lo | (hi << 16)) & (hh ? a.last_mask1 : a.last_mask0);       // bits of keys >= N
            }
            if (BYPRODUCTS && map_dst != nullptr) {
                // rows beyond N repeat row N - 1 and change nothing; key bits beyond N are not valid
                const uint32_t valid = x == T - 1 ? (hh ? a.last_mask1 : a.last_mask0) : 0xffffffffu;
                const uint32_t some = __builtin_amdgcn_ballot_w64(mine != 0u) != 0ull ? 1u : 0u;
                const uint32_t hole = __builtin_amdgcn_ballot_w64(mine != valid) != 0ull ? 1u : 0u;
                if constexpr (SPLIT) {
                    // the block's other 32 rows belong to another work-group: into the words at once, which were
                    // set to "nothing kept" and "everything kept" before the launch
                    if (lane == 0) {
                        if (some) atomicOr(map_dst + (x >> 5), 1u << (x & 31));
                        if (hole) atomicAnd(map_dst + TW + (x >> 5), ~(1u << (x & 31)));
                    }
                }
                some_acc |= some << (x & 31);
                hole_acc |= hole << (x & 31);
                if (SPLIT) {
                } else if ((x & 31) == 31 || x == T - 1) {
                    if (lane == 0) *(LDS_PTR(u32x2))(uintptr_t)(map_lds + (uint32_t)(x >> 5) * 8) = u32x2{some_acc, hole_acc};
                    some_acc = hole_acc = 0u;
                }
            }
            // lanes < 32 hold the word of keys 0..31, lanes >= 32 that of keys 32..63: both to both
            const auto r = __builtin_amdgcn_permlane32_swap(mine, mine, false, false);
            w.x = (uint32_t)r[0];
            w.y = (uint32_t)r[1];
            // A caller who will need the packed words (for the backward) gets them as a by-product.
            // Stored tile by tile they would leave as 4-byte pieces of 64 different rows; instead
            // the lower lane half keeps the words of tiles 4g and 4g + 1, the upper half those of
            // tiles 4g + 2 and 4g + 3, and after every fourth tile each lane stores 16 bytes: 32
            // consecutive bytes of each row per store instruction.
            if (SPLIT && BYPRODUCTS && words_out != nullptr && qrow < N && hh == 0) {
                words_out[2 * x] = w.x;
                if (2 * x + 1 < nw) words_out[2 * x + 1] = w.y;
            }
            if (!SPLIT && BYPRODUCTS && words_out != nullptr) {
                const int j = x & 3;
                const bool turn = hh == (j >> 1);
                if ((j & 1) == 0) {
                    pend.x = turn ? w.x : pend.x;
                    pend.y = turn ? w.y : pend.y;
                } else {
                    pend.z = turn ? w.x : pend.z;
                    pend.w = turn ? w.y : pend.w;
                }
                if (j == 3 || x == T - 1) {
                    // words of tiles beyond the last one have indices >= nw and stay unwritten
                    const int wb = 8 * (x >> 2) + 4 * hh;
                    if (qrow < N) {
                        typedef uint32_t u32x4_a4 __attribute__((ext_vector_type(4), aligned(4)));
                        if (wb + 3 < nw) {
                            __builtin_nontemporal_store((u32x4_a4)pend, reinterpret_cast<u32x4_a4 *>(words_out + wb));
                        } else {
                            if (wb < nw) words_out[wb] = pend.x;
                            if (wb + 1 < nw) words_out[wb + 1] = pend.y;
                            if (wb + 2 < nw) words_out[wb + 2] = pend.z;
                        }
                    }
                }
            }
        } else {
            w = lds_read_b64(maddr + slot * MASK_SLOT);
            if (UNLIKELY(x == cut_tile)) {
                w.x &= a.last_mask0;
                w.y &= a.last_mask1;
            }
        }
        return w;
    };
    auto narrow_swizzle = [](int row) __attribute__((always_inline)) { return (0x1320 >> (4 * ((row >> 2) & 3))) & 3; };      // 0, 2, 3, 1
    // ---- K/V tiles: async copies --------------------------------------------------------------
    // One global_load_lds_dwordx4 fills 1 KiB = 8 tile rows.  Wave w copies row blocks 2w, 2w+1 of
    // K and of V.  Lane i fills LDS chunk (row = 8*blk + i/8, position i%8) with the global chunk
    // position ^ swz(row):   K: swz(row) = (row >> 1) & 7      V: swz(row) = bitrev3((row >> 1) & 7)
    // (a chunk beyond the row's last is read as that one)
    auto chunk_at = [&](int c) __attribute__((always_inline)) -> uint32_t { return (uint32_t)(c < last_chunk ? c : last_chunk) << 4; };
    // NARROW (short rows in the second half): the second halves' tiles, K then V, as one series of pieces of 1 KiB (lane i: row i / 2 or i / 4 of it); at 64 bytes a row wave w copies piece w of
    // either, at 32 piece w of the four.  Their swizzle, K and V alike, is narrow_swizzle: none at 32 bytes.
    uint32_t kv_voff[2][2], kv_voff2[2][2];       // first and second column half
    auto row2_of = [&](int l) __attribute__((always_inline)) { return SECOND == 32 ? 32 * (wave & 1) + (l >> 1) : 16 * wave + (l >> 2); };      // the tile row of a lane's piece
#pragma unroll
    for (int j = 0; j < 2; ++j) {
        const int row = 8 * (SPLIT ? j : 2 * wave + j) + (lane >> 3);       // SPLIT: the wave copies rows 16i + these too
        const int pos = lane & 7;
        const int f = (row >> 1) & 7;
        const int fr = bitrev3(f);
        // row pitches are below 2^24 bytes (checked by the C-ABI layer): full-rate 24-bit multiplies
        kv_voff[0][j] = __umul24(row, k_rb) + chunk_at(pos ^ f);
        kv_voff[1][j] = __umul24(row, v_rb) + chunk_at(pos ^ fr);
        kv_voff2[0][j] = SAME_HALVES ? kv_voff[0][j] + 2 * HD : __umul24(row, k_rb) + chunk_at(8 + (pos ^ f));
        kv_voff2[1][j] = SAME_HALVES ? kv_voff[1][j] + 2 * HD : __umul24(row, v_rb) + chunk_at(8 + (pos ^ fr));
    }
    const bool takes_v2 = SECOND == 32 && wave >= 2;
    const uint32_t rb2 = takes_v2 ? v_rb : k_rb;
    if constexpr (NARROW) {
        const int row2 = row2_of(lane);
        const uint32_t c = chunk_at(SHORT_CHUNK + (SECOND == 32 ? lane & 1 : (lane & 3) ^ narrow_swizzle(row2)));
        kv_voff2[0][0] = __umul24(row2, rb2) + c;
        kv_voff2[1][0] = __umul24(row2, v_rb) + c;
    }
    const uint32_t kv_dst2 = lds0 + FIRST + (SECOND == 32 ? (takes_v2 ? C::OFF_V : 0) + (wave & 1) * 1024 : wave * 1024);
    const uint32_t kv_dst = lds0 + wave * 2048;
    auto issue_kv = [&](int t, auto stage_c) __attribute__((always_inline)) {
        constexpr int SO = decltype(stage_c)::value * STAGE_BYTES;
        const int key0 = t * BN;
        const uint16_t *ksrc = reinterpret_cast<const uint16_t *>(reinterpret_cast<const char *>(kb) + (uint32_t)key0 * k_rb);
        const uint16_t *vsrc = reinterpret_cast<const uint16_t *>(reinterpret_cast<const char *>(vb) + (uint32_t)key0 * v_rb);
        if (UNLIKELY(t == cut_tile)) {        // rows beyond N: copy row N-1 instead (zeroed later); no tile follows this one
            int last0 = key0;
            asm volatile("" : "+s"(last0));   // opaque: keeps this once-only arithmetic out of the loop's registers
            int l = lane;
            if constexpr (NARROW) asm volatile("" : "+v"(l));
#pragma unroll
            for (int j = 0; j < 2; ++j) {
                const int row = 8 * (2 * wave + j) + (l >> 3);
                const int over = last0 + row - (N - 1);
                if (over > 0) {
                    kv_voff[0][j] -= __umul24(over, k_rb); kv_voff[1][j] -= __umul24(over, v_rb);
                    if constexpr (!NARROW) { kv_voff2[0][j] -= __umul24(over, k_rb); kv_voff2[1][j] -= __umul24(over, v_rb); }
                }
            }
            if constexpr (NARROW) {
                const int over = last0 + row2_of(l) - (N - 1);
                if (over > 0) {
                    kv_voff2[0][0] -= __umul24(over, rb2);
                    kv_voff2[1][0] -= __umul24(over, v_rb);
                }
            }
        }
        // The two pieces of a row follow each other: its end and the next row's begin share lines, which two tiles a work-group are too short-lived to
        // find in the cache again.  K and V first, then their ends (and q likewise) -> this, us, at head dim 96, where rows all whole were the faster on
        // two tiles: inputs from memory, packed, 1024 heads, N = 104 20.9 -> 20.2 (whole 20.2), 384, N = 112 9.10 -> 8.88 (8.85);  boolean 384, N = 96
        // 9.44 -> 9.09 (9.16), 2048, N = 127 48.3 -> 48.1 (47.9), 256, N = 512 43.1 -> 42.4 (43.9).
        if constexpr (FIRST != 0) async_copy2_b128_at<SO, SO + 1024>(kv_dst, ksrc, kv_voff[0][0], kv_voff[0][1]);
        if constexpr (SAME_HALVES) {          // 128 bytes further along each row
            async_copy2_b128_at<SO + TILE_BYTES, SO + TILE_BYTES + 1024>(kv_dst, ksrc + HD, kv_voff[0][0], kv_voff[0][1]);
        } else if constexpr (SECOND == 64) {
            async_copy_b128_at<SO>(kv_dst2, ksrc, kv_voff2[0][0]);
        } else if constexpr (NH == 2 && !NARROW) {
            async_copy2_b128_at<SO + TILE_BYTES, SO + TILE_BYTES + 1024>(kv_dst, ksrc, kv_voff2[0][0], kv_voff2[0][1]);
        }
        if constexpr (FIRST != 0) async_copy2_b128_at<SO + C::OFF_V, SO + C::OFF_V + 1024>(kv_dst, vsrc, kv_voff[1][0], kv_voff[1][1]);
        if constexpr (SAME_HALVES) {
            async_copy2_b128_at<SO + C::OFF_V + TILE_BYTES, SO + C::OFF_V + TILE_BYTES + 1024>(kv_dst, vsrc + HD, kv_voff[1][0], kv_voff[1][1]);
        } else if constexpr (SECOND == 64) {
            async_copy_b128_at<SO + C::OFF_V>(kv_dst2, vsrc, kv_voff2[1][0]);
        } else if constexpr (SECOND == 32) {
            async_copy_b128_at<SO>(kv_dst2, takes_v2 ? vsrc : ksrc, kv_voff2[0][0]);
        } else if constexpr (NH == 2) {
            async_copy2_b128_at<SO + C::OFF_V + TILE_BYTES, SO + C::OFF_V + TILE_BYTES + 1024>(kv_dst, vsrc, kv_voff2[1][0], kv_voff2[1][1]);
        }
    };
    // SPLIT: all 64 rows of one matrix by one wavefront, 16 rows (two copies) at a time; the swizzles repeat
    // every 16 rows
    const uint32_t split_dst = lds0 + wave * STAGE_BYTES;
    auto issue_own = [&](int t, const uint16_t *mat, uint32_t sn, uint32_t rb, const uint32_t (&off)[2], const uint32_t (&off2)[2],
                         auto at_c) __attribute__((always_inline)) {
        constexpr int AT = decltype(at_c)::value;
        const int key0 = t * BN;
        const uint16_t *src = mat + (size_t)key0 * sn;
        const bool cut = t == cut_tile;
        auto group = [&](auto i_c) __attribute__((always_inline)) {
            constexpr int I = decltype(i_c)::value;
            uint32_t o[2] = {off[0], off[1]}, o2[2] = {off2[0], off2[1]};
            if (cut) {                        // rows beyond N: copy row N-1 instead (zeroed later)
#pragma unroll
                for (int j = 0; j < 2; ++j) {
                    const int r = 8 * j + (lane >> 3), over = key0 + 16 * I + r - (N - 1);
                    // what goes down by more than the lane's own rows is taken from the base's below
                    const uint32_t up = over > 0 ? __umul24(over, rb) : 0u;
                    o[j] += __umul24(16 * I, rb) - up;
                    o2[j] += __umul24(16 * I, rb) - up;
                }
            }
            const uint16_t *p = cut ? src : src + (size_t)(16 * I) * sn;
            async_copy_b128_at<AT + 2048 * I>(split_dst, p, o[0]);
            async_copy_b128_at<AT + 2048 * I + 1024>(split_dst, p, o[1]);
            if constexpr (NH == 2) {
                async_copy_b128_at<AT + TILE_BYTES + 2048 * I>(split_dst, p, o2[0]);
                async_copy_b128_at<AT + TILE_BYTES + 2048 * I + 1024>(split_dst, p, o2[1]);
            }
        };
        group(std::integral_constant<int, 0>{});
        group(std::integral_constant<int, 1>{});
        group(std::integral_constant<int, 2>{});
        group(std::integral_constant<int, 3>{});
    };
    auto issue_own_k = [&](int t) __attribute__((always_inline)) { issue_own(t, kb, k_sn, k_rb, kv_voff[0], kv_voff2[0], std::integral_constant<int, 0>{}); };
    auto issue_own_v = [&](int t) __attribute__((always_inline)) { issue_own(t, vb, v_sn, v_rb, kv_voff[1], kv_voff2[1], std::integral_constant<int, C::OFF_V>{}); };
    auto zero_own_rows = [&](int t, int at) __attribute__((always_inline)) {
        for (int r = (lane >> 3); r < BN; r += 8)
            if (t * BN + r >= N)
#pragma unroll
                for (int half = 0; half < NH; ++half)
                    *(LDS_PTR(u32x4))(uintptr_t)(split_dst + at + half * TILE_BYTES + r * 128 + (lane & 7) * 16) = u32x4{0u, 0u, 0u, 0u};
    };
    auto zero_tail_rows = [&](int t, int stage) __attribute__((always_inline)) {   // after the copies of the last tile have landed
        const int key0 = t * BN;
        int l = lane;
        if constexpr (NARROW) asm volatile("" : "+v"(l));        // as in issue_kv
#pragma unroll
        for (int j = 0; j < 2; ++j) {
            const int row = 8 * (2 * wave + j) + (l >> 3);
            if (FIRST != 0 && key0 + row >= N) {
                const uint32_t p = lds0 + stage * STAGE_BYTES + wave * 2048 + j * 1024 + l * 16;
                const u32x4 z = {0u, 0u, 0u, 0u};
#pragma unroll
                for (int part = 0; part < (NARROW ? 2 : 2 * NH); ++part)
                    *(LDS_PTR(u32x4))(uintptr_t)(p + (NARROW ? part * C::OFF_V : part * TILE_BYTES)) = z;
            }
        }
        if constexpr (NARROW) {
            if (key0 + row2_of(l) >= N) {
                const uint32_t p = kv_dst2 + stage * STAGE_BYTES + l * 16;
                const u32x4 z = {0u, 0u, 0u, 0u};
                *(LDS_PTR(u32x4))(uintptr_t)p = z;
                if constexpr (SECOND == 64) *(LDS_PTR(u32x4))(uintptr_t)(p + C::OFF_V) = z;
            }
        }
    };

    // ---- per-lane LDS read addresses (stage 0, first column half, first columns); everything else flips bits or is an immediate offset ----
    // K operand (block of 16 keys kb, step c): row 16kb + l16, chunk 4c + q4           -> (k_at ^ 64 (c % 2)) + 2048kb
    // V operand (16 columns db, block of 32 keys), read by ds_read_b64_tr_b16: the lane supplies
    //   rows 16x + 4q4 + (l16 >> 2), columns 16db + 4(l16 & 3) .. +3, x = 0, 1                -> (v_at ^ 32 (db % 4)) + 2048x
    // NARROW, second column half: K's row and chunk at k2_at + SECOND (rows beyond), V's at v2_at, ^ 32: 16 columns further
    uint32_t k_at, v_at, k2_at = 0u, v2_at = 0u;
    {
        const uint32_t own0 = SPLIT ? split_dst : lds0;
        const int r = 4 * q4 + (l16 >> 2);
        k_at = own0 + l16 * 128 + ((q4 ^ (l16 >> 1)) << 4);
        v_at = own0 + C::OFF_V + r * 128 + ((((l16 & 3) >> 1) ^ bitrev3(r >> 1)) << 4) + ((l16 & 1) << 3);
        if constexpr (NARROW) {
            // (80: what the lanes of the last two chunks read meets zeros of q, as where rows are whole; it is the row's last chunk there too)
            const int chunk = SECOND == 32 ? (q4 < 1 ? q4 : 1) : q4 ^ narrow_swizzle(l16);
            k2_at = own0 + FIRST + l16 * SECOND + (chunk << 4);
            v2_at = own0 + C::OFF_V + FIRST + r * SECOND + ((((l16 & 3) >> 1) ^ (SECOND == 32 ? 0 : narrow_swizzle(r))) << 4) + ((l16 & 1) << 3);
        }
    }
    const uint32_t nib_rotate = (4u * q4 + 28u) & 31u;     // right: the nibble of keys 4q4 .. 4q4 + 3 comes to bits 4 .. 7
    uint32_t nib_mask = 0xF0u, ones = E::ONES;             // in scalar registers: as literals they take four bytes more wherever they are used
    asm volatile("" : "+s"(nib_mask), "+s"(ones));

    // ================================ prologue: one memory round trip ================================
    constexpr int Q_HALF = SPLIT ? 4096 : 16384;         // between the column halves of the staged q
    // Requested at once, oldest first: q (this wave's 32 rows, staged through the second K/V stage,
    // which the prologue leaves unused, K-swizzled), then K/V and the mask words of tile 0.
    // WIDE_Q (q in fp32): the same pieces through registers, rounded once the copies below are on their way.  q is read by one
    // work-group alone, so this replaces a pass over it: 6 bytes an element instead of 8 with the rounded q kept, 4 without.  Conversion and
    // forward, separate pass -> this: 192 heads, N = 512, D = 128: 75.8 -> 69.8 us, D = 64: 42.9 -> 39.8; with the rounded q kept 81.2 -> 79.8 and
    // 46.4 -> 44.8.  Where it does not pay stands at its callers' rule (forward_rounds_q in binding.cpp).  What it could give and does not: the
    // compiler's waits for these loads also wait for the copies issued after them, which it knows nothing of.  As an instance of its own: decided at
    // run time, the other element types' loops came out 0.5 to 1 % slower.
    const uint32_t q_dst = SPLIT ? split_dst + C::OFF_V : lds0 + (NSTAGE - 1) * STAGE_BYTES + wave * 4096;
    // NARROW: the second half of q behind the four wavefronts' first halves, SECOND bytes a row, in as many pieces
    constexpr int Q2_PIECES = NARROW ? SECOND / 32 : 0;
    const uint32_t q2_dst = lds0 + (NSTAGE - 1) * STAGE_BYTES + 2 * FIRST + wave * (32 * SECOND);
    auto q2_row = [&](int j) __attribute__((always_inline)) { return SECOND == 32 ? lane >> 1 : 16 * j + (lane >> 2); };
    auto q2_chunk = [&](int j) __attribute__((always_inline)) { return SHORT_CHUNK + (SECOND == 32 ? lane & 1 : (lane & 3) ^ narrow_swizzle(q2_row(j))); };
    f32x4 wide[WIDE_Q ? 4 * NH : 1][2], wide2[WIDE_Q && NARROW ? Q2_PIECES : 1][2];
    constexpr int Q_PARTS = FIRST == 0 ? 0 : NARROW ? 1 : NH;             // column halves in whole rows
    static_assert(!NARROW || 2 * FIRST + 128 * SECOND <= STAGE_BYTES, "q fits a stage");
    {
        const int qbase = row_base < N ? row_base : N - 1;   // wave-uniform
        const uint16_t *qsrc = qb + (size_t)qbase * q_sn;
        const int last = N - 1 - qbase;                      // rows beyond N re-read row N-1
        const uint32_t dst = q_dst;
#pragma unroll
        for (int j = 0; j < 4; ++j) {
            const int row = 8 * j + (lane >> 3);
            const int pos = lane & 7;
            const int lrow = row < last ? row : last;
            const int c = pos ^ ((row >> 1) & 7);
            if constexpr (WIDE_Q) {
                const float *src = reinterpret_cast<const float *>(a.q.p) + ((size_t)bi * a.q.sb8 + (size_t)hi * a.q.sh8) * 8 +
                                   (size_t)(qbase + lrow) * q_sn;
#pragma unroll
                for (int half = 0; half < Q_PARTS; ++half) {
                    const f32x4 *x = reinterpret_cast<const f32x4 *>(src + (chunk_at(8 * half + c) >> 1));
                    wide[NH * j + half][0] = x[0];
                    wide[NH * j + half][1] = x[1];
                }
                continue;
            }
            if constexpr (FIRST != 0) async_copy_b128(dst + j * 1024, qsrc, __umul24(lrow, q_rb) + chunk_at(c));
            if constexpr (NH == 2 && !NARROW) async_copy_b128(dst + Q_HALF + j * 1024, qsrc, __umul24(lrow, q_rb) + chunk_at(8 + c));
            if constexpr (NARROW) {           // the rows' ends behind the last of their first pieces, as in issue_kv
                constexpr int EVERY = 4 / Q2_PIECES;
                const int i = j / EVERY, end_row = q2_row(i);
                if (j % EVERY == EVERY - 1)
                    async_copy_b128(q2_dst + i * 1024, qsrc, __umul24(end_row < last ? end_row : last, q_rb) + chunk_at(q2_chunk(i)));
            }
        }
        if constexpr (WIDE_Q && NARROW) {
#pragma unroll
            for (int j = 0; j < Q2_PIECES; ++j) {
                const int row = q2_row(j), lrow = row < last ? row : last;
                const float *src = reinterpret_cast<const float *>(a.q.p) + ((size_t)bi * a.q.sb8 + (size_t)hi * a.q.sh8) * 8 +
                                   (size_t)(qbase + lrow) * q_sn;
                const f32x4 *x = reinterpret_cast<const f32x4 *>(src + (chunk_at(q2_chunk(j)) >> 1));
                wide2[j][0] = x[0];
                wide2[j][1] = x[1];
            }
        }
    }
    using std::integral_constant;
    uint32_t live_w = has_map ? (first_w | first_w2) : 0xffffffffu;
    if ((T & 31) != 0 && TW == 1) live_w &= (1u << (T & 31)) - 1u;
    const uint32_t own_tiles = SPLIT ? 0x11111111u << wave : 0xffffffffu;
    live_w &= own_tiles;
    const int n_visits = !BYTEMASK && TW == 1 ? __builtin_popcount(live_w) : T;
    // (BYTEMASK: there is no map, and every tile, or every fourth of SPLIT, is visited.)
    // Walk over the set bits of the "live" words: `live_w` holds the bits of word `cur_w` that have
    // not been visited yet.  Words beyond the first (N > 2048) are fetched when the walk gets there.
    int base_t = 0, cur_w = 0;
    constexpr int STRIDE = SPLIT ? 4 : 1;
    int upcoming = SPLIT ? wave : 0;
    auto next_tile = [&]() __attribute__((always_inline)) -> int {     // next live tile, T if there is none; wave-uniform
        if constexpr (BYTEMASK) {
            const int t = upcoming < T ? upcoming : T;
            upcoming += STRIDE;
            return t;
        }
        while (UNLIKELY(live_w == 0u)) {
            if (++cur_w >= TW) return T;
            base_t = 32 * cur_w;
            uint32_t lv = 0xffffffffu, lv2 = 0u;
            if (mapw != nullptr)
                asm volatile("s_load_dword %0, %2, 0x0\n\ts_load_dword %1, %3, 0x0\n\ts_waitcnt lgkmcnt(0)"
                             : "=&s"(lv), "=&s"(lv2) : "s"(mapw + cur_w), "s"(mapw2 + cur_w) : "memory");
            lv |= lv2;
            if (cur_w == TW - 1 && (T & 31) != 0) lv &= (1u << (T & 31)) - 1u;
            live_w = lv & own_tiles;
        }
        const int b = __builtin_ctz(live_w);
        live_w &= live_w - 1u;
        return base_t + b;
    };
    const int t_first = next_tile();
    const bool even_progress = (NH == 1 || THIRD) && (int)blockIdx.x >= a.tail_start;   // three work-groups per CU, or four
    if (t_first < T) {
        if constexpr (SPLIT) {          // V waits until q, which sits in its buffer, has been read
            issue_own_k(t_first);
            issue_mask(t_first, integral_constant<int, 0>{});
        } else if constexpr (PAIRS) {   // the first pair's bytes before K/V: the walk below counts on that order
            issue_mask_pair(0);
            issue_kv(t_first, integral_constant<int, 0>{});
        } else {
            issue_kv(t_first, integral_constant<int, 0>{});
            issue_mask(t_first, integral_constant<int, 0>{});
        }
    }
    if constexpr (WIDE_Q) {
        uint16_t *q16 = a.q16.p != nullptr && (SPLIT ? wave == 0 : half == 0) ? slab(a.q16, bi, hi) : nullptr;
        auto land = [&](const f32x4 lo, const f32x4 hi4, uint32_t at, int row, int chunk) __attribute__((always_inline)) {
            const u32x4 t = {E::pack2_rne(lo.x, lo.y), E::pack2_rne(lo.z, lo.w), E::pack2_rne(hi4.x, hi4.y), E::pack2_rne(hi4.z, hi4.w)};
            *(LDS_PTR(u32x4))(uintptr_t)at = t;
            if (q16 != nullptr && row_base + row < N && chunk <= last_chunk)
                *reinterpret_cast<u32x4 *>(q16 + (size_t)(row_base + row) * a.q16.sn + 8 * chunk) = t;
        };
#pragma unroll
        for (int j = 0; j < 4; ++j) {
            const int row = 8 * j + (lane >> 3), c = (lane & 7) ^ ((row >> 1) & 7);
#pragma unroll
            for (int half = 0; half < Q_PARTS; ++half)
                land(wide[NH * j + half][0], wide[NH * j + half][1], q_dst + half * Q_HALF + j * 1024 + lane * 16, row, 8 * half + c);
        }
#pragma unroll
        for (int j = 0; j < Q2_PIECES; ++j) land(wide2[j][0], wide2[j][1], q2_dst + j * 1024 + lane * 16, q2_row(j), q2_chunk(j));
    }
    // small LDS table for the mask: entry n (16 B) holds four floats, float j = (bit j of n) ? 0 : -inf
    if (tid < 64)
        reinterpret_cast<float *>(smem)[tid] = (((tid >> 2) >> (tid & 3)) & 1) ? 0.f : -__builtin_inff();
    int yield_at = -1;                  // the visit at which this wave next lowers its priority
    if (even_progress && n_visits >= 4) {
        __builtin_amdgcn_s_setprio(3);
        yield_at = n_visits / 4;
    }
    if (SPLIT) { if (t_first < T) wait_vmcnt<8 * NH + C::MASK_COPIES>(); else wait_vmcnt<0>(); }
    else if (PAIRS) wait_vmcnt<C::KV_COPIES + (HALVES ? 2 : 4)>();      // q has landed; 4 (2) mask and the K/V copies may still be in flight
    else if (t_first < T) wait_vmcnt<COPIES>();        // q has landed; the copies of the first tile may still be in flight
    else wait_vmcnt<0>();
    // What only the end needs of the arguments, while q is on its way from LDS.  Requested with the others at the start (as the compiler has it) ->
    // behind the first copies -> here, the grid's size among the first arguments; small calls back to back: 2 heads, N = 128, D = 64 4.78 -> 4.64 ->
    // 4.55 us; D = 128: 224, N = 18 5.38 -> 5.15 -> 5.14, 32, N = 64 5.05 -> 4.89 -> 4.83.  (Where by-products are asked for, in training, as the
    // compiler has it: those kernels use all but a few scalar registers, and late costs them 192 heads, N = 577, D = 32 32.0 -> 32.2 us, fp32 queries, D = 80
    // 43.75 -> 44.1, of which two are then spilled.)
    Rows out = a.out, out32 = a.out32;
    float *lse = a.lse;
    if constexpr (!BYPRODUCTS) {
        const KernelArgs late = kernel_args();
        out = rows_of(late->out);
        out32 = rows_of(late->out32);
        lse = late->lse;
    }
    // ---- Q^T as MFMA B operands, scaled by scale*log2(e)/post_mul:
    //      lane holds query rows 16x + l16, d = 32*c + 8*q4 .. +7
    u32x4 qf[2][KS];
#pragma unroll
    for (int x = 0; x < 2; ++x)
#pragma unroll
        for (int c = 0; c < KS; ++c)
            qf[x][c] = NARROW && 4 * c == SHORT_CHUNK ? lds_read_b128(k2_at + FIRST + (NSTAGE - 1) * STAGE_BYTES + wave * (32 * SECOND) + 16 * SECOND * x)
                                        : lds_read_b128((k_at ^ (64 * (c & 1))) + 2048 * x +
                                     (SPLIT ? C::OFF_V + (c >> 1) * Q_HALF : (NSTAGE - 1) * STAGE_BYTES + (c >> 1) * Q_HALF + wave * 4096));
    // All requested before the first is converted.  Left alone, the compiler read, waited and converted one after the other, up to eight round trips
    // of LDS in a row: small calls back to back, that -> this, 2 heads, N = 128, D = 64 4.86 -> 4.78 us; D = 128: 224, N = 18 5.51 -> 5.38, 32, N = 64
    // 5.23 -> 5.05.  (fp32 queries: the same either way, 6.69 us of a call of two launches, and 96 heads, N = 577, D = 80 43.5 us left alone, 43.9 held.)
    if constexpr (!WIDE_Q) __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int x = 0; x < 2; ++x)
#pragma unroll
        for (int c = 0; c < KS; ++c) {
            u32x4 &t = qf[x][c];
#pragma unroll
            for (int i = 0; i < 4; ++i)
                t[i] = E::pack2_rne(E::up1((uint16_t)(t[i] & 0xffffu)) * a.q_scale, E::up1((uint16_t)(t[i] >> 16)) * a.q_scale);
            if ((!PACKED_ROWS || HDIM % 32 != 0) && 4 * c + q4 > last_chunk) t = u32x4{0u, 0u, 0u, 0u};      // beyond the row: adds nothing
        }

    if constexpr (SPLIT) {
        asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
        if (t_first < T) issue_own_v(t_first);
    }
    if constexpr (HALVES) {
        k_at += 4096 * half;
        v_at += 4096 * half;
        k2_at += 32 * SECOND * half;
        v2_at += 32 * SECOND * half;
    }

    // ---- running state: of the query rows 16x + l16 what the products and sums need, of the row l32 (in both lane halves) what is
    //      looked at once a tile ----
    f32x4 oacc[2][DB];                  // 16 columns each
#pragma unroll
    for (int x = 0; x < 2; ++x)
#pragma unroll
        for (int b = 0; b < DB; ++b) oacc[x][b] = f32x4{0.f, 0.f, 0.f, 0.f};
    float ref = 0.f;                    // reference point r, in accumulator units (log2 / pm)
    float rmax = -__builtin_inff();     // largest score seen when the maximum was last taken, minus r; -inf = no kept key yet
    int all_seen = 0;                   // wave-uniform: every row of this wavefront has met a kept key
    float l_run[2] = {0.f, 0.f};        // this lane's share of sum exp2(pm * (score - r))
    u32x2 refb[2] = {u32x2{0u, 0u}, u32x2{0u, 0u}};             // -r as four 16-bit terms (lanes 0 .. 15 only), B operand
    int ref_used = 0;                   // wave-uniform: 0 while r == 0 for every row: the extra MFMA is skipped

    auto set_ref = [&](float r_wanted) __attribute__((always_inline)) -> float {      // returns the value actually represented
        float rest = -r_wanted, sum = 0.f;
        uint16_t term[4];
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            const float clipped = __builtin_fminf(__builtin_fmaxf(rest, -E::TERM_MAX), E::TERM_MAX);
            term[i] = E::cvt1(clipped);
            const float got = E::up1(term[i]);
            rest -= got;
            sum += got;
        }
        const uint32_t keep = q4 == 0 ? 0xffffffffu : 0u;
        const RowPair lo = of_rows((uint32_t)term[0] | ((uint32_t)term[1] << 16)), hi = of_rows((uint32_t)term[2] | ((uint32_t)term[3] << 16));
#pragma unroll
        for (int x = 0; x < 2; ++x) refb[x] = u32x2{lo.w[x] & keep, hi.w[x] & keep};
        return -sum;
    };

    // One key tile for this wavefront.  `so` (LDS offset of the stage) is a compile-time constant
    // in every call, so all LDS addresses below are a register plus an immediate.
    // (SPLIT: `after_scores` runs when K has been read, `before_values` before V is.)
    constexpr int KB = HALVES ? 1 : 2;            // blocks of 32 keys that a wavefront takes of a tile
    auto compute_tile_with = [&](const u32x2 both, const uint32_t so, auto after_scores, auto before_values) __attribute__((always_inline)) {
        const u32x2 w2 = HALVES ? u32x2{half ? both.y : both.x, 0u} : both;       // of row l32
        if (UNLIKELY(__builtin_amdgcn_ballot_w64((w2.x | w2.y) != 0u) == 0ull)) {
            after_scores();
            return;
        }
        if constexpr (NARROW) asm volatile("" : "+v"(k2_at), "+v"(v2_at));
        asm volatile("" : "+v"(k_at), "+v"(v_at));       // or the compiler keeps a register for every address that follows from these
        // Steps of two products: S^T of 16 keys and 32 columns each, then O^T += V^T P^T of 16 columns and 32 keys.  The operands of a step are
        // requested AHEAD steps before it, and scheduling barriers hold that order: left alone, the compiler requests each just before
        // its use (it saves registers) and the wavefront sits out one LDS round trip after the other.
        constexpr int PH = 2 * KS, SCORES = KB * PH, VALUES = KB * DB;
        u32x4 k_ring[AHEAD + 1], v_ring[V_AHEAD + 1];
        auto fetch_k = [&](int n) __attribute__((always_inline)) {
            const int blk = n / PH, kb = n & 1, c = n % PH >> 1;
            if (NARROW && 4 * c == SHORT_CHUNK && n < SCORES) k_ring[n % (AHEAD + 1)] = lds_read_b128(k2_at + so + SECOND * (32 * blk + 16 * kb));
            else if (n < SCORES) k_ring[n % (AHEAD + 1)] = lds_read_b128((k_at ^ (64 * (c & 1))) + so + (c >> 1) * TILE_BYTES + 4096 * blk + 2048 * kb);
        };
        auto fetch_v = [&](int n) __attribute__((always_inline)) {
            if (n >= VALUES) return;
            const int blk = n / DB, b = n % DB;
            const bool second = NARROW && 2 * b >= SHORT_CHUNK;
            const uint32_t at = second ? (v2_at ^ (32 * (b & 3))) + so + 32 * SECOND * blk : (v_at ^ (32 * (b & 3))) + so + (b >> 2) * TILE_BYTES + 4096 * blk;
            const u32x2 lo = lds_read_tr16_b64(at), hi = lds_read_tr16_b64(at + (second ? 16 * SECOND : 2048));
            v_ring[n % (V_AHEAD + 1)] = u32x4{lo.x, lo.y, hi.x, hi.y};
        };
#pragma unroll
        for (int n = 0; n < AHEAD; ++n) fetch_k(n);
        __builtin_amdgcn_sched_barrier(0);
        constexpr int EARLY_V = SPLIT || (BYPRODUCTS && HDIM == 64) || THIRD ? 0 : HDIM <= 64 ? 2 : 4;       // of V before the exponentials, where there are registers
        // ---- S^T: sacc[blk][kb][x][j] = log2 weight / pm of (key 32blk + 16kb + 4q4 + j, query 16x + l16) ----
        f32x4 sacc[KB][2][2];
#pragma unroll
        for (int blk = 0; blk < KB; ++blk) {
            const uint32_t wl = blk == 0 ? w2.x : w2.y;
            const RowPair rows = of_rows(wl);
#pragma unroll
            for (int x = 0; x < 2; ++x) {
                const uint32_t wa = __builtin_amdgcn_alignbit(rows.w[x], rows.w[x], nib_rotate);
                sacc[blk][0][x] = __builtin_bit_cast(f32x4, lds_read_b128(lut_addr + (wa & nib_mask)));
                sacc[blk][1][x] = __builtin_bit_cast(f32x4, lds_read_b128(lut_addr + ((wa >> 16) & nib_mask)));
            }
        }
        if (UNLIKELY(ref_used)) {               // wave-uniform: some row of this wavefront has r != 0
            const u32x4 all_ones = {ones, ones, ones, ones};
#pragma unroll
            for (int blk = 0; blk < KB; ++blk)
#pragma unroll
                for (int kb = 0; kb < 2; ++kb)
#pragma unroll
                    for (int x = 0; x < 2; ++x) sacc[blk][kb][x] = E::mfma(all_ones, u32x4{refb[x].x, refb[x].y, 0u, 0u}, sacc[blk][kb][x]);
        }
#pragma unroll
        for (int n = 0; n < SCORES; ++n) {
            fetch_k(n + AHEAD);
            if (!SPLIT && n + EARLY_V >= SCORES) fetch_v(n + EARLY_V - SCORES);
            __builtin_amdgcn_sched_barrier(0);
            const int blk = n / PH, kb = n & 1, c = n % PH >> 1;
#pragma unroll
            for (int x = 0; x < 2; ++x) sacc[blk][kb][x] = E::mfma(k_ring[n % (AHEAD + 1)], qf[x][c], sacc[blk][kb][x]);
            __builtin_amdgcn_sched_barrier(0);
        }
        after_scores();
        // ---- the row maximum of the tile is taken only when it can matter ----
        // Moves the reference point when a row's scores leave the window [r-8, r+8] upwards, or when
        // the first kept score of a row lies below it.
        auto recentre = [&]() __attribute__((always_inline)) {
            float m[2];
#pragma unroll
            for (int x = 0; x < 2; ++x) {
                m[x] = -__builtin_inff();
#pragma unroll
                for (int blk = 0; blk < KB; ++blk)
#pragma unroll
                    for (int kb = 0; kb < 2; ++kb)
#pragma unroll
                        for (int j = 0; j < 4; ++j) m[x] = __builtin_fmaxf(m[x], sacc[blk][kb][x][j]);
            }
            const float mx = rows_max(m[0], m[1]);
            const float mxs = POSTMUL ? mx * pm : mx;
            const bool first = (rmax == -__builtin_inff());
            const bool move = (mxs > WINDOW_LOG2) | (first & (mxs < -WINDOW_LOG2) & (mx > -__builtin_inff()));
            const float top = __builtin_fmaxf(rmax, mx);
            if (UNLIKELY(__builtin_amdgcn_ballot_w64(move) != 0ull)) {
                // every row of the wavefront re-centres on its own largest score so far
                const bool any = top > -__builtin_inff();
                const float new_ref = set_ref(any ? ref + top : ref);
                const float delta = ref - new_ref;                       // ~ -top
                const float alpha = first ? 1.0f : __builtin_amdgcn_exp2f(POSTMUL ? delta * pm : delta);
                ref = new_ref;
                ref_used = 1;
                const RowPair da = of_rows(__builtin_bit_cast(uint32_t, delta)), al = of_rows(__builtin_bit_cast(uint32_t, alpha));
#pragma unroll
                for (int x = 0; x < 2; ++x) {
                    const float d = __builtin_bit_cast(float, da.w[x]), f = __builtin_bit_cast(float, al.w[x]);
                    l_run[x] *= f;
#pragma unroll
                    for (int b = 0; b < DB; ++b) oacc[x][b] *= f;
#pragma unroll
                    for (int blk = 0; blk < KB; ++blk)
#pragma unroll
                        for (int kb = 0; kb < 2; ++kb) sacc[blk][kb][x] += d;
                }
                rmax = top + delta;
            } else {
                rmax = top;
            }
        };
        // probabilities, packed as the B operands of the PV product, and this lane's sums of them
        u32x4 pb[KB][2];
        float lsum[2];
        auto exponentials = [&]() __attribute__((always_inline)) {
            lsum[0] = lsum[1] = 0.f;
#pragma unroll
            for (int blk = 0; blk < KB; ++blk)
#pragma unroll
                for (int kb = 0; kb < 2; ++kb)
#pragma unroll
                    for (int i = 0; i < 2; ++i)
#pragma unroll
                        for (int x = 0; x < 2; ++x) {
                            const float s0 = sacc[blk][kb][x][2 * i], s1 = sacc[blk][kb][x][2 * i + 1];
                            const float p0 = __builtin_amdgcn_exp2f(POSTMUL ? s0 * pm : s0);
                            const float p1 = __builtin_amdgcn_exp2f(POSTMUL ? s1 * pm : s1);
                            const uint32_t pk = E::pack2_prob(p0, p1);
                            pb[blk][x][2 * kb + i] = pk;
                            lsum[x] = E::add2(pk, ones, lsum[x]);
                        }
        };
        // A row needs the maximum when it meets its first kept key (to choose its reference point)
        // and when a score runs away above the window.  The first is known beforehand; the second
        // shows afterwards, in the sums of the exponentials (needed anyway): a weight above 2^14, an
        // infinity or a NaN makes a lane's sum of 32 weights exceed SUM_LIMIT, and no weight that
        // the window would have let pass (<= 2^8) can.  Only then are the maximum taken, the
        // reference moved and the exponentials redone.
        int with_max = 0;
        if (UNLIKELY(!all_seen)) {
            if (__builtin_amdgcn_ballot_w64((rmax == -__builtin_inff()) & ((w2.x | w2.y) != 0u)) != 0ull) {
                with_max = 1;
                recentre();
                all_seen = __builtin_amdgcn_readfirstlane(__builtin_amdgcn_ballot_w64(rmax == -__builtin_inff()) == 0ull ? 1 : 0);
            }
        }
        exponentials();
        if (UNLIKELY(__builtin_amdgcn_ballot_w64(!(lsum[0] + lsum[1] <= SUM_LIMIT)) != 0ull)) {
            if (!with_max) {
                recentre();
                exponentials();
            }
        }
        l_run[0] += lsum[0];
        l_run[1] += lsum[1];
        before_values();
        // ---- O^T += V^T * P^T : oacc[x][b][j] = out(query 16x + l16, d = 16b + 4q4 + j) ----
#pragma unroll
        for (int n = EARLY_V; n < V_AHEAD; ++n) fetch_v(n);
#pragma unroll
        for (int n = 0; n < VALUES; ++n) {
            fetch_v(n + V_AHEAD);
            __builtin_amdgcn_sched_barrier(0);
            const int blk = n / DB, b = n % DB;
#pragma unroll
            for (int x = 0; x < 2; ++x) oacc[x][b] = E::mfma(v_ring[n % (V_AHEAD + 1)], pb[blk][x], oacc[x][b]);
            __builtin_amdgcn_sched_barrier(0);
        }
    };

    auto compute_tile = [&](const u32x2 w2, const uint32_t so) __attribute__((always_inline)) {
        compute_tile_with(w2, so, [] {}, [] {});
    };

    // ================================ main loop ================================
    // What a visit spends beside its products and exponentials is scalar: some 60 instructions for the walk, the copies' addresses and the
    // rare cases.  The branches say which way they go (UNLIKELY), so that the usual way falls through and what rarely runs lies behind the
    // loop; wave-uniform flags are numbers in scalar registers, tile offsets 32 bits, and the copies of the tile that the keys end in change
    // the lanes' offsets in place, since none follows it.  Before -> now, one binary each in turn: 192 heads, D = 64, packed, N = 2048
    // 237.4 -> 229.5 us, N = 1024 64.4 -> 62.3, blocks with a map 38.0 -> 35.8; 8 heads, N = 3958, boolean 64.8 -> 58.7; D = 128, 128 heads,
    // N = 4096 1063 -> 1036, causal 619 -> 595; where the mask's bytes bound it (192, N = 512) 24.2 -> 23.9.
    // The tiles visited: every tile whose "some bit set" bit is on (all of them without a map), in
    // ascending order; the prologue has requested the first.  The i-th visit uses stage and mask
    // slot i % 2; the loop is unrolled by 2 so that these are constants.
    // In a visit of tile t:
    //   wait for the copies of tile t  ->  barrier  ->  request the copies of the next tile to be
    //   visited (K/V, then the mask words) into the stage the barrier has freed  ->  compute, unless
    //   this wave's 32 x 64 block of mask bits is empty.
    // (A ring of three stages, copies two tiles ahead, measured the same to 2 % slower on every
    // workload and costs 18 KB more LDS.)
    int visits = 0;
    // The hardware serves the oldest wave first, so of three co-resident work-groups one
    // finishes early and the last runs alone, at a worse rate than three together.  When
    // no other work-group waits for the slot, a wave therefore yields as it advances.
    auto progress = [&]() __attribute__((always_inline)) {
        if (UNLIKELY(visits == yield_at)) {
            if (visits == n_visits / 4) {
                __builtin_amdgcn_s_setprio(2);
                yield_at = n_visits / 2;
            } else if (visits == n_visits / 2) {
                __builtin_amdgcn_s_setprio(1);
                yield_at = (3 * n_visits) / 4;
            } else {
                __builtin_amdgcn_s_setprio(0);
            }
        }
        ++visits;
    };
    auto visit = [&](const int t, const int t_next, auto slot_c) __attribute__((always_inline)) {
        constexpr int SLOT = decltype(slot_c)::value;
        constexpr int SLOT2 = SLOT ^ 1;       // the stage freed by the barrier below
        progress();
        wait_vmcnt<0>();          // the copies of tile t have landed
        if (UNLIKELY(t == cut_tile)) zero_tail_rows(t, SLOT);
        __syncthreads();          // tile t landed for every wave; the stage of the previous visit is free
        const u32x2 w2 = mask_words(t, SLOT);
        if (LIKELY(t_next < T)) {       // K/V first: the MFMA operands are what the next visit needs first (1-2 % with a byte mask)
            issue_kv(t_next, integral_constant<int, SLOT2>{});
            issue_mask(t_next, integral_constant<int, SLOT2>{});
        }
        compute_tile(w2, (uint32_t)(SLOT * STAGE_BYTES));
    };
    if constexpr (SPLIT) {
        __syncthreads();              // the table of the mask bias
        for (int t = t_first, tn; t < T; t = tn) {
            tn = next_tile();
            wait_vmcnt<8 * NH>();     // K and the mask of tile t; its V may still be on its way
            if (UNLIKELY(t == cut_tile)) zero_own_rows(t, 0);
            const u32x2 w2 = mask_words(t, 0);
            compute_tile_with(w2, 0u,
                [&]() __attribute__((always_inline)) {
                    asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
                    if (tn < T) {
                        issue_own_k(tn);
                        issue_mask(tn, integral_constant<int, 0>{});
                    }
                },
                [&]() __attribute__((always_inline)) {
                    if (tn < T) wait_vmcnt<8 * NH + C::MASK_COPIES>(); else wait_vmcnt<0>();
                    if (UNLIKELY(t == cut_tile)) zero_own_rows(t, C::OFF_V);
                });
            asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
            if (tn < T) issue_own_v(tn);
        }
    } else if constexpr (PAIRS) {
        // Every tile is visited (there is no tile map with a boolean mask).
        // Copies in flight, oldest first, at the top of an even visit t: the bytes of the pair
        // (t, t + 1), then K/V of t; after its barrier K/V of t + 1 and then the bytes of the next
        // pair are requested, and the odd visit requests K/V of t + 2 after its barrier: the bytes of
        // a pair are always followed by exactly one tile's younger copies (KV_COPIES) when they are needed.  (The stores
        // of the by-products, when asked for, only add to the count: copies complete in the order of
        // their requests, so "at most so many outstanding" still means that all older copies are in.)
        // HALVES: a wavefront reads bytes that another has copied, behind the even visit's barrier; the next pair's are requested then
        // into the other slot, whose bytes were read before the odd visit's barrier.
        for (int t = 0; t < T; t += 2) {
            progress();
            u32x2 w_even, w_odd = {0u, 0u};
            auto words = [&]() __attribute__((always_inline)) {
                const int slot = HALVES ? (t >> 1) & 1 : 0;
                w_even = mask_words(t, slot, 0);
                if (WHOLE || t + 1 < T) w_odd = mask_words(t + 1, slot, 1);
            };
            if constexpr (!HALVES) {
                wait_vmcnt<C::KV_COPIES>();                   // this wave's bytes of the pair have landed
                words();
            }
            wait_vmcnt<0>();                                  // K/V of tile t
            if (!WHOLE && UNLIKELY(t == cut_tile)) zero_tail_rows(t, 0);
            __syncthreads();
            if constexpr (HALVES) words();
            if (WHOLE || t + 1 < T) issue_kv(t + 1, integral_constant<int, 1>{});
            if (LIKELY(t + 2 < T)) issue_mask_pair((t >> 1) + 1);     // the words above are in registers: the bytes may go
            compute_tile(w_even, 0u);
            if (!WHOLE && t + 1 >= T) break;
            progress();
            if (t + 2 < T) wait_vmcnt<HALVES ? 2 : 4>(); else wait_vmcnt<0>();   // K/V of tile t + 1 (the next pair's bytes may be on their way)
            if (!WHOLE && UNLIKELY(t + 1 == cut_tile)) zero_tail_rows(t + 1, 1);
            __syncthreads();
            if (LIKELY(t + 2 < T)) issue_kv(t + 2, integral_constant<int, 0>{});
            compute_tile(w_odd, (uint32_t)STAGE_BYTES);
        }
    } else
    for (int t = t_first; t < T;) {
        const int tn = next_tile();
        visit(t, tn, integral_constant<int, 0>{});
        if (tn >= T) break;
        t = next_tile();
        visit(tn, t, integral_constant<int, 1>{});
    }
    wait_vmcnt<0>();              // no copy may outlive the work-group's LDS allocation
    float l_row = rows_sum(l_run[0], l_run[1]);

    if constexpr (SPLIT) {
        // Wavefronts 1 to 3 leave their sums in their own buffers, wavefront 0 adds them to its own, all of them
        // moved to the largest reference point of those that have met a kept key.
        const f32x2 own = {rmax > -__builtin_inff() ? ref : -__builtin_inff(), l_row};
        if (wave != 0) {
#pragma unroll
            for (int x = 0; x < 2; ++x)
#pragma unroll
                for (int b = 0; b < DB; ++b)
                    *(LDS_PTR(f32x4))(uintptr_t)(split_dst + (x * DB + b) * 1024 + lane * 16) = oacc[x][b];
            *(LDS_PTR(f32x2))(uintptr_t)(split_dst + DB * 2048 + lane * 8) = own;
        }
        __syncthreads();
        if (wave != 0) return;
        f32x2 of_wave[4];
        of_wave[0] = own;
        float top = own.x;
#pragma unroll
        for (int w = 1; w < 4; ++w) {
            of_wave[w] = *(LDS_PTR(const f32x2))(uintptr_t)(lds0 + w * STAGE_BYTES + DB * 2048 + lane * 8);
            top = __builtin_fmaxf(top, of_wave[w].x);
        }
        ref = top > -__builtin_inff() ? top : 0.f;
        l_row = 0.f;
#pragma unroll
        for (int w = 0; w < 4; ++w) {
            // a wavefront that has met no kept key of the row has nothing to add (its factor is 0)
            const float d = of_wave[w].x - ref;
            const float f = __builtin_amdgcn_exp2f(POSTMUL ? d * pm : d);
            l_row = __builtin_fmaf(of_wave[w].y, f, l_row);
            const RowPair fx = of_rows(__builtin_bit_cast(uint32_t, f));
#pragma unroll
            for (int x = 0; x < 2; ++x)
#pragma unroll
                for (int b = 0; b < DB; ++b) {
                    const float g = __builtin_bit_cast(float, fx.w[x]);
                    if (w == 0) {
                        oacc[x][b] *= g;
                    } else {
                        const f32x4 o = *(LDS_PTR(const f32x4))(uintptr_t)(lds0 + w * STAGE_BYTES + (x * DB + b) * 1024 + lane * 16);
#pragma unroll
                        for (int j = 0; j < 4; ++j) oacc[x][b][j] = __builtin_fmaf(o[j], g, oacc[x][b][j]);
                    }
                }
        }
    }
    if constexpr (BYPRODUCTS && !SPLIT) {
        if (map_dst != nullptr) {
            const int rb = HALVES ? 0 : wave >> 1;             // block of 64 rows
            uint32_t before = 0u;
            if (lane == 0)
                before = __hip_atomic_fetch_add((LDS_PTR(uint32_t))(uintptr_t)(lds0 + C::OFF_MAP_ARRIVED + 4 * rb), 1u,
                                                __ATOMIC_ACQ_REL, __HIP_MEMORY_SCOPE_WORKGROUP);
            before = __builtin_amdgcn_readfirstlane(before);
            if (before == 1u && lane < TW && (HALVES || 2 * qt + rb < T)) {
                const int w = lane;                            // word of 32 key tiles
                const uint32_t src = lds0 + C::OFF_MAP + (uint32_t)(2 * rb) * (C::MAP_WORDS * 8) + (uint32_t)w * 8;
                const u32x2 x0 = lds_read_b64(src), x1 = lds_read_b64(src + C::MAP_WORDS * 8);
                const uint32_t in_range = (w == TW - 1 && (T & 31)) ? ((1u << (T & 31)) - 1u) : 0xffffffffu;
                uint32_t *dst = map_dst + (size_t)rb * 2 * TW;
                dst[w] = (x0.x | x1.x) & in_range;
                dst[TW + w] = ~(x0.y | x1.y) & in_range;
            }
        }
    }

    constexpr int HALF_SUMS = DB * 2048 + 1024;          // of one wavefront
    if constexpr (HALVES) {
        // Wavefronts 2 and 3 leave their sums for 0 and 1, which have the same rows, both moved to the larger reference point of
        // those that have met a kept key.
        const uint32_t sums = lds0 + (wave & 1) * HALF_SUMS;
        const f32x2 own = {rmax > -__builtin_inff() ? ref : -__builtin_inff(), l_row};
        __syncthreads();                                  // the last tile has been read by all
        if (half == 1) {
#pragma unroll
            for (int x = 0; x < 2; ++x)
#pragma unroll
                for (int b = 0; b < DB; ++b)
                    *(LDS_PTR(f32x4))(uintptr_t)(sums + (x * DB + b) * 1024 + lane * 16) = oacc[x][b];
            *(LDS_PTR(f32x2))(uintptr_t)(sums + DB * 2048 + lane * 8) = own;
        }
        __syncthreads();
        if (half == 1) return;
        const f32x2 other = *(LDS_PTR(const f32x2))(uintptr_t)(sums + DB * 2048 + lane * 8);
        const float top = __builtin_fmaxf(own.x, other.x);
        ref = top > -__builtin_inff() ? top : 0.f;
        // one that has met no kept key of the row has nothing to add (its factor is 0)
        const float dm = own.x - ref, d = other.x - ref;
        const float fm = __builtin_amdgcn_exp2f(POSTMUL ? dm * pm : dm), f = __builtin_amdgcn_exp2f(POSTMUL ? d * pm : d);
        l_row = __builtin_fmaf(other.y, f, l_row * fm);
        const RowPair mine = of_rows(__builtin_bit_cast(uint32_t, fm)), its = of_rows(__builtin_bit_cast(uint32_t, f));
#pragma unroll
        for (int x = 0; x < 2; ++x)
#pragma unroll
            for (int b = 0; b < DB; ++b) {
                const f32x4 o = *(LDS_PTR(const f32x4))(uintptr_t)(sums + (x * DB + b) * 1024 + lane * 16);
                const float g = __builtin_bit_cast(float, its.w[x]), gm = __builtin_bit_cast(float, mine.w[x]);
#pragma unroll
                for (int j = 0; j < 4; ++j) oacc[x][b][j] = __builtin_fmaf(o[j], g, oacc[x][b][j] * gm);
            }
    }

    // ---- epilogue ----
    // out = O / l.  The accumulator layout gives a lane 8-byte pieces of one row; written as they
    // are, a store instruction would touch 32 different 128-byte rows.  Each wave therefore
    // transposes its 32 x 64 block (one per column half) through 4 KiB of LDS and stores whole
    // 128-byte pieces of rows, non-temporally: the output is not read again here and should not
    // displace K, V and the mask.  The LDS used is the stage that tile T would have gone to: its
    // last occupant was tile T - 2, which every wave had finished before the barrier of the last
    // iteration, and no copy into it is in flight, so no further barrier is needed and a wave
    // that is done early stores early.
    const RowPair inv_of = of_rows(__builtin_bit_cast(uint32_t, l_row > 0.f ? 1.0f / l_row : 0.f));
    const float inv[2] = {__builtin_bit_cast(float, inv_of.w[0]), __builtin_bit_cast(float, inv_of.w[1])};
    {
        const int row0 = row_base;
        // Head dim 32, whose stages are smaller: through an area of the wavefront's own, with pairs of tiles' bytes that of the bytes; with one tile's
        // through both stages, behind a barrier.
        if constexpr (FIRST == 0 && BYTEMASK && !PAIRS && !HALVES) __syncthreads();
        const uint32_t ebase = FIRST == 0 && !HALVES ? lds0 + (PAIRS ? OFF_MASK : BYTEMASK ? 0 : C::OFF_MAP) + wave * 4096 : SPLIT ? lds0 : HALVES ? lds0 + 2 * HALF_SUMS + wave * 4096 : lds0 + (uint32_t)(visits & 1) * STAGE_BYTES + wave * 4096;
        store_rows<BF16>(oacc, inv, ebase, SPLIT ? 4096 : HALVES ? 8192 : NARROW ? 0 : 16384, block_dst(out, out32, bi, hi, row0, D), out.p != nullptr,
                             BF16 && out32.p != nullptr, row0, N, lane);       // fp32 callers compute in bf16
    }
    if (qrow < N) {
        if (lse != nullptr && hh == 0) {
            // log2 of the row's sum of exp(scale * score) is pm * r + log2(l)
            lse[(size_t)bh * N + qrow] =
                (l_row > 0.f) ? __builtin_fmaf(pm * ref, 0.6931471805599453f, __builtin_logf(l_row)) : -__builtin_inff();
            // (an explicit fma: left to the compiler, the sum was contracted in some instantiations of
            // this kernel and not in others, and their lse differed in the last bit)
        }
    }
}

}  // namespace

// The instance for (fp32 q, element type, post-multiplier, row strides) and the kind of mask: 0 packed words, 1
// boolean bytes, 2 the same with by-products, 3 and 4 those with two tiles' bytes per request, 5 to 7 the first
// three with the keys split between the wavefronts, 8 and 9 as 3 and 4 at any N; 10 to 14, 18 and 19 those ten less in halves.  This file is
// compiled once per head dim for the instances, side by side, and once for the launcher.
typedef void (*FwdKernel)(const AttnArgs);
#ifdef SMA_FWD_HEAD_DIM
template <int HDIM, bool BF16, bool POSTMUL, bool PACKED_ROWS, bool WIDE_Q = false> FwdKernel pick_mask_kind(int mask_kind)
{
    switch (mask_kind) {
    case 0: return attn_fwd_kernel<BF16, POSTMUL, PACKED_ROWS, HDIM, false, false, 0, false, WIDE_Q>;
    case 1: return attn_fwd_kernel<BF16, POSTMUL, PACKED_ROWS, HDIM, true, false, 0, false, WIDE_Q>;
    case 2: return attn_fwd_kernel<BF16, POSTMUL, PACKED_ROWS, HDIM, true, true, 0, false, WIDE_Q>;
    case 5: return attn_fwd_kernel<BF16, POSTMUL, PACKED_ROWS, HDIM, false, false, 0, true, WIDE_Q>;
    case 6: return attn_fwd_kernel<BF16, POSTMUL, PACKED_ROWS, HDIM, true, false, 0, true, WIDE_Q>;
    case 7: return attn_fwd_kernel<BF16, POSTMUL, PACKED_ROWS, HDIM, true, true, 0, true, WIDE_Q>;
    }
    if constexpr (HDIM <= 64) {
        switch (mask_kind) {
        case 3: return attn_fwd_kernel<BF16, POSTMUL, PACKED_ROWS, HDIM, true, false, 1, false, WIDE_Q>;
        case 4: return attn_fwd_kernel<BF16, POSTMUL, PACKED_ROWS, HDIM, true, true, 1, false, WIDE_Q>;
        case 8: return attn_fwd_kernel<BF16, POSTMUL, PACKED_ROWS, HDIM, true, false, 2, false, WIDE_Q>;
        case 9: return attn_fwd_kernel<BF16, POSTMUL, PACKED_ROWS, HDIM, true, true, 2, false, WIDE_Q>;
        case 13: return attn_fwd_kernel<BF16, POSTMUL, PACKED_ROWS, HDIM, true, false, 1, false, WIDE_Q, true>;
        case 14: return attn_fwd_kernel<BF16, POSTMUL, PACKED_ROWS, HDIM, true, true, 1, false, WIDE_Q, true>;
        case 18: return attn_fwd_kernel<BF16, POSTMUL, PACKED_ROWS, HDIM, true, false, 2, false, WIDE_Q, true>;
        case 19: return attn_fwd_kernel<BF16, POSTMUL, PACKED_ROWS, HDIM, true, true, 2, false, WIDE_Q, true>;
        }
    }
    if (mask_kind == 10) return attn_fwd_kernel<BF16, POSTMUL, PACKED_ROWS, HDIM, false, false, 0, false, WIDE_Q, true>;
    if constexpr (HDIM > 64) {
        switch (mask_kind) {
        case 11: return attn_fwd_kernel<BF16, POSTMUL, PACKED_ROWS, HDIM, true, false, 0, false, WIDE_Q, true>;
        case 12: return attn_fwd_kernel<BF16, POSTMUL, PACKED_ROWS, HDIM, true, true, 0, false, WIDE_Q, true>;
        }
    }
    return nullptr;
}
template <int HDIM> FwdKernel pick(int variant, int mask_kind)
{
    switch (variant) {
    case 0: return pick_mask_kind<HDIM, false, false, false>(mask_kind);
    case 1: return pick_mask_kind<HDIM, false, false, true>(mask_kind);
    case 2: return pick_mask_kind<HDIM, false, true, false>(mask_kind);
    case 3: return pick_mask_kind<HDIM, false, true, true>(mask_kind);
    case 4: return pick_mask_kind<HDIM, true, false, false>(mask_kind);
    case 5: return pick_mask_kind<HDIM, true, false, true>(mask_kind);
    case 6: return pick_mask_kind<HDIM, true, true, false>(mask_kind);
    case 7: return pick_mask_kind<HDIM, true, true, true>(mask_kind);
    case 12: return pick_mask_kind<HDIM, true, false, false, true>(mask_kind);
    case 13: return pick_mask_kind<HDIM, true, false, true, true>(mask_kind);
    case 14: return pick_mask_kind<HDIM, true, true, false, true>(mask_kind);
    default: return pick_mask_kind<HDIM, true, true, true, true>(mask_kind);
    }
}
#define SMA_NAME2(d) fwd_kernel_##d
#define SMA_NAME(d) SMA_NAME2(d)
FwdKernel SMA_NAME(SMA_FWD_HEAD_DIM)(int variant, int mask_kind) { return pick<SMA_FWD_HEAD_DIM>(variant, mask_kind); }
#else
FwdKernel fwd_kernel_32(int variant, int mask_kind);
FwdKernel fwd_kernel_64(int variant, int mask_kind);
FwdKernel fwd_kernel_80(int variant, int mask_kind);
FwdKernel fwd_kernel_96(int variant, int mask_kind);
FwdKernel fwd_kernel_128(int variant, int mask_kind);

// Number of compute units of the current device (cached per device ordinal).
int compute_units()
{
    static std::atomic<int> cached[64];      // 0 = not asked yet; threads may race to store the same value
    int dev = 0;
    if (hipGetDevice(&dev) != hipSuccess || dev < 0 || dev >= 64) return 0;
    int n = cached[dev].load(std::memory_order_relaxed);
    if (n == 0 && hipDeviceGetAttribute(&n, hipDeviceAttributeMultiprocessorCount, dev) == hipSuccess)
        cached[dev].store(n, std::memory_order_relaxed);
    return n;
}

hipError_t launch_attn_fwd(const AttnArgs &args, bool bf16, hipStream_t stream)
{
    AttnArgs a = args;
    a.div_H = make_fastdiv((uint32_t)a.H);
    long long groups = (long long)a.BH * a.qtiles;
    if (groups == 0) return hipSuccess;
    // Only a grid that is resident all at once with three work-groups (or four) on (almost) every CU evens out
    // its progress; with several rounds oldest-first is what frees slots for the waiting ones, and
    // applying it to the last round only measured neutral.
    const long long cus = compute_units();
    // Keys split between the wavefronts (SPLIT at the kernel): while all work-groups of 32 rows are resident
    // at once, two on a CU up to head dim 64 and one beyond, and there are three key tiles or more to share.  Beyond
    // that line the fewer, longer work-groups of 128 rows win (8 x 8 heads, N = 512, D = 64: 11.2 against 14.8 us).
    // By the shape alone, so that every way of giving the same mask gives the same bits.
    const bool split = a.N > 2 * BN && 2 * groups <= (a.D <= HD ? cus : cus / 2);
    if (split) {
        a.qtiles = (a.N + 31) / 32;
        groups = (long long)a.BH * a.qtiles;
        if (a.map_out != nullptr) {
            const hipError_t e = launch_tile_map_start(a.map_out, a.map_slabs, a.N, stream);
            if (e != hipSuccess) return e;
        }
    }
    // Beyond that line work-groups of 64 rows (HALVES at the kernel), `g64` of them:
    //   head dims beyond 64: while one on a CU holds them all.  With two on a CU they lose at 128 (8 x 8 heads, N = 512: 17.0 -> 17.8 us;
    //       32, N = 1024 22.9 -> 23.1, boolean 24.7 -> 25.3), but up to 96 they gain from 1024 rows on, as long as these are one round.  D = 96: 10 heads, N = 2048
    //       35.5 -> 30.7 (boolean 39.5 -> 36.6, untouched masks 42.1 -> 39.9), 32, N = 1024 20.5 -> 19.5 (22.3 -> 22.0, 24.7 -> 24.8); 64, N = 512 13.5 -> 14.0.  D = 80: 16, N = 2048
    //       32.9 -> 30.9 (boolean 36.3 -> 34.7, with by-products 41.3 -> 39.3, blocks with a map 23.0 -> 16.5, causal 31.6 -> 29.5), 20, N = 1600 36.5 -> 25.6 (boolean 39.5 -> 28.5); one loses
    //       there, 8, N = 4000 with by-products 81.5 -> 88.7.  Up to three on a CU, where that many share one at 80 and 96 (three_on_a_cu), by-products, which leave it at two, lose: D = 80, 24, N = 2000 packed
    //       47.2 -> 43.0, but boolean 55.9 -> 62.9, a training step 207 -> 235;
    //   up to 64, where three share a CU: when they are one round of two to three on a CU and work-groups of 128 rows would be one on some CUs and two on others.  Up
    //       to two on a CU, packed masks gain and boolean ones lose (32 heads, N = 1024: 16.4 -> 15.2; untouched 18.3 -> 18.7), and with a second
    //       round all do (28, N = 2048: 40.7 -> 45.8, boolean 44.6 -> 61.5; any number of rounds, but with a map only: blocks 192, N = 1024 36.9 -> 36.4, 384, N = 512 25.2 -> 27.0, causal
    //       42.6 -> 51.2).  Beyond ten tiles: 48, N = 1024 24.2 -> 20.3.  Shorter ones keep the order of their sums from before this rule; by time it could begin at four tiles (D = 64, N = 200
    //       to 640: 7 to 18 % less, blocks with a map up to 27; three tiles packed 7.6 -> 7.8).
    // Up to 128 keys there is nothing to share (6.6 us either way).  The split stays ahead where it fits: 8 heads, N = 1024 16.9 against 21.3 us.
    const long long g64 = (long long)a.BH * ((a.N + 63) / 64);
    const bool halves = !split && a.N > 2 * BN &&
                        (a.D > HD ? g64 <= (a.D <= 96 && a.N >= 1024 ? 2 * cus : cus) : a.N > 10 * BN && g64 > 2 * cus && g64 <= 3 * cus);
    if (halves) {
        a.qtiles = (a.N + 63) / 64;
        groups = (long long)a.BH * a.qtiles;
    }
    const int D = kernel_head_dim(a.D);
    const bool byproducts = a.mask_out != nullptr || a.map_out != nullptr, three = D <= HD || three_on_a_cu(D, a.byte_mask != 0, byproducts, a.q_f32 != 0);
    a.deal = make_deal(!split && !halves && !a.byte_mask && heads_alike(a.mask, a.H), a.BH, a.qtiles, (three ? 3 : 2) * cus, 4ll * a.N * a.D);
    // Four share a CU at head dim 32, but with by-products (132 to 137 registers): one round of those evens out its progress too.  Oldest first -> this, us: packed
    // 256 heads, N = 512 17.1 -> 15.5, causal 16.1 -> 14.5, blocks with a map 13.1 -> 11.8;  128, N = 1024 29.5 -> 27.2;  boolean 512, N = 256 13.9 -> 13.0, 132, N = 700 25.5 -> 23.0, 74, N = 1500
    // 53.1 -> 50.9;  fp32 149, N = 700 36.9 -> 34.7.  Not with a map of more than one word, from whose first alone a wavefront knows the visits ahead of it (32 heads, N = 4096, causal 55.5 -> 59.6).
    // The rest of the launcher stays with three: the deal keeps heads in turn on such a grid (its ends taken for a second round; without, 128, N = 1024, causal 18.1 -> 26.3), and the
    // boolean mask its pairs of tiles (one tile's bytes: 512, N = 256 13.0 -> 12.3, but 74, N = 1500 50.9 -> 58.3).
    const bool four = D == 32 && !byproducts && (a.tile_map == nullptr || a.N <= 32 * BN);
    a.tail_start = (!split && groups > 2 * cus && groups <= (four ? 4 : 3) * cus) ? 0 : (int)groups;
    a.groups = (int)groups;
    const dim3 grid((unsigned)groups), block(NTHREADS);
    const bool postmul = a.post_mul != 1.0f;
    const bool packed = a.D == D && (int)a.q.sn == D && (int)a.k.sn == D && (int)a.v.sn == D;
    if (!three) a.tail_start = (int)groups;                   // two work-groups per CU: nobody yields
    // two tiles' mask bytes per request (see PAIRS at the kernel), unless the grid is the single round of three work-groups on a CU in
    // step for which tail_start was set to 0 above
    const bool further = !split && a.byte_mask && D <= HD && (halves || a.tail_start != 0 || groups > 3 * cus);
    if (a.q_f32 && !bf16) return hipErrorInvalidValue;         // fp32 callers compute in bf16
    if (a.byte_mask && a.N < 16) return hipErrorInvalidValue;  // a row holds at least one 16-byte copy (checked by the C-ABI layer)
    const int mask_kind = (split ? 5 : halves ? 10 : 0) + (!a.byte_mask ? 0 : (!further ? 1 : a.N % (2 * BN) == 0 ? 3 : 8) + (byproducts ? 1 : 0));
    const int variant = (a.q_f32 ? 8 : 0) | (bf16 ? 4 : 0) | (postmul ? 2 : 0) | (packed ? 1 : 0);
    const FwdKernel kernel = D == 32 ? fwd_kernel_32(variant, mask_kind) : D == 64 ? fwd_kernel_64(variant, mask_kind)
                             : D == 80 ? fwd_kernel_80(variant, mask_kind) : D == 96 ? fwd_kernel_96(variant, mask_kind) : fwd_kernel_128(variant, mask_kind);
    // Three on a CU lose where the work is all bytes, two tiles a work-group and a head to each, over several rounds: 12 KiB more of LDS keep it at two.  D = 80, 2048 heads,
    // packed, two -> three on a CU: N = 112 38.3 -> 39.2 us, 128 42.4 -> 44.5 (boolean 47.3 -> 51.0), D = 96 42.9 -> 44.1;  512 heads 10.1 either way;  one tile, N = 64,
    // 19.3 -> 17.2, three, N = 136, 62.8 -> 55.3.
    const bool two = three && D > HD && !halves && !split && a.N > BN && a.N <= BM && groups > 3 * cus;
    hipLaunchKernelGGL(kernel, grid, block, two ? 12288 : 0, stream, a);
    return hipGetLastError();
}
#endif

}  // namespace sma
