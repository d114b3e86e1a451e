// Masked-attention backward for gfx950 (MI355X), head_dim 32, 64, 80, 96 or 128, fp16 / bf16, fp32 accumulate.
//
// The reference declares a backward launcher (csrc/sparse_attention.h:57-64) and its Python API
// calls sparse_attn_cuda.backward (python/sparse_attention.py:91-94), but neither was ever
// written; the formulas are those of its PyTorch fallback (python/sparse_attention.py:97-111):
//
//     P  = exp(scale * Q K^T - lse) on kept entries, 0 elsewhere      (lse saved by the forward)
//     dV = P^T dO          dP = dO V^T          delta_i = sum_d dO_id O_id  (= sum_j P_ij dP_ij)
//     dS = P o (dP - delta) * scale             dQ = dS K            dK = dS^T Q
//
// No atomics, bit-reproducible.  Sequences of which a work-group holds a whole head take attn_bwd_head.hip's kernel, others
// two, or both in one launch (attn_bwd_both_kernel):
//
//   attn_bwd_dq_kernel   one work-group = 128 query rows, walks the key tiles exactly like the
//                        forward: S^T = K Q^T and dP^T = V dO^T on the MFMA (a lane has two query rows, 16
//                        apart, so lse and delta are two scalars each and the mask enters as the accumulator's
//                        initial value), dS^T packed to 16 bit is the B operand of dQ^T += K^T dS^T
//                        (K^T by transposing LDS reads).  Also writes delta to the workspace.
//   attn_bwd_dkv_kernel  one work-group = 128 or 256 keys (a lane has two, 16 apart), walks the query tiles:
//                        S = Q K^T and dP = dO V^T with K, V fragments held in registers; -lse and
//                        -delta of the tile's rows are read from LDS (broadcast reads) straight
//                        into the accumulators as their initial values, so the products leave
//                        s - lse and dP - delta; the mask bit of (row, key) is bit (key % 32) of the
//                        row's word; P and dS packed to 16 bit are the B operands of
//                        dV^T += dO^T P and dK^T += Q^T dS.  The loop over the query tiles is
//                        unrolled by the two ring stages, so every LDS address in it is a
//                        register plus an immediate.
//
// Products of 16 x 16 x 32: what bounds these kernels at head dims 96 and 128 is the power the matrix cores draw, which lowers the clock, and a
// stream of these on random operands (benchprobe/) sustains 1968 TFLOP/s at 1.97 GHz where 32 x 32 x 16 sustains 1820 at 1.77.  A lane holds two rows (dQ) or two
// keys (dK/dV), 16 apart, and every operand that is read from LDS serves both; of lse, delta and mask words half as many reads are left.  They are short, so
// operands are requested two or three steps (of two products) ahead and the vector work of one step lies between the products of
// another; scheduling barriers hold that order.  The compiler's own order, each read just before its use: dK/dV 1878 -> 2090 us on 4 x 32 heads,
// N = 4096, D = 128; with it 1657, the matrix cores busy 62 % of the cycles at 2.03 GHz (before 57 % at 1.95); dQ 1405 -> 1345 -> 1275 us.
// The backward alone, 32 x 32 x 16 -> this, in us, random masks unless noted:
//   192 heads, N = 1024   D = 32 128 -> 120, 64 200 -> 184 (blocks, map 101 -> 97), 96 274 -> 254, 128 353 -> 318 (blocks, map 219 -> 200)
//   128 heads, N = 2048   D = 32 315 -> 294, 64 484 -> 440, 96 673 -> 613, 128 857 -> 780;  causal, N = 2000: 218 -> 210, 299 -> 280, 437 -> 410, 598 -> 550
//   8 heads, N = 3000     D = 32 64.8 -> 61.5, 64 81.0 -> 75.5, 96 113 -> 98, 128 174 -> 155
//
// Tiles (64 rows x 64 x 16 bit) are copied global -> LDS by global_load_lds_dwordx4 into two
// stages, one tile ahead; the 16-byte chunks of a row are XOR-swizzled with swizzle16((row >> 1) & 7),
// which keeps both the row reads (ds_read_b128) and the transposing reads (ds_read_b64_tr_b16) of
// the same tile free of bank conflicts.
//
// Head dim 128 (NH = 2) is handled as two column halves of 64: every streamed matrix is kept in LDS
// as two 64-column tiles, the products that contract over the head dim (S, dP) run over both
// halves, the others (dQ, dK, dV) fill one pair of accumulators per half.  Head dim 32 uses half a tile: the copies fill the upper half of
// every LDS row with copies of the row's last 16 bytes, which are never read;
// contractions over the head dim take one MFMA step and the outputs have two 16-column blocks.  Head dim 96
// is 128 with such a half tile as its second half: three steps, six blocks; 80 the same with five.
#include "attn_bwd_common.h"

namespace sma {
namespace {

constexpr int HD = 64;             // columns of one LDS tile: the head dim, or one half of a head dim of 128
constexpr int BM = 128;            // rows (queries or keys) per work-group
constexpr int BN = 64;             // rows per streamed tile
constexpr int NTHREADS = 256;
constexpr int TILE_BYTES = BN * HD * 2;
constexpr int NSTAGE = 2;
constexpr int AUX_BYTES = 2048;                             // small per-tile data of a stage

// LDS map (bytes) for head dim 64 * NH: a stage holds the NH column halves of the first streamed
// matrix, then those of the second.
template <int NH> struct Cfg {
    static constexpr int STAGE_BYTES = 2 * NH * TILE_BYTES;
    static constexpr int OFF_B = NH * TILE_BYTES;           // second matrix inside a stage
    static constexpr int OFF_AUX = NSTAGE * STAGE_BYTES;
    static constexpr int OFF_LUT = OFF_AUX + NSTAGE * AUX_BYTES;
    static constexpr int LDS_BYTES = OFF_LUT + 256;
};

// Per-lane constants of the tile copies: wave w copies row blocks 2w and 2w+1 (8 rows each) of a
// 64-row tile; lane i fills LDS chunk (row 8*blk + i/8, position i%8) with global chunk
// position ^ swizzle16((row >> 1) & 7).
struct TileCopy {
    uint32_t chunk[2];      // byte offset of the lane's global chunk inside its row
    uint32_t chunk2[2];     // the same for the second column half
    int row[2];
};
// last_chunk: the row's last 16-byte chunk, which stands in for those beyond it
__device__ __forceinline__ TileCopy make_tile_copy(int wave, int lane, int last_chunk)
{
    TileCopy c;
#pragma unroll
    for (int j = 0; j < 2; ++j) {
        const int row = 8 * (2 * wave + j) + (lane >> 3);
        const int pos = lane & 7;
        c.row[j] = row;
        const int chunk = pos ^ swizzle16((row >> 1) & 7);
        c.chunk[j] = (uint32_t)(chunk < last_chunk ? chunk : last_chunk) << 4;
        c.chunk2[j] = (uint32_t)(chunk + 8 < last_chunk ? chunk + 8 : last_chunk) << 4;
    }
    return c;
}
// Copy the tile whose first row is row r0 of the N-row matrix `mat` (row stride sn elements, below
// 2^23); rows >= N re-read row N-1 (they are zeroed after landing).
template <int NH>
__device__ __forceinline__ void issue_tile(uint32_t dst, const uint16_t *mat, uint32_t sn, int r0,
                                           int N, const TileCopy &c, int wave)
{
    const uint16_t *src = mat + (size_t)r0 * sn;
    const int last = N - 1 - r0;
#pragma unroll
    for (int j = 0; j < 2; ++j) {
        const int r = c.row[j] < last ? c.row[j] : last;
        const uint32_t row = __umul24(r, 2u * sn);
        async_copy_b128(dst + wave * 2048 + j * 1024, src, row + c.chunk[j]);
        if constexpr (NH == 2) async_copy_b128(dst + TILE_BYTES + wave * 2048 + j * 1024, src, row + c.chunk2[j]);
    }
}
// Zero the rows >= N of the `parts` consecutive 64-column tiles that start at dst.
__device__ __forceinline__ void zero_tile_tail(uint32_t dst, int parts, int r0, int N, const TileCopy &c,
                                               int wave, int lane)
{
#pragma unroll
    for (int j = 0; j < 2; ++j)
        if (r0 + c.row[j] >= N) {
            const u32x4 z = {0u, 0u, 0u, 0u};
            for (int part = 0; part < parts; ++part)
                *(LDS_PTR(u32x4))(uintptr_t)(dst + part * TILE_BYTES + wave * 2048 + j * 1024 + lane * 16) = z;
        }
}

// ------------------------------------------------------------------------------------------------
// dQ (and delta)
// ------------------------------------------------------------------------------------------------
// Two products of 16-bit pairs more.  Delta is formed in the same order, and so with the same bits, by the dQ kernel and by attn_bwd_delta_kernel:
// by fmas over the 8 elements of a chunk and then of the one 8 chunks further, then chunks 2s and 2s + 1, then pairs of these.
template <bool BF16> __device__ __forceinline__ float add_products(uint32_t x, uint32_t y, float sum)
{
    using E = Elem<BF16>;
    sum = __builtin_fmaf(E::up1((uint16_t)(x & 0xffffu)), E::up1((uint16_t)(y & 0xffffu)), sum);
    return __builtin_fmaf(E::up1((uint16_t)(x >> 16)), E::up1((uint16_t)(y >> 16)), sum);
}
// HAVE_DELTA: attn_bwd_delta_kernel has left it
template <bool BF16, int HDIM, bool WIDE, bool HAVE_DELTA>
__device__ __forceinline__ void dq_rows(const AttnBwdArgs &a, unsigned char *smem, int bh, int qt)
{
    using E = Elem<BF16>;
    constexpr int NH = HDIM > 64 ? 2 : 1;         // 64-column tiles per matrix
    constexpr int KS = (HDIM + 31) / 32;          // MFMA steps of a contraction over the head dim
    constexpr int DB = HDIM / 16;                 // 16-column accumulator blocks of an output
    constexpr int AHEAD = HDIM <= 64 ? 2 : 3;     // steps by which an operand is requested before its use
    using C = Cfg<NH>;
    constexpr int STAGE_BYTES = C::STAGE_BYTES, OFF_AUX = C::OFF_AUX, OFF_LUT = C::OFF_LUT;
    const uint32_t lds0 = (uint32_t)(uintptr_t)(LDS_PTR(unsigned char))smem;

    const int tid = threadIdx.x;
    const int lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int l16 = lane & 15, q4 = lane >> 4;
    const int N = a.N, nw = (N + 31) >> 5;
    const int T = (N + BN - 1) / BN;
    const bool ragged = (N & (BN - 1)) != 0;
    const float pm = a.post_mul;

    const int bi = (int)fastdiv((uint32_t)bh, a.div_H), hi = bh - bi * a.H;
    const uint16_t *kb = slab(a.k, bi, hi), *vb = slab(a.v, bi, hi);
    const uint16_t *qb = slab(a.q, bi, hi), *dob = slab(a.dout, bi, hi), *ob = slab(a.out, bi, hi);
    const uint32_t *mb = slab(a.mask, bi, hi);

    // ---- this lane's two query rows: q^T and dO^T fragments (B operands), delta, lse ----
    u32x4 qf[2][KS], dof[2][KS];
    float L[2];                         // p = exp2(pm * s - L); rows that kept nothing (lse = -inf) and rows beyond N get L = +inf
    f32x4 from_delta[2];                // what the dP accumulators start from
#pragma unroll
    for (int qb_ = 0; qb_ < 2; ++qb_) {
        const int qrow = qt * BM + wave * 32 + 16 * qb_ + l16;
        const int qr = qrow < N ? qrow : N - 1;
        u32x4 of[KS];
        load_row(qf[qb_], qb, a.q.sn, qr, q4, a.D);
        load_row(dof[qb_], dob, a.dout.sn, qr, q4, a.D);
        float delta = 0.f, d2[2] = {0.f, 0.f};
        if constexpr (HAVE_DELTA) delta = a.delta[(size_t)bh * N + qr];
        else load_row(of, ob, a.out.sn, qr, q4, a.D);
#pragma unroll
        for (int s = 0; s < KS; ++s)
#pragma unroll
            for (int i = 0; i < 4; ++i) {
                if constexpr (!HAVE_DELTA) d2[s & 1] = add_products<BF16>(dof[qb_][s][i], of[s][i], d2[s & 1]);
                qf[qb_][s][i] = E::pack2_rne(E::up1((uint16_t)(qf[qb_][s][i] & 0xffffu)) * a.q_scale, E::up1((uint16_t)(qf[qb_][s][i] >> 16)) * a.q_scale);
            }
        if constexpr (!HAVE_DELTA) {
            delta = xhalf_sum(xrow_sum(d2[0])) + xhalf_sum(xrow_sum(d2[1]));
            if (qrow < N && q4 == 0) a.delta[(size_t)bh * N + qrow] = delta;
        }
        const float lse_row = a.lse[(size_t)bh * N + qr];
        L[qb_] = (qrow >= N || lse_row == -__builtin_inff()) ? __builtin_inff() : lse_row * LOG2E;
        from_delta[qb_] = f32x4{-delta, -delta, -delta, -delta};
    }
    // kept, the first MFMAs of a tile read them in place
    asm volatile("" : "+v"(from_delta[0]), "+v"(from_delta[1]));

    // ---- copies ----
    const TileCopy tc = make_tile_copy(wave, lane, (a.D >> 3) - 1);
    const int mrow = qt * BM + wave * 32 + (lane >> 1);
    const uint32_t m_voff = (uint32_t)(((size_t)(mrow < N ? mrow : N - 1) * nw + (lane & 1)) * 4);
    auto issue = [&](int t, int st) {
        uint32_t voff = m_voff;
        if (2 * t + 1 >= nw) voff -= (lane & 1) * 4;          // odd word count: re-read the last word
        async_copy_b32(lds0 + OFF_AUX + st * AUX_BYTES + wave * 256, mb + 2 * t, voff);
        issue_tile<NH>(lds0 + st * STAGE_BYTES, kb, a.k.sn, t * BN, N, tc, wave);
        issue_tile<NH>(lds0 + st * STAGE_BYTES + C::OFF_B, vb, a.v.sn, t * BN, N, tc, wave);
    };
    // With a tile map only the key tiles that hold a set mask bit for this work-group's rows are
    // visited (the map has one row of "live" bits per block of 64 query rows: two of them are ORed);
    // without one, all.  Wave-uniform walk over the set bits, a word (32 tiles) at a time.
    const int TW = (T + 31) >> 5;
    const uint32_t *mapw = nullptr, *mapw2 = nullptr;
    if (a.tile_map != nullptr) {
        mapw = a.tile_map + bi * a.map_sb + hi * a.map_sh + (size_t)(2 * qt) * 2 * TW;
        mapw2 = (2 * qt + 1 < T) ? mapw + 2 * TW : mapw;
    }
    int cur_w = -1;
    uint32_t live_w = 0u;
    auto next_tile = [&]() __attribute__((always_inline)) -> int {     // next live tile, T if there is none
        while (live_w == 0u) {
            if (++cur_w >= TW) return T;
            uint32_t lv = 0xffffffffu;
            if (mapw != nullptr) lv = __builtin_amdgcn_readfirstlane(mapw[cur_w] | mapw2[cur_w]);
            if (cur_w == TW - 1 && (T & 31) != 0) lv &= (1u << (T & 31)) - 1u;
            live_w = lv;
        }
        const int b = __builtin_ctz(live_w);
        live_w &= live_w - 1u;
        return 32 * cur_w + b;
    };
    const int t_first = next_tile();
    if (t_first < T) issue(t_first, 0);
    if (tid < 64)
        reinterpret_cast<float *>(smem + OFF_LUT)[tid] = (((tid >> 2) >> (tid & 3)) & 1) ? 0.f : -__builtin_inff();

    f32x4 oacc[2][DB];                  // 16 columns of dQ of 16 rows each
#pragma unroll
    for (int x = 0; x < 2; ++x)
#pragma unroll
        for (int b = 0; b < DB; ++b) oacc[x][b] = f32x4{0.f, 0.f, 0.f, 0.f};
    const uint32_t lut_addr = lds0 + OFF_LUT;
    const uint32_t nib_rotate = (4u * q4 + 28u) & 31u;     // right: the nibble of keys 4q4 .. 4q4 + 3 comes to bits 4 .. 7

    uint32_t row_at = make_tile_read(lane).row, col_at = make_tile_read(lane).col;
    // one key tile; the ring stage is a compile-time constant, as in the dK/dV kernel, so that every LDS address is a register plus an
    // immediate.  4 x 32 heads, N = 4096, D = 128: 1275 us, 1.29 PFLOP/s, the matrix cores busy two thirds of the time at 1.86 GHz
    auto tile = [&](int t, int t_next, auto st_c) __attribute__((always_inline)) {
        constexpr int st = decltype(st_c)::value;
        const uint32_t so = lds0 + st * STAGE_BYTES;
        WAIT_VMCNT(0);
        if (ragged && t == T - 1) zero_tile_tail(so, 2 * NH, t * BN, N, tc, wave, lane);
        __syncthreads();          // tile t of every wave landed; the other stage is free
        if (t_next < T) issue(t_next, st ^ 1);

        // Steps of two products each: S^T of 32 keys (mask bias as initial value), dP^T of them, then the same of the other 32, then dQ^T += K^T dS^T.
        // Element j of [kb][x] <-> key 32blk + 16kb + 4q4 + j, row 16x + l16.
        asm volatile("" : "+v"(row_at), "+v"(col_at));       // or the compiler keeps a register for every address that follows from these
        auto k_row = [&](int blk, int n) __attribute__((always_inline)) {        // step n: key block n & 1, columns 32 (n >> 1)
            return lds_read_b128((row_at ^ (64 * ((n >> 1) & 1))) + so + (n >> 2) * TILE_BYTES + 4096 * blk + 2048 * (n & 1));
        };
        auto v_row = [&](int blk, int n) __attribute__((always_inline)) {
            return lds_read_b128((row_at ^ (64 * ((n >> 1) & 1))) + so + C::OFF_B + (n >> 2) * TILE_BYTES + 4096 * blk + 2048 * (n & 1));
        };
        auto k_col = [&](int blk, int b) __attribute__((always_inline)) {
            const uint32_t ko = (col_at ^ (32 * (b & 3))) + so + (b >> 2) * TILE_BYTES + 4096 * blk;
            const u32x2 lo = lds_read_tr16_b64(ko), hi = lds_read_tr16_b64(ko + 2048);
            return u32x4{lo.x, lo.y, hi.x, hi.y};
        };
        // The operands of a step are requested AHEAD steps before it, and scheduling barriers hold that order: left alone, the compiler
        // requests each just before its use.
        constexpr int PH = 2 * KS;                    // steps of a phase
        u32x4 ring[AHEAD + 1];
        auto fetch = [&](int n) __attribute__((always_inline)) {
            u32x4 &r = ring[n % (AHEAD + 1)];
            if (n < PH) r = k_row(0, n);
            else if (n < 2 * PH) r = v_row(0, n - PH);
            else if (n < 3 * PH) r = k_row(1, n - 2 * PH);
            else if (n < 4 * PH) r = v_row(1, n - 3 * PH);
            else if (n < 4 * PH + DB) r = k_col(0, n - 4 * PH);
            else if (n < 4 * PH + 2 * DB) r = k_col(1, n - 4 * PH - DB);
        };
        u32x2 w2[2];
#pragma unroll
        for (int x = 0; x < 2; ++x) w2[x] = lds_read_b64(lds0 + OFF_AUX + st * AUX_BYTES + wave * 256 + 128 * x + l16 * 8);
#pragma unroll
        for (int n = 0; n < AHEAD; ++n) fetch(n);
        __builtin_amdgcn_sched_barrier(0);
#pragma unroll
        for (int x = 0; x < 2; ++x)
            if (t == T - 1) { w2[x].x &= a.last_mask0; w2[x].y &= a.last_mask1; }
        if (__builtin_amdgcn_ballot_w64((w2[0].x | w2[0].y | w2[1].x | w2[1].y) != 0u) == 0ull) return;

        u32x4 pb[2][2];
        f32x4 sacc[2][2][2], dacc[2][2][2];           // [blk]: a block's registers are free again when its dS is packed
        auto bias = [&](int blk) __attribute__((always_inline)) {
#pragma unroll
            for (int x = 0; x < 2; ++x) {
                const uint32_t w = blk == 0 ? w2[x].x : w2[x].y;
                const uint32_t wa = __builtin_amdgcn_alignbit(w, w, nib_rotate);
                sacc[blk][0][x] = __builtin_bit_cast(f32x4, lds_read_b128(lut_addr + (wa & 0xF0u)));
                sacc[blk][1][x] = __builtin_bit_cast(f32x4, lds_read_b128(lut_addr + ((wa >> 16) & 0xF0u)));
            }
        };
        auto weight = [&](int blk, int e) __attribute__((always_inline)) {       // element e of 16
            const int kb = e >> 3, x = (e >> 2) & 1, j = e & 3;
            sacc[blk][kb][x][j] = __builtin_amdgcn_exp2f(__builtin_fmaf(sacc[blk][kb][x][j], pm, -L[x]));
        };
        auto dscore = [&](int blk, int i) __attribute__((always_inline)) {       // dS^T / scale = P^T o (dP^T - delta), pair i of 8, packed as B operand
            const int kb = i >> 2, x = (i >> 1) & 1, j = 2 * (i & 1);
            pb[blk][x][2 * kb + (i & 1)] = E::pack2_rne(sacc[blk][kb][x][j] * dacc[blk][kb][x][j], sacc[blk][kb][x][j + 1] * dacc[blk][kb][x][j + 1]);
        };
        bias(0);
#pragma unroll
        for (int n = 0; n < 4 * PH + 2 * DB; ++n) {
            fetch(n + AHEAD);
            if (n == 2 * PH - 2) bias(1);
            __builtin_amdgcn_sched_barrier(0);
            const u32x4 &r = ring[n % (AHEAD + 1)];
            const int ph = n / PH, m = n % PH, blk = ph >> 1, kb = m & 1, c = m >> 1;
            if (n >= 4 * PH) {
                const int k = n - 4 * PH, b = k % DB;
#pragma unroll
                for (int x = 0; x < 2; ++x) oacc[x][b] = E::mfma(r, pb[k / DB][x], oacc[x][b]);
                if (k < DB) {
#pragma unroll
                    for (int i = 0; i < (8 + DB - 1) / DB; ++i)
                        if (k * ((8 + DB - 1) / DB) + i < 8) dscore(1, k * ((8 + DB - 1) / DB) + i);
                }
            } else if (ph == 0 || ph == 2) {
#pragma unroll
                for (int x = 0; x < 2; ++x) sacc[blk][kb][x] = E::mfma(r, qf[x][c], sacc[blk][kb][x]);
                if (ph == 2) {
#pragma unroll
                    for (int i = 0; i < (8 + PH - 1) / PH; ++i)
                        if (m * ((8 + PH - 1) / PH) + i < 8) dscore(0, m * ((8 + PH - 1) / PH) + i);
                }
            } else {
#pragma unroll
                for (int x = 0; x < 2; ++x) dacc[blk][kb][x] = E::mfma(r, dof[x][c], c == 0 ? from_delta[x] : dacc[blk][kb][x]);
#pragma unroll
                for (int i = 0; i < (16 + PH - 1) / PH; ++i)
                    if (m * ((16 + PH - 1) / PH) + i < 16) weight(blk, m * ((16 + PH - 1) / PH) + i);
            }
            __builtin_amdgcn_sched_barrier(0);
        }
    };
    for (int t = t_first; t < T;) {
        const int tn = next_tile();
        tile(t, tn, std::integral_constant<int, 0>{});
        if (tn >= T) break;
        t = next_tile();
        tile(tn, t, std::integral_constant<int, 1>{});
    }
    WAIT_VMCNT(0);
    __syncthreads();              // every wave is done reading the stages
    const int row0 = qt * BM + wave * 32;
    if (row0 < N) {
        store_gradient<BF16, WIDE>(oacc, a.scale, lds0 + wave * 4096, a, a.dq, bi, hi, row0, lane);
    }
}

template <bool BF16, int HDIM, bool WIDE>
__global__ __launch_bounds__(NTHREADS, HDIM > 64 ? 2 : 3) void attn_bwd_dq_kernel(const AttnBwdArgs a)
{
    __shared__ __attribute__((aligned(1024))) unsigned char smem[Cfg<(HDIM > 64 ? 2 : 1)>::LDS_BYTES];
    const Dealt d = deal(a.deal, a.qtiles, renumber_block());
    dq_rows<BF16, HDIM, WIDE, false>(a, smem, d.head, a.qtiles - 1 - d.tile);      // last rows first, as in the forward
}

// ------------------------------------------------------------------------------------------------
// dK and dV
// ------------------------------------------------------------------------------------------------
// NW wavefronts of 32 keys each.  The K fragments of a wavefront's keys stay in registers, and the V fragments where they
// fit.  VLDS: they wait in LDS, 16 bytes per lane and fragment in the order the lanes read them.
//   128  the accumulators of dK and dV take 128 registers; both gradients in one kernel form S once where a kernel
//        for each formed it twice: 2783 -> 2032 us on 4 x 32 heads, N = 4096 (now 1657, 1.33 PFLOP/s over four products)
//   64   166 registers instead of 198: three work-groups on a CU instead of two, where the grid has them (see the
//        launcher): 16 x 12 heads, N = 512, this kernel alone on warm inputs: 41.0 -> 37.3 us (691 TFLOP/s)
template <int HDIM, int NW, bool VLDS> struct DkvCfg {
    static constexpr int NH = HDIM > 64 ? 2 : 1;
    static constexpr int KS = (HDIM + 31) / 32;             // MFMA steps of a contraction over the head dim
    static constexpr int STAGE_BYTES = 2 * NH * TILE_BYTES;
    static constexpr int OFF_B = NH * TILE_BYTES;           // dO inside a stage
    static constexpr int AUX = NW * 256 + 512;              // per wavefront its mask words of 64 rows, then lse, delta
    static constexpr int OFF_AUX = NSTAGE * STAGE_BYTES;
    static constexpr int OFF_FRAG = OFF_AUX + NSTAGE * AUX; // V fragments of each wavefront
    static constexpr int FRAG = VLDS ? 2 * KS * 1024 : 0;   // of two blocks of 16 keys
    static constexpr int LDS_BYTES = OFF_FRAG + NW * FRAG;
};
template <bool BF16, int HDIM, int NW, bool VLDS, bool POSTMUL, bool WIDE, bool HALVES = false>
__device__ __forceinline__ void dkv_keys(const AttnBwdArgs &a, unsigned char *smem, int bh, int kt)
{
    using E = Elem<BF16>;
    constexpr int NH = HDIM > 64 ? 2 : 1;
    using C = DkvCfg<HDIM, NW, VLDS>;
    constexpr int KS = C::KS;
    constexpr int DB = HDIM / 16;
    constexpr int AHEAD = VLDS || HDIM == 32 ? 2 : 3;             // one more where there are registers for it
    constexpr int STAGE_BYTES = C::STAGE_BYTES, OFF_AUX = C::OFF_AUX, AUX_BYTES = C::AUX;
    constexpr int OFF_LSE = NW * 256, OFF_DELTA = OFF_LSE + 256;       // inside the small data of a stage
    const uint32_t lds0 = (uint32_t)(uintptr_t)(LDS_PTR(unsigned char))smem;

    const int tid = threadIdx.x;
    const int lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int l16 = lane & 15, q4 = lane >> 4;
    const int N = a.N, nw = (N + 31) >> 5;
    const int T = (N + BN - 1) / BN;
    const bool ragged = (N & (BN - 1)) != 0;
    const float pm = POSTMUL ? a.post_mul : 1.0f;
    const float lse_mul = -LOG2E / pm;                // pm is a power of two: exact

    const int bi = (int)fastdiv((uint32_t)bh, a.div_H), hi = bh - bi * a.H;
    const uint16_t *qb = slab(a.q, bi, hi), *dob = slab(a.dout, bi, hi);
    const uint16_t *kb_ = slab(a.k, bi, hi), *vb = slab(a.v, bi, hi);
    const uint32_t *mb = slab(a.mask, bi, hi);
    const float *lse_b = a.lse + (size_t)bh * N, *delta_b = a.delta + (size_t)bh * N;

    // ---- this lane's two keys: K^T (scaled) and V^T fragments, B operands ----
    // HALVES: a work-group of half the keys, in which the wavefronts of either half take 32 rows of every tile and their sums are added at the
    // end.  One CU holds one work-group of eight wavefronts, so a grid just beyond a round took two: its last heads, where work-groups of 128 keys
    // hold them all at once, come in such ones, each three quarters as long as a whole one.  The backward alone, before -> now, in us:
    //   36 heads, N = 2048: 377 -> 343 (causal 281 -> 247);  48: 394 -> 365;  68: 596 -> 560;  72, N = 1000: 206 -> 192;  18, N = 4000,
    //   causal: 489 -> 421;  forward + backward, 40, N = 2048, one mask in blocks: 276 -> 248.  Of 70 grids of 17 to 96 heads, random, causal and causal
    //   with a map, one lost: 24 heads, N = 3000, causal without a map, whose short work-groups fill the second round by themselves: 271 -> 286 (with a
    //   map 254 either way, random 514 -> 462).
    static_assert(!HALVES || (NW == 8 && VLDS && DB * 4096 * 4 <= C::LDS_BYTES), "four wavefronts' sums fit the LDS");
    constexpr int KW = HALVES ? 4 : NW;               // wavefronts side by side on different keys
    const int half = HALVES ? wave >> 2 : 0;          // ... and which 32 rows of every tile this one takes
    const int key0 = kt * (32 * KW) + (HALVES ? wave & 3 : wave) * 32;
    const bool wave_valid = key0 < N;                 // wave-uniform: some key of this wave exists
    const uint32_t wave_keys = N - key0 >= 32 ? 0xffffffffu : N > key0 ? (1u << (N - key0)) - 1u : 0u;      // of them the existing ones
    const int wi = (key0 >> 5) < nw ? (key0 >> 5) : nw - 1;     // this wave's mask word of a row
    const uint32_t frag = lds0 + C::OFF_FRAG + wave * C::FRAG + lane * 16;
    u32x4 kf[2][KS], vf[2][VLDS ? 1 : KS];
#pragma unroll
    for (int kb = 0; kb < 2; ++kb) {
        const int key = key0 + 16 * kb + l16;         // a key beyond N has sums that are not stored
        u32x4 v_all[KS];
        load_row(kf[kb], kb_, a.k.sn, key < N ? key : N - 1, q4, a.D);
        load_row(v_all, vb, a.v.sn, key < N ? key : N - 1, q4, a.D);
#pragma unroll
        for (int s = 0; s < KS; ++s) {
#pragma unroll
            for (int i = 0; i < 4; ++i) {
                kf[kb][s][i] = E::pack2_rne(E::up1((uint16_t)(kf[kb][s][i] & 0xffffu)) * a.q_scale, E::up1((uint16_t)(kf[kb][s][i] >> 16)) * a.q_scale);
            }
            if constexpr (VLDS) *(LDS_PTR(u32x4))(uintptr_t)(frag + (kb * KS + s) * 1024) = v_all[s];
            else vf[kb][VLDS ? 0 : s] = v_all[s];
        }
    }

    // ---- copies: Q tile, dO tile; per wave its mask word of the 64 rows; lse (wave 0), delta (wave 1)
    // (eight wavefronts: the first four copy Q, the others dO)
    const int cw = wave & 3;
    const TileCopy tc = make_tile_copy(cw, lane, (a.D >> 3) - 1);
    auto issue = [&](int t, int st) {
        const int r0 = t * BN;
        const int row = r0 + lane < N ? r0 + lane : N - 1;
        const uint32_t aux = lds0 + OFF_AUX + st * AUX_BYTES;
        async_copy_b32(aux + wave * 256, mb + wi, (uint32_t)((size_t)row * nw * 4));
        if (wave == 0) async_copy_b32(aux + OFF_LSE, lse_b, (uint32_t)(row * 4));
        if (wave == 1) async_copy_b32(aux + OFF_DELTA, delta_b, (uint32_t)(row * 4));
        if (NW == 4 || wave < 4) issue_tile<NH>(lds0 + st * STAGE_BYTES, qb, a.q.sn, r0, N, tc, cw);
        if (NW == 4 || wave >= 4) issue_tile<NH>(lds0 + st * STAGE_BYTES + C::OFF_B, dob, a.dout.sn, r0, N, tc, cw);
    };
    // With a tile map only the blocks of 64 query rows in which the mask keeps something for this
    // work-group's keys (KW / 2 key tiles: neighbouring bits of one word of the row block's "live"
    // bits) are visited: lane r of a wavefront looks at row block 64c + r, a
    // ballot turns the 64 answers into the bits that are walked.  Every wavefront does the same.
    const int TW = (T + 31) >> 5;
    const uint32_t *mapc = a.tile_map != nullptr
        ? a.tile_map + bi * a.map_sb + hi * a.map_sh + ((KW / 2 * kt) >> 5) : nullptr;
    int cur_c = -1;
    unsigned long long live_c = 0ull;
    auto next_tile = [&]() __attribute__((always_inline)) -> int {     // next live row block, T if there is none
        while (live_c == 0ull) {
            if (64 * ++cur_c >= T) return T;
            const int r = 64 * cur_c + lane;
            bool lv = r < T;
            if (mapc != nullptr && lv) lv = ((mapc[(size_t)r * 2 * TW] >> ((KW / 2 * kt) & 31)) & ((1u << (KW / 2)) - 1u)) != 0u;
            live_c = __builtin_amdgcn_ballot_w64(lv);
        }
        const int b = __builtin_ctzll(live_c);
        live_c &= live_c - 1ull;
        return 64 * cur_c + b;
    };
    const int t_first = next_tile();
    if (t_first < T) issue(t_first, 0);

    f32x4 dkacc[2][DB], dvacc[2][DB];     // 16 columns of 16 keys each
#pragma unroll
    for (int kb = 0; kb < 2; ++kb)
#pragma unroll
        for (int b = 0; b < DB; ++b) dkacc[kb][b] = dvacc[kb][b] = f32x4{0.f, 0.f, 0.f, 0.f};

    // bases of this lane's reads of the small data; opaque, because beyond 64 KiB the compiler would otherwise
    // keep a register for every sum of base and offset (40 of them) instead of using the offset field, and at 64
    // three work-groups on a CU leave no register to spare
    uint32_t aux_rows = lds0 + OFF_AUX + 16 * q4, aux_words = aux_rows + wave * 256, aux_lane = lds0 + OFF_AUX + 4 * lane;
    aux_rows += 128 * half;
    aux_words += 128 * half;
    if constexpr (VLDS || OFF_AUX >= 65536) asm volatile("" : "+v"(aux_rows), "+v"(aux_words), "+v"(aux_lane));

    uint32_t row_at = make_tile_read(lane).row + 4096 * half, col_at = make_tile_read(lane).col + 4096 * half;
    // one q tile; the ring stage is a compile-time constant so that every LDS address of the body is
    // a register plus an immediate
    auto tile = [&](int t, int t_next, auto st_c) __attribute__((always_inline)) {
        constexpr int st = decltype(st_c)::value;
        const uint32_t so = lds0 + st * STAGE_BYTES;
        WAIT_VMCNT(0);
        if (wave == 0) {
            // lse of the tile's rows -> what the score accumulators start from, -lse * log2(e) / pm, so
            // that exp2(pm * accumulator) is the probability; rows that kept nothing or lie beyond N
            // -> -inf (probability 0)
            const uint32_t p = aux_lane + st * AUX_BYTES + OFF_LSE;
            const float l = *(LDS_PTR(float))(uintptr_t)p;
            const bool dead = (t * BN + lane >= N) || (l == -__builtin_inff());
            *(LDS_PTR(float))(uintptr_t)p = dead ? -__builtin_inff() : l * lse_mul;
        }
        if (wave == 1) {
            // -delta: the dP accumulators start from it
            const uint32_t p = aux_lane + st * AUX_BYTES + OFF_DELTA;
            *(LDS_PTR(float))(uintptr_t)p = -*(LDS_PTR(float))(uintptr_t)p;
        }
        if (ragged && t == T - 1) {
            if (NW == 4) zero_tile_tail(so, 2 * NH, t * BN, N, tc, cw, lane);
            else zero_tile_tail(so + (wave >> 2) * C::OFF_B, NH, t * BN, N, tc, cw, lane);
        }
        __syncthreads();
        if (t_next < T) issue(t_next, st ^ 1);
        if (!wave_valid) return;

        // which rows keep any of this wavefront's keys, by one word a lane
        const uint32_t w = *(LDS_PTR(const uint32_t))(uintptr_t)(aux_lane + wave * 256 + st * AUX_BYTES);
        const unsigned long long live_rows = __builtin_amdgcn_ballot_w64((w & wave_keys) != 0u) >> (32 * half);
#pragma unroll
        for (int blk = 0; blk < (HALVES ? 1 : 2); ++blk) {
            if ((uint32_t)(live_rows >> (32 * blk)) == 0u) continue;
            asm volatile("" : "+v"(row_at), "+v"(col_at));
            // Element j of [rb][kb] <-> query row 32blk + 16rb + 4q4 + j of the tile, key 16kb + l16.
            // Steps of two products each: S (PH of them), dP (as many), dV (DB), dK (DB).  The operands of a step are requested AHEAD steps
            // before it, and scheduling barriers hold that order: left alone, the compiler requests each just before its use.  The exponentials
            // go beside dP's products, dS is formed beside dV's.
            constexpr int PH = 2 * KS;
            auto row = [&](int n) __attribute__((always_inline)) -> uint32_t {           // row block n & 1, columns 32 (n >> 1)
                return (row_at ^ (64 * ((n >> 1) & 1))) + so + (n >> 2) * TILE_BYTES + 4096 * blk + 2048 * (n & 1);
            };
            auto col = [&](int b, int off) __attribute__((always_inline)) {
                const uint32_t at = (col_at ^ (32 * (b & 3))) + so + off + (b >> 2) * TILE_BYTES + 4096 * blk;
                const u32x2 lo = lds_read_tr16_b64(at), hi = lds_read_tr16_b64(at + 2048);
                return u32x4{lo.x, lo.y, hi.x, hi.y};
            };
            auto rows_data = [&](int off, int rb) __attribute__((always_inline)) {
                return __builtin_bit_cast(f32x4, lds_read_b128(aux_rows + st * AUX_BYTES + off + 128 * blk + 64 * rb));
            };
            auto mask_words = [&](int rb) __attribute__((always_inline)) { return lds_read_b128(aux_words + st * AUX_BYTES + 128 * blk + 64 * rb); };
            u32x4 ring[AHEAD + 1], vs[2][2], mw[2], pp[2], ps[2];
            auto fetch = [&](int n) __attribute__((always_inline)) {
                u32x4 &r = ring[n % (AHEAD + 1)];
                if (n < PH) r = lds_read_b128(row(n));
                else if (n < 2 * PH) r = lds_read_b128(row(n - PH) + C::OFF_B);
                else if (n < 2 * PH + DB) r = col(n - 2 * PH, C::OFF_B);
                else if (n < 2 * PH + 2 * DB) r = col(n - 2 * PH - DB, 0);
            };
            auto fetch_v = [&](int c) __attribute__((always_inline)) {
#pragma unroll
                for (int kb = 0; kb < 2; ++kb) vs[c & 1][kb] = VLDS ? lds_read_b128(frag + (kb * KS + c) * 1024) : vf[kb][VLDS ? 0 : c];
            };
            // the accumulators start from the rows' -lse (scaled) and -delta (the same for both blocks of keys): the products then leave
            // s - lse and dP - delta, with no subtraction per element
            f32x4 sacc[2][2], dacc[2][2];
#pragma unroll
            for (int rb = 0; rb < 2; ++rb) sacc[rb][0] = sacc[rb][1] = rows_data(OFF_LSE, rb);
#pragma unroll
            for (int n = 0; n < AHEAD; ++n) fetch(n);
#pragma unroll
            for (int n = 0; n < 2 * PH + 2 * DB; ++n) {
                fetch(n + AHEAD);
                const int m = n % PH, rb = m & 1, c = m >> 1;
                if (n == PH - 2) {
                    fetch_v(0);
#pragma unroll
                    for (int i = 0; i < 2; ++i) dacc[i][0] = dacc[i][1] = rows_data(OFF_DELTA, i);
                }
                if (n == PH - 1) mw[0] = mask_words(0);
                if (n == PH + PH / 2 - 1) mw[1] = mask_words(1);
                if (n >= PH && n < 2 * PH && rb == 0 && c + 1 < KS) fetch_v(c + 1);
                __builtin_amdgcn_sched_barrier(0);
                const u32x4 &r = ring[n % (AHEAD + 1)];
                if (n < PH) {
#pragma unroll
                    for (int kb = 0; kb < 2; ++kb) sacc[rb][kb] = E::mfma(r, kf[kb][c], sacc[rb][kb]);
                } else if (n < 2 * PH) {
#pragma unroll
                    for (int kb = 0; kb < 2; ++kb) dacc[rb][kb] = E::mfma(r, vs[c & 1][kb], dacc[rb][kb]);
#pragma unroll
                    for (int i = 0; i < (16 + PH - 1) / PH; ++i) {
                        const int e = m * ((16 + PH - 1) / PH) + i, er = e >> 3, ek = (e >> 2) & 1, j = e & 3;
                        if (e < 16) {
                            const uint32_t keep = (uint32_t)__builtin_amdgcn_sbfe((int)mw[er][j], (uint32_t)(l16 + 16 * ek), 1u);
                            const float x = __builtin_amdgcn_exp2f(POSTMUL ? sacc[er][ek][j] * pm : sacc[er][ek][j]);
                            float p = __builtin_bit_cast(float, __builtin_bit_cast(uint32_t, x) & keep);
                            asm volatile("" : "+v"(p));              // here: the compiler would keep both operands of all 16 for the first use
                            sacc[er][ek][j] = p;
                        }
                    }
                    if (n == 2 * PH - 1) {
#pragma unroll
                        for (int i = 0; i < 8; ++i)
                            pp[(i >> 1) & 1][2 * (i >> 2) + (i & 1)] =
                                E::pack2_rne(sacc[i >> 2][(i >> 1) & 1][2 * (i & 1)], sacc[i >> 2][(i >> 1) & 1][2 * (i & 1) + 1]);
                    }
                } else if (n < 2 * PH + DB) {          // dV^T += dO^T P
                    const int b = n - 2 * PH;
#pragma unroll
                    for (int kb = 0; kb < 2; ++kb) dvacc[kb][b] = E::mfma(r, pp[kb], dvacc[kb][b]);
#pragma unroll
                    for (int q = 0; q < (8 + DB - 1) / DB; ++q) {
                        const int i = b * ((8 + DB - 1) / DB) + q, ir = i >> 2, ik = (i >> 1) & 1, j = 2 * (i & 1);
                        if (i < 8)
                            ps[ik][2 * ir + (i & 1)] = E::pack2_rne(sacc[ir][ik][j] * dacc[ir][ik][j], sacc[ir][ik][j + 1] * dacc[ir][ik][j + 1]);
                    }
                } else {                               // dK^T += Q^T dS
                    const int b = n - 2 * PH - DB;
#pragma unroll
                    for (int kb = 0; kb < 2; ++kb) dkacc[kb][b] = E::mfma(r, ps[kb], dkacc[kb][b]);
                }
                __builtin_amdgcn_sched_barrier(0);
            }
        }
    };
    for (int t = t_first; t < T;) {
        const int tn = next_tile();
        tile(t, tn, std::integral_constant<int, 0>{});
        if (tn >= T) break;
        t = next_tile();
        tile(tn, t, std::integral_constant<int, 1>{});
    }
    WAIT_VMCNT(0);
    __syncthreads();
    if constexpr (HALVES) {
        // the sums over the other 32 rows of every tile, from the wavefront that has the same keys
        const uint32_t sums = lds0 + (wave & 3) * (DB * 4096) + lane * 16;
        if (half == 1 && wave_valid) {
#pragma unroll
            for (int kb = 0; kb < 2; ++kb)
#pragma unroll
                for (int b = 0; b < DB; ++b) {
                    *(LDS_PTR(f32x4))(uintptr_t)(sums + (kb * DB + b) * 1024) = dkacc[kb][b];
                    *(LDS_PTR(f32x4))(uintptr_t)(sums + ((2 + kb) * DB + b) * 1024) = dvacc[kb][b];
                }
        }
        __syncthreads();
        if (half == 1 || !wave_valid) return;
        // One gradient after the other: with both sums in registers at once 17 to 20 of them were spilled, here and because of their allocation to the
        // whole kernel, which took 256 registers for 246 (36 heads, N = 2048, the backward alone: 329.6 -> 327.8 us; 128, N = 4096: 3326 -> 3308).
        auto add = [&](f32x4 (&acc)[2][DB], uint32_t at) __attribute__((always_inline)) {
#pragma unroll
            for (int kb = 0; kb < 2; ++kb)
#pragma unroll
                for (int b = 0; b < DB; ++b) {
                    if (b % 4 == 0) __builtin_amdgcn_sched_barrier(0);        // four blocks' sums in registers at a time
                    acc[kb][b] += *(LDS_PTR(const f32x4))(uintptr_t)(at + (kb * DB + b) * 1024);
                }
        };
        add(dkacc, sums);
        store_gradient<BF16, WIDE>(dkacc, a.scale, lds0 + wave * (DB * 4096), a, a.dk, bi, hi, key0, lane);      // over its own sums
        __builtin_amdgcn_sched_barrier(0);
        add(dvacc, sums + DB * 2048);
        store_gradient<BF16, WIDE>(dvacc, 1.0f, lds0 + wave * (DB * 4096), a, a.dv, bi, hi, key0, lane);
        return;
    }
    if (wave_valid) {
        store_gradient<BF16, WIDE>(dkacc, a.scale, lds0 + wave * 4096, a, a.dk, bi, hi, key0, lane);
        store_gradient<BF16, WIDE>(dvacc, 1.0f, lds0 + wave * 4096, a, a.dv, bi, hi, key0, lane);
    }
}

// (head dim 32: 128 registers, four work-groups on a CU; with the 136 that the compiler takes by itself three, 126 heads, N = 1664,
// dQ and dK/dV: 233.5 -> 238.6 us)
template <bool BF16, int HDIM, int NW, bool VLDS, bool POSTMUL, bool WIDE>
__global__ __launch_bounds__(64 * NW, HDIM == 128 ? NW / 4 : HDIM == 32 ? 4 : VLDS ? 3 : 2) void attn_bwd_dkv_kernel(const AttnBwdArgs a)
{
    __shared__ __attribute__((aligned(1024))) unsigned char smem[DkvCfg<HDIM, NW, VLDS>::LDS_BYTES];
    if constexpr (HDIM == 128 && NW == 8) {
        const int late = (int)blockIdx.x - a.whole_groups;
        if (late >= 0) {
            const int i = renumber_block(late, (int)gridDim.x - a.whole_groups);
            const int h = (int)fastdiv((uint32_t)i, a.div_qtiles);
            dkv_keys<BF16, HDIM, NW, VLDS, POSTMUL, WIDE, true>(a, smem, a.whole_heads + h, i - h * a.qtiles);
            return;
        }
    }
    const Dealt d = deal(a.deal, a.ktiles, HDIM == 128 && NW == 8 ? renumber_block((int)blockIdx.x, a.whole_groups) : renumber_block());
    dkv_keys<BF16, HDIM, NW, VLDS, POSTMUL, WIDE>(a, smem, d.head, d.tile);
}

// ------------------------------------------------------------------------------------------------
// both in one launch
// ------------------------------------------------------------------------------------------------
// The work-groups of a head follow each other, those of its keys (which take longer) first.  What that gives: a grid that is
// resident all at once runs both kinds side by side instead of one after the other; where rows and keys have unequal work the ends of the
// one fill with the other; and q, k, v and dO of a head come from memory once.  What it costs: delta beforehand, in a
// launch of its own, and dK/dV at the occupancy of both.  The backward alone, two launches -> this, in us:
//   one round     8 heads, N = 512: 29.6 -> 20.1;  64, N = 700: 51.3 -> 46.4;  20, N = 2048: 118 -> 105;  1, N = 4096: 173 -> 105;  D = 32: 8 heads, N = 333: 19.2 ->
//                 12.9;  D = 128: 16 heads, N = 512: 44.4 -> 30.4;  4, N = 4096: 259 -> 168
//   blocks, map   forward + backward, 12 heads, N = 1024: batch 16 156 -> 149, 8 86.7 -> 82.0, 4 66.9 -> 55.2;
//                 16 x 12, N = 700: 104.9 -> 95.2;  2 x 8, N = 4096: 178 -> 165
//   random, map   (one of a mask in which nothing can be skipped) 16 x 12 heads, N = 1024: 274.2 -> 275.5;  4 x 32, N = 2048: 687.7 -> 685.1;
//                 4 x 8, N = 4096: 672 -> 646;  3 x 12, N = 2048: 228.8 -> 206.5
//   up to a third beyond full rounds, with a map    random masks lose, those that a map is made for gain: 16 heads, N = 4096 random 260 -> 272, causal
//                 229 -> 185, blocks 135 -> 117;  13, N = 4096 237 -> 251, 220 -> 173, 131 -> 113;  64, N = 1024 79.1 -> 82.0, 68.2 -> 63.2, 52.5 ->
//                 49.1;  70, N = 700 52.5 -> 55.1, 44.1 -> 43.4, 42.1 -> 36.6
// Beyond one round and without a map it is left off: 192 heads, N = 1024: 214 -> 221; 60, N = 1000 (1.25 rounds): 74 -> 84 (causal masks would gain:
// 128, N = 1000: 125 -> 109, but the launcher doesn't see them; D = 32 with a map: 384 heads, N = 600: 94.2 -> 96.6;
// D = 96 with a map: blocks 8 x 12, N = 1024 145 -> 131, but 8 x 16, N = 2048 443 -> 447, and a random mask 907 -> 932).
//
// Delta of every row, eight lanes a row: whole lines at once (two lanes a row, with the fragments' access, took 10 us more of 150 on 16 x 12
// heads, N = 1024)
template <bool BF16> __global__ __launch_bounds__(NTHREADS) void attn_bwd_delta_kernel(const AttnBwdArgs a)
{
    const int N = a.N, bh = (int)fastdiv(blockIdx.x, a.div_qtiles), bi = (int)fastdiv((uint32_t)bh, a.div_H), hi = bh - bi * a.H;
    const uint16_t *dob = slab(a.dout, bi, hi), *ob = slab(a.out, bi, hi);
    const int c = threadIdx.x & 7;
#pragma unroll
    for (int j = 0; j < 4; ++j) {
        const int row = ((int)blockIdx.x - bh * a.qtiles) * BM + 32 * j + (int)(threadIdx.x >> 3), r = row < N ? row : N - 1;
        float d = 0.f;
        for (int chunk = c; 8 * chunk < a.D; chunk += 8) {
            const u32x4 x = *reinterpret_cast<const u32x4 *>(dob + (size_t)r * a.dout.sn + 8 * chunk);
            const u32x4 y = *reinterpret_cast<const u32x4 *>(ob + (size_t)r * a.out.sn + 8 * chunk);
#pragma unroll
            for (int i = 0; i < 4; ++i) d = add_products<BF16>(x[i], y[i], d);
        }
        // lane ^ 1, then lane ^ 2, then 7 - lane
        d += __builtin_bit_cast(float, __builtin_amdgcn_update_dpp(0, __builtin_bit_cast(int, d), 0xB1, 0xf, 0xf, true));
        d += __builtin_bit_cast(float, __builtin_amdgcn_update_dpp(0, __builtin_bit_cast(int, d), 0x4E, 0xf, 0xf, true));
        d += __builtin_bit_cast(float, __builtin_amdgcn_update_dpp(0, __builtin_bit_cast(int, d), 0x141, 0xf, 0xf, true));
        if (row < N && c == 0) a.delta[(size_t)bh * N + row] = d;
    }
}
template <bool BF16, int HDIM, bool POSTMUL, bool WIDE>
__global__ __launch_bounds__(NTHREADS, HDIM == 128 ? 1 : HDIM > 64 ? 2 : 3) void attn_bwd_both_kernel(const AttnBwdArgs a)
{
    constexpr bool VLDS = HDIM == 64 || HDIM == 128;
    constexpr int DQ = Cfg<(HDIM > 64 ? 2 : 1)>::LDS_BYTES, DKV = DkvCfg<HDIM, 4, VLDS>::LDS_BYTES;
    __shared__ __attribute__((aligned(1024))) unsigned char smem[DQ > DKV ? DQ : DKV];
    const Dealt d = deal(a.deal, a.ktiles, renumber_block());
    if (d.tile < a.qtiles) dkv_keys<BF16, HDIM, 4, VLDS, POSTMUL, WIDE>(a, smem, d.head, d.tile);
    else dq_rows<BF16, HDIM, WIDE, true>(a, smem, d.head, 2 * a.qtiles - 1 - d.tile);
}

template <bool BF16, int HDIM, bool POSTMUL, bool WIDE>
void launch_pair(hipStream_t stream, const AttnBwdArgs &args)
{
    AttnBwdArgs a = args;
    const long long groups = (long long)a.BH * a.qtiles, cus = compute_units();
    const bool alike = heads_alike(a.mask, a.H);
    // Both kinds of work-groups in one launch (see attn_bwd_both_kernel): while all are resident at once, or with a tile map
    if (2 * groups <= (HDIM == 128 ? 1 : HDIM > 64 ? 2 : 3) * cus ||
        (a.tile_map != nullptr && HDIM == 64 && groups < (1ll << 30))) {
        a.ktiles = 2 * a.qtiles;
        a.deal = make_deal(alike, a.BH, a.ktiles, (HDIM == 128 ? 1 : HDIM > 64 ? 2 : 3) * cus, 8ll * a.N * a.D);
        hipLaunchKernelGGL((attn_bwd_delta_kernel<BF16>), dim3((unsigned)groups), dim3(NTHREADS), 0, stream, a);
        hipLaunchKernelGGL((attn_bwd_both_kernel<BF16, HDIM, POSTMUL, WIDE>), dim3((unsigned)(2 * groups)), dim3(NTHREADS), 0, stream, a);
        return;
    }
    // dQ first: it also fills the delta workspace that the dK/dV kernel reads (same stream)
    a.deal = make_deal(alike, a.BH, a.qtiles, (HDIM > 64 ? 2 : HDIM == 64 ? 3 : 4) * cus, 4ll * a.N * a.D);
    hipLaunchKernelGGL((attn_bwd_dq_kernel<BF16, HDIM, WIDE>), dim3((unsigned)(a.BH * a.qtiles)), dim3(NTHREADS), 0, stream, a);
    auto dkv = [&](auto nw_c, auto vlds_c) {
        constexpr int NW = decltype(nw_c)::value;
        a.ktiles = (a.N + 32 * NW - 1) / (32 * NW);
        long long launched = (long long)a.BH * a.ktiles;
        int whole = a.BH;
        if constexpr (HDIM == 128 && NW == 8) {
            // heads beyond the last full round in work-groups of 128 keys, if these are one round at most (see HALVES at the kernel)
            const long long full = cus > 0 ? (launched - 1) / cus * cus / a.ktiles : a.BH, rest = a.BH - full;
            a.whole_heads = rest * a.qtiles <= cus ? (int)full : a.BH;
            whole = a.whole_heads;
            a.whole_groups = a.whole_heads * a.ktiles;
            launched = a.whole_groups + (long long)(a.BH - a.whole_heads) * a.qtiles;
        }
        a.deal = make_deal(alike, whole, a.ktiles, (HDIM == 128 ? 1 : HDIM == 32 ? 4 : decltype(vlds_c)::value ? 3 : 2) * cus, 4ll * a.N * a.D);
        hipLaunchKernelGGL((attn_bwd_dkv_kernel<BF16, HDIM, NW, decltype(vlds_c)::value, POSTMUL, WIDE>),
                           dim3((unsigned)launched), dim3(64 * NW), 0, stream, a);
    };
    using four = std::integral_constant<int, 4>;
    if constexpr (HDIM == 128) {
        // Eight wavefronts read Q and dO once per 256 keys and keep two of themselves on a SIMD, four leave a CU to one work-group:
        // 16 x 12 heads, N = 1024: 373 against 431 us.  A grid that four fill no more than once takes eight on 128 keys (the rows between
        // them, HALVES) from 641 keys on: 16 heads, N = 2048 145 -> 136 us, 6, N = 4000 256 -> 232, 28, N = 1088 81.0 -> 79.4;
        // 40, N = 700 57.2 either way, 60, N = 512 46.6 -> 47.9.  Four stay there, and on short keys of which 256 at a
        // time would leave a sixth or more idle (300 heads, N = 384, by halves: 134 -> 141).
        if (groups > cus ? a.qtiles % 2 == 0 || a.qtiles >= 5 : a.qtiles > 5) dkv(std::integral_constant<int, 8>{}, std::true_type{});
        else dkv(four{}, std::true_type{});
    } else if (HDIM == 64 && groups > 2 * cus && (2 * groups <= 7 * cus || groups > 4 * cus)) {
        // Three work-groups on a CU.  A grid that two of them on each CU hold does not need the third and pays for the reads
        // (128 heads, N = 448, the backward alone: 39.0 against 38.1 us), and from 3.5 to 4 per CU two full rounds of two
        // are as fast as one and a third of three.  Forward + backward, inputs from memory, two -> three: 2 to 3 per CU gain 2.5 to
        // 6.5 % (172 heads, N = 300: 59.3 -> 55.6 us; 192, N = 512: 95.6 -> 92.5; 48, N = 2048: 296 -> 288), 3 to 3.5 nothing (224,
        // N = 512: 117.6 either way) to 1.2 % the other way (56, N = 2048: 374.6 -> 379.3), beyond 4 1 to 3.5 % (400, N = 300:
        // 100.6 -> 97.2; 96, N = 2048: 570 -> 561).
        dkv(four{}, std::integral_constant<bool, HDIM == 64>{});
    } else {
        dkv(four{}, std::false_type{});
    }
}
template <int HDIM>
void launch_head_dim(bool bf16, hipStream_t stream, const AttnBwdArgs &a)
{
    const bool postmul = a.post_mul != 1.0f;       // exp2(pm * s) needs its multiplication only then
    if (a.grads_f32)                               // fp32 callers compute in bf16
        postmul ? launch_pair<true, HDIM, true, true>(stream, a) : launch_pair<true, HDIM, false, true>(stream, a);
    else if (bf16)
        postmul ? launch_pair<true, HDIM, true, false>(stream, a) : launch_pair<true, HDIM, false, false>(stream, a);
    else
        postmul ? launch_pair<false, HDIM, true, false>(stream, a) : launch_pair<false, HDIM, false, false>(stream, a);
}

}  // namespace

hipError_t launch_attn_bwd(const AttnBwdArgs &args, bool bf16, hipStream_t stream)
{
    AttnBwdArgs a = args;
    a.div_qtiles = make_fastdiv((uint32_t)a.qtiles);
    a.div_H = make_fastdiv((uint32_t)a.H);
    if ((long long)a.BH * a.qtiles == 0) return hipSuccess;
    if (a.grads_f32 && !bf16) return hipErrorInvalidValue;
    if (launch_attn_bwd_head(a, bf16, stream)) return hipGetLastError();
    switch (kernel_head_dim(a.D)) {
    case 128: launch_head_dim<128>(bf16, stream, a); break;
    case 96: launch_head_dim<96>(bf16, stream, a); break;
    case 80: launch_head_dim<80>(bf16, stream, a); break;
    case 64: launch_head_dim<64>(bf16, stream, a); break;
    default: launch_head_dim<32>(bf16, stream, a); break;
    }
    return hipGetLastError();
}

}  // namespace sma
