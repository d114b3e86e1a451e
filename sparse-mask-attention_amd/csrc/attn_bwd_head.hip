// dQ, dK and dV of a whole head in one work-group: sequences of at most 128 (head dims 96 and 128, four wavefronts), 256
// (eight) or 512 keys (head dims 32 and 64, 64 keys to a wavefront).  The formulas are those at the top of attn_bwd.hip.
//
// S, dP and the exponentials are formed once where the two kernels of attn_bwd.hip form them twice (five N x N x D products
// instead of seven), q, k, v and dO come from memory once, and there is one launch.  No sums between work-groups:
// bit-reproducible.
//   wavefront    32 KB keys, KB = 1 or 2, products of 16 x 16 x 32 (a lane has the keys lane % 16 and 16 more, as in the dK/dV kernel); dK and dV
//                are its accumulators, V fragments stay in registers.  Every operand that is read from LDS serves two products, those of dV
//                and dK 2 KB.
//   rows         32 at a time, in a ring of two stages: Q, dO, the mask words of each wavefront's keys.  The wavefront that has copied
//                eight rows also forms their delta (O comes with them) and Q scaled and rounded as the forward does it, so that
//                the probabilities fit its lse, in the place of O.  Delta of all rows before the first, as the two kernels have it,
//                made every work-group begin with twice the bytes while nothing is computed: 64.6 -> 57.7 us on 192 heads, N = 512,
//                D = 64, 175 -> 156 on 1024, N = 256, D = 128.  Scaling by every wavefront for itself: 4 us more on the first.
//   K            all of it in LDS, both as the operand of S and, read transposed, of dQ
//   dS           to LDS as [key][row], 64 bytes a key; after the next barrier the wavefronts share dQ^T = K^T dS^T of the 32 rows
//                in blocks of 16 x 16.  Eight wavefronts have two such buffers and one barrier for 32 rows; four have one,
//                so that two work-groups share a CU, and two barriers.
// Swizzles: Q and dO as everywhere in the backward (swizzle16 of row / 2), K by 16 bytes with the bits (2 ^ 1, 0, 1) of row / 2
// and dS by 8 bytes with the bits (1, 0, 2) of key / 4: the row accesses (see swizzle16) and the transposing reads of 16 keys x 16
// columns that dQ needs, keys 8q4 + 0 .. 3 and then + 4 .. 7 of the sixteens q4, stay free of bank conflicts.  The 8-byte writes don't: those of dS
// (eight a wavefront for 32 rows) and of the epilogue's transposes meet in pairs on the 32 banks that a write sees, 4 cycles more each.  These are all that the counter shows, on
// 192 heads, N = 512, D = 64 786432 + 196608 cycles of 9968640 in which LDS is active.
//
// The backward alone, inputs in turn, in us, before (two kernels, up to 256 keys at head dims up to 64 an earlier form of this
// one) -> now:
//   D =  64   N = 512: 192 heads 69.5 -> 57.7, 256: 93.6 -> 66.4;  N = 256: 1024 heads 102.4 -> 81.6, causal 95.7 -> 75.6, 256: 26.8 -> 24.7;
//             2048 heads, N = 32: 26.6 -> 20.0
//   D = 128   N = 256: 256 heads 54.0 -> 40.4, 1024: 212 -> 156;  1024 heads: N = 128 98.8 -> 64.3, N = 64 54.9 -> 31.9
//   D =  32   1024 heads, N = 256: 66.1 -> 53.7;  192, N = 512: 45.3 -> 39.8;   D = 96   1024 heads, N = 128: 57.1 -> 48.1
// Products of 32 x 32 x 16 and exp2(fma(s, post_mul, -lse)) -> products of 16 x 16 x 32, the exponentials of one block of keys beside the products of
// dP and dS beside dV's, accumulators that start from -lse, no multiplication where post_mul is 1 (the backward alone, us):
//   D =  64   N = 512: 192 heads 52.1 -> 50.1, 256 58.6 -> 55.1, causal 49.2 -> 46.7;  640, N = 400: 131.9 -> 123.5;  1024, N = 256, causal 62.7 ->
//             60.8;  1024, N = 128 28.2 -> 26.9;  192, N = 512, blocks 45.6 -> 42.7
//   D = 128   1024 heads, N = 256 154 -> 146, 256 35.6 -> 34.1;  up to 128 keys, bound by memory, the same (1024, N = 128 50.3, 50.4)
//   D =  32   192 heads, N = 512 37.6 -> 36.4;  1024, N = 256 47.0 -> 45.3
// What bounds it: on 192 heads, N = 512, D = 64 some 5900 cycles for 32 rows: dQ's 16 products a wavefront 1400 to 2000 of them (LDS round trips and, for the
// wavefronts that copy, the addresses of the mask words, 64 lines a copy), S to dK 4000 (of a SIMD's two wavefronts 2050 cycles of products, 1800 of vector ALU,
// and LDS round trips that no registers are left to hide), the rest for delta, scaling and the barrier.  Starting half of the wavefronts with
// dQ and half with S changed nothing; nor did four or six of dQ's operands on their way instead of two (57.2 us with the registers it took).  Prologue
// and epilogue, some 20000 cycles of 115000, move 256 KB of every CU at what memory gives.
#include <type_traits>

#include "attn_bwd_common.h"

namespace sma {
namespace {

template <int HDIM, int NW, int KB> struct HeadCfg {
    static constexpr int NH = HDIM > 64 ? 2 : 1;                    // column halves of 64
    static constexpr int KEYS = 32 * NW * KB;                       // and rows, at most
    static constexpr int K_HALF = KEYS * 128;
    static constexpr int OFF_DS = NH * K_HALF;
    static constexpr int DS_BYTES = KEYS * 64;                      // dS of 32 rows: [key][row]
    static constexpr int DS_BUFS = NW == 8 ? 2 : 1;
    static constexpr int PART = NH * 4096;                          // 32 rows of one matrix
    static constexpr bool LAND = !(NW == 4 && NH == 2);             // scaled Q in LDS (there two work-groups would not fit)
    // a stage: Q, dO, scaled Q (before that O, of which delta is formed), each wavefront's mask words, lse and delta
    static constexpr int OFF_WORDS = (LAND ? 3 : 2) * PART;
    static constexpr int OFF_LSE = OFF_WORDS + NW * 256, OFF_DELTA = OFF_LSE + 256;       // (a copy fills 64 places of lse)
    static constexpr int STAGE_BYTES = OFF_DELTA + 128;
    static constexpr int OFF_STAGE = OFF_DS + DS_BUFS * DS_BYTES;
    static constexpr int OFF_LIVE = OFF_STAGE + 2 * STAGE_BYTES;    // [buffer][wavefront]
    static constexpr int LDS_BYTES = OFF_LIVE + 64;
};

__device__ __forceinline__ u32x4 tr_pair(uint32_t lo, uint32_t hi)
{
    const u32x2 x = lds_read_tr16_b64(lo), y = lds_read_tr16_b64(hi);
    return u32x4{x.x, x.y, y.x, y.y};
}

template <bool BF16, int HDIM, int NW, int KB, bool POSTMUL, bool WIDE>
__global__ __launch_bounds__(64 * NW, HDIM <= 64 && KB == 1 && NW == 4 ? 3 : 2) void attn_bwd_head_kernel(const AttnBwdArgs a)
{
    using E = Elem<BF16>;
    using C = HeadCfg<HDIM, NW, KB>;
    constexpr int NH = C::NH, KS = HDIM / 32, DB = HDIM / 16;
    __shared__ __attribute__((aligned(1024))) unsigned char smem[C::LDS_BYTES];
    const uint32_t lds0 = (uint32_t)(uintptr_t)(LDS_PTR(unsigned char))smem;

    const int tid = threadIdx.x;
    const int lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int l16 = lane & 15, q4 = lane >> 4;
    const int bh = renumber_block();
    const int N = a.N, nw = (N + 31) >> 5;
    const int RB = (N + 31) >> 5;                     // blocks of 32 rows
    const float pm = POSTMUL ? a.post_mul : 1.0f, lse_mul = -LOG2E / pm;        // pm is a power of two: exact

    const int bi = (int)fastdiv((uint32_t)bh, a.div_H), hi = bh - bi * a.H;
    const uint16_t *qb = slab(a.q, bi, hi), *dob = slab(a.dout, bi, hi), *ob = slab(a.out, bi, hi);
    const uint16_t *kb_ = slab(a.k, bi, hi), *vb = slab(a.v, bi, hi);
    const uint32_t *mb = slab(a.mask, bi, hi);

    // ---- copies
    const int last_chunk = (a.D >> 3) - 1;
    auto chunk_at = [&](int c) __attribute__((always_inline)) -> uint32_t { return (uint32_t)(c < last_chunk ? c : last_chunk) << 4; };
    auto k_swizzle = [](int row) __attribute__((always_inline)) { const int p = (row >> 1) & 7; return ((p ^ (p << 1)) & 4) | ((p & 1) << 1) | ((p >> 1) & 1); };
    const int key0 = wave * (32 * KB);                // this wavefront's keys
    const bool wave_valid = key0 < N;                 // wave-uniform
    const int part = wave & 3;
    u32x4 o_next[C::LAND ? 1 : NH];                   // O where it does not go through LDS
    auto issue = [&](int i, auto st_c) __attribute__((always_inline)) {
        constexpr int SO = C::OFF_STAGE + decltype(st_c)::value * C::STAGE_BYTES;
        int ln = lane;
        asm volatile("" : "+v"(ln));                  // the few sums below are made again each time instead of kept
        const int prow = 8 * part + (ln >> 3);        // the row of a stage that this lane copies 16 bytes of
        const int pc = (ln & 7) ^ swizzle16((prow >> 1) & 7);
        const uint32_t pchunk = chunk_at(pc), pchunk2 = chunk_at(8 + pc);
        const int row = 32 * i + prow < N ? 32 * i + prow : N - 1;
        auto rows = [&](auto off_c, const uint16_t *mat, uint32_t sn) __attribute__((always_inline)) {
            constexpr int AT = SO + decltype(off_c)::value;
            const uint32_t r = __umul24(row, 2u * sn);
            async_copy_b128_at<AT>(lds0 + part * 1024, mat, r + pchunk);
            if constexpr (NH == 2) async_copy_b128_at<AT + 4096>(lds0 + part * 1024, mat, r + pchunk2);
        };
        if (wave < 4) {
            rows(std::integral_constant<int, 0>{}, qb, a.q.sn);
            rows(std::integral_constant<int, C::PART>{}, dob, a.dout.sn);
            if constexpr (C::LAND) {
                rows(std::integral_constant<int, 2 * C::PART>{}, ob, a.out.sn);
            } else {
                const uint32_t r = __umul24(row, 2u * a.out.sn);
                o_next[0] = *reinterpret_cast<const u32x4 *>(reinterpret_cast<const unsigned char *>(ob) + (r + pchunk));
                o_next[NH - 1] = *reinterpret_cast<const u32x4 *>(reinterpret_cast<const unsigned char *>(ob) + (r + pchunk2));
            }
        }
        if (wave == NW - 1) {
            const int lrow = 32 * i + (ln & 31) < N ? 32 * i + (ln & 31) : N - 1;
            async_copy_b32_at<SO + C::OFF_LSE>(lds0, a.lse + (size_t)bh * N, (uint32_t)(lrow * 4));
        }
        const int mword = KB == 2 ? wave * 2 + (ln >> 5) : wave, wi = mword < nw ? mword : nw - 1;
        const int mrow = 32 * i + (ln & 31) < N ? 32 * i + (ln & 31) : N - 1;
        async_copy_b32_at<SO + C::OFF_WORDS>(lds0 + wave * 256, mb, (uint32_t)((mrow * nw + wi) * 4));
    };
#pragma unroll
    for (int j = 0; j < 4 * KB; ++j) {                // its rows of K
        const int row = key0 + 8 * j + (lane >> 3), r = row < N ? row : N - 1;
        const int chunk = (lane & 7) ^ k_swizzle(row);
        const uint32_t off = __umul24(r, 2u * a.k.sn);
        async_copy_b128(lds0 + key0 * 128 + j * 1024, kb_, off + chunk_at(chunk));
        if constexpr (NH == 2) async_copy_b128(lds0 + C::K_HALF + key0 * 128 + j * 1024, kb_, off + chunk_at(8 + chunk));
    }
    issue(0, std::integral_constant<int, 0>{});

    // ---- V^T fragments of this lane's keys
    u32x4 vf[2 * KB][KS];                             // blocks of 16 keys
#pragma unroll
    for (int k = 0; k < 2 * KB; ++k) {
        const int key = key0 + 16 * k + l16, kr = key < N ? key : N - 1;
        const uint16_t *vp = vb + (size_t)kr * a.v.sn;
#pragma unroll
        for (int c = 0; c < KS; ++c) {                // columns beyond the row's end: its last ones, set to zero
            const int col = 32 * c + 8 * q4;
            vf[k][c] = *reinterpret_cast<const u32x4 *>(vp + (col < a.D ? col : a.D - 8)) & (col < a.D ? 0xffffffffu : 0u);
        }
    }
    if (tid < 16) *(LDS_PTR(uint32_t))(uintptr_t)(lds0 + C::OFF_LIVE + 4 * tid) = 0u;
    const bool keys_end = key0 + 32 * KB > N;         // wave-uniform: some of this wavefront's keys do not exist

    f32x4 dkacc[KB][2][DB], dvacc[KB][2][DB];
#pragma unroll
    for (int kb = 0; kb < KB; ++kb)
#pragma unroll
        for (int k = 0; k < 2; ++k)
#pragma unroll
            for (int b = 0; b < DB; ++b) dkacc[kb][k][b] = dvacc[kb][k][b] = f32x4{0.f, 0.f, 0.f, 0.f};

    // ---- read addresses
    // One register per pattern: a step along a row flips bits of the swizzled chunk, eight (four) rows further down flip
    // another and add their bytes; the rest is an immediate.
    uint32_t row_at = lds0 + C::OFF_STAGE + make_tile_read(lane).row, col_at = lds0 + C::OFF_STAGE + make_tile_read(lane).col;
    uint32_t key_at = lds0 + (key0 + l16) * 128 + ((q4 ^ k_swizzle(l16)) << 4);
    auto ds_swizzle = [](int key) __attribute__((always_inline)) { const int x = key >> 2; return ((x & 3) << 1) | ((x >> 2) & 1); };
    uint32_t ds_at = lds0 + C::OFF_DS + (key0 + l16) * 64 + ((q4 ^ ds_swizzle(l16)) << 3);
    uint32_t part_at = lds0 + 16 * q4, lane_at = lds0 + 4 * lane;      // rows 4q4 .. of the small data; this lane's word

    // dQ^T = K^T dS^T in blocks of 16 columns x 16 rows
    constexpr int NDB = HDIM / 16;
    constexpr int RH = NW >= 2 * NDB ? 1 : 2;         // row halves of a wavefront
    constexpr int PASSES = (NDB + NW - 1) / NW;   // its blocks of columns, NW apart: 64 columns
    static_assert(PASSES == 1 || NW == 4, "the blocks of a wavefront lie in different column halves");
    const int db = RH == 1 ? wave % NDB : wave, rh0 = RH == 1 ? wave / NDB : 0;
    unsigned char *dq_slab = reinterpret_cast<unsigned char *>(a.dq.p) + ((size_t)bi * a.dq.sb8 + (size_t)hi * a.dq.sh8) * (WIDE ? 32 : 16);
    const bool dq_wave = RH == 1 ? wave < 2 * NDB : wave < NDB;
    uint32_t dq_k, dq_s;
    {
        const int i16 = lane & 15, key = 8 * (lane >> 4) + (i16 >> 2);
        dq_k = lds0 + (db >> 2) * C::K_HALF + key * 128 + (((2 * (db & 3) + ((i16 & 3) >> 1)) ^ k_swizzle(key)) << 4) + ((i16 & 1) << 3);
        dq_s = lds0 + C::OFF_DS + key * 64 + (((4 * rh0 + (i16 & 3)) ^ ds_swizzle(key)) << 3);
    }

    // q as the forward multiplies it (scaled, rounded once more), so that the probabilities fit its lse
    auto scaled = [&](u32x4 x) __attribute__((always_inline)) {
#pragma unroll
        for (int j = 0; j < 4; ++j)
            x[j] = E::pack2_rne(E::up1((uint16_t)(x[j] & 0xffffu)) * a.q_scale, E::up1((uint16_t)(x[j] >> 16)) * a.q_scale);
        return x;
    };
    // after the copies of 32 rows, by the wavefronts that have made them: delta, scaled Q (in the place of O), lse
    auto land = [&](int i, auto st_c) __attribute__((always_inline)) {
        constexpr int SO = C::OFF_STAGE + decltype(st_c)::value * C::STAGE_BYTES;
        if (wave < 4) {
            int ln = lane;
            asm volatile("" : "+v"(ln));
            const int prow = 8 * part + (ln >> 3), chunk = (ln & 7) ^ swizzle16((prow >> 1) & 7);
            const uint32_t at = lds0 + 16 * ln + (SO + part * 1024);
            float delta = 0.f;
#pragma unroll
            for (int half = 0; half < NH; ++half) {
                const u32x4 x = lds_read_b128(at + C::PART + half * 4096);
                const u32x4 o = C::LAND ? lds_read_b128(at + 2 * C::PART + half * 4096) : o_next[C::LAND ? 0 : half];
                float d = 0.f;
#pragma unroll
                for (int j = 0; j < 4; ++j) {
                    d = __builtin_fmaf(E::up1((uint16_t)(x[j] & 0xffffu)), E::up1((uint16_t)(o[j] & 0xffffu)), d);
                    d = __builtin_fmaf(E::up1((uint16_t)(x[j] >> 16)), E::up1((uint16_t)(o[j] >> 16)), d);
                }
                delta += chunk + 8 * half <= last_chunk ? d : 0.f;            // beyond the row's end its last columns stand once more
                if constexpr (C::LAND) *(LDS_PTR(u32x4))(uintptr_t)(at + 2 * C::PART + half * 4096) = scaled(lds_read_b128(at + half * 4096));
            }
            // the eight lanes of a row
            delta += __builtin_bit_cast(float, __builtin_amdgcn_update_dpp(0, __builtin_bit_cast(int, delta), 0xB1, 0xf, 0xf, true));
            delta += __builtin_bit_cast(float, __builtin_amdgcn_update_dpp(0, __builtin_bit_cast(int, delta), 0x4E, 0xf, 0xf, true));
            delta += __builtin_bit_cast(float, __builtin_amdgcn_update_dpp(0, __builtin_bit_cast(int, delta), 0x141, 0xf, 0xf, true));
            if ((ln & 7) == 0) {
                *(LDS_PTR(float))(uintptr_t)(lds0 + (SO + C::OFF_DELTA) + 4 * prow) = -delta;
                if (32 * i + prow < N) a.delta[(size_t)bh * N + 32 * i + prow] = delta;
            }
        }
        if (wave == NW - 1 && lane < 32) {
            const uint32_t at = lane_at + (SO + C::OFF_LSE);
            const float l = *(LDS_PTR(float))(uintptr_t)at;
            // rows that kept nothing or lie beyond N: probability 0
            *(LDS_PTR(float))(uintptr_t)at = 32 * i + lane >= N || l == -__builtin_inff() ? -__builtin_inff() : l * lse_mul;
        }
    };
    // ---- 32 query rows: dV, dK, and dS into LDS
    auto rows32 = [&](auto st_c) __attribute__((always_inline)) {
        constexpr int st = decltype(st_c)::value;
        constexpr int DS = C::DS_BUFS == 2 ? st * C::DS_BYTES : 0;
        constexpr int SB = st * C::STAGE_BYTES;
        // opaque: the compiler would keep a register for every address that follows from these
        asm volatile("" : "+v"(row_at), "+v"(col_at), "+v"(key_at), "+v"(ds_at), "+v"(part_at), "+v"(lane_at));
        const uint32_t word_at = lane_at + (C::OFF_STAGE + SB + C::OFF_WORDS + wave * 256), words_at = part_at + (C::OFF_STAGE + SB + C::OFF_WORDS + wave * 256);
        uint32_t word = *(LDS_PTR(const uint32_t))(uintptr_t)(word_at);
        if (keys_end) {                               // nothing is kept of keys beyond N, whatever their bits
            int ln = lane;
            asm volatile("" : "+v"(ln));
            const int left = N - key0 - (KB == 2 ? ln & 32 : 0);
            word &= left >= 32 ? 0xffffffffu : left > 0 ? (1u << left) - 1u : 0u;
            *(LDS_PTR(uint32_t))(uintptr_t)(word_at) = word;
        }
        // Steps of two products (four where both blocks of 32 keys take part), kb = 0, 1 in turn: S (PH of them), dP (as many); then dV and dK (DB
        // each).  Operands are requested AHEAD steps before their use, and scheduling barriers hold that order: left alone, the compiler
        // requests each just before it is needed, since registers are short, and the wavefront sits out some 30 LDS round
        // trips one after the other.  The eight wavefronts go through these phases together, so what a wavefront's vector ALU does beside its own
        // products counts: the exponentials of kb lie in its dP, its dS in the S of the next or in dV.
        constexpr int PH = 2 * KS, SCORES = 2 * PH * KB, STEPS = SCORES + 2 * DB, AHEAD = KB == 2 ? HDIM == 64 ? 1 : 2 : 3;
        const uint32_t rows = part_at + (C::OFF_STAGE + SB + C::OFF_LSE);
        u32x4 ring[AHEAD + 1], kf[2][2];
        auto fetch = [&](int n) __attribute__((always_inline)) {
            u32x4 &r = ring[n % (AHEAD + 1)];
            if (n < SCORES) {                             // row block m & 1, columns 32 (m >> 1) of Q or dO
                const int m = n % PH, dp = n / PH & 1;
                r = lds_read_b128((row_at ^ (64 * ((m >> 1) & 1))) + SB + (dp ? C::PART : C::LAND ? 2 * C::PART : 0) + (m >> 2) * 4096 + 2048 * (m & 1));
            } else if (n < STEPS) {                       // dO^T, then Q^T, 16 columns
                const int b = (n - SCORES) % DB;
                const uint32_t at = (col_at ^ (32 * (b & 3))) + SB + (n - SCORES < DB ? C::PART : 0) + (b >> 2) * 4096;
                r = tr_pair(at, at + 2048);
            }
        };
        auto fetch_k = [&](int kb, int c) __attribute__((always_inline)) {
#pragma unroll
            for (int k = 0; k < 2; ++k) kf[c & 1][k] = lds_read_b128((key_at ^ (64 * (c & 1))) + (c >> 1) * C::K_HALF + 4096 * kb + 2048 * k);
        };
        u32x4 mw[2];                                      // mask words of 16 rows
        f32x4 sacc[KB][2][2], dacc[KB][2][2];             // [kb][rb][k]: rows 16rb + 4q4 + j, key 32kb + 16k + l16
        u32x4 pp[KB][2], ps[KB][2];
        auto weight = [&](int kb, int e) __attribute__((always_inline)) {           // element e of 16
            const int rb = e >> 3, k = (e >> 2) & 1, j = e & 3;
            const uint32_t keep = (uint32_t)__builtin_amdgcn_sbfe((int)mw[rb][j], (uint32_t)(l16 + 16 * k), 1u);
            const float x = __builtin_amdgcn_exp2f(POSTMUL ? sacc[kb][rb][k][j] * pm : sacc[kb][rb][k][j]);
            float p = __builtin_bit_cast(float, __builtin_bit_cast(uint32_t, x) & keep);
            asm volatile("" : "+v"(p));                   // here: the compiler would keep both operands of all 16 for the first use
            sacc[kb][rb][k][j] = p;
        };
        auto pack_weights = [&](int kb, int i) __attribute__((always_inline)) {     // pair i of 8
            const int rb = i >> 2, k = (i >> 1) & 1, j = 2 * (i & 1);
            pp[kb][k][2 * rb + (i & 1)] = E::pack2_rne(sacc[kb][rb][k][j], sacc[kb][rb][k][j + 1]);
        };
        auto dscore = [&](int kb, int i) __attribute__((always_inline)) {
            const int rb = i >> 2, k = (i >> 1) & 1, j = 2 * (i & 1);
            ps[kb][k][2 * rb + (i & 1)] = E::pack2_rne(sacc[kb][rb][k][j] * dacc[kb][rb][k][j], sacc[kb][rb][k][j + 1] * dacc[kb][rb][k][j + 1]);
            if (i & 1)
                *(LDS_PTR(u32x2))(uintptr_t)((ds_at ^ (32 * rb + 8 * k)) + DS + 2048 * kb + 1024 * k) = u32x2{ps[kb][k][2 * rb], ps[kb][k][2 * rb + 1]};
        };
        // the accumulators start from -lse (over pm) and -delta: the products leave s - lse and dP - delta, with no addition per element
        auto from_lse = [&](int kb) __attribute__((always_inline)) {
#pragma unroll
            for (int i = 0; i < 2; ++i) sacc[kb][i][0] = sacc[kb][i][1] = __builtin_bit_cast(f32x4, lds_read_b128(rows + 64 * i));
        };
        if (NW == 8) __builtin_amdgcn_s_setprio(0);
        from_lse(0);
        fetch_k(0, 0);
#pragma unroll
        for (int n = 0; n < AHEAD; ++n) fetch(n);
        __builtin_amdgcn_sched_barrier(0);                // requested before the words are looked at
        const bool live = __builtin_amdgcn_ballot_w64(word != 0u) != 0ull;         // dQ leaves out the others
        if (lane == 0) *(LDS_PTR(uint32_t))(uintptr_t)(lds0 + C::OFF_LIVE + (C::DS_BUFS == 2 ? 32 * st : 0) + 4 * wave) = live ? 1u : 0u;
        if (!live) return;
        static_assert(C::LAND || KB == 1, "one S of rows as they are");
        if constexpr (!C::LAND) ring[0] = scaled(ring[0]);
#pragma unroll
        for (int n = 0; n < STEPS; ++n) {
            fetch(n + AHEAD);
            const int kb = n / (2 * PH), m = n % PH, rb = m & 1, c = m >> 1;
            const bool dp = n / PH & 1;
            if (n < SCORES) {
                if (!dp && rb == 0 && c + 1 < KS) fetch_k(kb, c + 1);
                if (dp && kb + 1 < KB && m == PH - 1) fetch_k(kb + 1, 0);
                if (!dp && m == PH - 2) {
#pragma unroll
                    for (int i = 0; i < 2; ++i) {
                        dacc[kb][i][0] = __builtin_bit_cast(f32x4, lds_read_b128(rows + (C::OFF_DELTA - C::OFF_LSE) + 64 * i));
                        dacc[kb][i][1] = dacc[kb][i][0];
                    }
                }
                if (!dp && m == PH - 1) mw[0] = lds_read_b128(words_at + 128 * kb);
                if (dp && m == PH / 2 - 1) mw[1] = lds_read_b128(words_at + 128 * kb + 64);
                if (dp && kb + 1 < KB && m == PH - 2) from_lse(kb + 1);
            }
            __builtin_amdgcn_sched_barrier(0);
            if (n < SCORES && !dp) {
#pragma unroll
                for (int k = 0; k < 2; ++k) sacc[kb][rb][k] = E::mfma(ring[n % (AHEAD + 1)], kf[c & 1][k], sacc[kb][rb][k]);
                if constexpr (!C::LAND) {                 // the next step's
                    if (m + 1 < PH) ring[(n + 1) % (AHEAD + 1)] = scaled(ring[(n + 1) % (AHEAD + 1)]);
                }
            } else if (n < SCORES) {
                constexpr int EACH = (16 + PH - 1) / PH;
#pragma unroll
                for (int k = 0; k < 2; ++k) dacc[kb][rb][k] = E::mfma(ring[n % (AHEAD + 1)], vf[2 * kb + k][c], dacc[kb][rb][k]);
#pragma unroll
                for (int e = m * EACH; e < (m + 1) * EACH && e < 16; ++e) weight(kb, e);
                if (m == PH - 1) {
#pragma unroll
                    for (int i = 0; i < 8; ++i) {
                        pack_weights(kb, i);
                        if (kb + 1 < KB) dscore(kb, i);   // (at once: the registers that this frees are needed)
                    }
                }
            } else {
                const int b = (n - SCORES) % DB;
                const u32x4 &r = ring[n % (AHEAD + 1)];
#pragma unroll
                for (int x = 0; x < KB; ++x)
#pragma unroll
                    for (int k = 0; k < 2; ++k) {
                        if (n - SCORES < DB) dvacc[x][k][b] = E::mfma(r, pp[x][k], dvacc[x][k][b]);
                        else dkacc[x][k][b] = E::mfma(r, ps[x][k], dkacc[x][k][b]);
                    }
                if (n - SCORES < DB) {
                    constexpr int EACH = (8 + DB - 1) / DB;
#pragma unroll
                    for (int i = b * EACH; i < (b + 1) * EACH && i < 8; ++i) dscore(KB - 1, i);
                }
            }
            __builtin_amdgcn_sched_barrier(0);
        }
    };
    // ---- dQ of the 32 rows whose dS is complete
    auto dq32 = [&](int i, auto buf_c) __attribute__((always_inline)) {
        constexpr int BUF = C::DS_BUFS == 2 ? decltype(buf_c)::value : 0;
        if (!dq_wave) return;
        // The hardware serves the oldest wavefronts first; here the others would wait twice as long for their LDS reads, and all
        // of them for those at the next barrier: 61.9 -> 57.9 us on 192 heads, N = 512, D = 64
        if (NW == 8 && wave >= NW / 2) __builtin_amdgcn_s_setprio(1);
        int ln = lane;
        asm volatile("" : "+v"(ln));
        const uint32_t flag = *(LDS_PTR(const uint32_t))(uintptr_t)(lds0 + (C::OFF_LIVE + 32 * BUF) + 4 * (ln & (NW - 1)));
#pragma unroll
        for (int pass = 0; pass < PASSES; ++pass) {
            if (pass > 0 && wave + NW * pass >= NDB) break;
            constexpr int CH = RH == 1 ? 2 : 1;           // chains of products of a block
            f32x4 acc[RH][CH];
#pragma unroll
            for (int r = 0; r < RH; ++r)
#pragma unroll
                for (int c = 0; c < CH; ++c) acc[r][c] = f32x4{0.f, 0.f, 0.f, 0.f};
            asm volatile("" : "+v"(dq_k), "+v"(dq_s));
            constexpr int DEPTH = 2;                      // products whose operands are on their way
            u32x4 kt[DEPTH], dst[DEPTH][RH];
            auto fetch = [&](int ks) __attribute__((always_inline)) {
                constexpr int AT = BUF * C::DS_BYTES;
                kt[ks % DEPTH] = tr_pair(dq_k + (pass * C::K_HALF + 4096 * ks), (dq_k ^ 80) + (pass * C::K_HALF + 4096 * ks + 512));
#pragma unroll
                for (int r = 0; r < RH; ++r)
                    dst[ks % DEPTH][r] = tr_pair((dq_s ^ (32 * r)) + (AT + 2048 * ks), (dq_s ^ (32 * r + 16)) + (AT + 2048 * ks + 256));
            };
            auto product = [&](int ks) __attribute__((always_inline)) {
#pragma unroll
                for (int r = 0; r < RH; ++r) acc[r][ks % CH] = E::mfma(kt[ks % DEPTH], dst[ks % DEPTH][r], acc[r][ks % CH]);
            };
#pragma unroll
            for (int d = 0; d < DEPTH; ++d) fetch(d);     // before the flags are looked at
            __builtin_amdgcn_sched_barrier(0);
            const uint32_t live = (uint32_t)__builtin_amdgcn_ballot_w64(flag != 0u) & ((1u << NW) - 1u);
            if (live == (1u << NW) - 1u) {
#pragma unroll
                for (int ks = 0; ks < NW * KB; ++ks) {
                    __builtin_amdgcn_sched_barrier(0);
                    product(ks);
                    if (ks + DEPTH < NW * KB) fetch(ks + DEPTH);
                }
                __builtin_amdgcn_sched_barrier(0);
            } else {
#pragma unroll
                for (int w = 0; w < NW; ++w)
                    if (live >> w & 1u) {
#pragma unroll
                        for (int kb = 0; kb < KB; ++kb) {
                            fetch(w * KB + kb);
                            product(w * KB + kb);
                        }
                    }
            }
            const int col = 16 * db + 64 * pass + 4 * (ln >> 4);
#pragma unroll
            for (int r = 0; r < RH; ++r) {
                if constexpr (CH == 2) acc[r][0] += acc[r][1];
                const int row = 32 * i + 16 * (rh0 + r) + (ln & 15);
                if (row >= N || col >= a.D) continue;
                const uint32_t at = (uint32_t)row * a.dq.sn + (uint32_t)col;          // elements: a slab's bytes fit 31 bits
                const u32x2 h = {E::pack2_rne(acc[r][0][0] * a.scale, acc[r][0][1] * a.scale), E::pack2_rne(acc[r][0][2] * a.scale, acc[r][0][3] * a.scale)};
                if constexpr (WIDE)
                    *reinterpret_cast<f32x4 *>(dq_slab + 4 * at) = f32x4{E::up1((uint16_t)(h.x & 0xffffu)), E::up1((uint16_t)(h.x >> 16)),
                                                                  E::up1((uint16_t)(h.y & 0xffffu)), E::up1((uint16_t)(h.y >> 16))};
                else
                    *reinterpret_cast<u32x2 *>(dq_slab + 2 * at) = h;
            }
        }
    };

    WAIT_VMCNT(0);
    if (a.D < HDIM && lane < 32 * KB) {               // columns of K beyond the row's end add nothing to the scores
        for (int c = last_chunk + 1; c < 4 * KS; ++c)
            *(LDS_PTR(u32x4))(uintptr_t)(lds0 + (c >> 3) * C::K_HALF + (key0 + lane) * 128 + (((c & 7) ^ k_swizzle(lane)) << 4)) = u32x4{0u, 0u, 0u, 0u};
    }
    auto iteration = [&](int i, auto st_c) __attribute__((always_inline)) {
        constexpr int st = decltype(st_c)::value;
        using same = std::integral_constant<int, st>;
        using other = std::integral_constant<int, st ^ 1>;
        __syncthreads();                              // these 32 rows have landed; the other stage is done with
        if (i + 1 < RB) issue(i + 1, other{});
        if constexpr (C::DS_BUFS == 2) {
            if (i > 0) dq32(i - 1, other{});
            if (wave_valid && i < RB) rows32(same{});
            WAIT_VMCNT(0);
            if (i + 1 < RB) land(i + 1, other{});
        } else {
            if (wave_valid) rows32(same{});
            WAIT_VMCNT(0);
            if (i + 1 < RB) land(i + 1, other{});
            __syncthreads();
            dq32(i, same{});                          // its stores are nothing that the next rows wait for
        }
    };
    land(0, std::integral_constant<int, 0>{});
    constexpr int EXTRA = C::DS_BUFS == 2 ? 1 : 0;    // dQ of the last rows
    for (int i = 0; i < RB + EXTRA; i += 2) {
        iteration(i, std::integral_constant<int, 0>{});
        if (i + 1 < RB + EXTRA) iteration(i + 1, std::integral_constant<int, 1>{});
    }
    __syncthreads();
    if (wave_valid) {
#pragma unroll
        for (int kb = 0; kb < KB; ++kb) {
            if (key0 + 32 * kb >= N) break;
            store_gradient<BF16, WIDE>(dkacc[kb], a.scale, lds0 + wave * 4096, a, a.dk, bi, hi, key0 + 32 * kb, lane);
            store_gradient<BF16, WIDE>(dvacc[kb], 1.0f, lds0 + wave * 4096, a, a.dv, bi, hi, key0 + 32 * kb, lane);
        }
    }
}

template <bool BF16, int HDIM, int NW, int KB, bool WIDE> void launch(hipStream_t stream, const AttnBwdArgs &a)
{
    // exp2(pm * s) needs its multiplication only then
    const auto kernel = a.post_mul != 1.0f ? attn_bwd_head_kernel<BF16, HDIM, NW, KB, true, WIDE> : attn_bwd_head_kernel<BF16, HDIM, NW, KB, false, WIDE>;
    hipLaunchKernelGGL(kernel, dim3((unsigned)a.BH), dim3(64 * NW), 0, stream, a);
}
template <bool BF16, bool WIDE> bool pick(hipStream_t stream, const AttnBwdArgs &a)
{
    // Backward alone, inputs in turn, the kernels of attn_bwd.hip against this one, in us:
    // up to 256 keys always (D = 64, N = 256: 85 heads 19.1, 18.9, 256: 31.0, 24.0; 8 heads, N = 128: 9.8, 9.2; D = 128: 85 heads 30.9, 27.8).  From
    // 129 keys on few heads, of which the others give the rows and the keys a CU each, side by side in one launch, would be faster there (8
    // heads, N = 256: D = 64 13.3, 17.5, D = 128 20.0, 25.2; 64 heads 15.0, 18.5; more than 64 not), but dK and dV would be further from 64 bits than
    // they are: the others' dK/dV kernel scales and rounds k where the forward rounded scaled q (relative 2-norm of dK, bf16, N = 256, D = 64: 0.00312
    // against 0.00287; 0.00052 against 0.00050 in fp16 at N = 512).
    // 129 to 256 keys at head dims up to 64: eight wavefronts of 32 keys while every head has a CU of its own (256 heads 25.5, four
    // wavefronts of 64 keys 27.9), beyond that the four, two work-groups to a CU (300: 44.4 against 38.4).
    // 257 to 512 keys: a work-group has a CU for itself and a round takes the same time however few heads it holds, so that
    // most of the places must be taken, `need` of 32: more up to 384 keys, where a quarter or more of the wavefronts have no keys, and after
    // the first round at head dims up to 32, whose products are cheaper.  With a tile map the others visit only the tiles that hold
    // something, where here all rows are visited and wavefronts skip; but the gradients are the same bits with and without a map, so the line is
    // one for all masks.  Random masks without a map, and after the stroke blocks kept by a quarter, with one:
    //   D = 64   N = 512: 128 heads 46.5, 51.7;  160 59.2, 52.7 / 42.0, 48.0;  330 111, 106 / 73, 91;  400 134, 117 / 83, 94;  480 155, 125;
    //            600 188, 167 / 121, 138
    //            N = 320: 160 heads 32.1, 33.8;  175 38.3, 34.3;  400 69.0, 71.1;  440 79.3, 73.5 / 53.9, 59.6;  1000 155, 149 / 111, 118;
    //            1300 193, 210 (N = 300)
    //   D = 32   N = 512: 160 heads 41.8, 38.2;  320 69.4, 77.7;  400 88.6, 80.0 / 57.7, 66.3;  600 124, 121 / 80, 98;  700 137, 125 / 88, 100
    //            N = 384: 400 heads 54.7, 59.5;  480 63.4, 62.8;  768 92.5, 91.5 / 67.5, 79.2;  1300 148, 159 (N = 350)
    // Over 2000 such grids, masks and maps the kernel taken is on average 0.6 % behind the better one for random and causal masks, 2.7 % for
    // blocks with a map.
    const int D = kernel_head_dim(a.D), N = a.N;
    const long long cus = compute_units(), rounds = cus > 0 ? (a.BH + cus - 1) / cus : 1;
    const bool own_cu = a.BH <= cus;
    const int need = rounds == 1 ? (N > 384 ? 20 : 22) : N > 384 ? (D == 64 ? 23 : rounds == 2 ? 24 : 26) : D == 64 ? (rounds == 2 ? 27 : 29)
                                                                                                              : rounds == 2 ? 30 : 33;
    const bool filled = 32 * (long long)a.BH >= need * rounds * cus;
    auto narrow = [&](auto d_c) {
        constexpr int HDIM = decltype(d_c)::value;
        if (N <= 128) launch<BF16, HDIM, 4, 1, WIDE>(stream, a);
        else if (N <= 256) own_cu ? launch<BF16, HDIM, 8, 1, WIDE>(stream, a) : launch<BF16, HDIM, 4, 2, WIDE>(stream, a);
        else if (N <= 512 && filled) launch<BF16, HDIM, 8, 2, WIDE>(stream, a);
        else return false;
        return true;
    };
    auto wide = [&](auto d_c) {
        constexpr int HDIM = decltype(d_c)::value;
        if (N <= 128) launch<BF16, HDIM, 4, 1, WIDE>(stream, a);
        else if (N <= 256) launch<BF16, HDIM, 8, 1, WIDE>(stream, a);
        else return false;
        return true;
    };
    return D == 32 ? narrow(std::integral_constant<int, 32>{}) : D == 64 ? narrow(std::integral_constant<int, 64>{})
           : D <= 96 ? wide(std::integral_constant<int, 96>{}) : wide(std::integral_constant<int, 128>{});
}

}  // namespace

bool launch_attn_bwd_head(const AttnBwdArgs &a, bool bf16, hipStream_t stream)
{
    return a.grads_f32 ? pick<true, true>(stream, a) : bf16 ? pick<true, false>(stream, a) : pick<false, false>(stream, a);
}

}  // namespace sma
