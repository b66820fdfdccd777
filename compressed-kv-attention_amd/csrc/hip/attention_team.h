// The team split kernel (templates): one workgroup of two or four waves per
// split, instantiated per head_dim and score order in
// attention_team_d<D>_o<O>.hip.
#pragma once
// gfx950 fused decode attention at head_dim 80 to 256 (see kTeam), scalar/AVX2
// and AVX-512 BF16 score orders. The one-wave kernel (attention_wave.h) holds
// a chunk's rows, every row group's accumulators of every channel and a tile
// of 64 whole rows in one wave, which at these sizes leaves one or two waves
// per SIMD. Here W waves (2 up to head_dim 128, 4 above) share the chunk's
// tile and split its work, so that three or four waves fit a SIMD at every size
// (kTeamOcc):
//   1. wave w decodes rows [64 w / W, 64 (w + 1) / W) of the chunk's K rows
//      from registers into the tile and writes the escapes of its rows over
//      them, then requests its rows of the next chunk's K;
//   2. every wave takes all 64 tokens (lane = token) through its share of the
//      score chains: in the scalar order chains j with j % 4 in
//      [4 w / W, 4 (w + 1) / W) (whose sums are whole brackets of hsum8's
//      tree), in the AVX-512 order the quads of chains of the same numbers
//      (whole a_i of its tree), on the matrix cores as the one-wave kernel
//      does. The tile keeps each wave's channels of a K row together; when a
//      wave has read its own, it leaves the G partial scores in their place;
//   3. wave w adds the partial scores of query rows w, w + W, ... in the
//      tree's order and turns them into e and alpha;
//   4. wave w decodes its rows of V into the tile and requests the next ones;
//   5. wave w folds the chunk's tokens in order into D / W channels
//      (lane = channel); wave 0 also carries l.
// The operations of every score, coefficient and accumulator are those of
// the one-wave kernel in the same order, so the outputs are its bits.
//
// Bound: instruction issue, then HBM (SQ counters: the vector and matrix pipes
// are busy 77 % of a launch at head_dim 128, 68 % at 96 and 51 % at eight rows
// of 256, where three waves per SIMD wait at five barriers per chunk). Measured,
// per attention call, before (one wave per split at 128 and 256, a four-wave
// kernel on the vector ALU at the other sizes) and with teams: 64 heads x 4
// queries, head_dim 128, 65,536 tokens: 373 -> 332-338 us (4.8-4.9 TB/s);
// four sequences of up to 25,003 tokens x 8 heads x 8 queries, head_dim 256:
// 204 -> 90 us; 64 heads x 4 queries, head_dim 96, 16,411 tokens: 735 -> 83 us.
// At head_dim 64 one wave stays: half the lanes of a two-wave team's fold
// would carry no channel.
//
// An octet of channels is kept as four dwords, dword p = channels p and
// p + 4 of the octet: the pairs that share a bracket of hsum8's tree, and
// the ones a 4-bit octet's codes give without a byte select
// ((codes >> 4 p) & 0x000F000F).
#include "attention_wave.h"

namespace kvexp_dev {
namespace team {
using namespace wave;

template <int D>
struct TShape {
    static_assert(D % 16 == 0 && D >= 64 && D <= 256, "16-channel pieces; partial scores need 32 bytes per wave and row");
    static constexpr int W = D <= 128 ? 2 : 4;        // waves per workgroup
    static_assert(W == 2 || D % 32 == 0, "four K sub-rows start on 16 bytes");
    static constexpr int RO = kChunk / W;             // rows a wave decodes
    static constexpr int NP = D / 16;                 // 16-channel pieces per row
    static constexpr int RS = kWave / NP;             // whole rows per register
    static constexpr int NL = RS * NP;                // their lanes
    static constexpr int NR = (RO + RS - 1) / RS;     // registers of a wave's rows
    static constexpr int Last = (RO - RS * (NR - 1)) * NP - 1; // last register: the lane of the rows' last piece
    static constexpr int CW = D / W;                  // channels per wave (scores and fold)
    static constexpr int QR = (CW + 15) / 16;         // query operand registers per row group
    static constexpr int TS = 2 * D + 16;             // bytes per tile row
    static constexpr int RawRows = kChunk / 2;        // rows of a raw block per chunk (16-byte registers only)
};

template <int G, int D>
struct alignas(16) TeamLds {
    uint64_t exptab[32];
    uint8_t tile[kChunk * TShape<D>::TS];
    float eT[G][kRowPad]; // e of token t, row g (0 past the chunk's end)
    float aT[G][kRowPad]; // alpha of token t, row g (1 where no running maximum moves)
    uint64_t am[4];       // per wave: tokens that move a running maximum of its rows
    uint32_t low[4];      // AVX-512 order, plain BF16 rows: whether the wave's rows need the flushing scores
};

// Workgroup barrier for LDS traffic only: the global loads in flight stay in
// flight (the fence of __syncthreads would wait for them).
__device__ __forceinline__ void team_sync() {
    asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
    __builtin_amdgcn_s_barrier();
    asm volatile("" ::: "memory");
}

template <int D>
struct TRows {
    uint4 s[TShape<D>::NR]; // 16 sign/mantissa bytes of the lane's piece (raw block: 16 bytes of its rows)
    uint2 c[TShape<D>::NR]; // the 8 bytes that end with the piece's codes
    uint32_t sx, cx;        // shifted rows: the dwords that hold the wave's last two bytes of each stream
};

// The wave's rows of the next chunk: rows [r0 + RO w, r0 + RO (w + 1)) of the
// cursor's block, of the `rows` that the chunk may take from r0. Register k
// of lane l: piece l + NL k of them. A raw block's rows are split among the
// waves as its RawRows: bytes 1024 k + 16 l of the wave's run. Where the block
// holds a whole chunk of coded rows the addresses are the streams' starts plus
// the lane's offset (the lanes of the last register past the wave's rows
// repeat its last piece); elsewhere loads past the chunk's rows repeat their
// last piece. Both paths issue the same loads, which stay in the block but for
// the half dword named below.
//
// Blocks are 2-byte aligned, and loads of 16 or 8 bytes at an address that is
// not a multiple of 4 keep the CU's address unit about four times as long
// (cache-resident, 9.4 against 35.7 TB/s). So where a whole chunk of 4- or
// 2-bit rows starts 2 bytes past a multiple of 4, its streams are read from
// 2 bytes below (c.shift): the decode picks the sign/mantissa bytes with other
// byte selects and moves only the codes, and the two bytes that a piece lacks
// are in the next lane's first dword (the last lane's: in sx and cx, aligned
// dwords that start with them). Where a block without escapes ends with the
// wave's codes, the upper half of cx lies past the block, and past the container
// if it is the last one: an aligned dword whose lower half is inside is in the
// same page, so it can be read, and the upper half is not used. (Kept inside by
// 2-byte loads, or by the dword that ends with the codes and a shift, eight rows
// of head_dim 256 took 91.5 for 90.4 us, and three rows of one head x 4,096
// tokens 25.7 for 25.0.)
template <int D>
__device__ __forceinline__ void load_team_rows(Cursor &c, int w, int r0, int rows, TRows<D> &R) {
    using S = TShape<D>;
    const int mode = c.mode();
    const bool raw = mode == 0;
    c.lrows = rows;
    rows = max(rows, 1);
    const int lane = lane_here();
    const int cbytes = mode * (D / 8), cw = 2 * mode;
    const int cd = D + c.ntok() * D + cw - 8; // the load that ends with the codes of the block's piece 0
    c.shift = 0;
    // the dwords with the last bytes of the wave's rows (shifted rows; else any aligned dword of the block)
    const uint8_t *px = reinterpret_cast<const uint8_t *>(reinterpret_cast<uintptr_t>(c.blk + 8) & ~uintptr_t(3));
    const uint8_t *pc = px;
    if (!raw && c.ntok() - r0 >= kChunk) {
        const uint8_t *sb = c.blk + 8 + (D + (r0 + S::RO * w) * D);
        const uint8_t *cb = c.blk + 8 + (cd + (r0 + S::RO * w) * cbytes);
        if ((reinterpret_cast<uintptr_t>(c.blk) & 3u) == 2u && mode != 3) {
            c.shift = 1;
            sb -= 2;
            cb -= 2;
            px = sb + S::RO * D;
            pc = cb + (S::RO * cbytes + 8 - cw);
        }
        const int ll = S::Last < kWave - 1 ? min(lane, S::Last) : lane;
        const uint32_t cl = uint32_t(cw * lane);
#pragma unroll
        for (int k = 0; k < S::NR; ++k) {
            const bool end = k == S::NR - 1;
            R.s[k] = ld16(sb + 16 * S::NL * k + uint32_t(16 * (end ? ll : lane)));
            R.c[k] = ld8(cb + (uint32_t(cw * S::NL * k) + (end ? uint32_t(cw * ll) : cl)));
        }
    } else {
        const uint8_t *b = c.blk + 8;
        int s0, se, ss, c0, ce, cs;
        if (!raw) {
            s0 = D + (r0 + S::RO * w) * D;
            se = D + (r0 + rows) * D - 16;
            ss = 16 * S::NL;
            c0 = cd + (r0 + S::RO * w) * cbytes;
            ce = cd + (r0 + rows) * cbytes - cw;
            cs = cw * S::NL;
        } else {
            const int rn = min(rows, S::RawRows);
            s0 = (r0 + S::RawRows / S::W * w) * (2 * D);
            se = (r0 + rn) * (2 * D) - 16;
            ss = 1024;
            cs = 0;
            c0 = ce = r0 * (2 * D);
        }
        const uint32_t ls = uint32_t(16 * lane), lc = uint32_t(cw * lane);
#pragma unroll
        for (int k = 0; k < S::NR; ++k) {
            const int bs = min(s0 + ss * k, se), bc = min(c0 + cs * k, ce);
            R.s[k] = ld16(b + bs + min(ls, uint32_t(se - bs)));
            R.c[k] = ld8(b + bc + min(lc, uint32_t(ce - bc)));
        }
    }
    R.sx = *(g_u32 *)(px);
    R.cx = *(g_u32 *)(pc);
}

// The pair words of an octet of raw BF16 channels (four natural pairs).
__device__ __forceinline__ uint4 raw_octet(const uint4 &n) {
    return make_uint4(__builtin_amdgcn_perm(n.z, n.x, 0x05040100u), __builtin_amdgcn_perm(n.z, n.x, 0x07060302u),
                      __builtin_amdgcn_perm(n.w, n.y, 0x05040100u), __builtin_amdgcn_perm(n.w, n.y, 0x07060302u));
}

// An octet's codes with its second half at bits 16 and up: code p at bits
// [MODE p, ...) and code p + 4 sixteen bits above it.
template <int MODE>
__device__ __forceinline__ uint32_t spread_codes(const uint2 &c, int o) {
    if constexpr (MODE == 4) return o == 0 ? c.x : c.y;
    else if constexpr (MODE == 2) // the octet's two bytes are bytes 2o, 2o + 1 of c.y
        return __builtin_amdgcn_perm(c.y, c.y, o == 0 ? 0x0c010c00u : 0x0c030c02u);
    else { // 24 bits: bytes 2 + 3o .. 4 + 3o of c
        const uint32_t w = o == 0 ? __builtin_amdgcn_alignbyte(c.y, c.x, 2u) : c.y >> 8;
        return (w & 0xFFFu) | ((w << 4) & 0x0FFF0000u);
    }
}

// x << K plus b in one instruction (the compiler would shift before the mask
// that made x, which takes one more).
template <int K>
__device__ __forceinline__ uint32_t lshl_add(uint32_t x, uint32_t b) {
    uint32_t r;
    asm("v_lshl_add_u32 %0, %1, %3, %2" : "=v"(r) : "v"(x), "v"(b), "n"(K));
    return r;
}

// The exponent pairs of an octet (at bits 14:7 and 30:23) from its spread
// codes and its base words: codes + base, each pair's codes masked where they
// stand and shifted up by the add (4-bit codes: 29.7 issue cycles per octet;
// 36.4 with a shift, a mask and an add for each pair).
template <int MODE>
__device__ __forceinline__ void octet_exponents(uint32_t cw, const uint32_t *bp, uint32_t (&t)[4]) {
    constexpr uint32_t M = ((1u << MODE) - 1u) * 0x10001u;
    t[0] = lshl_add<7>(cw & M, bp[0]);
    t[1] = lshl_add<7 - MODE>(cw & (M << MODE), bp[1]);
    if constexpr (MODE == 4) {
        const uint32_t hi = cw >> 5; // pairs 2 and 3 at bits 3 and 7
        t[2] = lshl_add<4>(hi & (M << 3), bp[2]);
        t[3] = (hi & (M << 7)) + bp[3];
    } else {
        t[2] = lshl_add<7 - 2 * MODE>(cw & (M << (2 * MODE)), bp[2]);
        if constexpr (MODE == 2) t[3] = lshl_add<1>(cw & (M << 6), bp[3]);
        else t[3] = ((cw >> 2) & (M << 7)) + bp[3];
    }
}

// A pair of an octet: the channels whose sign/mantissa bytes are byte b of s0
// and of s1, with the exponent pair t.
__device__ __forceinline__ uint32_t team_pair(uint32_t s0, uint32_t s1, uint32_t b, uint32_t t, uint32_t smm) {
    const uint32_t s = __builtin_amdgcn_perm(s1, s0, ((4u + b) << 24) | ((4u + b) << 16) | (b << 8) | b);
    return __builtin_amdgcn_bitop3_b32(s, t, smm, 0xE4);
}

// Writes the two octets of a piece (column c of its row) to the tile row:
// PLAIN (V, and K in the AVX-512 order): octet o's pair words at 16 o; else
// (K in the scalar order) the pair words of wave w's chains of every octet
// together, at 2 D / W w.
template <int D, bool PLAIN>
__device__ __forceinline__ void store_piece(uint8_t *row, int c, const uint4 &a, const uint4 &b) {
    if constexpr (PLAIN) {
        reinterpret_cast<uint4 *>(row + 32 * c)[0] = a;
        reinterpret_cast<uint4 *>(row + 32 * c)[1] = b;
    } else if constexpr (TShape<D>::W == 2) {
        *reinterpret_cast<uint4 *>(row + 16 * c) = make_uint4(a.x, a.y, b.x, b.y);
        *reinterpret_cast<uint4 *>(row + D + 16 * c) = make_uint4(a.z, a.w, b.z, b.w);
    } else {
        *reinterpret_cast<uint2 *>(row + 8 * c) = make_uint2(a.x, b.x);
        *reinterpret_cast<uint2 *>(row + D / 2 + 8 * c) = make_uint2(a.y, b.y);
        *reinterpret_cast<uint2 *>(row + D + 8 * c) = make_uint2(a.z, b.z);
        *reinterpret_cast<uint2 *>(row + 3 * (D / 2) + 8 * c) = make_uint2(a.w, b.w);
    }
}
// One octet o of a row (raw rows).
template <int D, bool PLAIN>
__device__ __forceinline__ void store_octet(uint8_t *row, int o, const uint4 &a) {
    if constexpr (PLAIN) {
        *reinterpret_cast<uint4 *>(row + 16 * o) = a;
    } else if constexpr (TShape<D>::W == 2) {
        *reinterpret_cast<uint2 *>(row + 8 * o) = make_uint2(a.x, a.y);
        *reinterpret_cast<uint2 *>(row + D + 8 * o) = make_uint2(a.z, a.w);
    } else {
        *reinterpret_cast<uint32_t *>(row + 4 * o) = a.x;
        *reinterpret_cast<uint32_t *>(row + D / 2 + 4 * o) = a.y;
        *reinterpret_cast<uint32_t *>(row + D + 4 * o) = a.z;
        *reinterpret_cast<uint32_t *>(row + 3 * (D / 2) + 4 * o) = a.w;
    }
}
// Byte of channel d in a tile row.
template <int D, bool PLAIN>
__device__ __forceinline__ uint32_t channel_byte(uint32_t d) {
    const uint32_t o = d >> 3, p = d & 3u, half = (d >> 2) & 1u;
    if constexpr (PLAIN) return 16 * o + 4 * p + 2 * half;
    else if constexpr (TShape<D>::W == 2) return (p >> 1) * D + 8 * o + 4 * (p & 1u) + 2 * half;
    else return p * (D / 2) + 4 * o + 2 * half;
}

// The first dword of the next piece of a shifted stream: x is the lane's dword
// that the next lane's piece starts with, y the same of the next register
// (lane 63's next piece is that register's lane 0), or the stream's last
// dword in the last register. Every lane must call it (lane moves).
template <int D, bool END>
__device__ __forceinline__ uint32_t next_dword(uint32_t x, uint32_t y) {
    using S = TShape<D>;
    const uint32_t n = uint32_t(dpp_i32<0x134>(0, int(x))); // wave_rol:1: the next lane's
    if constexpr (END) return lane_here() == S::Last ? y : n;
    else if constexpr (S::NL == kWave) {
        const uint32_t n2 = uint32_t(dpp_i32<0x134>(0, int(y)));
        return lane_here() == kWave - 1 ? n2 : n;
    } else return n; // the lanes past the whole rows hold the next register's first pieces
}

template <int D, bool PLAIN, int MODE, bool SHIFT>
__device__ __forceinline__ void decode_team_mode(const TRows<D> &R, const uint32_t (&bp)[8], uint8_t *tile, int w,
                                                 uint32_t smm) {
    using S = TShape<D>;
    const int lane = lane_here();
    const int lr = lane / S::NP, col = lane - lr * S::NP;
    uint8_t *dst = tile + (S::RO * w + lr) * S::TS;
    static_for<0, S::NR>([&](auto K) {
        constexpr int k = decltype(K)::value, kn = k + 1 < S::NR ? k + 1 : k;
        constexpr bool end = k == S::NR - 1;
        const uint4 sm = R.s[k];
        uint2 cd = R.c[k];
        uint32_t s4 = 0;
        if constexpr (SHIFT) {
            s4 = next_dword<D, end>(sm.x, end ? R.sx : R.s[kn].x);
            if constexpr (MODE == 4) {
                const uint32_t c2 = next_dword<D, end>(cd.x, end ? R.cx : R.c[kn].x);
                cd = make_uint2(__builtin_amdgcn_alignbit(cd.y, cd.x, 16), __builtin_amdgcn_alignbit(c2, cd.y, 16));
            } else { // the lane's codes are the upper four of its 8 bytes, the next lane's 8 start 4 further on
                const uint32_t c2 = next_dword<D, end>(cd.y, end ? R.cx : R.c[kn].y);
                cd.y = __builtin_amdgcn_alignbit(c2, cd.y, 16);
            }
        }
        uint4 o[2];
#pragma unroll
        for (int h = 0; h < 2; ++h) {
            const uint32_t cw = spread_codes<MODE>(cd, h);
            uint32_t t[4];
            octet_exponents<MODE>(cw, bp + 4 * h, t);
            const uint32_t s0 = comp(sm, 2 * h), s1 = comp(sm, 2 * h + 1);
            if constexpr (SHIFT) { // the octet's bytes: s0 >> 16, s1, s2 & 0xFFFF
                const uint32_t s2 = h == 0 ? sm.z : s4;
                o[h] = make_uint4(team_pair(s0, s1, 2, t[0], smm), team_pair(s0, s1, 3, t[1], smm),
                                  team_pair(s1, s2, 0, t[2], smm), team_pair(s1, s2, 1, t[3], smm));
            } else {
                o[h] = make_uint4(team_pair(s0, s1, 0, t[0], smm), team_pair(s0, s1, 1, t[1], smm),
                                  team_pair(s0, s1, 2, t[2], smm), team_pair(s0, s1, 3, t[3], smm));
            }
        }
        // not stored: the pieces past a register's whole rows (the next
        // register's first ones, whose next lane is lane 0 here) and the last
        // register's past the wave's rows
        constexpr int rows = S::RS * (k + 1) > S::RO ? S::RO - S::RS * k : S::RS;
        if (rows * S::NP >= kWave || lr < rows) store_piece<D, PLAIN>(dst + S::RS * k * S::TS, col, o[0], o[1]);
    });
}

// -0 in every channel of the wave's tile rows at and past `rows`.
template <int D>
__device__ __forceinline__ void negzero_rows(uint8_t *tile, int w, int rows) {
    using S = TShape<D>;
    const int row = S::RO * w + lane_here();
    if (rows < S::RO * (w + 1) && lane_here() < S::RO && row >= rows) fill_negzero<D>(tile + row * S::TS);
}

// The wave's rows held in R into the tile; V: rows past the chunk's end get
// -0 in every channel.
template <int D, bool PLAIN, bool V>
__device__ __forceinline__ void decode_team_rows(const Cursor &c, const TRows<D> &R, uint8_t *tile, int w, int rows) {
    using S = TShape<D>;
    const int mode = c.mode();
    if (mode != 0) {
        const uint32_t smm = sm_mask_vgpr();
        // base words of the lane's column: pair p of octet h is channels
        // 8h + p, 8h + p + 4, bytes p of the column's base dwords 2h, 2h + 1
        const int lane = lane_here();
        uint32_t bp[8];
#pragma unroll
        for (int h = 0; h < 2; ++h) {
            const int at = 4 * (lane % S::NP + 2 * S::NP * h);
            const uint32_t b0 = uint32_t(__builtin_amdgcn_ds_bpermute(at, int(c.basew)));
            const uint32_t b1 = uint32_t(__builtin_amdgcn_ds_bpermute(at + 4 * S::NP, int(c.basew)));
#pragma unroll
            for (uint32_t p = 0; p < 4; ++p)
                bp[4 * h + p] = __builtin_amdgcn_perm(b1, b0, 0x0c000c00u | ((4u + p) << 16) | p) << 7;
        }
        if (mode == 4) {
            if (c.shift) decode_team_mode<D, PLAIN, 4, true>(R, bp, tile, w, smm);
            else decode_team_mode<D, PLAIN, 4, false>(R, bp, tile, w, smm);
        } else if (mode == 2) {
            if (c.shift) decode_team_mode<D, PLAIN, 2, true>(R, bp, tile, w, smm);
            else decode_team_mode<D, PLAIN, 2, false>(R, bp, tile, w, smm);
        } else {
            decode_team_mode<D, PLAIN, 3, false>(R, bp, tile, w, smm);
        }
    } else {
        // raw rows: the wave's RawRows / W rows, 16 bytes (an octet) per register
        constexpr int RW = S::RawRows / S::W;
        const int lane = lane_here();
#pragma unroll
        for (int k = 0; k < S::NR; ++k) {
            const int o = 64 * k + lane, r = o / (D / 8);
            if (r < RW && RW * w + r < min(c.lrows, S::RawRows))
                store_octet<D, PLAIN>(tile + (RW * w + r) * S::TS, o - r * (D / 8), raw_octet(R.s[k]));
        }
        if constexpr (V) team_sync(); // the rows below may be another wave's
    }
    if constexpr (V) negzero_rows<D>(tile, w, rows);
}

// Writes the escape words of rows [r0, r0 + n) of the cursor's block that lie
// in the wave's rows over their elements and moves the cursor past all of
// them. The first 64 records, one per lane, were loaded with the rows (a chunk
// of head_dim 256 holds about 49 at a rate of 0.3 %); the later ones
// (escape-dense blocks) are loaded here, 256 at a time. Every wave walks every
// record of the chunk, so the cursors (and, with CHK, the answer: whether any
// word is a nonzero value below the exponent bound that `low` encodes, see
// low_bf16) agree without an exchange.
template <int D, bool PLAIN, bool CHK = false>
__device__ __forceinline__ bool patch_team(Cursor &c, int r0, int n, uint8_t *tile, int w, uint32_t low = 0) {
    using S = TShape<D>;
    const int nesc = c.nesc();
    if (c.ecur >= nesc) return false;
    const int lane = lane_id();
    const uint32_t hi = uint32_t((r0 + n) * D), own = uint32_t((r0 + S::RO * w) * D);
    bool bad = false;
    // record `at` of the block, if it lies in the chunk: its word to its
    // element when that is in the wave's rows; returns the chunk's records
    auto take = [&](int at, uint32_t rec) {
        const uint32_t pos = rec & 0xFFFFu, word = rec >> 16;
        const bool in = at < nesc && pos < hi;
        if (in && pos - own < uint32_t(S::RO * D)) {
            const uint32_t row = pos / D, col = pos - row * D;
            *reinterpret_cast<uint16_t *>(tile + (int(row) - r0) * S::TS + channel_byte<D, PLAIN>(col)) =
                uint16_t(word);
        }
        if (CHK) bad |= __ballot(in && low_bf16(word, low)) != 0;
        return __popcll(__ballot(in));
    };
    int got = take(c.ecur + lane, c.erec.x);
    c.ecur += got;
    if (got < kWave) return bad;
    while (c.ecur < nesc) {
        u32x4 r = {0u, 0u, 0u, 0u};
        if (4 * lane < nesc - c.ecur) r = *(g_u32x4 *)(c.esc + c.ecur + 4 * lane);
        got = 0;
#pragma unroll
        for (int j = 0; j < 4; ++j) got += take(c.ecur + 4 * lane + j, r[j]);
        c.ecur += got;
        if (got < 4 * kWave) break;
    }
    return bad;
}

// block_vectors with one record per lane (in erec.x).
template <int D>
__device__ __forceinline__ void team_block_vectors(Cursor &c) {
    constexpr int NP = TShape<D>::NP;
    const int lane = lane_here();
    c.basew = *(g_u32 *)(c.blk + 8 + 16 * (lane % NP) + 4 * ((lane / NP) & 3));
    uint32_t r = 0u;
    if (lane < c.nesc() - c.ecur || lane == 0) r = *(g_u32 *)(c.esc + c.ecur + lane);
    c.erec.x = r;
}

// Channel of the wave's score operand i (0 .. CW - 1).
template <int D, int ORDER>
__device__ __forceinline__ int score_channel(int w, int i) {
    if constexpr (ORDER == 0) {
        if constexpr (TShape<D>::W == 2) return 8 * (i >> 2) + 2 * w + ((i >> 1) & 1) + 4 * (i & 1);
        else return 8 * (i >> 1) + w + 4 * (i & 1);
    } else {
        if constexpr (TShape<D>::W == 2) return 32 * (i >> 4) + 16 * w + (i & 15);
        else return 32 * (i >> 3) + 8 * w + (i & 7);
    }
}

// Partial scores of the lane's token over the wave's chains, scalar order:
// chains j with j % 4 in the wave's share, each over octets in order, then
// their brackets of hsum8's tree. sub: the wave's part of the lane's tile row.
template <int G, int D>
__device__ __forceinline__ void team_scores(const uint8_t *sub, const float (&qa)[kGroups<G>][TShape<D>::QR],
                                            f4 (&p)[kGroups<G>]) {
    using S = TShape<D>;
    constexpr int NG = kGroups<G>, NC = 8 / S::W; // chains: octet elements (q, q + 4), q in the wave's share
    f4 ch[NG][NC];
#pragma unroll
    for (int rg = 0; rg < NG; ++rg)
#pragma unroll
        for (int j = 0; j < NC; ++j) ch[rg][j] = f4{0.0f, 0.0f, 0.0f, 0.0f};
    static_for<0, S::CW / 8>([&](auto I) {
        constexpr int i0 = 8 * decltype(I)::value;
        const uint4 kb = *reinterpret_cast<const uint4 *>(sub + 2 * i0);
        const float k[8] = {lo_f32(kb.x), hi_f32(kb.x), lo_f32(kb.y), hi_f32(kb.y),
                            lo_f32(kb.z), hi_f32(kb.z), lo_f32(kb.w), hi_f32(kb.w)};
        static_for<0, 8>([&](auto J) {
            constexpr int i = i0 + decltype(J)::value;
#pragma unroll
            for (int rg = 0; rg < NG; ++rg)
                ch[rg][i % NC] = mfma_rank1<i % 16>(qa[rg][i / 16], k[J], ch[rg][i % NC]);
        });
        __builtin_amdgcn_sched_group_barrier(0x002, 8, 0);
        __builtin_amdgcn_sched_group_barrier(0x008, 8 * NG, 0);
    });
#pragma unroll
    for (int rg = 0; rg < NG; ++rg) {
        p[rg] = ch[rg][0] + ch[rg][1];
        if constexpr (NC == 4) p[rg] = p[rg] + (ch[rg][2] + ch[rg][3]);
    }
}

// Channel e of an octet of pair words.
__device__ __forceinline__ float octet_elem(const uint4 &x, int e) {
    const uint32_t d = comp(x, e & 3);
    return e < 4 ? lo_f32(d) : hi_f32(d);
}

// The same in the AVX-512 BF16 order without flushes (see scores_dp_of): the
// wave's quads of chains, each octet's odd channels before its even ones.
template <int G, int D>
__device__ __forceinline__ void team_scores_dp(const uint8_t *row, int w, const float (&qa)[kGroups<G>][TShape<D>::QR],
                                               f4 (&p)[kGroups<G>]) {
    using S = TShape<D>;
    constexpr int NG = kGroups<G>, NQ = 4 / S::W;
    static_for<0, NQ>([&](auto X) {
        constexpr int x = decltype(X)::value;
        f4 ch[NG][4];
#pragma unroll
        for (int rg = 0; rg < NG; ++rg)
#pragma unroll
            for (int j = 0; j < 4; ++j) ch[rg][j] = f4{0.0f, 0.0f, 0.0f, 0.0f};
        static_for<0, D / 32>([&](auto C) {
            constexpr int i0 = 8 * NQ * decltype(C)::value + 8 * x; // operand of the octet's channel 0
            const uint4 kb = *reinterpret_cast<const uint4 *>(row + 16 * (4 * decltype(C)::value + NQ * w + x));
            static_for<0, 2>([&](auto E) {
                static_for<0, 4>([&](auto J) {
                    constexpr int e = 2 * decltype(J)::value + 1 - decltype(E)::value;
                    const float k = octet_elem(kb, e);
#pragma unroll
                    for (int rg = 0; rg < NG; ++rg)
                        ch[rg][J] = mfma_rank1<(i0 + e) % 16>(qa[rg][(i0 + e) / 16], k, ch[rg][J]);
                });
            });
            // octet by octet (all octets read ahead spilled above four rows; one
            // head x 4,096 tokens, three rows of head_dim 128: 26.6 us with, 26.2 without)
            if constexpr (NG > 1 || S::W == 4) {
                __builtin_amdgcn_sched_group_barrier(0x002, 8, 0);
                __builtin_amdgcn_sched_group_barrier(0x008, 8 * NG, 0);
            }
        });
#pragma unroll
        for (int rg = 0; rg < NG; ++rg) {
            const f4 a = (ch[rg][0] + ch[rg][1]) + (ch[rg][2] + ch[rg][3]);
            if constexpr (x == 0) p[rg] = a;
            else p[rg] = p[rg] + a;
        }
    });
}

// Whether the wave's channels of any `in` lane's tile row hold an element below
// the bound (see low_bf16). A wave's own chains flush or do not: the others'
// answers may differ.
template <int D>
__device__ __forceinline__ bool team_row_low(const uint8_t *row, int w, bool in, uint32_t low) {
    constexpr int NQ = 4 / TShape<D>::W;
    low_min_t lo = kLowMinNone;
#pragma unroll 1
    for (int c = 0; c < D / 32; ++c)
#pragma unroll
        for (int x = 0; x < NQ; ++x)
            lo = low_min(lo, *reinterpret_cast<const uint4 *>(row + 16 * (4 * c + NQ * w + x)));
    return any_low(in ? lo : kLowMinNone, low);
}

// The same with every flush applied (scores_dp_flush), on the vector ALU.
template <int G, int D>
__device__ __forceinline__ void team_scores_dp_flush(const uint8_t *row, int w, const uint16_t *q,
                                                     f4 (&p)[kGroups<G>]) {
    using S = TShape<D>;
    constexpr int NQ = 4 / S::W;
    static_for<0, G>([&](auto GI) {
        constexpr int g = decltype(GI)::value;
        float r = 0.0f;
#pragma unroll 1
        for (int x = 0; x < NQ; ++x) {
            float t[4] = {0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll 1
            for (int c = 0; c < D / 32; ++c) {
                const int o = 4 * c + NQ * w + x;
                const uint4 kb = *reinterpret_cast<const uint4 *>(row + 16 * o);
                const uint16_t *qo = q + size_t(g) * D + 8 * o;
#pragma unroll
                for (int j = 0; j < 4; ++j) {
                    const float q1 = __uint_as_float(uint32_t(qo[2 * j + 1]) << 16);
                    const float q0 = __uint_as_float(uint32_t(qo[2 * j]) << 16);
                    t[j] = flush_tiny(fmaf(flush_tiny(octet_elem(kb, 2 * j + 1)), flush_tiny(q1), t[j]));
                    t[j] = flush_tiny(fmaf(flush_tiny(octet_elem(kb, 2 * j)), flush_tiny(q0), t[j]));
                }
            }
            const float a = (t[0] + t[1]) + (t[2] + t[3]);
            r = x == 0 ? a : r + a;
        }
        p[g / 4][g % 4] = r;
    });
}

// Byte of partial score g (0 .. 7, 16-byte runs of four) of wave w in a tile
// row: inside the K channels that only wave w reads.
template <int D, int ORDER>
__device__ __forceinline__ int partial_byte(int w, int g) {
    if constexpr (ORDER == 0) return 2 * TShape<D>::CW * w + 4 * g;
    else if constexpr (TShape<D>::W == 2) return 32 * w + 4 * g;
    else return 16 * w + 64 * (g >> 2) + 4 * (g & 3);
}

// Operands of the fold in flight (one channel per lane): V of the next quads
// of four tokens, e of four tokens (wave 0).
struct TFoldIn {
    uint2 vq[3];
    f4 e4[2];
};

// Token T of the ordered fold (see fold_token), one channel per lane. L: the
// wave also carries l.
template <int G, int D, int T, bool MOVE, bool L, bool AHEAD>
__device__ __forceinline__ void team_fold_token(const TeamLds<G, D> &S, lds_f32 *eb, lds_f32 *ab, const uint8_t *trb,
                                                const uint32_t (&am)[2], const float (&ea)[kGroups<G>][4], TFoldIn &in,
                                                f4 &a4, f4 (&acc)[kGroups<G>], float &lvec) {
    constexpr int NG = kGroups<G>, TS = TShape<D>::TS, Q = T / 4;
    if constexpr (T % 4 == 0) {
        if constexpr (4 * (Q + 2) < kChunk) in.vq[(Q + 2) % 3] = load_tr(trb + 4 * (Q + 2) * TS);
        if constexpr (L && AHEAD && 4 * (Q + 1) < kChunk)
            in.e4[(Q + 1) & 1] = *reinterpret_cast<lds_f4 *>(eb + 4 * (Q + 1));
        if constexpr (L && MOVE) a4 = *reinterpret_cast<lds_f4 *>(ab + 4 * Q);
    }
    const float v = quad_f32<T % 4>(in.vq[Q % 3]);
    if constexpr (MOVE) {
        if ((am[T / 32] & (1u << (T % 32))) != 0) {
            // (the empty asm keeps this a branch: at two rows the compiler read
            // and selected the alphas of all 64 tokens instead, and spilled)
            if constexpr (G == 2) asm volatile("");
            float av[G];
#pragma unroll
            for (int g = 0; g < G; ++g) av[g] = S.aT[g][T];
#pragma unroll
            for (int g = 0; g < G; ++g) acc[g / 4][g % 4] *= av[g];
        }
    }
    if constexpr (L) {
        const float el = in.e4[AHEAD ? Q & 1 : 0][T % 4];
        if constexpr (MOVE) lvec = fmaf(lvec, a4[T % 4], el);
        else lvec = lvec + el;
        asm volatile("" : "+v"(lvec)); // the l chain in token order (see fold_token)
        if constexpr (!AHEAD && T % 4 == 3 && T + 1 < kChunk) in.e4[0] = *reinterpret_cast<lds_f4 *>(eb + T + 1);
    }
#pragma unroll
    for (int rg = 0; rg < NG; ++rg) acc[rg] = mfma_rank1<T % 16>(ea[rg][T / 16], v, acc[rg]);
}

template <int G, int D, int T, bool L, bool AHEAD>
__device__ __forceinline__ void team_fold(const TeamLds<G, D> &S, lds_f32 *eb, lds_f32 *ab, const uint8_t *trb,
                                          const uint32_t (&am)[2], const float (&ea)[kGroups<G>][4], TFoldIn &in,
                                          f4 (&acc)[kGroups<G>], float &lvec) {
    constexpr int GS = 16, NG = kGroups<G>;
    if constexpr (T < kChunk) {
        constexpr uint32_t gm = uint32_t(((1ull << GS) - 1ull) << (T % 32));
        f4 a4;
        if ((am[T / 32] & gm) == 0) {
            static_for<0, GS>([&](auto K) {
                team_fold_token<G, D, T + decltype(K)::value, false, L, AHEAD>(S, eb, ab, trb, am, ea, in, a4, acc, lvec);
            });
            static_for<0, GS / 4>([&](auto) {
                __builtin_amdgcn_sched_group_barrier(0x002, L ? 8 : 4, 0);
                __builtin_amdgcn_sched_group_barrier(0x008, 4 * NG, 0);
            });
        } else {
            static_for<0, GS>([&](auto K) {
                team_fold_token<G, D, T + decltype(K)::value, true, L, AHEAD>(S, eb, ab, trb, am, ea, in, a4, acc, lvec);
                // (two rows: quad by quad, or registers of the rows in flight are moved and spilled)
                if constexpr (G == 2 && decltype(K)::value % 4 == 3) asm volatile("" : "+v"(acc[0]));
            });
        }
        team_fold<G, D, T + GS, L, AHEAD>(S, eb, ab, trb, am, ea, in, acc, lvec);
    }
}

// Plain BF16 rows of the wave: register j of lane l holds bytes
// 1024 j + 16 l of its RO rows from token t (rows past `avail` of the chunk
// repeat the last one).
template <int D>
constexpr int kTeamRawRegs = (TShape<D>::RO * D / 8 + kWave - 1) / kWave;

template <int D>
__device__ __forceinline__ void load_team_raw(const uint16_t *base, int w, int t, int avail,
                                              uint4 (&R)[kTeamRawRegs<D>]) {
    const uint8_t *b = reinterpret_cast<const uint8_t *>(base + size_t(t) * D);
    const int lane = lane_here();
#pragma unroll
    for (int j = 0; j < kTeamRawRegs<D>; ++j) {
        const int o = 64 * j + lane, r = o / (D / 8);
        R[j] = ld16(b + uint32_t(min(TShape<D>::RO * w + r, avail - 1) * (2 * D) + 16 * (o - r * (D / 8))));
    }
}

template <int D, bool PLAIN>
__device__ __forceinline__ void store_team_raw(const uint4 (&R)[kTeamRawRegs<D>], uint8_t *tile, int w) {
    const int lane = lane_here();
#pragma unroll
    for (int j = 0; j < kTeamRawRegs<D>; ++j) {
        const int o = 64 * j + lane, r = o / (D / 8);
        if ((64 * j + 63) / (D / 8) >= TShape<D>::RO && r >= TShape<D>::RO) continue;
        store_octet<D, PLAIN>(tile + (TShape<D>::RO * w + r) * TShape<D>::TS, o - r * (D / 8), raw_octet(R[j]));
    }
}

// acc * inv with a NaN of inv before one of acc: a row whose l is NaN gives
// l's NaN in every channel, as the one-wave kernel does (the operand order of
// a plain product is the compiler's).
__device__ __forceinline__ float scale_by(float inv, float acc) {
    float r;
    asm("v_mul_f32_e32 %0, %1, %2" : "=v"(r) : "v"(inv), "v"(acc));
    return r;
}

template <bool XKV, int D> struct TRegsOf { typedef TRows<D> T; };
template <int D> struct TRegsOf<false, D> { typedef uint4 T[kTeamRawRegs<D>]; };

// Four waves per SIMD (128 registers); three (168) at more than four query
// rows, whose second row group would spill 14 to 84 registers at four (64
// plain heads x 24,000 tokens of head_dim 128, five rows: 171 -> 207 us),
// except at the sizes whose rows take three registers per stream and wave
// instead of four (80 and 160). A spill or a move of a register that a row in
// flight is loaded into waits for the load, which cost two rows at head_dim
// 128 a quarter of the call (plain 186 -> 146 us, AVX-512 XKV 171 -> 131
// without them).
template <int G, int D>
constexpr int kTeamOcc = G > 4 && TShape<D>::NR > 3 ? 3 : 4;

// Whether wave 0 reads e of a quad of tokens a whole quad ahead. Not at four
// plain rows of head_dim 256: those four registers would spill two that rows
// are in flight to (64 heads x 65,536 tokens: 774 us, 735 without).
template <int G, int D, bool XKV>
constexpr bool kFoldAhead = XKV || D < 256 || G != 4;

template <int G, int D, bool XKV, int ORDER>
__global__ __launch_bounds__(TShape<D>::W * 64) __attribute__((amdgpu_waves_per_eu(kTeamOcc<G, D>)))
void attn_team_kernel(const HeadDev *__restrict__ heads, const WorkItem *__restrict__ items,
                      const BlockDesc *__restrict__ desc, const uint16_t *__restrict__ q_all,
                      float *__restrict__ out_all, float *__restrict__ lse_all, float *__restrict__ ws) {
    using SH = TShape<D>;
    constexpr int TS = SH::TS, W = SH::W, NG = kGroups<G>, CW = SH::CW;
    constexpr bool KP = ORDER == 1;          // layout of a K row in the tile (store_piece)
    constexpr int RQ = (G + W - 1) / W;      // query rows whose softmax a wave computes
    __shared__ TeamLds<G, D> S;
    if (threadIdx.x < 64) kvexp_exp_table_to_lds(S.exptab);

    const int lane = lane_id();
    const int w = __builtin_amdgcn_readfirstlane(int(threadIdx.x) >> 6);
    const WorkItem wi = load_scalar(items + blockIdx.x);
    const HeadDev hd = load_scalar(heads + wi.head);
    const uint16_t *qh = q_all + size_t(hd.q_row) * D;
    // The query rows widened to FP32 as the A operands of the wave's score
    // products: qa[rg][j] at lane 4b + r holds row 4 rg + r at the channel of
    // the wave's operand 16 j + b (0 for rows past G and operands past CW).
    float qa[NG][SH::QR];
    uint32_t klow = 0, kmin = 0;
    {
        const int r = lane & 3, b = lane >> 2;
#pragma unroll
        for (int rg = 0; rg < NG; ++rg) {
            const int g = min(4 * rg + r, G - 1);
#pragma unroll
            for (int j = 0; j < SH::QR; ++j) {
                const int i = min(16 * j + b, CW - 1);
                float qv = __uint_as_float(uint32_t(qh[size_t(g) * D + score_channel<D, ORDER>(w, i)]) << 16);
                if constexpr (ORDER == 1) qv = flush_tiny(qv);
                qa[rg][j] = 4 * rg + r < G && 16 * j + b < CW ? qv : 0.0f;
            }
        }
    }
    if constexpr (ORDER == 1) {
        // the K exponent bound of the fast score path over all of the head's
        // query elements (see attn_wave_kernel)
        int qe = 255;
        for (int i = lane; i < G * D; i += kWave) {
            const int e = (qh[i] >> 7) & 0xFF; // 0: zero or denormal, read as zero
            if (e != 0) qe = min(qe, e);
        }
        qe = wave_min_i32(qe);
        kmin = uint32_t(max(1, 142 - qe));
        klow = (kmin << 7) - 1u;
    }

    f4 acc[NG];
#pragma unroll
    for (int rg = 0; rg < NG; ++rg) acc[rg] = f4{0.0f, 0.0f, 0.0f, 0.0f};
    float msc[RQ]; // running maximum of the wave's query rows w + W r (wave-uniform)
#pragma unroll
    for (int r = 0; r < RQ; ++r) msc[r] = -__builtin_inff();
    float lvec = 0.0f; // wave 0: lane g < G holds l of query row g

    Cursor kc{}, vc{};
    typename TRegsOf<XKV, D>::T RK, RV;
    int t = wi.tok_begin;
    if constexpr (XKV) {
        enter_block(kc, desc + wi.kdi, t);
        enter_block(vc, desc + wi.vdi, t);
        team_block_vectors<D>(kc);
        load_team_rows<D>(kc, w, 0, min(kChunk, min(kc.t1, wi.tok_end) - t), RK);
        team_block_vectors<D>(vc);
        load_team_rows<D>(vc, w, 0, min(kChunk, min(vc.t1, wi.tok_end) - t), RV);
    } else {
        load_team_raw<D>(hd.kraw, w, t, min(kChunk, wi.tok_end - t), RK);
        load_team_raw<D>(hd.vraw, w, t, min(kChunk, wi.tok_end - t), RV);
    }

    // phase trace (builds with KVEXP_PHASE_TRACE; see attn_wave_kernel): per
    // wave of the scalar-order XKV kernel, cycles in the phases that
    // bench.py names
    constexpr bool TR = KVEXP_TRACE_ON(XKV, ORDER);
    unsigned long long ph[12] = {0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0};
    const unsigned long long tw0 = TR ? __builtin_readcyclecounter() : 0ull;
    unsigned long long tprev = tw0;
    auto stamp = [&](int i) {
        if constexpr (TR) {
            const unsigned long long now = __builtin_readcyclecounter();
            ph[i] += now - tprev;
            tprev = now;
        }
    };
    auto after = [&](uint32_t x) {
        if constexpr (TR) asm volatile("" ::"v"(x));
    };
    (void)stamp;
    (void)after;

    // issue priority by progress (see attn_wave_kernel)
    const int quarter = (wi.tok_end - wi.tok_begin + 3) / 4;
    int prio = -1;
    while (t < wi.tok_end) {
        const int ln = lane_here();
        {
            const int want = priority_of(wi.tok_end - t, quarter);
            if (want != prio) {
                if (want == 3) __builtin_amdgcn_s_setprio(3);
                else if (want == 2) __builtin_amdgcn_s_setprio(2);
                else if (want == 1) __builtin_amdgcn_s_setprio(1);
                else __builtin_amdgcn_s_setprio(0);
                prio = want;
            }
        }
        int n = min(kChunk, wi.tok_end - t);
        if constexpr (XKV) {
            n = min(n, min(kc.t1 - t, vc.t1 - t));
            if (kc.mode() == 0 || vc.mode() == 0) n = min(n, SH::RawRows);
        }
        if (n <= 0) break; // unreachable with plan-checked descriptors (n_tokens > 0); the same in every wave
        const int tn = t + n, tp = min(tn, wi.tok_end - 1);

        // 1. the wave's K rows -> tile, the next ones requested
        bool flush = false, kraw = false; // kraw: rows of a raw block, checked in the tile
        if constexpr (XKV) after(RK.c[SH::NR - 1].y);
        stamp(0); // K rows arrived
        if constexpr (XKV) {
            if constexpr (ORDER == 1) {
                if (kc.mode() != 0) {
                    const uint32_t bw = kc.basew;
                    const u16x2 e = __builtin_bit_cast(u16x2, bw & 0x00FF00FFu);
                    const u16x2 o = __builtin_bit_cast(u16x2, (bw >> 8) & 0x00FF00FFu);
                    const u16x2 bmin = __builtin_elementwise_min(e, o), bmax = __builtin_elementwise_max(e, o);
                    const uint32_t top = 256u - (1u << kc.mode());
                    flush = __ballot(uint32_t(min(bmin.x, bmin.y)) < kmin || uint32_t(max(bmax.x, bmax.y)) > top) != 0;
                } else if constexpr (kRawChecked<D>) {
                    kraw = true;
                } else {
                    flush = true;
                }
            }
            decode_team_rows<D, KP, false>(kc, RK, S.tile, w, n);
            wave_sync();
            flush |= patch_team<D, KP, ORDER == 1>(kc, t - kc.t0, n, S.tile, w, klow);
            stamp(1); // K decoded, its escapes written
            if (tp >= kc.t1) enter_block(kc, kc.d + 1, kc.t1);
            team_block_vectors<D>(kc);
            load_team_rows<D>(kc, w, tp - kc.t0, min(kChunk, min(kc.t1, wi.tok_end) - tp), RK);
        } else {
            if constexpr (ORDER == 1) {
                low_min_t lo = kLowMinNone;
#pragma unroll
                for (int j = 0; j < kTeamRawRegs<D>; ++j) {
                    const int r = (64 * j + ln) / (D / 8);
                    if (r < SH::RO && SH::RO * w + r < n) lo = low_min(lo, RK[j]);
                }
                const bool low = any_low(lo, klow);
                if (ln == 0) S.low[w] = low ? 1u : 0u;
            }
            store_team_raw<D, KP>(RK, S.tile, w);
            load_team_raw<D>(hd.kraw, w, tp, min(kChunk, wi.tok_end - tp), RK);
        }
        stamp(2); // next K rows requested
        team_sync(); // K tile whole
        stamp(3);

        // 2. the wave's share of the scores, lane = token
        {
            f4 p[NG];
            uint8_t *row = S.tile + ln * TS;
            if constexpr (ORDER == 0) {
                team_scores<G, D>(row + 2 * CW * w, qa, p);
            } else {
                if constexpr (!XKV) {
                    uint32_t any = 0;
#pragma unroll
                    for (int i = 0; i < W; ++i) any |= S.low[i];
                    flush = __builtin_amdgcn_readfirstlane(any) != 0;
                }
                if constexpr (XKV && kRawChecked<D>) {
                    if (kraw) flush = team_row_low<D>(row, w, ln < n, klow);
                }
                if (!flush) team_scores_dp<G, D>(row, w, qa, p);
                else team_scores_dp_flush<G, D>(row, w, qh, p);
            }
            wave_sync();
#pragma unroll
            for (int rg = 0; rg < NG; ++rg)
                *reinterpret_cast<f4 *>(row + partial_byte<D, ORDER>(w, 4 * rg)) = p[rg];
        }
        stamp(4); // partial scores
        team_sync(); // partial scores whole
        stamp(5);

        // 3. softmax coefficients of query rows w + W r, lane = token (see
        // attn_wave_kernel; a wave without a row left repeats row G - 1, to
        // the same values)
        const uint64_t nmask = n >= kChunk ? ~0ull : ((1ull << n) - 1ull);
        uint64_t amask = 0;
        {
            float s[RQ], mi[RQ];
            const uint8_t *row = S.tile + ln * TS;
#pragma unroll
            for (int r = 0; r < RQ; ++r) {
                const int g = min(w + W * r, G - 1);
                float x[W];
#pragma unroll
                for (int i = 0; i < W; ++i)
                    x[i] = *reinterpret_cast<const float *>(row + partial_byte<D, ORDER>(i, g));
                if constexpr (W == 2) s[r] = x[0] + x[1];
                else s[r] = (x[0] + x[1]) + (x[2] + x[3]);
                mi[r] = s[r];
            }
            wave_scan_max_rows<RQ>(mi);
            float m[RQ], mp[RQ], x[RQ];
            double kd[RQ], rr[RQ];
            uint64_t tb[RQ];
#pragma unroll
            for (int r = 0; r < RQ; ++r) {
                m[r] = max_f32(mi[r], msc[r]);
                mp[r] = wave_shift_up(m[r], msc[r]);
                x[r] = lane_select(__ballot(s[r] > mp[r]), mp[r] - s[r], s[r] - m[r]);
                kvexp_expf_reduce(x[r], kd[r], rr[r]);
                tb[r] = S.exptab[uint32_t(__double_as_longlong(kd[r])) & 31u];
            }
#pragma unroll
            for (int r = 0; r < RQ; ++r) {
                const int g = min(w + W * r, G - 1);
                float y = kvexp_expf_finish(kd[r], rr[r], tb[r]);
                y = lane_select_or0(__ballot(!(x[r] < -0x1.9fe368p6f)), y);
                const float dg = mp[r] - m[r];
                amask |= __ballot(!(dg == 0.0f)) & nmask;
                const uint64_t mv = __ballot(s[r] > mp[r]);
                const float e = lane_select(mv, (s[r] - m[r]) + 1.0f, y);
                const float al = lane_select(mv, y, dg + 1.0f);
                S.eT[g][ln] = lane_select_or0(nmask, e);
                S.aT[g][ln] = lane_select_or1(nmask, al);
                msc[r] = readlane_f32(m[r], n - 1);
            }
            if (ln == 0) S.am[w] = amask;
        }
        stamp(6); // coefficients
        team_sync(); // coefficients whole, partial scores read
        stamp(7);
        if constexpr (XKV) after(RV.c[SH::NR - 1].y);
        stamp(8); // V rows arrived

        // 4. the wave's V rows -> tile, the next ones requested
        if constexpr (XKV) {
            decode_team_rows<D, true, true>(vc, RV, S.tile, w, n);
            wave_sync();
            patch_team<D, true>(vc, t - vc.t0, n, S.tile, w);
            stamp(9); // V decoded, its escapes written
            if (tp >= vc.t1) enter_block(vc, vc.d + 1, vc.t1);
            team_block_vectors<D>(vc);
            load_team_rows<D>(vc, w, tp - vc.t0, min(kChunk, min(vc.t1, wi.tok_end) - tp), RV);
        } else {
            store_team_raw<D, true>(RV, S.tile, w);
            wave_sync();
            negzero_rows<D>(S.tile, w, n);
            load_team_raw<D>(hd.vraw, w, tp, min(kChunk, wi.tok_end - tp), RV);
        }
        team_sync(); // V tile whole
        stamp(10); // next V rows requested, V tile whole

        // 5. ordered fold, lane = the wave's channel
        {
            int lq = ln;
            asm volatile("" : "+v"(lq));
            float ea[NG][4];
#pragma unroll
            for (int rg = 0; rg < NG; ++rg) {
                const int g = min(4 * rg + (lq & 3), G - 1);
#pragma unroll
                for (int j = 0; j < 4; ++j) ea[rg][j] = S.eT[g][16 * j + (ln >> 2)];
            }
            uint64_t all = 0;
#pragma unroll
            for (int i = 0; i < W; ++i) all |= S.am[i];
            uint32_t am[2] = {uint32_t(__builtin_amdgcn_readfirstlane(int(uint32_t(all)))),
                              uint32_t(__builtin_amdgcn_readfirstlane(int(uint32_t(all >> 32))))};
            asm volatile("" : "+s"(am[0]), "+s"(am[1]));
            const int gl = min(ln & 7, G - 1);
            lds_f32 *eb = (lds_f32 *)&S.eT[gl][0];
            lds_f32 *ab = (lds_f32 *)&S.aT[gl][0];
            const int sl = ln & 15;
            const uint8_t *trb = S.tile + ((sl >> 2) * TS + 32 * (ln >> 4) + 8 * (sl & 3) + 2 * CW * w);
            TFoldIn in;
#pragma unroll
            for (int k = 0; k < 2; ++k) in.vq[k] = load_tr(trb + 4 * k * TS);
            if (w == 0) {
                in.e4[0] = *reinterpret_cast<lds_f4 *>(eb);
                team_fold<G, D, 0, true, kFoldAhead<G, D, XKV>>(S, eb, ab, trb, am, ea, in, acc, lvec);
            } else {
                team_fold<G, D, 0, false, true>(S, eb, ab, trb, am, ea, in, acc, lvec);
            }
        }
        after(__float_as_uint(acc[0].x));
        stamp(11); // folded
        team_sync(); // V tile read
        stamp(10);
        t = tn;
    }
#if defined(KVEXP_PHASE_TRACE)
    if constexpr (TR) {
        const int slot = int(blockIdx.x) * W + w;
        if (lane == 0 && slot < kTraceWaves) {
            unsigned long long *o = g_phase_trace + size_t(slot) * kTraceWords;
            o[0] = tw0;
            o[1] = __builtin_readcyclecounter();
            for (int i = 0; i < kTracePhases; ++i) o[2 + i] = ph[i];
            o[kTracePhases + 2] = (unsigned long long)__smid() | ((unsigned long long)wi.head << 16) |
                                  ((unsigned long long)wi.split << 40);
        }
    }
#endif

    // ---- epilogue: m of every row (its wave) and l (wave 0) to every wave
#pragma unroll
    for (int r = 0; r < RQ; ++r)
        if (lane == 0) S.aT[0][min(w + W * r, G - 1)] = msc[r];
    if (w == 0 && lane < G) S.eT[0][lane] = lvec;
    team_sync();
    // tile position CW w + lane of a V row: channels p, p + 4 of an octet side by side
    const int pos = CW * w + lane;
    const int d = (pos & ~7) + ((pos & 7) >> 1) + 4 * (pos & 1);
    if (hd.n_splits == 1) {
        if (lane < CW) {
#pragma unroll
            for (int g = 0; g < G; ++g)
                out_all[(size_t(hd.q_row) + g) * D + d] = scale_by(1.0f / S.eT[0][g], acc[g / 4][g % 4]);
        }
        if (lse_all != nullptr && w == 0 && lane < G) lse_all[hd.q_row + lane] = S.aT[0][lane] + logf(lvec);
        return;
    }
    float *slot = ws + size_t(hd.ws_base + wi.split) * Shape<D>::kSlotFloats;
    if (w == 0 && lane < G) {
        slot[lane] = S.aT[0][lane];
        slot[kSlotQ + lane] = lvec;
    }
    if (lane < CW) {
#pragma unroll
        for (int g = 0; g < G; ++g) slot[2 * kSlotQ + g * D + d] = acc[g / 4][g % 4];
    }
}

} // namespace team
} // namespace kvexp_dev

namespace kvexp_launch {
using namespace kvexp_dev;

template <int G, int D, bool XKV, int ORDER>
static hipError_t launch_team_g(const HeadDev *heads, const WorkItem *items, int n_items,
                                const BlockDesc *desc,
                                const uint16_t *q, float *out, float *lse, float *ws, hipStream_t s) {
    hipLaunchKernelGGL((team::attn_team_kernel<G, D, XKV, ORDER>), dim3(n_items), dim3(team::TShape<D>::W * 64), 0, s,
                       heads, items, desc, q, out, lse, ws);
    return hipGetLastError();
}

template <int D, bool XKV, int ORDER>
static hipError_t launch_team_x(int G, const HeadDev *heads, const WorkItem *items, int n_items,
                                const BlockDesc *desc,
                                const uint16_t *q, float *out, float *lse, float *ws, hipStream_t s) {
    switch (G) {
    case 1: return launch_team_g<1, D, XKV, ORDER>(heads, items, n_items, desc, q, out, lse, ws, s);
    case 2: return launch_team_g<2, D, XKV, ORDER>(heads, items, n_items, desc, q, out, lse, ws, s);
    case 3: return launch_team_g<3, D, XKV, ORDER>(heads, items, n_items, desc, q, out, lse, ws, s);
    case 4: return launch_team_g<4, D, XKV, ORDER>(heads, items, n_items, desc, q, out, lse, ws, s);
    case 5: return launch_team_g<5, D, XKV, ORDER>(heads, items, n_items, desc, q, out, lse, ws, s);
    case 6: return launch_team_g<6, D, XKV, ORDER>(heads, items, n_items, desc, q, out, lse, ws, s);
    case 7: return launch_team_g<7, D, XKV, ORDER>(heads, items, n_items, desc, q, out, lse, ws, s);
    case 8: return launch_team_g<8, D, XKV, ORDER>(heads, items, n_items, desc, q, out, lse, ws, s);
    default: return hipErrorInvalidValue;
    }
}

#define KVEXP_TEAM_UNIT(D, O)                                                                                        \
    hipError_t attention_team_d##D##_o##O(bool xkv, int G, const HeadDev *heads, const WorkItem *items,             \
                                         int n_items, const BlockDesc *desc, const uint16_t *q,        \
                                         float *out, float *lse, float *ws, hipStream_t s) {                        \
        return xkv ? launch_team_x<D, true, O>(G, heads, items, n_items, desc, q, out, lse, ws, s)                   \
                   : launch_team_x<D, false, O>(G, heads, items, n_items, desc, q, out, lse, ws, s);                 \
    }                                                                                                                \
    KVEXP_TRACE_READER(team, D, O)

} // namespace kvexp_launch
