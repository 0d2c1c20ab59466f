// gemm_split.hpp -- the fp32 tile GEMM kernel of gfx950, on its bf16 matrix
// cores.
//
// An fp32 value x of 2^-110 and above is the exact sum of three bf16 values (8
// significant bits each, rounded to nearest): x = x0 + x1 + x2 with
// |x1| <= 2^-8 |x0| and |x2| <= 2^-17 |x0|.  (Below that it is one if its last
// bit is 2^-133 or more, bf16's smallest value; see redo_flag for the
// others.)  A product of two such sums has nine terms; the six largest,
//     a2 b0 + a0 b2 + a1 b1 + a1 b0 + a0 b1 + a0 b0,
// leave out less than 2^-24 of |a b|.  Each is one bf16 MFMA; the six of a 32-k
// tile add up from zero (the smallest terms among the first), and that sum
// goes to the accumulator with one fp32 addition.  (Six MFMAs straight into
// the accumulator are 5 % faster, and as exact as the fp32 MFMA chain for
// independent operands, but a term like a1 b1 with one sign throughout -- a row
// times itself, SYRK's diagonal -- is lost to rounding once the accumulator
// is 2^18 times its tile sum: the 8192^2 SYRK was off by 2.0e-6, the fp32
// chain by 1.5e-6.)
//   Error of K-term dot products against 64-bit sums, 2-norm, fp32 MFMA
// chain -> this sum (256 x 256, uniform on [-1, 1) / on [0, 1) / normal):
//     K = 32     1.0e-7 / 8.4e-8 / 1.0e-7  ->  3.6e-8 / 3.4e-8 / 3.8e-8
//     K = 512    4.1e-7 / 3.1e-7 / 4.1e-7  ->  8.6e-8 / 6.0e-8 / 8.9e-8
//     K = 8192   1.6e-6 / 1.2e-6 / 1.6e-6  ->  3.0e-7 / 2.1e-7 / 3.1e-7
//   The bf16 MFMAs run at 16 times the fp32 ones' rate (2.5 PFLOP/s against
// 157 TFLOP/s), so six of them per product take 3/8 of the time; what the chip
// holds of that is bound by its power (the clock falls to 1.8-2.0 GHz), so work
// beside the MFMAs (LDS traffic, the split itself) is what the layout below
// saves.
#pragma once

#include "gemm_mfma.hpp"

// every lambda of the kernel is inlined, whatever its size: its arrays are registers
#define SBX_INLINE __attribute__((always_inline))

namespace sbx {

typedef __bf16 bf16x2 __attribute__((ext_vector_type(2)));
typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));

// The bf16 MFMA with the fp32 16x16x4's result layout (Mfma<float, 1>).
//   A operand: lane l holds A[i = l % 16][k = 8 * (l / 16) + 0..7], B likewise.
// (32x32x16 has the same peak rate, but the chip holds less of it: 1920
// against 2170 TFLOP/s, operands in registers, both bound by power.)
__device__ inline f32x4 split_mma(bf16x8 a, bf16x8 b, f32x4 c)
{
    return __builtin_amdgcn_mfma_f32_16x16x32_bf16(a, b, c, 0, 0, 0);
}

// Two fp32 values -> their three bf16 pieces, packed (first value in the low
// half).  The differences are exact.  An infinity, or a value that rounds to
// one, leaves NaNs (see redo_flag).
// lost: gathers the last remainders' bits.  A remainder of 2^-126 and more has 8
// significant bits and none in its word's lower half; a smaller one is a
// multiple of 2^-149 whose bits below 2^-133, those that bf16 has no place for,
// are that lower half.  So the split of every value was exact if and only if
// the lower half of `lost` is still 0 (checked on the device over all
// magnitudes from 2^-149 to 2^-90).
__device__ inline void split_pair(float a, float b, uint32_t& p0, uint32_t& p1, uint32_t& p2,
                                  uint32_t& lost)
{
    auto pack = [](float x, float y) {
        const bf16x2 v = {(__bf16)x, (__bf16)y};
        uint32_t p = __builtin_bit_cast(uint32_t, v);
        // (opaque: otherwise each value taken back out of the pair is
        // converted a second time on its own, 13 instructions for 11)
        asm("" : "+v"(p));
        return p;
    };
    auto lo = [](uint32_t p) { return __builtin_bit_cast(float, p << 16); };
    auto hi = [](uint32_t p) { return __builtin_bit_cast(float, p & 0xffff0000u); };
    p0 = pack(a, b);
    const float a1 = a - lo(p0), b1 = b - hi(p0);
    p1 = pack(a1, b1);
    const float a2 = a1 - lo(p1), b2 = b1 - hi(p1);
    // (one instruction, in place: as an expression the remainders of a whole
    // tile are kept to be joined at its end, and spill)
    asm("v_or3_b32 %0, %0, %1, %2" : "+v"(lost) : "v"(a2), "v"(b2));
    p2 = pack(a2, b2);
}

constexpr uint32_t kLostBits = 0xffff;

// Largest magnitude among four values, and whether the split of one is inexact.
__device__ inline void gather_stats(f32x4 w, float& mx, uint32_t& lost)
{
    mx = fmaxf(fmaxf(mx, fmaxf(fabsf(w[0]), fabsf(w[1]))), fmaxf(fabsf(w[2]), fabsf(w[3])));
    uint32_t p0, p1, p2;
    split_pair(w[0], w[1], p0, p1, p2, lost);
    split_pair(w[2], w[3], p0, p1, p2, lost);
}

// The lane's index, computed anew at each use: what the k loop's tail and the
// epilogue derive from it is then not kept in registers over the loop, which
// has none to spare.
__device__ inline int lane_id()
{
    int l;
    asm volatile("v_mbcnt_lo_u32_b32 %0, -1, 0\n\tv_mbcnt_hi_u32_b32 %0, -1, %0" : "=v"(l));
    return l;
}

// f(Int<I>{}) for I = A .. B - 1.
template <int A, int B, typename F>
__device__ __forceinline__ void static_for(F&& f)
{
    if constexpr (A < B) {
        f(Int<A>{});
        static_for<A + 1, B>(f);
    }
}

// Descriptor of an operand whose 32 k rows may span more than 2 GiB (leading
// dimensions from 2^24 on): offsets and sizes are unsigned.  kOobOffset then
// no longer lies past its end; a lane that holds rows outside C reads some of the
// operand instead, and its results are not stored.
template <bool KC>
__device__ inline __amdgpu_buffer_rsrc_t operand_rsrc(const float* base, int64_t bytes)
{
    constexpr uint32_t most = KC ? (uint32_t)kMaxRecords : 0xfffffff0u;
    // (32-bit compares: 64-bit ones take vector registers)
    const int hi = (int)(bytes >> 32);
    const uint32_t lo = (uint32_t)bytes;
    const uint32_t n = hi < 0 ? 0 : hi > 0 || lo > most ? most : lo;
    return __builtin_amdgcn_make_buffer_rsrc(const_cast<float*>(base), (short)0, (int)n, kRsrcWord3);
}

// N rows of an x-contiguous operand at one k.  (One is a plain float: an array of one-element
// vectors ends up in memory.)
template <int N>
struct RowVec {
    typedef float type __attribute__((ext_vector_type(N)));
    __device__ static inline float get(type x, int u) { return x[u]; }
};
template <>
struct RowVec<1> {
    typedef float type;
    __device__ static inline float get(float x, int) { return x; }
};

// The operand that the waves share: global -> registers -> three bf16 planes
// in LDS, 32 k at a time.
//   X: tile extent; NB: its 16-row blocks a wave multiplies (all that are
//   computed); KC: k is contiguous in memory.
// LDS holds the tile in MFMA fragment order: per plane, blocks of 16 tile
// rows; a block is 4 octets of 16 slots of 16 bytes, octet q of a slot being
// k = 16h + 4q + e (h < 2, e < 4) of one row, so a wave reads a fragment as one
// contiguous 16 bytes per lane.  U blocks interleave (block u holds rows
// U*i + u, as in Frag), so a lane's results lie in U consecutive rows.
// A thread holds 4 consecutive k of a row, half an octet: 8 bytes per plane.
// That 16 consecutive lanes fill 128 bytes of distinct banks with them takes
//   KC:  (two rows) the slot index XORed with 2 * octet, and for U > 1, where
//        the rows lie in neighbouring blocks, a block pad of 16 bytes;
//   !KC: lane bit 3 choosing the half, so that 8 slots' both halves are
//        written, and where a thread's XV rows are not all U blocks a block
//        pad that moves its neighbours' blocks.
template <int X, int NB, bool KC, bool KTAIL, int NTHR, int PF, int CPOL>
struct SplitOperand {
    static constexpr int BK = 32;
    static constexpr int NF = X * BK / NTHR;  // floats per thread and k tile
    static constexpr int U = NB % 4 == 0 ? 4 : NB % 2 == 0 ? 2 : 1;
    static constexpr int XV = KC ? 1 : (U < NF / 4 ? U : NF / 4);  // !KC: rows per load
    static constexpr int NG = NF / (4 * XV);       // groups of 4 k (x XV rows) per thread
    static constexpr int VPR = BK / 4;             // KC: 16-byte vectors per row
    static constexpr int RSTEP = NTHR / VPR;       // KC: rows per sweep
    // KC: sweeps inside one group of interleaved blocks (their slots differ)
    static constexpr int NLG = KC && RSTEP < 16 * U ? 16 * U / RSTEP : 1;
    static constexpr int NL = NLG < NG ? NLG : NG;
    static constexpr int XCH = X / XV;             // !KC: chunks of XV rows
    static constexpr int OSTEP = KC ? 1 : NTHR / XCH / 2;  // !KC: octets per sweep
    static constexpr int PAD = KC ? (U > 1 ? 16 : 0) : (XV < U ? 128 / U : 0);
    static constexpr int BLK = 1024 + PAD;  // bytes of a block
    static constexpr int PLANE = (X / 16) * BLK;
    static constexpr int BYTES = 3 * PLANE;  // one k tile
    static constexpr int NROW = KC ? NG : XV;  // rows a thread holds values of
    static_assert(NF % 4 == 0 && NF >= 4, "at least one group of 4 k per thread");
    static_assert(KC ? (RSTEP * NG == X && (NL == 1 || NL * RSTEP == 16 * U || NL == NG))
                     : (XCH % 8 == 0 && XCH * OSTEP * 2 == NTHR && OSTEP * NG == 4),
                  "thread map must cover the tile");

    int voff;       // byte offset from the tile's base; out of range where X is masked
    int row_bytes;  // KC: bytes between sweeps; !KC: between k rows
    int lds0[NL];           // LDS offsets of this thread's first NL groups
    uint32_t lost = 0;      // see split_pair
    typedef RowVec<XV> xvec;
    f32x4 stage[KC ? PF : 1][KC ? NG : 1];       // KC: PF tiles in flight, 4 k of a row each
    typename xvec::type xstage[KC ? 1 : PF][KC ? 1 : NG][4];  // !KC: likewise, XV rows at one k each

    // KC: first k of this thread's vectors
    __device__ static inline int first_k() { return 4 * (lane_id() % VPR); }
    // !KC: chunk of rows of thread tid
    __device__ static inline int chunk(int tid) { return (tid & 7) | ((tid >> 4) % (XCH / 8)) << 3; }

    __device__ inline void init(int tid, int64_t ld, int x_rem)
    {
        int x, o, h, k0;
        if constexpr (KC) {
            x = tid / VPR;
            o = tid % 4;
            h = tid / 4 % 2;
            k0 = 4 * (tid % VPR);
            // (rows past X's end lie past the descriptor's)
            voff = (int)((x * ld + k0) * 4);
            row_bytes = (int)(RSTEP * ld * 4);
        } else {
            x = chunk(tid) * XV;
            h = (tid >> 3) & 1;
            o = tid / (2 * XCH);
            k0 = 16 * h + 4 * o;
            voff = x < x_rem ? (int)((k0 * ld + x) * 4) : kOobOffset;
            row_bytes = (int)(ld * 4);
        }
#pragma unroll
        for (int l = 0; l < NL; ++l) {
            const int xl = x + l * RSTEP;
            const int blk = xl / (16 * U) * U + xl % U;
            const int slot = xl % (16 * U) / U ^ (KC ? 2 * o : 0);
            lds0[l] = blk * BLK + (o * 16 + slot) * 16 + h * 8;
        }
    }

    // Load a k tile through `rs`, moved by the scalar byte offset `soff`.
    // CHECK: only its first k_rem k are inside K.
    template <int S, bool CHECK>
    __device__ inline void load(__amdgpu_buffer_rsrc_t rs, int soff, int k_rem)
    {
#pragma unroll
        for (int g = 0; g < NG; ++g) {
            if constexpr (KC) {
                const int off = !CHECK || first_k() < k_rem ? voff + g * row_bytes : kOobOffset;
                stage[S][g] = __builtin_bit_cast(
                    f32x4, __builtin_amdgcn_raw_buffer_load_b128(rs, off, soff, CPOL));
            } else {
#pragma unroll
                for (int kk = 0; kk < 4; ++kk) {
                    // CHECK: as in DirectOperand
                    const int r = g * OSTEP * 4 + kk;
                    const int off = CHECK ? (int)((uint32_t)voff + (uint32_t)r * (uint32_t)row_bytes) : voff;
                    const int so = CHECK ? soff : soff + r * row_bytes;
                    if constexpr (XV == 4)
                        xstage[S][g][kk] = __builtin_bit_cast(
                            f32x4, __builtin_amdgcn_raw_buffer_load_b128(rs, off, so, CPOL));
                    else if constexpr (XV == 2)
                        xstage[S][g][kk] = __builtin_bit_cast(
                            f32x2, __builtin_amdgcn_raw_buffer_load_b64(rs, off, so, CPOL));
                    else
                        xstage[S][g][kk] = __builtin_bit_cast(
                            float, __builtin_amdgcn_raw_buffer_load_b32(rs, off, so, CPOL));
                }
            }
        }
    }

    // Four consecutive k of a row: group g of staging set S, its row u.
    // MASK: they may straddle K (a k-contiguous vector past K holds the next
    // row's first elements).
    template <int S, bool MASK>
    __device__ inline f32x4 value(int g, int u, int k_rem) const
    {
        f32x4 w;
        if constexpr (KC) {
            w = stage[S][g];
        } else {
#pragma unroll
            for (int e = 0; e < 4; ++e) w[e] = xvec::get(xstage[S][g][e], u);
        }
        if constexpr (KC && KTAIL && MASK) {
            const int lim = k_rem - first_k();
#pragma unroll
            for (int d = 1; d < 4; ++d) w[d] = d < lim ? w[d] : 0.0f;
        }
        return w;
    }

    // Split group g of staging set S and write its pieces to the k tile at `lds`.
    template <int S, bool MASK>
    __device__ inline void store(char* lds, int g, int k_rem)
    {
#pragma unroll
        for (int u = 0; u < XV; ++u) {
            const f32x4 w = value<S, MASK>(g, u, k_rem);
            u32x2 p[3];
            uint32_t a0, a1, a2, b0, b1, b2;
            split_pair(w[0], w[1], a0, a1, a2, lost);
            split_pair(w[2], w[3], b0, b1, b2, lost);
            p[0] = u32x2{a0, b0}; p[1] = u32x2{a1, b1}; p[2] = u32x2{a2, b2};
            const int at = KC ? lds0[g % NL] + g / NL * (NL * RSTEP / 16) * BLK
                              : lds0[0] + u * BLK + g * OSTEP * 256;
#pragma unroll
            for (int t = 0; t < 3; ++t) *reinterpret_cast<u32x2*>(lds + at + t * PLANE) = p[t];
        }
    }

    // The k tile unsplit, for fp32 MFMAs: per 16-row block two halves of 4 octets
    // of 16 slots of 16 bytes (4 k each), the slots XORed with octet and half so
    // that 8 consecutive lanes' writes (KC: one row's) and reads meet no bank twice.
    static constexpr int RAW_BLK = 2048;
    static_assert((X / 16) * RAW_BLK <= BYTES, "a raw tile takes a split one's place");
    template <int S>
    __device__ inline void store_raw(char* lds, int tid, int k_rem) const
    {
        const int x0 = KC ? tid / VPR : chunk(tid) * XV;
        const int h = KC ? tid / 4 % 2 : (tid >> 3) & 1;
        const int o0 = KC ? tid % 4 : tid / (2 * XCH);
#pragma unroll
        for (int g = 0; g < NG; ++g)
#pragma unroll
            for (int u = 0; u < XV; ++u) {
                const int x = x0 + (KC ? g * RSTEP : u), o = o0 + (KC ? 0 : g * OSTEP);
                const int blk = x / (16 * U) * U + x % U, slot = x % (16 * U) / U;
                *reinterpret_cast<f32x4*>(lds + blk * RAW_BLK + h * 1024 + (o * 16 + (slot ^ (o | 4 * h))) * 16) =
                    value<S, true>(g, u, k_rem);
            }
    }
    // A lane's fragment of half h in a raw block.
    __device__ static inline int raw_off(int lane, int h)
    {
        const int i = lane % 16, o = lane / 16;
        return h * 1024 + (o * 16 + (i ^ (o | 4 * h))) * 16;
    }

    // The staged tile's part in its rows' statistics; next() may stage another.
    template <int S, typename F>
    __device__ inline void stats(float (&mx)[NROW], uint32_t (&ls)[NROW], int k_rem, F&& next)
    {
        f32x4 w[NG][XV];
#pragma unroll
        for (int g = 0; g < NG; ++g)
#pragma unroll
            for (int u = 0; u < XV; ++u) w[g][u] = value<S, true>(g, u, k_rem);
        next();
#pragma unroll
        for (int g = 0; g < NG; ++g)
#pragma unroll
            for (int u = 0; u < XV; ++u) gather_stats(w[g][u], mx[KC ? g : u], ls[KC ? g : u]);
    }

    // Tile row of slot i of block b.
    __device__ static inline int map(int b, int i)
    {
        return (b / U) * U * 16 + U * i + (b % U);
    }
    // Byte offset of a lane's fragment in a block.
    __device__ static inline int frag_off(int lane)
    {
        const int i = lane % 16, o = lane / 16;
        return (o * 16 + (KC ? i ^ (2 * o) : i)) * 16;
    }
    // tile row of this thread's row i
    __device__ static inline int row_of(int tid, int i, int)
    {
        return KC ? tid / VPR + i * RSTEP : chunk(tid) * XV + i;
    }
};

// An operand that no two waves share (the tile has one wave along the other
// dimension): each wave loads its own NB blocks of 16 rows straight into the
// MFMA lane layout and splits them in registers, with no LDS in between.
// Lane (i, q) holds, of a 32-k tile, k = 16h + 4q + e (h < 2, e < 4) of row
// map(b, i) -- the k order SplitOperand's 16-row blocks use.
// U blocks interleave (row U*i + u of a group is slot i of block u).
//   KC:  two 16-byte loads per block.  PF == 1: each covers 64 bytes of 16
//        rows.  PF > 1 (streaming from HBM): each covers the whole 128 bytes of 8
//        rows: load h brings lane (i, q) floats 4q + 16 (i / 8) of slot 8h + i % 8,
//        and the lanes i and i ^ 8 then trade halves (one DPP move a
//        register; 65536 x 32 x 4096: 214 -> 185 us; 8192^3, which does not
//        stream, is 1.5 % faster without).  One descriptor per block, clipped to the operand: rows
//        past its end read as zeros.
//   !KC: eight loads of U rows at one k each.
template <int NB, bool KC, bool KTAIL, int PF, int CPOL>
struct DirectOperand {
    static constexpr bool TRADE = KC && PF > 1;
    static constexpr int NPC = PF > 1 ? 2 : 1;
    static constexpr int U = NB % 4 == 0 ? 4 : NB % 2 == 0 ? 2 : 1;
    static constexpr int NW = KC ? 1 : NB / U;  // !KC: groups of interleaved blocks
    static constexpr int NROW = NB;  // rows a lane holds values of
    int voff[KC ? 2 : NW];
    uint32_t lost = 0;  // see split_pair
    typedef RowVec<U> xvec;
    f32x4 stage[KC ? PF : 1][KC ? NB : 1][2];     // KC: PF tiles in flight
    typename xvec::type xstage[KC ? 1 : PF][KC ? 1 : NW][8];  // !KC: likewise, U rows at one k each
    bf16x8 pc[NPC][NB][3];

    // 4q, and the first k of lane l's KC loads
    __device__ static inline int first_k() { return lane_id() / 16 * 4; }
    __device__ static inline int load_k(int l)
    {
        return l / 16 * 4 + (TRADE ? l % 16 / 8 * 16 : 0);
    }

    __device__ inline void init(int lane, int64_t ld, int x_rem)
    {
        const int i = lane % 16, k0 = lane / 16 * 4, kl = load_k(lane);
        if constexpr (KC) {
            voff[0] = (int)((U * (TRADE ? i % 8 : i) * ld + kl) * 4);
            voff[1] = TRADE ? voff[0] + (int)(8 * U * ld * 4) : voff[0];
        } else {
#pragma unroll
            for (int w = 0; w < NW; ++w) {
                const int x = w * 16 * U + U * i;
                voff[w] = x < x_rem ? (int)((k0 * ld + x) * 4) : kOobOffset;
            }
        }
    }

    // A k tile through rs[b] (KC: block b's descriptor; else rs[0]).
    template <int S, bool CHECK>
    __device__ inline void load(const __amdgpu_buffer_rsrc_t (&rs)[KC ? NB : 1], int soff,
                                int row_bytes, int k_rem)
    {
        if constexpr (KC) {
            const int kl = CHECK ? load_k(lane_id()) : 0;
#pragma unroll
            for (int b = 0; b < NB; ++b)
#pragma unroll
                for (int h = 0; h < 2; ++h) {
                    const int off = !CHECK || kl + (TRADE ? 0 : 16 * h) < k_rem ? voff[h] : kOobOffset;
                    stage[S][b][h] = __builtin_bit_cast(
                        f32x4, __builtin_amdgcn_raw_buffer_load_b128(
                                   rs[b], off, TRADE ? soff : soff + 64 * h, CPOL));
                }
        } else {
#pragma unroll
            for (int w = 0; w < NW; ++w)
#pragma unroll
                for (int n = 0; n < 8; ++n) {
                    const int h = n / 4, e = n % 4;
                    // CHECK: a row past K lies past the descriptor's end (the
                    // row's offset then goes where that is tested for certain)
                    const int r = 16 * h + e;
                    const int off = CHECK ? (int)((uint32_t)voff[w] + (uint32_t)r * (uint32_t)row_bytes) : voff[w];
                    const int so = CHECK ? soff : soff + r * row_bytes;
                    if constexpr (U == 4)
                        xstage[S][w][n] = __builtin_bit_cast(
                            f32x4, __builtin_amdgcn_raw_buffer_load_b128(rs[0], off, so, CPOL));
                    else if constexpr (U == 2)
                        xstage[S][w][n] = __builtin_bit_cast(
                            f32x2, __builtin_amdgcn_raw_buffer_load_b64(rs[0], off, so, CPOL));
                    else
                        xstage[S][w][n] = __builtin_bit_cast(
                            float, __builtin_amdgcn_raw_buffer_load_b32(rs[0], off, so, CPOL));
                }
        }
    }

    // The trade of halves, once per staged tile, before value().
    template <int S>
    __device__ inline void arrange()
    {
        if constexpr (TRADE)
#pragma unroll
            for (int b = 0; b < NB; ++b)
#pragma unroll
                for (int d = 0; d < 4; ++d) {
                    constexpr int kRor8 = 0x128;  // lane i takes lane i ^ 8's, of 16
                    const float xf = stage[S][b][0][d], yf = stage[S][b][1][d];
                    const int x = __builtin_bit_cast(int, xf), y = __builtin_bit_cast(int, yf);
                    // lanes 8-15 take y, lanes 0-7 take x
                    stage[S][b][0][d] = __builtin_bit_cast(
                        float, __builtin_amdgcn_update_dpp(x, y, kRor8, 0xf, 0xc, false));
                    stage[S][b][1][d] = __builtin_bit_cast(
                        float, __builtin_amdgcn_update_dpp(y, x, kRor8, 0xf, 0x3, false));
                }
    }

    // k = 16h + 4q + 0..3 of block b's row.  MASK: they may straddle K.
    template <int S, bool MASK>
    __device__ inline f32x4 value(int b, int h, int k_rem) const
    {
        f32x4 w;
        if constexpr (KC) {
            w = stage[S][b][h];
        } else {
#pragma unroll
            for (int e = 0; e < 4; ++e) w[e] = xvec::get(xstage[S][b / U][4 * h + e], b % U);
        }
        if constexpr (KC && KTAIL && MASK) {
            const int lim = k_rem - first_k() - 16 * h;
#pragma unroll
            for (int d = 1; d < 4; ++d) w[d] = d < lim ? w[d] : 0.0f;
        }
        return w;
    }

    // Split the staged tile into the MFMA operands pc[P].
    template <int S, int P, bool MASK>
    __device__ inline void split(int k_rem)
    {
        arrange<S>();
        u32x4 p[NB][3];
        auto half = [&](int b, int h) SBX_INLINE {
            const f32x4 w = value<S, MASK>(b, h, k_rem);
#pragma unroll
            for (int d = 0; d < 2; ++d) {
                uint32_t q0, q1, q2;
                split_pair(w[2 * d], w[2 * d + 1], q0, q1, q2, lost);
                p[b][0][2 * h + d] = q0; p[b][1][2 * h + d] = q1; p[b][2][2 * h + d] = q2;
            }
        };
        // in the order that frees the loads' registers soonest
        if constexpr (KC) {
#pragma unroll
            for (int b = 0; b < NB; ++b) { half(b, 0); half(b, 1); }
        } else {
#pragma unroll
            for (int h = 0; h < 2; ++h) {
#pragma unroll
                for (int b = 0; b < NB; ++b) half(b, h);
                if constexpr (PF == 1) __builtin_amdgcn_sched_barrier(0);
            }
        }
#pragma unroll
        for (int b = 0; b < NB; ++b)
#pragma unroll
            for (int t = 0; t < 3; ++t) pc[P][b][t] = __builtin_bit_cast(bf16x8, p[b][t]);
    }

    // The staged tile's part in its rows' statistics; next() may stage another.
    template <int S, typename F>
    __device__ inline void stats(float (&mx)[NROW], uint32_t (&ls)[NROW], int k_rem, F&& next)
    {
        arrange<S>();
        f32x4 w[NB][2];
#pragma unroll
        for (int b = 0; b < NB; ++b)
#pragma unroll
            for (int h = 0; h < 2; ++h) w[b][h] = value<S, true>(b, h, k_rem);
        next();
#pragma unroll
        for (int b = 0; b < NB; ++b)
#pragma unroll
            for (int h = 0; h < 2; ++h) gather_stats(w[b][h], mx[b], ls[b]);
    }

    __device__ static inline int map(int b, int i)
    {
        return (b / U) * U * 16 + U * i + (b % U);
    }
    __device__ static inline int row_of(int tid, int i, int w0) { return w0 + map(i, tid % 16); }
};

// Shorter sums are left to fp32 MFMAs: with few terms the rounding
// of the result is most of the error, and a split adds its own to it.  One k
// tile holds them.
constexpr int kSplitMinK = 32;

// Whether a tile has to be computed again with fp32 MFMAs.  Two things show
// that the split did not hold its values:
// (1) Every infinity and NaN of an operand, every value that rounds to an
//     infinite bf16 and every overflow leaves a non-finite accumulator (inf * 0
//     and inf - inf are NaN).
// (2) A value whose split is inexact (split_pair's lost: it lies below 2^-110)
//     is held to within 2^-134.  Over K' terms that moves a result by
//         2^-134 K' (max of its column, if its row holds such a value,
//                    + max of its row, if its column does),
//     which is let pass where it is below 2^-24 of the result, as a product's
//     own dropped terms are.  Tails of a softmax, 2^-120 beside 1, pass; rows
//     that are tiny as a whole, or whose other values meet zeros, do not.
// redo_flag: a thread's own view (1, 2: lost bits of the direct, the shared
// operand; 4: a non-finite accumulator), all that a tile without them pays.
template <typename MF, int NBM, int NBN>
__device__ __forceinline__ int redo_flag(const typename MF::acc_t (&acc)[NBM][NBN], uint32_t lost_d,
                                uint32_t lost_s)
{
    float z = 0.0f;  // 0 * acc is not 0 where acc is not finite
#pragma unroll
    for (int i = 0; i < NBM; ++i)
#pragma unroll
        for (int j = 0; j < NBN; ++j)
#pragma unroll
            for (int r = 0; r < MF::NACC; ++r) z = fmaf(acc[i][j][r], 0.0f, z);
    return (z == 0.0f ? 0 : 4) | ((lost_s & kLostBits) != 0 ? 2 : 0) | ((lost_d & kLostBits) != 0 ? 1 : 0);
}

// redo_fails: a lane's accumulators against (1) and (2): 0, or how many fail
// (in bits 16 and up; a non-finite one counts as two) over the last one's code.
// row: largest magnitude of each of the tile's BM rows of A and BN columns of
// B, as bits; low: not 0 where that row or column holds a value with an inexact
// split, kOutside where it lies outside C: that comes of the memory beside the
// operands and counts for nothing.  terms: K'.
constexpr unsigned kOutside = 1u << 31;
template <typename MF, typename OpA, typename OpB, int BM, int NBM, int NBN>
__device__ __forceinline__ int redo_fails(const typename MF::acc_t (&acc)[NBM][NBN], const unsigned* row,
                                 const unsigned* low, int terms, int wm0, int wn0, int lane)
{
    const float unit = 0x1p-110f * (float)terms;  // 2^24 * 2^-134 K'
    int fails = 0;
#pragma unroll
    for (int j = 0; j < NBN; ++j) {
        const int n = wn0 + OpB::map(j, lane % 16);
        const float cmax = __builtin_bit_cast(float, row[BM + n]);
        const unsigned clow = low[BM + n];
#pragma unroll
        for (int i = 0; i < NBM; ++i)
#pragma unroll
            for (int r = 0; r < MF::NACC; ++r) {
                const int m = wm0 + OpA::map(i, MF::row(r, lane / 16));
                const unsigned rlow = low[m];
                const float least = unit * ((rlow != 0 ? cmax : 0.0f) +
                                            (clow != 0 ? __builtin_bit_cast(float, row[m]) : 0.0f));
                const float v = fabsf(acc[i][j][r]);
                int step = v <= __FLT_MAX__ ? (v >= least ? 0 : 0x10000) : 0x20000;
                if ((int)(rlow | clow) < 0) step = 0;
                fails = step ? (fails & ~0xffff) + step + ((j * NBM + i) * MF::NACC + r) : fails;
                // (opaque: otherwise each term is kept until the end, and spills)
                asm volatile("" : "+v"(fails));
            }
        __builtin_amdgcn_sched_barrier(0);
    }
    return fails;
}

// A sum of ordinary terms may cancel to nothing (one result in 10^8 at K =
// 4096): up to kRedoSingles failing results of a wave, one a lane, are
// looked at by themselves, the wave's lanes taking K between them: such a one
// passes where 2^-134 per value with an inexact split is below 2^-24 of its sum of magnitudes.
constexpr int kRedoSingles = 8;

template <typename MF, typename OpA, typename OpB, bool A_KC, bool B_KC, int NBM>
__device__ __forceinline__ bool redo_needed(const GemmArgs<float>& p, int fails, const float* A, const float* B,
                                   int m0, int n0, int wm0, int wn0, int k_begin, int k_end, int lane)
{
    unsigned long long who = __ballot(fails != 0);
    if (__ballot(fails >= 0x20000) != 0 || __popcll(who) > kRedoSingles) return true;
    for (; who != 0; who &= who - 1) {
        const int src = __ffsll(who) - 1;
        const int code = __builtin_amdgcn_readlane(fails, src) & 0xffff;
        const int i = code / MF::NACC % NBM, j = code / MF::NACC / NBM;
        const int64_t m = m0 + wm0 + OpA::map(i, MF::row(code % MF::NACC, src / 16));
        const int64_t n = n0 + wn0 + OpB::map(j, src % 16);
        float sum = 0.0f, loss = 0.0f;
#pragma unroll 1
        for (int64_t k = k_begin + lane; k < k_end; k += 64) {
            const float a = A[A_KC ? m * p.lda + k : k * p.lda + m];
            const float b = B[B_KC ? n * p.ldb + k : k * p.ldb + n];
            float ma = 0.0f, mb = 0.0f;
            uint32_t la = 0, lb = 0;
            gather_stats(f32x4{a, a, a, a}, ma, la);
            gather_stats(f32x4{b, b, b, b}, mb, lb);
            sum = fmaf(ma, mb, sum);
            loss += ((la & kLostBits) != 0 ? mb : 0.0f) + ((lb & kLostBits) != 0 ? ma : 0.0f);
        }
        for (int d = 32; d > 0; d >>= 1) {
            sum += __shfl_xor(sum, d);
            loss += __shfl_xor(loss, d);
        }
        if (!(0x1p-110f * loss <= sum)) return true;
    }
    return false;
}

// BM x BN tile, 32 k per step, WAVES_M x WAVES_N waves, one of them 1; BMC, BNC:
// rows and columns of the tile that are computed (fewer than BM, BN where the
// host knows that M <= BMC or N <= BNC, one tile row or column: a 48-wide C
// then does not pay for 64 columns of MFMAs); PF: see step1 and step; WPE: waves per SIMD; STREAM: the operand whose loads
// are non-temporal.
// One wave along N: each wave's rows of A are its own (A_DIRECT; one along M:
// its columns of B), and that operand goes from memory to the wave's
// registers (DirectOperand); only the other one, which all waves share, goes
// through LDS (SplitOperand).  Against both through LDS that takes nearly
// half of the LDS traffic: 8192^3 5.13 -> 4.55 ms (with the 16x16x32 MFMAs).
template <int BM, int BN, int WAVES_M, int WAVES_N, bool A_KC, bool B_KC, bool KTAIL, int PF,
          int WPE, int STREAM, int BNC, int BMC>
__global__ void __launch_bounds__(WAVES_M * WAVES_N * 64) __attribute__((amdgpu_waves_per_eu(WPE, WPE)))
gemm_split_kernel(GemmArgs<float> p)
{
    typedef Mfma<float, 1> MF;
    constexpr bool A_DIRECT = WAVES_N == 1;
    static_assert(A_DIRECT || WAVES_M == 1, "one operand belongs to the waves");
    constexpr int MB = 16, BK = 32;
    constexpr int WTM = BMC / WAVES_M, WTN = BNC / WAVES_N;
    constexpr int NBM = WTM / MB, NBN = WTN / MB;
    constexpr int NTHR = WAVES_M * WAVES_N * 64;
    constexpr int CA = STREAM == 1 ? kNonTemporal : 0, CB = STREAM == 2 ? kNonTemporal : 0;
    constexpr bool D_KC = A_DIRECT ? A_KC : B_KC, S_KC = A_DIRECT ? B_KC : A_KC;
    constexpr int NBD = A_DIRECT ? NBM : NBN, NBS = A_DIRECT ? NBN : NBM;
    constexpr int XS = A_DIRECT ? BN : BM;
    typedef DirectOperand<NBD, D_KC, KTAIL, PF, A_DIRECT ? CA : CB> OpD;
    typedef SplitOperand<XS, NBS, S_KC, KTAIL, NTHR, PF, A_DIRECT ? CB : CA> OpS;
    typedef typename std::conditional<A_DIRECT, OpD, OpS>::type OpA;
    typedef typename std::conditional<A_DIRECT, OpS, OpD>::type OpB;

    __shared__ __attribute__((aligned(16))) char smem[2 * OpS::BYTES];
    __shared__ int redo;
    static_assert(2 * OpS::BYTES >= 8 * (BM + BN), "the rows' statistics lie there after the k loop");

    const int tid = threadIdx.x;
    const int lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int wm0 = (wave / WAVES_N) * WTM;
    const int wn0 = (wave % WAVES_N) * WTN;

    const TileUnit t = tile_unit(p);
    const int m0 = t.tm * BM, n0 = t.tn * BN;
    const float* A;
    const float* B;
    float* C;
    batch_bases(p, (int64_t)blockIdx.z, A, B, C);

    const int64_t a_span = A_KC ? ((int64_t)(p.M - 1) * p.lda + p.K) * 4
                                : ((int64_t)(p.K - 1) * p.lda + p.M) * 4;
    const int64_t b_span = B_KC ? ((int64_t)(p.N - 1) * p.ldb + p.K) * 4
                                : ((int64_t)(p.K - 1) * p.ldb + p.N) * 4;
    const int64_t a_org = A_KC ? (int64_t)m0 * p.lda : (int64_t)m0;
    const int64_t b_org = B_KC ? (int64_t)n0 * p.ldb : (int64_t)n0;

    // the direct operand from the wave's first row, the shared one from the tile's
    const float* const D = A_DIRECT ? A : B;
    const float* const S = A_DIRECT ? B : A;
    const int64_t ld_d = A_DIRECT ? p.lda : p.ldb, ld_s = A_DIRECT ? p.ldb : p.lda;
    const int64_t d_span = A_DIRECT ? a_span : b_span, s_span = A_DIRECT ? b_span : a_span;
    const int w0 = A_DIRECT ? wm0 : wn0;
    const int64_t d_org = (A_DIRECT ? a_org : b_org) + (D_KC ? (int64_t)w0 * ld_d : (int64_t)w0);
    const int64_t s_org = A_DIRECT ? b_org : a_org;
    const int64_t d_step = D_KC ? BK : (int64_t)BK * ld_d;
    const int64_t s_step = S_KC ? BK : (int64_t)BK * ld_s;

    typename MF::acc_t acc[NBM][NBN];
#pragma unroll
    for (int i = 0; i < NBM; ++i)
#pragma unroll
        for (int j = 0; j < NBN; ++j)
#pragma unroll
            for (int r = 0; r < MF::NACC; ++r) acc[i][j][r] = 0;

    const int nk_all = (p.K + BK - 1) / BK;
    const int kt0 = t.is_split ? (int)((int64_t)t.part * nk_all / p.split) : 0;
    const int nk = t.is_split ? (int)((int64_t)(t.part + 1) * nk_all / p.split) : nk_all;

    OpD opd;
    OpS ops;
    // (again after the k loop, whose registers then hold nothing for later)
    auto init = [&](int ln) SBX_INLINE {
        opd.init(ln, ld_d, (A_DIRECT ? p.M - m0 : p.N - n0) - w0);
        ops.init(wave * 64 + ln, ld_s, A_DIRECT ? p.N - n0 : p.M - m0);
    };
    init(lane);
    if (tid == 0) redo = 0;

    // Fixed descriptors for the k tiles that are full and not the last,
    // moving ones for the rest (as in gemm_mfma_kernel).  A k-contiguous
    // direct operand takes one descriptor per block of 16 rows.
    constexpr int ND = D_KC ? NBD : 1;
    auto d_rsrc = [&](int64_t org, __amdgpu_buffer_rsrc_t (&r)[ND]) SBX_INLINE {
#pragma unroll
        for (int b = 0; b < ND; ++b) {
            const int64_t o = org + (int64_t)OpD::map(b, 0) * ld_d;
            r[b] = operand_rsrc<D_KC>(D + o, d_span - o * 4);
        }
    };
    __amdgpu_buffer_rsrc_t rd0[ND];
    // (the fixed ones by make_rsrc: where they are used 2 GiB is enough, and with
    // operand_rsrc's selects before the loop 8192^3 read 15 % more from beyond
    // L2 and took 4496 us against 4442)
#pragma unroll
    for (int b = 0; b < ND; ++b) {
        const int64_t o = d_org + (int64_t)OpD::map(b, 0) * ld_d;
        rd0[b] = make_rsrc(D + o, d_span - o * 4);
    }
    const __amdgpu_buffer_rsrc_t rs0 = make_rsrc(S + s_org, s_span - s_org * 4);
    const int d_row_bytes = (int)(ld_d * 4);
    const int64_t d_tile = D_KC ? (int64_t)NBD * 16 * ld_d + BK : (int64_t)BK * ld_d + NBD * 16;
    const int64_t s_tile = S_KC ? (int64_t)XS * ld_s + BK : (int64_t)BK * ld_s + XS;
    const bool fixed_ok = ((int64_t)nk * d_step + d_tile) * 4 < kMaxRecords - 64 &&
                          ((int64_t)nk * s_step + s_tile) * 4 < kMaxRecords - 64;
    auto issue_d = [&](auto SET, int kt, auto FIXED) SBX_INLINE {
        constexpr int st = decltype(SET)::value;
        if constexpr (decltype(FIXED)::value) {
            opd.template load<st, false>(rd0, (int)(kt * d_step * 4), d_row_bytes, BK);
        } else {
            __amdgpu_buffer_rsrc_t r[ND];
            d_rsrc(d_org + kt * d_step, r);
            opd.template load<st, true>(r, 0, d_row_bytes, p.K - kt * BK);
        }
    };
    auto issue_s = [&](auto SET, int kt, auto FIXED) SBX_INLINE {
        constexpr int st = decltype(SET)::value;
        if constexpr (decltype(FIXED)::value) {
            ops.template load<st, false>(rs0, (int)(kt * s_step * 4), BK);
        } else {
            const int64_t ps = s_org + kt * s_step;
            ops.template load<st, true>(operand_rsrc<S_KC>(S + ps, s_span - ps * 4), 0, p.K - kt * BK);
        }
    };
    auto commit = [&](auto SET, int kt, int buf, auto MASK) SBX_INLINE {
#pragma unroll
        for (int g = 0; g < OpS::NG; ++g)
            ops.template store<decltype(SET)::value, decltype(MASK)::value>(
                smem + buf * OpS::BYTES, g, p.K - kt * BK);
    };
    bf16x8 fs[PF][3];  // fragments of one shared block (PF > 1: and of the next)
    auto read_s = [&](auto F, int at, int j, int u) SBX_INLINE {
        fs[decltype(F)::value][u] = *reinterpret_cast<const bf16x8*>(smem + at + j * OpS::BLK + u * OpS::PLANE);
    };
    // Products of piece u of a shared block and piece v of the direct
    // operand's N blocks from i0 on, into their sums t of this k tile (C:
    // the first, from zero).
    auto mma = [&](auto P, auto F, auto C, int i0, int u, int v, auto& t) SBX_INLINE {
        constexpr int pp = decltype(P)::value, f = decltype(F)::value;
        constexpr int n = (int)(sizeof(t) / sizeof(t[0]));
        const f32x4 zero = {0, 0, 0, 0};
#pragma unroll
        for (int i = 0; i < n; ++i) {
            const f32x4 c = decltype(C)::value ? zero : t[i];
            if constexpr (A_DIRECT) t[i] = split_mma(opd.pc[pp][i0 + i][v], fs[f][u], c);
            else t[i] = split_mma(fs[f][u], opd.pc[pp][i0 + i][v], c);
        }
    };
    auto add = [&](int i0, int j, const auto& t) SBX_INLINE {
        constexpr int n = (int)(sizeof(t) / sizeof(t[0]));
#pragma unroll
        for (int i = 0; i < n; ++i)
#pragma unroll
            for (int r = 0; r < 4; ++r) {
                if constexpr (A_DIRECT) acc[i0 + i][j][r] += t[i][r];
                else acc[j][i0 + i][r] += t[i][r];
            }
    };
    constexpr bool kTight = NBM * NBN >= 32;  // 128 accumulators: no register to spare
    static_assert(NBD % 2 == 0 && PF <= 2, "direct blocks are multiplied two side by side");
    // PF == 1 (registers are short): the tile's direct operand is staged,
    // its shared one in LDS buffer cur.  The next tile's shared loads run
    // over the first half of the MFMAs, its direct ones over the second.
    // Piece u of the next shared block is read when this block's MFMAs
    // have used it.
    auto step1 = [&](int kt, int cur, auto MASK, auto FIXED) SBX_INLINE {
        constexpr Int<0> z{};
        opd.template split<0, 0, decltype(MASK)::value>(p.K - kt * BK);
        __builtin_amdgcn_sched_barrier(0);
        issue_s(z, kt + 1, FIXED);
        __builtin_amdgcn_sched_barrier(0);
        const int at = cur * OpS::BYTES + OpS::frag_off(kTight ? lane_id() : lane);
#pragma unroll
        for (int u = 2; u >= 0; --u) read_s(z, at, 0, u);
        static_for<0, NBS>([&](auto J) SBX_INLINE {
            constexpr int j = decltype(J)::value;
            static_for<0, NBD / 2>([&](auto H) SBX_INLINE {
                constexpr int i0 = decltype(H)::value * 2;
                // the six products: by piece of the shared operand, small ones first
                f32x4 t[2];
                static_for<0, 3>([&](auto W) SBX_INLINE {
                    constexpr int u = 2 - decltype(W)::value;
                    static_for<0, 3 - u>([&](auto V) SBX_INLINE {
                        mma(z, z, Int<u == 2>{}, i0, u, 2 - u - decltype(V)::value, t);
                    });
                    if constexpr (j + 1 < NBS && i0 + 2 == NBD) read_s(z, at, j + 1, u);
                });
                add(i0, j, t);
                __builtin_amdgcn_sched_barrier(0);
            });
            if constexpr (j == NBS / 2 - 1) {
                commit(z, kt + 1, cur ^ 1, MASK);
                __builtin_amdgcn_sched_barrier(0);
                issue_d(z, kt + 1, FIXED);
                __builtin_amdgcn_sched_barrier(0);
            }
        });
        __syncthreads();
    };
    // PF > 1: the tile's direct operand is split already (pc[par]), its
    // shared one in LDS buffer par.  The next tile, in staging set SET, is
    // split among this tile's MFMAs (the waves of a workgroup run in step:
    // split first, multiplied then, each unit would wait for the other),
    // and the set refilled PF tiles on.
    auto step = [&](auto SET, auto P, int kt, auto MASK, auto FIXED) SBX_INLINE {
        constexpr int par = decltype(P)::value;
        const int at = par * OpS::BYTES + OpS::frag_off(lane);
#pragma unroll
        for (int u = 2; u >= 0; --u) read_s(Int<0>{}, at, 0, u);
        opd.template split<decltype(SET)::value, par ^ 1, decltype(MASK)::value>(p.K - (kt + 1) * BK);
        commit(SET, kt + 1, par ^ 1, MASK);
        issue_s(SET, kt + 1 + PF, FIXED);
        issue_d(SET, kt + 1 + PF, FIXED);
        static_for<0, NBS>([&](auto J) SBX_INLINE {
            constexpr int j = decltype(J)::value, f = j % 2;
            if constexpr (j + 1 < NBS)
#pragma unroll
                for (int u = 2; u >= 0; --u) read_s(Int<(j + 1) % 2>{}, at, j + 1, u);
            f32x4 t[NBD];
            static_for<0, 3>([&](auto W) SBX_INLINE {
                constexpr int u = 2 - decltype(W)::value;
                static_for<0, 3 - u>([&](auto V) SBX_INLINE {
                    mma(P, Int<f>{}, Int<u == 2>{}, 0, u, 2 - u - decltype(V)::value, t);
                });
            });
            add(0, j, t);
        });
        // Nothing of the next step moves up: its splits would wait for the
        // youngest loads.
        __builtin_amdgcn_sched_barrier(0);
        __syncthreads();
        __builtin_amdgcn_sched_barrier(0);
    };

    constexpr std::false_type kNo{};
    constexpr std::true_type kYes{};
    // The wave's tile over this unit's k with fp32 MFMAs, in the place of what is
    // in acc: sums shorter than kSplitMinK from the start (4096^2 x 16 17.5 us,
    // 1024 x 8192 x 31 12.7; the fp32 MFMA tile kernels 16.5 and 12.4), and tiles
    // the split cannot hold after it (4096^3 of NaN 1.52 ms, with one infinity
    // 1.58; those kernels 0.91 and 1.02).  LDS double buffer, one barrier per 32 k.  The next tile's loads run over this one's MFMAs where there are
    // registers for them; a large tile's MFMAs take 8 us per 32 k, its loads 1.
    auto fp32_pass = [&]() SBX_INLINE {
        constexpr Int<0> z{};
        const int ln = lane_id(), td = wave * 64 + ln;
        init(ln);
#pragma unroll
        for (int i = 0; i < NBM; ++i)
#pragma unroll
            for (int j = 0; j < NBN; ++j)
#pragma unroll
                for (int r = 0; r < MF::NACC; ++r) acc[i][j][r] = 0;
        auto issue = [&](int kt) SBX_INLINE {
            issue_s(z, kt, kNo);
            issue_d(z, kt, kNo);
        };
        if constexpr (!kTight) issue(kt0);
        int cur = 0;
#pragma unroll 1
        for (int kt = kt0; kt < nk; ++kt, cur ^= 1) {
            const int k_rem = p.K - kt * BK;
            char* const buf = smem + cur * OpS::BYTES;
            if constexpr (kTight) issue(kt);
            ops.template store_raw<0>(buf, td, k_rem);
            opd.template arrange<0>();
            f32x4 fd[2][NBD];
#pragma unroll
            for (int h = 0; h < 2; ++h)
#pragma unroll
                for (int i = 0; i < NBD; ++i) fd[h][i] = opd.template value<0, true>(i, h, k_rem);
            if constexpr (!kTight) issue(kt + 1);
            __syncthreads();
#pragma unroll
            for (int h = 0; h < 2; ++h) {
                if (h == 1 && k_rem <= 16) break;
                const int off = OpS::raw_off(ln, h);
                constexpr int JW = !kTight && NBS % 2 == 0 ? 2 : 1;  // blocks side by side
                static_for<0, NBS / JW>([&](auto G) SBX_INLINE {
                    constexpr int j0 = decltype(G)::value * JW;
                    f32x4 fs[JW];
#pragma unroll
                    for (int j = 0; j < JW; ++j)
                        fs[j] = *reinterpret_cast<const f32x4*>(buf + off + (j0 + j) * OpS::RAW_BLK);
#pragma unroll
                    for (int e = 0; e < 4; ++e)
#pragma unroll
                        for (int j = 0; j < JW; ++j)
#pragma unroll
                            for (int i = 0; i < NBD; ++i) {
                                if constexpr (A_DIRECT)
                                    acc[i][j0 + j] = MF::mma(fd[h][i][e], fs[j][e], acc[i][j0 + j]);
                                else
                                    acc[j0 + j][i] = MF::mma(fs[j][e], fd[h][i][e], acc[j0 + j][i]);
                            }
                    __builtin_amdgcn_sched_barrier(0);
                });
            }
        }
    };

    bool again = p.K < kSplitMinK;
    if (!again) {
        // tile t is staged in set (t - kt0) % PF
        static_for<0, PF>([&](auto I) SBX_INLINE {
            issue_s(I, kt0 + decltype(I)::value, kNo);
            issue_d(I, kt0 + decltype(I)::value, kNo);
        });
        commit(Int<0>{}, kt0, 0, kYes);
        if constexpr (PF > 1) {
            opd.template split<0, 0, true>(p.K - kt0 * BK);
            issue_s(Int<0>{}, kt0 + PF, kNo);
            issue_d(Int<0>{}, kt0 + PF, kNo);
        }
        __syncthreads();
        probe_mark(p, 0);
        int kt = kt0;
        if constexpr (PF == 1) {
            // (one copy of the step: two in turn, with fixed LDS buffers, take
            // more registers than there are)
            int cur = 0;
            // every tile a step loads (kt + 1) is full and not the last
            if (fixed_ok)
                for (; kt + 1 < nk - 1; ++kt, cur ^= 1) step1(kt, cur, kNo, kYes);
            for (; kt < nk; ++kt, cur ^= 1) step1(kt, cur, kYes, kNo);
        } else {
            // every tile a step loads (up to kt + 1 + PF) is full and not the last
            if (fixed_ok)
                for (; kt + 2 + PF < nk - 1; kt += 2)
                    static_for<0, 2>([&](auto I) SBX_INLINE {
                        constexpr int i = decltype(I)::value;
                        step(Int<(i + 1) % PF>{}, Int<i>{}, kt + i, kNo, kYes);
                    });
            for (; kt < nk; kt += 2)
                static_for<0, 2>([&](auto I) SBX_INLINE {
                    constexpr int i = decltype(I)::value;
                    if (kt + i < nk) step(Int<(i + 1) % PF>{}, Int<i>{}, kt + i, kYes, kNo);
                });
        }
        probe_mark(p, 1);
        // (all waves are past their last use of smem)
        const int flag = redo_flag<MF>(acc, opd.lost, ops.lost);
        if (flag) atomicOr(&redo, flag);
        __syncthreads();
        const int flags = __builtin_amdgcn_readfirstlane(redo);
        // Two looks.  The first takes every row of an operand with an inexact
        // split (be it in what lies beside the matrix) to hold one, and reads the
        // other operand again for its magnitudes: it lets pass no less than the
        // second, which reads both.
        for (int look = (flags & 3) != 0 ? 0 : 1; __builtin_expect(flags != 0, 0) && look < 2; ++look) {
            const int ln = lane_id(), td = wave * 64 + ln;
            init(ln);
            unsigned* const row = reinterpret_cast<unsigned*>(smem);
            unsigned* const low = row + BM + BN;
            const int d0 = A_DIRECT ? 0 : BM, s0 = A_DIRECT ? BM : 0;
            const bool lost_a = (flags & (A_DIRECT ? 1 : 2)) != 0, lost_b = (flags & (A_DIRECT ? 2 : 1)) != 0;
            for (int i = td; i < BM + BN; i += NTHR) {
                row[i] = 0;
                const bool inside = i < BM ? i < p.M - m0 : i - BM < p.N - n0;
                low[i] = !inside ? kOutside : look == 0 && (i < BM ? lost_a : lost_b);
            }
            __syncthreads();
            const bool see_d = look == 0 ? (flags & 2) != 0 : (flags & 3) != 0;
            const bool see_s = look == 0 ? (flags & 1) != 0 : (flags & 3) != 0;
            constexpr Int<0> z{};
            // the next tile's loads run over this one's statistics
            if (see_d) {
                float mx[OpD::NROW] = {};
                uint32_t ls[OpD::NROW] = {};
                issue_d(z, kt0, kNo);
                for (kt = kt0; kt < nk; ++kt)
                    opd.template stats<0>(mx, ls, p.K - kt * BK, [&]() SBX_INLINE { issue_d(z, kt + 1, kNo); });
#pragma unroll
                for (int i = 0; i < OpD::NROW; ++i) {
                    const int x = d0 + OpD::row_of(td, i, w0);
                    atomicMax(row + x, __builtin_bit_cast(unsigned, mx[i]));
                    atomicOr(low + x, ls[i] & kLostBits);
                }
            }
            if (see_s) {
                float mx[OpS::NROW] = {};
                uint32_t ls[OpS::NROW] = {};
                issue_s(z, kt0, kNo);
                for (kt = kt0; kt < nk; ++kt)
                    ops.template stats<0>(mx, ls, p.K - kt * BK, [&]() SBX_INLINE { issue_s(z, kt + 1, kNo); });
#pragma unroll
                for (int i = 0; i < OpS::NROW; ++i) {
                    const int x = s0 + OpS::row_of(td, i, 0);
                    atomicMax(row + x, __builtin_bit_cast(unsigned, mx[i]));
                    atomicOr(low + x, ls[i] & kLostBits);
                }
            }
            __syncthreads();
            const int fails = redo_fails<MF, OpA, OpB, BM>(acc, row, low, (nk - kt0) * BK, wm0, wn0, ln);
            if (redo_needed<MF, OpA, OpB, A_KC, B_KC, NBM>(p, fails, A, B, m0, n0, wm0, wn0, kt0 * BK,
                                                           min(nk * BK, p.K), ln))
                atomicOr(&redo, 8 << look);
            __syncthreads();
            again = (__builtin_amdgcn_readfirstlane(redo) & 8 << look) != 0;
            if (!again) break;
        }
    }
    if (__builtin_expect(again, 0)) fp32_pass();
    store_tile<float, MF, OpA, OpB, BM, BN, WTM, WTN, NBM, NBN>(p, acc, t, m0, n0, wm0, wn0, lane_id(), C);
}

}  // namespace sbx
