// Long kernels (11 to 31 taps) in bf16 on the matrix cores (gfx950, wave64).
//
// On the vector ALU a conv of 31 taps is bound by its FMAs, not by HBM. As a contraction it is four output rows of one
// channel at a time:
//     y[4g + i] = sum over window rows r of A[i][r] * x[4g - FRONT + r],     A[i][r] = w[tap r - i, zero outside the taps]
// (a band of the channel's Toeplitz matrix), four window rows per instruction. v_mfma_f32_4x4x4_16b_bf16 does that for 16
// channels (its 16 blocks) and 4 neighbouring groups of four output rows (the 4 columns of a block) in one instruction:
// lane 4 b + n holds row n (A) or column n (B) of block b, that is channel b's window rows of output rows 4n .. 4n + 3. One
// instruction makes 1024 products of which 31/36 are taps at 31 taps, and issues every 4.5 ns per SIMD, where the same
// products take 14 v_fmac_f32 of 1 ns. Products of bf16 values are exact and the sums are fp32, as on the vector ALU.
//
// Where data crosses lanes: nowhere. A lane reads its Q channels of four window rows out of LDS (8 bytes a row at Q = 4)
// and packs pairs of rows per channel with v_perm_b32 (a 4 x 4 transpose of 16-bit values in registers).
//
// Zeros and non-finite values: the band's zeros multiply rows that are not in an output row's taps, so an Inf or NaN there
// would reach it. Every sum that holds such a product is itself not finite; the kernels test their sums and form those of a pass
// again without the factors that are not finite, then add the products with such factors that belong, one at a time. So sums
// that none of them belongs to keep their bits, whatever shares a pass with them.
//
// Sequence boundaries: one wave of a block leaves for every tile a bit string, one bit per staged row, set where a sequence
// begins. A wave whose window holds no bit runs unmasked; otherwise every lane finds the rows of its four output rows'
// sequences from the bits around them (shifts and bit counts), clears the others with an AND on the packed rows and makes
// one pass per sequence among its four rows.
//
// No counterpart in the reference (peymanvahidi/nanoplm 0.1.6 has no convolution); tensor contract:
// modeling.py:339,421-439 and collator.py:322-325,405-458.
#pragma once
#include "dwconv_lds_split_kernels.h"

namespace nplm {

typedef short s16x4 __attribute__((ext_vector_type(4)));

// The band of KT taps inside the plan of KP = 15 or 31: window row r of output row group g is row 4g - (KP-1)/2 + r. Only
// the 4-row chunks CK0 .. CK0 + NCK - 1 hold taps; they start where those of KP start, so sums group the same products
// whatever KT is.
template <int KT>
struct MfmaTaps {
    static_assert(KT == 11 || KT == 15 || KT == 21 || KT == 31, "built sizes");
    static constexpr int KP = KT <= 15 ? 15 : 31;
    static constexpr int PP = (KP - 1) / 2, P = (KT - 1) / 2;
    static constexpr int CK0 = (PP - P) / 4;
    static constexpr int LAST = PP + 3 + P;                  // last window row with a tap (output row 3, last tap)
    static constexpr int NCK = LAST / 4 - CK0 + 1;
    static constexpr int FRONT = PP - 4 * CK0;               // rows staged in front of a tile's first output row
    static constexpr int LASTROWS = LAST % 4 + 1;            // rows of the last chunk that hold taps
    static constexpr int HALO = 4 * (NCK - 2) + LASTROWS;    // staged rows beyond the tile's own
    static constexpr int WSTR = 2 * NCK + 3;                 // dwords per channel of the weight table (odd: no bank conflicts)
};

constexpr int kMfmaCb = 512;           // bytes of a row in one column block: 256 channels
constexpr int kMfmaCh = kMfmaCb / 2;
constexpr int kMfmaGatedCb = 256;      // gated kernels: 128 channels (three tiles in each of two buffers)
constexpr int kMfmaGatedRows = 64;
constexpr int kMfmaGatedSteps = 16;    // gated forward: steps of 64 rows in a run, at most
constexpr int kMfmaQ = 4;              // channels of a lane: 8 bytes of a row
constexpr int kMfmaFwdRows = 64;       // output rows of a forward tile
// Offset of a store that is to be dropped: beyond the descriptor of a group of output rows (less than 2 GiB) whatever
// the row. A branch around the store instead splits the schedule and costs registers.
constexpr int kMfmaNoStore = (int)0x80000000;
__device__ __forceinline__ rsrc_t mfma_out_rsrc(void* out, int row0, int rows, int rowb) {
    return make_rsrc(reinterpret_cast<char*>(out) + (size_t)row0 * (size_t)rowb, (uint32_t)(rows * rowb));
}
constexpr int kMfmaWords = 8;          // 32-bit words of a tile's boundary bits (lanes read up to 2 words past the last row)

// One chunk (four rows) of a lane's Q channels as matrix operands: per channel rows 0, 1 and rows 2, 3.
// The two bf16 of a dword, zero in the place of one that is not finite.
__device__ __forceinline__ uint32_t non_finite_bf16x2(uint32_t v) { return ((v & 0x7f807f80u) + 0x00800080u) & 0x80008000u; }
__device__ __forceinline__ uint32_t finite_bf16x2(uint32_t v) {
    const uint32_t bad = non_finite_bf16x2(v);                                  // sign bit of each half: its exponent is all ones
    return v & ~((bad << 1) - (bad >> 15));                                     // (the bits spread over their halves)
}
__device__ __forceinline__ u32x2 finite_bf16x4(u32x2 v) { return u32x2{finite_bf16x2(v.x), finite_bf16x2(v.y)}; }

template <int Q = kMfmaQ>
struct MfmaChunk {
    u32x2 b[Q];
    __device__ __forceinline__ s16x4 op(int q) const { return __builtin_bit_cast(s16x4, b[q]); }
    __device__ __forceinline__ void drop_non_finite() {
#pragma unroll
        for (int q = 0; q < Q; ++q) b[q] = finite_bf16x4(b[q]);
    }
};
template <int Q = kMfmaQ> struct MfmaRaw { uint32_t r[4][Q / 2]; };

// (lds_u32x2 loads: one ds_read_b64 per row, rows 512 bytes apart)
typedef const __attribute__((address_space(3))) u32x2* lds_u32x2;
__device__ __forceinline__ u32x2 mfma_lds(uint32_t at) { return *(lds_u32x2)(uintptr_t)at; }
template <int Q>
__device__ __forceinline__ void mfma_pack(const MfmaRaw<Q>& r, MfmaChunk<Q>& c) {
#pragma unroll
    for (int h = 0; h < Q / 2; ++h) {
        c.b[2 * h].x = __builtin_amdgcn_perm(r.r[1][h], r.r[0][h], 0x05040100);
        c.b[2 * h].y = __builtin_amdgcn_perm(r.r[3][h], r.r[2][h], 0x05040100);
        c.b[2 * h + 1].x = __builtin_amdgcn_perm(r.r[1][h], r.r[0][h], 0x07060302);
        c.b[2 * h + 1].y = __builtin_amdgcn_perm(r.r[3][h], r.r[2][h], 0x07060302);
    }
}
__device__ __forceinline__ f32x4 mfma4(s16x4 a, s16x4 b, f32x4 c) { return __builtin_amdgcn_mfma_f32_4x4x4bf16_1k(a, b, c, 0, 0, 0); }

// Staging: rows of a column block of CB = 512 (gated: 256) bytes, two (four) per 1 KiB direct load. The 16-byte pieces of a row are permuted (by the
// lanes' global addresses, inside the row) so that lanes which read four rows at once read different banks: byte b of row
// r lies at b ^ mfma_place(swz(r)). SWZ_ROW: swz = r & 3 (readers at distance 1 row); SWZ_QUAD: (r >> 2) & 3 (distance 4 rows);
// SWZ_BOTH: (r + (r >> 2)) & 3 (distance 4 rows, and at most two on a bank at distance 1).
// place() is linear (place(a ^ b) = place(a) ^ place(b)) and sets 16 lanes that read one slice of 32 bytes of four rows 32 bytes
// apart from one another (modulo 128), 32 lanes that read 64 bytes of each 64 bytes apart (modulo 256): an 8-byte read takes 16 lanes
// at a time. With s << 6 alone rows 0 and 2 met in every such read (LDS conflicts for 0.28 of the cycles, now 0.02).
__host__ __device__ constexpr int mfma_place(int s) { return (s << 6 | s << 4) & 0xe0; }
enum MfmaSwz { SWZ_QUAD = 0, SWZ_ROW = 1, SWZ_BOTH = 2 };
template <MfmaSwz SWZ>
__device__ __forceinline__ int mfma_swz(int row) {
    return (SWZ == SWZ_ROW ? row : SWZ == SWZ_QUAD ? row >> 2 : row + (row >> 2)) & 3;
}
// Every one of the NLW loader waves issues the same number of loads (a surplus one repeats the last rows), so that "all but
// the newest tile's have landed" is a compile-time wait.
template <int NROWS, int NLW, MfmaSwz SWZ, int ONCE_AUX, int CB = kMfmaCb>
__device__ __forceinline__ void mfma_stage(const void* __restrict__ src, char* dst, int first_row, int T, size_t row_bytes,
                                           int col_byte0, int valid_bytes, int lw, int lane, int edge) {
    constexpr int RPL = 1024 / CB, NL = (NROWS + RPL - 1) / RPL, CNT = (NL + NLW - 1) / NLW;
    const int rb = first_row > 0 ? first_row : 0;
    const rsrc_t rs = rows_rsrc(src, rb, T, row_bytes);
    const int rowb = (int)row_bytes;
    const int lrow = lane / (CB / 16), lpiece = lane % (CB / 16);
    // Rows outside [0, T) are not clamped. Those from T on lie outside the descriptor, which ends with the tensor's last row, and land
    // as zeros: GatedDw's sums take them in (dy to db, h and dy to a sequence of their own). The offsets of rows in front of 0
    // fall outside the descriptor too, or, on a tensor beyond 4 GiB, on other rows of it: what lands for them is never used.
#pragma unroll
    for (int i = 0; i < CNT; ++i) {
        const int gi = lw + i * NLW < NL ? lw + i * NLW : NL - 1;
        const int row = RPL * gi + lrow;
        const int piece = lpiece ^ (mfma_place(mfma_swz<SWZ>(row)) >> 4);
        const bool once = gi * RPL >= edge && gi * RPL + RPL <= NROWS - edge;
        if ((NROWS % RPL == 0 || row < NROWS) && piece * 16 < valid_bytes)
            load_to_lds<ONCE_AUX>(rs, dst + gi * 1024, (first_row - rb + row) * rowb + col_byte0 + piece * 16, 0, once);
    }
}

// Boundary bits of the rows [a, a + n): bit p of `words` is set iff a sequence begins at row a + p (0 < p < n); the tensor's
// first and one-past-last row count. One whole wave (walk_starts()).
struct MfmaMarks {
    const int32_t* __restrict__ cu;
    uint32_t* words;
    int a, n, lane;
    __device__ __forceinline__ void mark(int row) const {
        const uint32_t p = (uint32_t)row - (uint32_t)a;      // (unsigned: cu may hold anything)
        if (row > a && p < (uint32_t)n) __hip_atomic_fetch_or(words + (p >> 5), 1u << (p & 31), __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
    }
    __device__ __forceinline__ uint64_t above(uint32_t lo, uint32_t step, uint32_t end, int row) const {
        const uint32_t i = lo + ((uint32_t)lane + 1) * step - 1;
        return __builtin_amdgcn_ballot_w64(cu[i < end ? i : end] > row);
    }
    __device__ __forceinline__ int take(uint32_t lo, uint32_t end, int& first) const {
        const uint32_t i = lo + (uint32_t)lane;
        const int v = cu[i < end ? i : end];
        mark(v);
        first = __builtin_amdgcn_readfirstlane(v);
        return __builtin_amdgcn_readlane(v, 63);
    }
};
template <int NWORDS = kMfmaWords>
__device__ __forceinline__ void mfma_bounds(const int32_t* __restrict__ cu, int S, int T, int a, int n, uint32_t* words, int lane) {
    if (lane < NWORDS) words[lane] = 0;
    MfmaMarks m{cu, words, a, n, lane};
    if (lane == 0) m.mark(0);
    if (lane == 1) m.mark(T);
    walk_starts(m, S, T, a, n);
}

// Boundary bits of a lane's window: bit r is set iff a sequence begins at window row r (r < 64).
struct MfmaBits { uint32_t lo, hi; };
// Rows [lo, hi) of a window that belong to the sequence of window row p < 31; hi may lie up to 21 rows behind p, beyond any
// window. (32-bit operations only, no compares.)
__device__ __forceinline__ void mfma_row_bounds(MfmaBits w, int p, int& lo, int& hi) {
    const uint32_t below = (w.lo & ((2u << p) - 1u)) | 1u;
    const uint32_t above = __builtin_amdgcn_alignbit(w.hi, w.lo, p + 1) | 1u << 20;
    lo = 31 - (int)__builtin_clz(below);
    hi = p + 1 + (int)__builtin_ctz(above);
}
// The rows [lo, hi) as bits (lo < 32, 0 < hi <= 63).
__device__ __forceinline__ MfmaBits mfma_row_mask(int lo, int hi) {
    const int h0 = hi < 32 ? hi : 32, h1 = hi > 32 ? hi - 32 : 0;
    return MfmaBits{(0xffffffffu >> (32 - h0)) & (0xffffffffu << lo), ~(0xffffffffu << h1)};
}

// OR and AND of the four columns' masks, as scalars (the blocks hold the same four).
__device__ __forceinline__ void mfma_columns(MfmaBits v, uint64_t& some, uint64_t& every) {
    some = 0;
    every = ~0ull;
#pragma unroll
    for (int n = 0; n < 4; ++n) {
        const uint64_t c = (uint64_t)(uint32_t)__builtin_amdgcn_readlane((int)v.lo, n) |
                           (uint64_t)(uint32_t)__builtin_amdgcn_readlane((int)v.hi, n) << 32;
        some |= c;
        every &= c;
    }
}

// The caller's weight (bf16) of channel c at tap m of the plan (0 .. KP-1), as the conv takes it (FLIP: the transposed conv of dx).
template <int KP, bool FLIP>
__device__ __forceinline__ float mfma_weight(const void* __restrict__ w, int w_flags, int c, int m, bool res) {
    const int off = w_tap_off(w_flags), kw = KP - 2 * off;
    const int r = (FLIP ? KP - 1 - m : m) - off;
    float v = 0.f;
    if (r >= 0 && r < kw) {
        const uint32_t i = (uint32_t)(c * kw + r) * 2;       // bytes (bf16 weights; C * K is below 2^28)
        v = bf16_to_f32(*reinterpret_cast<const uint16_t*>(reinterpret_cast<const char*>(w) + i));
    }
    return v + (res && m == (KP - 1) / 2 ? 1.f : 0.f);
}

// Gated forward: h is taken kGateUp times as large, weights (and the identity) as much smaller.
constexpr float kGateUp = 65536.f, kGateDown = 1.f / kGateUp;
// kGateUp * u * silu(g), in the steps of gate_mul()
__device__ __forceinline__ float gate_mul_up(float u, float g) {
    return u * g * __builtin_amdgcn_rcpf(__builtin_fmaf(__builtin_amdgcn_exp2f(-1.44269504088896341f * g), kGateDown, kGateDown));
}
// A weight as the gated forward's table holds it
__device__ __forceinline__ uint32_t mfma_weight_down(float w) { return __float_as_uint(w * kGateDown) & 0xffff0000u; }

// Weight table of a column block in LDS, [channel][WSTR] dwords of two bf16: entry e of a channel is plan tap e - 4 + 4 CK0. Behind it
// one word of each of the NW waves that fill it, not zero where it met a weight that is not finite. DOWN: weights for gate_mul_up(), and
// those below 2^-110, which lose bits there, count with the ones that are not finite.
template <int KT, int CH, int NW, bool DOWN = false>
struct MfmaWeights {
    using TP = MfmaTaps<KT>;
    static constexpr int MARKS_AT = CH * TP::WSTR, BYTES = (MARKS_AT + NW) * 4;
    template <bool FLIP>
    __device__ __forceinline__ static void fill(uint32_t* tab, const void* __restrict__ w, int w_flags, int ch0, int nch, int tid) {
        uint32_t odd = 0;
        for (int i = tid; i < CH * TP::WSTR; i += NW * 64) {
            const int c = i / TP::WSTR, p = i - c * TP::WSTR;
            uint32_t t = 0;
            if (c < nch) {
#pragma unroll
                for (int h = 0; h < 2; ++h) {
                    const int m = 2 * p + h - 4 + 4 * TP::CK0;
                    if (m >= 0 && m < TP::KP) {
                        const float v = mfma_weight<TP::KP, FLIP>(w, w_flags, ch0 + c, m, false);
                        t |= ((DOWN ? mfma_weight_down(v) : __float_as_uint(v)) >> 16) << (16 * h);
                        if constexpr (DOWN) odd |= __float_as_uint(v * kGateDown) & 0xffffu;
                    }
                }
            }
            odd |= non_finite_bf16x2(t);
            tab[i] = t;
        }
        const bool any = __builtin_amdgcn_ballot_w64(odd != 0) != 0;
        if ((tid & 63) == 0) tab[MARKS_AT + tid / 64] = any ? 1 : 0;
    }
    // NaN if one of the block's weights is not finite (DOWN: or too small), else 0 (after the barrier that follows fill())
    __device__ __forceinline__ static float odd(const uint32_t* tab) {
        uint32_t any = 0;
#pragma unroll
        for (int i = 0; i < NW; ++i) any |= tab[MARKS_AT + i];
        return __int_as_float(__builtin_amdgcn_readfirstlane((int)(any ? 0x7fc00000u : 0u)));
    }
};

// Ring of chunks (four rows of 128 channels) of h = u * silu(g) in the LDS, as matrix operands: a record holds, per term and channel,
// the four rows' bf16. Records lie 64 bytes off a multiple of 256 apart, so that the four lanes of a block, which read records one
// apart, are on different banks (LDS conflict cycles a call of T=131072, C=2048, 31 taps by that offset: 16 8.6e7, 32 4.2e7, 64 1.1e7,
// which are the stores' ds_bpermute; 397, 379 and 357 us).
// In phase p the producers write records 16 p - PRE on, 16 of them, and the consumers read the window of the step that begins at
// record 16 (p - 2): the two ranges are adjacent and fill the ring.
template <int KT>
struct MfmaRing {
    using TP = MfmaTaps<KT>;
    static constexpr int R = kMfmaGatedRows, CH = kMfmaGatedCb / 2;
    static constexpr int TERM = CH * 8, REC = 3 * TERM + 64;
    static constexpr int NWIN = (R + TP::HALO + 3) / 4, PRE = 2 * (R / 4) - NWIN, LEN = NWIN + R / 4;
    static constexpr int BYTES = LEN * REC;
    static_assert(PRE >= 0, "a run's first window is written in two phases");
    // LDS address of an offset that may lie up to one length behind the ring's end (the ring begins the kernel's LDS)
    __device__ __forceinline__ static uint32_t at(uint32_t x) {
        const uint32_t w = x - BYTES;                        // (huge in front of the end)
        return w < x ? w : x;
    }
    __device__ __forceinline__ static int next(int slot) { return slot + R / 4 < LEN ? slot + R / 4 : slot + R / 4 - LEN; }
};

// One wave's conv over staged rows: 16 Q channels, groups of 16 NSTEP output rows. FLIP: dx from dy. RES: the identity is one
// more band (a single 1 per row), since a bf16 weight plus one is not one in bf16.
// GATED (backward): the rows are dh; what is stored are the two halves of dz = [dh * silu(g) | dh * u * silu'(g)], with u and
// g of the row out of their LDS tiles; 256-byte column blocks.
// LINES: stores with `nt`, for output rows of whole cache lines (see mfma_lines()).
// TERMS = 3 (gated forward): the rows are kGateUp * h in fp32, as three bf16 terms that add up to it, out of a ring of chunks that are
// already packed (MfmaRing); the weights are kGateDown times the caller's.
template <int KT, int NSTEP, bool FLIP, bool RES, bool LINES, bool GATED = false, int TERMS = 1>
struct MfmaConv {
    using TP = MfmaTaps<KT>;
    static constexpr bool RING = TERMS > 1;
    using RG = MfmaRing<KT>;
    static constexpr int Q = GATED || RING ? 2 : kMfmaQ, NCK = TP::NCK, CB = GATED ? kMfmaGatedCb : kMfmaCb;
    static constexpr MfmaSwz SWZ = GATED ? SWZ_BOTH : SWZ_QUAD;
    static constexpr int ROWS = 16 * NSTEP;                  // output rows of a group
    struct Source { const void* z; int row0, T; };           // RING: z [T, 2C] and the row of the group's first output row
    static_assert(ROWS % 32 == 0, "a group's boundary bits start at a word");
    static constexpr int NCHUNK = 4 * (NSTEP - 1) + NCK;     // chunks that the steps of a group read (per lane)
    static constexpr int IDC = (TP::FRONT + 0) / 4;          // chunk of the identity's first row
    static constexpr int IDN = (TP::FRONT + 3) / 4 - IDC + 1;
    struct Chunk {
        MfmaChunk<Q> t[TERMS];
        __device__ __forceinline__ void mask(uint32_t m0, uint32_t m1) {
#pragma unroll
            for (int i = 0; i < TERMS; ++i)
#pragma unroll
                for (int q = 0; q < Q; ++q) { t[i].b[q].x &= m0; t[i].b[q].y &= m1; }
        }
        __device__ __forceinline__ void drop_non_finite() {
#pragma unroll
            for (int i = 0; i < TERMS; ++i) t[i].drop_non_finite();
        }
    };
    using Raw = std::conditional_t<RING, Chunk, MfmaRaw<Q>>;
    // a group's (or step's) first window row: its address in the tile (RING: the offset in the ring of the lane's slice of its chunk,
    // or that plus the ring's length)
    using At = std::conditional_t<RING, uint32_t, const char*>;
    __device__ __forceinline__ static At step_at(At lp, int s) { return lp + (RING ? 4 * s * RG::REC : 16 * s * CB); }
    __device__ __forceinline__ static void pack(const Raw& r, Chunk& c) {
        if constexpr (RING) c = r; else mfma_pack(r, c.t[0]);
    }
    s16x4 A[NCK][Q];
    s16x4 I[RES ? IDN : 1];
    f32x4 bias;            // where the sums start (dx: 0)
    uint32_t slice;        // RING: the lane's slice of chunk n from the ring's start
    int off[4];            // LDS offset of the lane's slice of chunk c, by c & 3 (without c * 4 rows)
    int n;                 // the lane's column: output rows 4 n .. 4 n + 3 of a step
    int c0;                // its first channel
    int swap;              // stores: the lane whose output goes out through this one (x 4)
    int out_at;            // byte offset of that lane's slice of output row 4 n, or kMfmaNoStore
    bool active;
    float odd;             // NaN: a weight of the block is not finite (MfmaWeights::odd), else 0
    const void* w;
    int w_flags;

    __device__ __forceinline__ void init(const uint32_t* tab, float odd_, const void* w_, int w_flags_, const void* b, int wc, int lane, int ch0, int nch, int rowb) {
        odd = odd_;
        n = lane & 3;
        const int blk = lane >> 2;
        const int lc = (wc * 16 + blk) * Q;
        active = lc < nch;
        const int lcc = active ? lc : nch - Q;
        c0 = ch0 + lcc;
        swap = ((lane >> 4) + 4 * (lane & 15)) * 4;
        const int lcs = (wc * 16 + (lane & 15)) * Q;
        out_at = lcs < nch ? 4 * (lane >> 4) * (GATED ? 2 * rowb : rowb) + (ch0 + lcs) * 2 : kMfmaNoStore;
        w = w_;
        w_flags = w_flags_;
#pragma unroll
        for (int k = 0; k < 4; ++k) off[k] = RING ? 0 : 4 * n * CB + ((lcc * 2) ^ mfma_place((n + k) & 3));
        slice = n * RG::REC + lcc * 8;
        const int p0 = (4 - n) >> 1, sh = (n & 1) * 16;
#pragma unroll
        for (int q = 0; q < Q; ++q) {
            const uint32_t* row = tab + (lcc + q) * TP::WSTR + p0;
            uint32_t d = row[0];
#pragma unroll
            for (int k = 0; k < NCK; ++k) {
                const uint32_t d1 = row[2 * k + 1], d2 = row[2 * k + 2];
                const u32x2 v = {__builtin_amdgcn_alignbit(d1, d, sh), __builtin_amdgcn_alignbit(d2, d1, sh)};
                A[k][q] = __builtin_bit_cast(s16x4, v);
                d = d2;
            }
        }
        if constexpr (RES) {
#pragma unroll
            for (int k = 0; k < IDN; ++k)
#pragma unroll
                for (int e = 0; e < 4; ++e) I[k][e] = (4 * (IDC + k) + e == TP::FRONT + n) ? (short)(RING ? 0x3780 : 0x3f80) : (short)0;      // (RING: kGateDown)
        }
#pragma unroll
        for (int q = 0; q < Q; ++q) {
            bias[q] = 0.f;
            if (b) bias[q] = (w_flags & W_BF16) ? bf16_to_f32(reinterpret_cast<const uint16_t*>(b)[c0 + q]) : reinterpret_cast<const float*>(b)[c0 + q];
        }
        // here and not at every step, where stores are under way (T=131072, C=1024, 11 taps, 24 rows a sequence: 110 us there, 99)
        if constexpr (!FLIP) wait_vmem_all();
    }

    __device__ __forceinline__ f32x4 start(int q) const {
        if constexpr (FLIP) return f32x4{0.f, 0.f, 0.f, 0.f};
        float b = bias[q];
        asm volatile("" : "+v"(b));                          // (else four copies of it stay in registers)
        return f32x4{b, b, b, b};
    }
    // acc += the products of window chunk k (FINITE: without the weights that are not finite)
    // (term and channel i of the TERMS * Q alone)
    template <int k, bool FINITE = false>
    __device__ __forceinline__ void tap(f32x4 (&acc)[Q], const Chunk& x, int i) const {
        const int q = i % Q;
        s16x4 w4 = A[k][q];
        if constexpr (FINITE) {
            u32x2 t = __builtin_bit_cast(u32x2, w4);
            asm volatile("" : "+v"(t.x), "+v"(t.y));         // (not formed ahead of the steps and kept in registers)
            w4 = __builtin_bit_cast(s16x4, finite_bf16x4(t));
        }
        acc[q] = mfma4(w4, x.t[i / Q].op(q), acc[q]);
        if constexpr (RES && k >= IDC && k < IDC + IDN) acc[q] = mfma4(I[k - IDC], x.t[i / Q].op(q), acc[q]);
    }
    template <int k, bool FINITE = false>
    __device__ __forceinline__ void taps(f32x4 (&acc)[Q], const Chunk& x) const {
#pragma unroll
        for (int i = TERMS * Q - 1; i >= 0; --i) tap<k, FINITE>(acc, x, i);      // (the smaller terms first)
    }
    // window chunk c of the lane, its first ROWS rows
    template <int c, int ROWS = 4>
    __device__ __forceinline__ void read(At lp, Raw& o) const {
        if constexpr (RING) {
            const uint32_t at = RG::at(lp + c * RG::REC);
#pragma unroll
            for (int i = 0; i < TERMS; ++i) {
                const u32x4 v = *(const __attribute__((address_space(3))) u32x4*)(uintptr_t)(at + i * RG::TERM);
                o.t[i].b[0] = u32x2{v.x, v.y};
                o.t[i].b[1] = u32x2{v.z, v.w};
            }
            if constexpr (ROWS < 4) o.mask(ROWS == 1 ? 0xffffu : ~0u, ROWS == 3 ? 0xffffu : 0u);
            return;
        } else {
#pragma unroll
        for (int r = 0; r < 4; ++r) {
            if (r < ROWS) {
                RowVec<true, Q> t;
                t.load(lp + off[(c + (SWZ == SWZ_BOTH ? r : 0)) & 3] + (c * 4 + r) * CB);
#pragma unroll
                for (int h = 0; h < Q / 2; ++h) o.r[r][h] = t.d[h];
            } else {
#pragma unroll
                for (int h = 0; h < Q / 2; ++h) o.r[r][h] = 0;
            }
        }
        }
    }
    // Adjacent lanes of a sum are rows 0, 4, 8, 12; they trade places first, so that 16 adjacent lanes store the 32 Q bytes
    // of one row (as 4-row pieces of 8 bytes the memory pipeline takes four times the requests: T=131072, C=2048, 31 taps
    // 223 us against 200).
    __device__ __forceinline__ void store_at(rsrc_t ro, int at, int soff, const float (&v)[Q]) const {
        RowVec<true, Q> o;
        o.from_f32(v);
#pragma unroll
        for (int h = 0; h < Q / 2; ++h) o.d[h] = (uint32_t)__builtin_amdgcn_ds_bpermute(swap, (int)o.d[h]);
        constexpr int aux = LINES ? kStoreAux : 0;
        if constexpr (Q == 4) __builtin_amdgcn_raw_buffer_store_b64(u32x2{o.d[0], o.d[1]}, ro, at, soff, aux);
        else __builtin_amdgcn_raw_buffer_store_b32(o.d[0], ro, at, soff, aux);
    }
    // output row 4 n + row of the group; up = the group's first row in the u tile
    __device__ __forceinline__ void store(rsrc_t ro, int at, int rowb, const char* up, int row, const float (&v)[Q]) const {
        if constexpr (GATED) {
            float u[Q], g[Q], du[Q], dg[Q];
            RowVec<true, Q> ru, rg;
            ru.load(up + off[0] + row * CB);
            rg.load(up + off[0] + (row + kMfmaGatedRows) * CB);
            ru.to_f32(u);
            rg.to_f32(g);
#pragma unroll
            for (int q = 0; q < Q; ++q) {
                const float sg = sigmoid_f32(g[q]);
                du[q] = v[q] * (g[q] * sg);
                dg[q] = v[q] * (u[q] * sg * (1.f + g[q] * (1.f - sg)));
            }
            store_at(ro, at, row * 2 * rowb, du);
            store_at(ro, at, row * 2 * rowb + rowb, dg);
        } else {
            store_at(ro, at, row * rowb, v);
        }
    }

    // boundary bits of this lane's window in step s (rows 16 s + 4 n on) of a group whose bits start at wp
    __device__ __forceinline__ MfmaBits window_bits(const uint32_t* wp, int s) const {
        const int at = 16 * s + 4 * n;
        const uint32_t* d = wp + (at >> 5);
        const uint32_t d0 = d[0], d1 = d[1], d2 = d[2];
        return MfmaBits{__builtin_amdgcn_alignbit(d1, d0, at & 31), __builtin_amdgcn_alignbit(d2, d1, at & 31)};
    }

    // Boundaries among a group's window rows, read by the wave as scalars. wp: its boundary bits (bit 0 is no boundary).
    static constexpr int SPAN = 16 * NSTEP + TP::HALO;       // window rows of the group
    // Up to 15 taps a step's passes have too few chunks to leave out. With three sequences the plain kernels' steps are as fast as three
    // sweeps and faster where sequences are short (T=131072, C=2048, 16 rows a sequence, none / two / three swept: 21 taps 289 / 287 / 307 us, 31 taps
    // 326 / 328 / 340; 32 rows 253 / 243 / 244 and 289 / 268 / 266); the gated ones gain (forward of 31 taps, T=16384, C=1024, 24 rows, two / three: 55 / 50,
    // backward, C=2048, 48 rows 127 / 124).
    static constexpr int kFewSequences = NCK < 7 ? 0 : GATED || RING ? 3 : 2;
    // whether at most kFewSequences sequences own rows of the group
    __device__ __forceinline__ static bool few_sequences(const uint32_t* wp) {
        int n = 1;
        if constexpr (GATED || RING) {                       // (short sequences, 4 rows: gated forward 54.5 and 53.2 us, T=16384, C=1024)
            constexpr int A = TP::FRONT + 1;                 // rows FRONT + 1 .. FRONT + ROWS - 1
#pragma unroll
            for (int i = 0; i < ROWS; i += 32) {
                const uint32_t w = __builtin_amdgcn_alignbit(wp[(A + i) / 32 + 1], wp[(A + i) / 32], (A + i) & 31);
                n += __builtin_popcount((uint32_t)__builtin_amdgcn_readfirstlane((int)(i + 32 < ROWS ? w : w & 0x7fffffffu)));
            }
        } else {                                             // (plain forward of 21 taps, 75 rows, T=131072, C=2048: that way 211, this one 209)
#pragma unroll
            for (int i = 0; i * 32 < TP::FRONT + ROWS; ++i) {    // rows FRONT + 1 .. FRONT + ROWS - 1
                constexpr int A = TP::FRONT + 1, B = TP::FRONT + ROWS;
                const uint32_t from = A > 32 * i ? (A - 32 * i < 32 ? ~0u << (A & 31) : 0u) : ~0u;
                const uint32_t to = B < 32 * i + 32 ? (1u << (B & 31)) - 1u : ~0u;
                n += __builtin_popcount((uint32_t)__builtin_amdgcn_readfirstlane((int)(wp[i] & from & to)));
            }
        }
        return n <= kFewSequences;
    }
    // first window row of the sequence that holds row `at` (0: it began before), at < 32
    __device__ __forceinline__ static int start_of(const uint32_t* wp, int at) {
        const uint32_t w = (uint32_t)__builtin_amdgcn_readfirstlane((int)wp[0]);
        return 31 - (int)__builtin_clz((w & ((2u << at) - 1u)) | 1u);
    }
    // first window row behind row `at` where a sequence begins (SPAN: none)
    __device__ __forceinline__ static int start_behind(const uint32_t* wp, int at) {
        int r = SPAN;
#pragma unroll
        for (int i = (SPAN + 31) / 32 - 1; i >= 0; --i) {
            const int sh = at + 1 - 32 * i;                  // bits from here on lie behind `at`
            uint32_t w = (uint32_t)__builtin_amdgcn_readfirstlane((int)wp[i]);
            w = sh <= 0 ? w : sh < 32 ? w & (~0u << sh) : 0u;
            if (w) r = 32 * i + (int)__builtin_ctz(w);
        }
        return r < SPAN ? r : SPAN;
    }
    // Packed masks of a lane's window rows 4 (c + n) .. + 3 against [lo, hi) (uniform).
    __device__ __forceinline__ void chunk_masks(int c, int lo, int hi, uint32_t& m0, uint32_t& m1) const {
        const int o = lo > 4 * c ? lo - 4 * c : 0, e = hi - 4 * c < 16 ? hi - 4 * c : 16;      // (o < 16, e > 0: some rows are in)
        const uint32_t v = (((1u << e) - 1u) & (~0u << o)) >> (4 * n);
        m0 = __builtin_amdgcn_perm((uint32_t)((int)(v << 30) >> 31), (uint32_t)((int)(v << 31) >> 31), 0x05040100);
        m1 = __builtin_amdgcn_perm((uint32_t)((int)(v << 28) >> 31), (uint32_t)((int)(v << 29) >> 31), 0x05040100);
    }
    // The group's output rows, chunk after chunk of its window, each chunk for all the steps it belongs to. PART: only the rows of one
    // sequence, window rows [lo, hi): chunks without any of its rows are left out, those at its ends masked, rows outside it not
    // stored. Returns whether all sums are finite (those that are not have to be formed again).
    template <bool PART>
    __device__ __forceinline__ bool sweep(At lp, int lo, int hi, rsrc_t ro, int rowb, const char* up) const {
        float chk = PART || RING ? odd : 0.f;
        f32x4 acc[(NCK + 3) / 4][Q];
        Raw raw;
        read<0>(lp, raw);
        int range = 0;                                       // output rows [o, e) of the group, relative to the storing lane's first
        if constexpr (PART) range = __builtin_amdgcn_ds_bpermute(swap, 4 * n);
        static_for<NCHUNK>([&](auto c_c) __attribute__((always_inline)) {
            constexpr int c = decltype(c_c)::value;
            const Raw cur = raw;
            if constexpr (c + 1 < NCHUNK)
                read<c + 1, (c + 1 == NCHUNK - 1 ? TP::LASTROWS : 4)>(lp, raw);
            static_for<NSTEP>([&](auto s_c) __attribute__((always_inline)) {
                constexpr int s = decltype(s_c)::value;
                if constexpr (c == 4 * s) {
#pragma unroll
                    for (int q = 0; q < Q; ++q) acc[s % ((NCK + 3) / 4)][q] = start(q);
                }
            });
            if (!PART || (4 * c < hi && 4 * c + 16 > lo)) {
                Chunk x;
                pack(cur, x);
                if (PART && (4 * c < lo || 4 * c + 16 > hi)) {
                    uint32_t m0, m1;
                    chunk_masks(c, lo, hi, m0, m1);
                    x.mask(m0, m1);
                }
                // (the sums of all steps by turns: a product waits for the one before it in its sum)
#pragma unroll
                for (int i = TERMS * Q - 1; i >= 0; --i)
                    static_for<NSTEP>([&](auto s_c) __attribute__((always_inline)) {
                        constexpr int s = decltype(s_c)::value;
                        constexpr int k = c - 4 * s;
                        if constexpr (k >= 0 && k < NCK) tap<k>(acc[s % ((NCK + 3) / 4)], x, i);
                    });
            }
            static_for<NSTEP>([&](auto s_c) __attribute__((always_inline)) {
                constexpr int s = decltype(s_c)::value;
                if constexpr (c - 4 * s == NCK - 1) {
                    const f32x4 (&a)[Q] = acc[s % ((NCK + 3) / 4)];
                    if (!PART || (lo < TP::FRONT + 16 * s + 16 && hi > TP::FRONT + 16 * s)) {
#pragma unroll
                        for (int q = 0; q < Q; ++q) chk = __builtin_fmaf(a[q][0], 0.f, chk);
#pragma unroll
                        for (int i = 0; i < 4; ++i) {
                            float v[Q];
#pragma unroll
                            for (int q = 0; q < Q; ++q) v[q] = a[q][i];
                            int at = out_at;
                            if constexpr (PART) {
                                const int r = TP::FRONT + 16 * s + i + range;
                                at = r >= lo && r < hi ? out_at : kMfmaNoStore;
                            }
                            store(ro, at, rowb, up, 16 * s + i, v);
                        }
                    }
                }
            });
            __builtin_amdgcn_sched_barrier(0);
        });
        return __builtin_amdgcn_ballot_w64(active && !__builtin_isfinite(chk)) == 0;
    }

    // One group of output rows: lp = the group's first window row in LDS, words = the tile's boundary bits, p0 = the window row's
    // place among them; ro = descriptor of the group's output rows (those in front of T).
    // GATED: up = the group's first row in the u tile; the g tile lies kMfmaGatedRows rows behind it. RING: src = where h comes from.
    __device__ __forceinline__ void rows(At lp, const uint32_t* words, int p0, rsrc_t ro, int rowb, const char* up = nullptr,
                                         const Source& src = Source{}) const {
        const uint32_t* wp = words + (p0 >> 5);              // p0 is a multiple of 32
        bool open;                                           // no boundary inside the window (a bit at its first row is none)
        {
            uint32_t any = 0;
#pragma unroll
            for (int i = 0; i * 32 < SPAN; ++i) any |= wp[i] & (i == 0 ? ~1u : SPAN - i * 32 >= 32 ? ~0u : (1u << (SPAN & 31)) - 1u);
            open = __builtin_amdgcn_readfirstlane((int)any) == 0;
        }
        if (open) {
            if (sweep<false>(lp, 0, SPAN, ro, rowb, up)) return;
        } else if (kFewSequences > 0 && few_sequences(wp)) {
            // One sweep per sequence that owns rows of the group.
            int lo = start_of(wp, TP::FRONT);
            bool done = true;
            do {
                const int hi = start_behind(wp, lo > TP::FRONT ? lo : TP::FRONT);
                done = sweep<true>(lp, lo, hi, ro, rowb, up) && done;
                lo = hi;
            } while (lo < TP::FRONT + ROWS);
            if (done) return;
        }
#pragma nounroll
        for (int s = 0; s < NSTEP; ++s) {
            const MfmaBits bits = window_bits(wp, s);
            const At sp = step_at(lp, s);
            int i0 = 0;
            do {
                int lo, hi;
                mfma_row_bounds(bits, TP::FRONT + (i0 < 4 ? i0 : 3), lo, hi);
                f32x4 acc[Q];
                pass<false>(sp, lo, hi, acc);
                const int i1 = hi - TP::FRONT < 4 ? hi - TP::FRONT : 4;
                // (a row that is not finite meets all four sums; a weight meets each in another chunk, and chunks are left out here)
                float chk = odd;
#pragma unroll
                for (int q = 0; q < Q; ++q) chk = __builtin_fmaf(acc[q][0], 0.f, chk);
                if (__builtin_expect(__builtin_amdgcn_ballot_w64(active && !__builtin_isfinite(chk)) != 0, 0)) {
                    pass<true>(sp, lo, hi, acc);
                    const int range = __builtin_amdgcn_ds_bpermute(swap, i0 | i1 << 8);
#pragma nounroll
                    for (int i = 0; i < 4; ++i) {
                        float v[Q];
#pragma unroll
                        for (int q = 0; q < Q; ++q) v[q] = i < 2 ? (i == 0 ? acc[q][0] : acc[q][1]) : i == 2 ? acc[q][2] : acc[q][3];
                        if constexpr (RING) add_apart(src, rowb, 16 * s + i, i, lo, hi, v);
                        else add_non_finite(sp, i, lo, hi, v);
                        store(ro, i >= (range & 255) && i < (range >> 8) ? out_at : kMfmaNoStore, rowb, up, 16 * s + i, v);
                    }
                } else {
                    const int range = __builtin_amdgcn_ds_bpermute(swap, i0 | i1 << 8);     // rows of the pass in the lane that stores them
#pragma unroll
                    for (int i = 0; i < 4; ++i) {
                        float v[Q];
#pragma unroll
                        for (int q = 0; q < Q; ++q) v[q] = acc[q][i];
                        store(ro, i >= (range & 255) && i < (range >> 8) ? out_at : kMfmaNoStore, rowb, up, 16 * s + i, v);
                    }
                }
                i0 = i0 < 4 ? i1 : 4;
            } while (__builtin_amdgcn_ballot_w64(i0 < 4) != 0);
        }
    }

    // The sums of a step (sp: its first window row) over the window rows [lo, hi) alone. FINITE: products of finite factors alone.
    template <bool FINITE>
    __device__ __forceinline__ void pass(At sp, int lo, int hi, f32x4 (&acc)[Q]) const {
        const MfmaBits in = mfma_row_mask(lo, hi);
        // window rows that some lane's pass takes, and those that every lane's takes (lanes of a column hold the same):
        // a chunk that none takes is skipped, one that all take whole needs no mask
        uint64_t some, every;
        mfma_columns(in, some, every);
#pragma unroll
        for (int q = 0; q < Q; ++q) acc[q] = start(q);
        Raw raw;
        if constexpr (!FINITE) {
            read<0>(sp, raw);
            asm volatile("" ::: "memory");                   // (else the reads move into the first chunk's branch, in front of their use)
        }
        static_for<NCK>([&](auto k_c) __attribute__((always_inline)) {
            constexpr int k = decltype(k_c)::value;
            if constexpr (FINITE) read<k, (k == NCK - 1 ? TP::LASTROWS : 4)>(sp, raw);      // (rarely run: few registers)
            const Raw cur = raw;
            if constexpr (!FINITE && k + 1 < NCK)
                read<k + 1, (k + 1 == NCK - 1 ? TP::LASTROWS : 4)>(sp, raw);
            if ((some >> (4 * k)) & 15) {
                Chunk x;
                pack(cur, x);
                if (((every >> (4 * k)) & 15) != 15) {
                    const uint32_t b4 = 4 * k < 32 ? in.lo >> (4 * k & 31) : in.hi >> (4 * k & 31);
                    const uint32_t m0 = __builtin_amdgcn_perm((uint32_t)((int)(b4 << 30) >> 31), (uint32_t)((int)(b4 << 31) >> 31), 0x05040100);
                    const uint32_t m1 = __builtin_amdgcn_perm((uint32_t)((int)(b4 << 28) >> 31), (uint32_t)((int)(b4 << 29) >> 31), 0x05040100);
                    x.mask(m0, m1);
                }
                if constexpr (FINITE) x.drop_non_finite();
                taps<k, FINITE>(acc, x);
            }
            __builtin_amdgcn_sched_barrier(0);
        });
    }
    // v += the products of output row 4 n + i of the step that are in its pass's window rows [lo, hi) and have a factor that is not finite
    __device__ __forceinline__ void add_non_finite(At sp, int i, int lo, int hi, float (&v)[Q]) const {
        const int koff = w_tap_off(w_flags), kw = TP::KP - 2 * koff;
        const bool res = (w_flags & W_RESIDUAL) != 0;
#pragma nounroll
        for (int m = koff; m < koff + kw; ++m) {
            const int p = TP::FRONT + i - TP::PP + m;           // window row of tap m
            if (p < lo || p >= hi || !active) continue;
            // (the lane's row 4 n + p of the step: its piece is where the chunk of that row has it)
            float f[Q];
            const char* a = sp + (off[0] ^ mfma_place((((p >> 2) + (SWZ == SWZ_BOTH ? p : 0) + n) & 3) ^ n)) + p * CB;
            RowVec<true, Q> x;
            x.load(a);
            x.to_f32(f);
#pragma unroll
            for (int q = 0; q < Q; ++q) {
                const float wq = mfma_weight<TP::KP, FLIP>(w, w_flags, c0 + q, m, res);
                if (!__builtin_isfinite(f[q]) || !__builtin_isfinite(wq)) v[q] = __builtin_fmaf(wq, f[q], v[q]);
            }
        }
    }
    // The same for the gated forward, h once more from z: products that the finite terms and weights lack are those with a kGateUp * h or a
    // weight that is not finite and, of weights too small for the table, what it holds too little. (row: output row 4 n + row of the group)
    __device__ __forceinline__ void add_apart(const Source& src, int rowb, int row, int i, int lo, int hi, float (&v)[Q]) const {
        const int koff = w_tap_off(w_flags), kw = TP::KP - 2 * koff;
        const bool res = (w_flags & W_RESIDUAL) != 0;
#pragma nounroll
        for (int m = koff; m < koff + kw; ++m) {
            const int p = TP::FRONT + i - TP::PP + m;           // window row of tap m
            const int t = src.row0 + 4 * n + row + m - TP::PP;  // its row of z
            if (p < lo || p >= hi || !active || t < 0 || t >= src.T) continue;
            const char* a = reinterpret_cast<const char*>(src.z) + (size_t)t * 2 * (size_t)rowb + (size_t)c0 * 2;
            const uint32_t u = *reinterpret_cast<const uint32_t*>(a), g = *reinterpret_cast<const uint32_t*>(a + rowb);
#pragma unroll
            for (int q = 0; q < Q; ++q) {
                const float uq = q == 0 ? bf16_lo(u) : bf16_hi(u), gq = q == 0 ? bf16_lo(g) : bf16_hi(g), h = gate_mul(uq, gq);
                const float wq = mfma_weight<TP::KP, FLIP>(w, w_flags, c0 + q, m, false);
                if (!__builtin_isfinite(gate_mul_up(uq, gq)) || !__builtin_isfinite(wq))
                    v[q] = __builtin_fmaf(wq + (res && m == TP::PP ? 1.f : 0.f), h, v[q]);
                else
                    v[q] = __builtin_fmaf(wq - __uint_as_float(mfma_weight_down(wq)) * kGateUp, h, v[q]);
            }
        }
    }
};

// Forward: 64-row tiles, 8 compute waves (4 wave-columns x 2 groups of 32 rows), 3 loader waves and one that finds the
// boundaries of the next tile; two tile buffers.
// Bound by HBM from 64 row tiles on: T=131072, C=2048, 31 taps, one sequence 182 us (5.9 TB/s), 248 on the vector ALU; log-normal
// lengths 189 (216 with neither the sweeps over single sequences nor rows 32 bytes apart). More rows
// per tile, three buffers or 1 KiB column blocks measured the same or slower (a tile's compute already hides the next one's
// loads); one scout wave costs nothing that the loaders would use.
template <int KT>
struct MfmaFwdShape {
    using TP = MfmaTaps<KT>;
    static constexpr int NCW = kMfmaCh / (16 * kMfmaQ), NWC = 8, NRG = NWC / NCW, NWL = 3;
    static constexpr int NT = (NWC + NWL + 1) * 64;
    static constexpr int R = kMfmaFwdRows, RW = R / NRG, NROWS = R + TP::HALO;
    static constexpr int BUF_BYTES = NROWS * kMfmaCb;
    static constexpr int TAB_AT = 2 * BUF_BYTES + 2 * kMfmaWords * 4;      // two tiles, their boundary bits, the weight table
    using W = MfmaWeights<KT, kMfmaCh, NWC>;
    static constexpr int LDS_BYTES = TAB_AT + W::BYTES;
    static_assert(LDS_BYTES <= kLdsBytes, "fits the LDS");
    static_assert((NROWS + 31) / 32 + 2 <= kMfmaWords, "lanes read two words past the one of their window's first row");
};

template <int KT, bool RES, bool LINES>
__global__ void __launch_bounds__(MfmaFwdShape<KT>::NT)
dwconv_fwd_mfma_kernel(const void* __restrict__ x, const int32_t* __restrict__ cu, const void* __restrict__ w,
                       const void* __restrict__ bias, void* __restrict__ y, const LdsGeo g) {
    using SH = MfmaFwdShape<KT>;
    using TP = MfmaTaps<KT>;
    constexpr int R = SH::R;
    extern __shared__ __attribute__((aligned(16))) char lds_raw[];
    uint32_t* words = reinterpret_cast<uint32_t*>(lds_raw + 2 * SH::BUF_BYTES);
    uint32_t* tab = reinterpret_cast<uint32_t*>(lds_raw + SH::TAB_AT);
    const int lane = (int)(threadIdx.x & 63);
    const int wv = wave_id();
    int cb, tb;
    lds_block_coords(g, cb, tb);
    const int T = g.T, S = g.S, C = g.C;
    const int rowb = C * 2;
    const int col_byte0 = cb * kMfmaCb;
    const int valid_bytes = rowb - col_byte0 < kMfmaCb ? rowb - col_byte0 : kMfmaCb;
    const int ntl = (g.ntiles + g.nbt - 1) / g.nbt;
    int q = tb;

    if (wv >= SH::NWC) {
        // they go ahead of the compute waves of their SIMD: the loads of the next tile leave as soon as the tiles change
        // (31 taps, T=131072, C=2048, one sequence: 195 us without, 183 with)
        __builtin_amdgcn_s_setprio(3);
        const int lw = wv - SH::NWC;
        auto prepare = [&](int par, int t0) __attribute__((always_inline)) {
            if (lw < SH::NWL) {
                mfma_stage<SH::NROWS, SH::NWL, SWZ_QUAD, kLoadAuxOnceFwd>(x, lds_raw + par * SH::BUF_BYTES, t0 - TP::FRONT, T, (size_t)rowb,
                                                                       col_byte0, valid_bytes, lw, lane, TP::HALO);
            } else {
                mfma_bounds(cu, S, T, t0 - TP::FRONT, SH::NROWS, words + par * kMfmaWords, lane);
            }
        };
        prepare(0, tb * R);
        lds_barrier();                       // the weight table is written
        for (int it = 0; it < ntl; ++it) {
            if (lw < SH::NWL) wait_vmem_all();
            lds_barrier();                   // tile `it` has landed, the buffer of the tile before is free
            q = lds_next_slot(g, q);
            const int t0 = it + 1 < ntl ? lds_tile_row0(g, it + 1, q, R) : T;
            if (t0 < T) prepare((it + 1) & 1, t0);
        }
        return;
    }
    const int wc = wv % SH::NCW, r0 = wv / SH::NCW * SH::RW;
    const int nch = valid_bytes / 2;
    SH::W::template fill<false>(tab, w, g.w_flags, cb * kMfmaCh, nch, (int)threadIdx.x);
    lds_barrier();
    MfmaConv<KT, SH::RW / 16, false, RES, LINES> conv;
    conv.init(tab, SH::W::odd(tab), w, g.w_flags, bias, wc, lane, cb * kMfmaCh, nch, rowb);
    for (int it = 0; it < ntl; ++it) {
        lds_barrier();
        const int tf = lds_tile_row0(g, it, q, R) + r0;
        if (tf < T)
            conv.rows(lds_raw + (it & 1) * SH::BUF_BYTES + r0 * kMfmaCb, words + (it & 1) * kMfmaWords, r0,
                      mfma_out_rsrc(y, tf, T - tf < SH::RW ? T - tf : SH::RW, rowb), rowb);
        q = lds_next_slot(g, q);
    }
}

// ---- backward --------------------------------------------------------------------------------------------------------
// dw of a plan tap m sums x[t] * dy[t - (KP-1)/2 + m] over the rows t of one sequence. As a contraction over rows:
//     D[i][j] += sum over k of x[4c + k - i] * dy_staged[4(c + d + j) + k],  d = 0, 4:  the lag is m = 4 CK0 + 4d + 4j + i
// so the four lanes of a block hold x at distance one row and dy at distance four rows, and 32 taps (16 at KP = 15) of 16
// channels take two instructions (one) per four rows. db is the product of dy's chunks with ones. A tile's sums are formed
// from zero and join the block's when they are finite; otherwise the tile is summed again without the values that are not, and the
// products with those are added one at a time (sums that none of them belongs to keep their bits).
template <int KT>
struct MfmaDw {
    using TP = MfmaTaps<KT>;
    static constexpr int Q = kMfmaQ, R = 64;
    static constexpr int ND = TP::KP == 15 ? 1 : 2;          // groups of 16 lags
    static constexpr int NCX = R / 4 + 1;                    // x chunks: a lane's rows are shifted by up to 3
    static constexpr int ROWB = kMfmaCb, SPAN = R + TP::HALO; // (staged rows)
    f32x4 tot[ND][Q];
    float dbs[Q];              // the lane's share of db
    uint32_t ady[4], ax[4];    // LDS addresses of the lane's slice: of dy chunk c by c & 3, of row k of an x chunk (chunk 0, the tile at hand)
    int n, c0;
    bool active;

    __device__ __forceinline__ void init(const char* lds, int wc, int lane, int ch0, int nch, int x_at) {
        n = lane & 3;
        const int lc = (wc * 16 + (lane >> 2)) * Q;
        active = lc < nch;
        const int lcc = active ? lc : nch - Q;
        c0 = ch0 + lcc;
#pragma unroll
        for (int k = 0; k < 4; ++k) {
            const uint32_t base = (uint32_t)(uintptr_t)(const __attribute__((address_space(3))) char*)lds;
            ady[k] = base + 4 * n * ROWB + ((lcc * 2) ^ mfma_place((n + k) & 3));
            ax[k] = base + x_at + (k - n) * ROWB + ((lcc * 2) ^ mfma_place((k - n) & 3));
        }
#pragma unroll
        for (int q = 0; q < Q; ++q) {
            dbs[q] = 0.f;
#pragma unroll
            for (int d = 0; d < ND; ++d) tot[d][q] = f32x4{0.f, 0.f, 0.f, 0.f};
        }
    }
    __device__ __forceinline__ void read_x(int chunk, MfmaRaw<Q>& o) const {
#pragma unroll
        for (int k = 0; k < 4; ++k) {
            const u32x2 t = mfma_lds(ax[k] + chunk * 4 * ROWB);
            o.r[k][0] = t.x; o.r[k][1] = t.y;
        }
    }
    __device__ __forceinline__ void read_dy(int chunk, MfmaRaw<Q>& o) const {
#pragma unroll
        for (int k = 0; k < 4; ++k) {
            const u32x2 t = mfma_lds(ady[chunk & 3] + (chunk * 4 + k) * ROWB);
            o.r[k][0] = t.x; o.r[k][1] = t.y;
        }
    }
    __device__ __forceinline__ void next_buffer(int by) {
#pragma unroll
        for (int k = 0; k < 4; ++k) { ady[k] += by; ax[k] += by; }
    }
    // Packed masks of a lane's rows r0 + at .. r0 + at + 3 against [lo, hi); r0, lo, hi are uniform, at + 4 <= 16.
    __device__ __forceinline__ static void row_masks(int r0, int at, int lo, int hi, uint32_t& m0, uint32_t& m1) {
        const int o = lo > r0 ? lo - r0 : 0, e = hi - r0 < 16 ? hi - r0 : 16;
        uint32_t in = (uint32_t)__builtin_amdgcn_readfirstlane((int)(e > o ? ((1u << e) - 1u) & ~((1u << o) - 1u) : 0u));
        asm volatile("" : "+s"(in));                         // (not computed ahead of the tiles and kept in registers)
        const uint32_t v = in >> at;
        m0 = __builtin_amdgcn_perm((uint32_t)((int)(v << 30) >> 31), (uint32_t)((int)(v << 31) >> 31), 0x05040100);
        m1 = __builtin_amdgcn_perm((uint32_t)((int)(v << 28) >> 31), (uint32_t)((int)(v << 29) >> 31), 0x05040100);
    }
    __device__ __forceinline__ static void mask(MfmaChunk<Q>& c, uint32_t m0, uint32_t m1) {
#pragma unroll
        for (int q = 0; q < Q; ++q) { c.b[q].x &= m0; c.b[q].y &= m1; }
    }
    __device__ __forceinline__ void add_db(const MfmaChunk<Q>& dy) {
        const s16x4 one = {(short)0x3f80, (short)0x3f80, (short)0x3f80, (short)0x3f80};
#pragma unroll
        for (int q = 0; q < Q; ++q) {
            dbs[q] += mfma4(one, dy.op(q), f32x4{0.f, 0.f, 0.f, 0.f})[0];
            asm volatile("" : "+v"(dbs[q]));                 // one product's registers at a time
        }
    }

    // acc += the sums of a tile with boundaries: one pass per sequence that owns rows of the tile, over the chunks that hold them; the
    // next chunk is on its way while one is summed. FINITE: products of finite factors alone.
    template <bool FINITE>
    __device__ __forceinline__ void passes(uint64_t w0, uint64_t w1, int nrow, f32x4 (&acc)[ND][Q]) const {
        const uint32_t col = ady[0] ^ mfma_place(n);              // the lane's address of dy chunk 0 without the permutation of its rows
        uint32_t m0, m1;
        int a = sequence_of(w0, w1, TP::FRONT);
        while (a < TP::FRONT + nrow) {
            int b = next_sequence(w0, w1, a);
            if (b > SPAN) b = SPAN;                          // (staged rows end there)
            const int t0 = a > TP::FRONT ? a - TP::FRONT : 0, t1 = b - TP::FRONT < nrow ? b - TP::FRONT : nrow;
            const int c1 = (t1 + 2) >> 2;
            MfmaRaw<Q> rx, rd[ND];
            auto fetch = [&](int c) __attribute__((always_inline)) {
                const uint32_t at = (col + 4 * c * ROWB) ^ mfma_place((n + c) & 3);
#pragma unroll
                for (int k = 0; k < 4; ++k) {
                    u32x2 t = mfma_lds(ax[k] + c * 4 * ROWB);
                    rx.r[k][0] = t.x; rx.r[k][1] = t.y;
#pragma unroll
                    for (int d = 0; d < ND; ++d) {
                        t = mfma_lds(at + (16 * d + k) * ROWB);
                        rd[d].r[k][0] = t.x; rd[d].r[k][1] = t.y;
                    }
                }
            };
            int c = t0 >> 2;
            fetch(c);
#pragma nounroll
            for (; c <= c1; ++c) {
                MfmaChunk<Q> x, dy[ND];
                mfma_pack(rx, x);
#pragma unroll
                for (int d = 0; d < ND; ++d) mfma_pack(rd[d], dy[d]);
                fetch(c < c1 ? c + 1 : c);
                if (4 * c - 3 < t0 || 4 * c + 3 >= t1) {
                    row_masks(4 * c - 3, 3 - n, t0, t1, m0, m1);
                    mask(x, m0, m1);
                }
                if constexpr (FINITE) x.drop_non_finite();
#pragma unroll
                for (int d = 0; d < ND; ++d) {
                    const int r0 = 4 * (c + 4 * d);
                    if (r0 < a || r0 + 16 > b) {
                        row_masks(r0, 4 * n, a, b, m0, m1);
                        mask(dy[d], m0, m1);
                    }
                    if constexpr (FINITE) dy[d].drop_non_finite();
#pragma unroll
                    for (int q = 0; q < Q; ++q) acc[d][q] = mfma4(x.op(q), dy[d].op(q), acc[d][q]);
                }
            }
            a = b;
        }
    }
    // Whether at most kFewSequences sequences own rows of the tile.
    static constexpr int kFewSequences = ND == 2 ? 2 : 0;    // (with one group of lags the loop of passes() is as fast)
    __device__ __forceinline__ static bool few_sequences(uint64_t w0, uint64_t w1) {
        return __builtin_popcountll(w0 >> (TP::FRONT + 1)) + __builtin_popcountll(w1 & ((1ull << TP::FRONT) - 1ull)) < kFewSequences;
    }
    // acc += a tile's sums, chunk after chunk of dy, db with them; each chunk of x is packed once and meets the chunks of dy of both groups of lags.
    // PART: those of one sequence alone, staged rows [a, b): chunks that hold none of its rows are left out, those at its ends masked.
    // Every chunk is a place of its own in the code, so that neither addresses nor registers are moved: with one wave per SIMD
    // every instruction counts, and the loop of passes() spends 170 on a chunk where this spends 45.
    template <bool PART>
    __device__ __forceinline__ void sweep(int a, int b, int nrow, f32x4 (&acc)[ND][Q]) {
        constexpr int NR = 4 * (ND - 1) + 1, NCD = NCX + 4 * (ND - 1);
        // rows of x and the chunks they lie in (a lane's rows are shifted by up to 3)
        const int t0 = PART && a > TP::FRONT ? a - TP::FRONT : 0, t1 = !PART ? R : b - TP::FRONT < nrow ? b - TP::FRONT : nrow;
        // (PART, db: the chunks 0, 4, ... that hold the sequence's rows of the tile are among those visited, x0 .. x1 + 4: the first of
        // these rows is FRONT + t0)
        const int d0 = (TP::FRONT + t0) >> 4 << 2;
        const int x0 = !PART ? 0 : TP::FRONT < 15 && d0 < t0 >> 2 ? d0 : t0 >> 2, x1 = PART ? (t1 + 2) >> 2 : NCX - 1;
        MfmaRaw<Q> rd, rx;
        MfmaChunk<Q> ring[NR];                               // x chunks c - 4 .. c (of one group of lags: c)
        if (!PART || x0 == 0) {
            read_dy(0, rd);
            read_x(0, rx);
        }
        static_for<NCD>([&](auto c_c) __attribute__((always_inline)) {
            constexpr int c = decltype(c_c)::value;
            auto next = [&]() __attribute__((always_inline)) {
                if constexpr (c + 1 < NCD) read_dy(c + 1, rd);
                if constexpr (c + 1 < NCX) read_x(c + 1, rx);
            };
            if (!PART || (c >= x0 && c <= x1 + 4 * (ND - 1))) {
                MfmaChunk<Q> dy;
                uint32_t m0, m1;
                mfma_pack(rd, dy);
                if constexpr (c < NCX) {
                    mfma_pack(rx, ring[c % NR]);
                    if (PART ? 4 * c - 3 < t0 || 4 * c + 3 >= t1 : c == 0 || c == NCX - 1) {
                        row_masks(4 * c - 3, 3 - n, t0, t1, m0, m1);
                        mask(ring[c % NR], m0, m1);
                    }
                }
                // (what follows the staged rows meets only masked x, but may hold a NaN)
                if (PART ? 4 * c < a || 4 * c + 16 > b : 4 * c + 16 > SPAN) {
                    row_masks(4 * c, 4 * n, PART ? a : 0, PART ? b : SPAN, m0, m1);
                    mask(dy, m0, m1);
                }
                next();
                if constexpr (c < NCX) {
                    if (!PART || c <= x1) {
#pragma unroll
                        for (int q = 0; q < Q; ++q) acc[0][q] = mfma4(ring[c % NR].op(q), dy.op(q), acc[0][q]);
                    }
                }
                if constexpr (ND == 2 && c >= 4) {
                    if (!PART || c - 4 >= x0) {
#pragma unroll
                        for (int q = 0; q < Q; ++q) acc[ND - 1][q] = mfma4(ring[(c - 4) % NR].op(q), dy.op(q), acc[ND - 1][q]);
                    }
                }
                // db: staged rows 4c .. 4c + 15 in the four columns
                if constexpr (c % 4 == 0 && c < NCX) {
                    if constexpr (c == 0 || c == NCX - 1) {
                        row_masks(4 * c, 4 * n, TP::FRONT, TP::FRONT + R, m0, m1);
                        mask(dy, m0, m1);
                    }
                    add_db(dy);
                }
            } else if (c + 1 == x0) {
                next();
            }
            __builtin_amdgcn_sched_barrier(0);
        });
    }
    // words = the tile's boundary bits; nrow = its rows in front of T
    __device__ __forceinline__ void tile(const uint32_t* words, int nrow) {
        uint64_t w0, w1;                                     // boundary bits of staged rows 0 .. 63 and 64 on
        {
            uint32_t v[4];
#pragma unroll
            for (int i = 0; i < 4; ++i) v[i] = (uint32_t)__builtin_amdgcn_readfirstlane((int)words[i]);
            w0 = ((uint64_t)v[0] | (uint64_t)v[1] << 32) & ~1ull;
            w1 = (uint64_t)v[2] | (uint64_t)v[3] << 32;
        }
        f32x4 acc[ND][Q];
#pragma unroll
        for (int d = 0; d < ND; ++d)
#pragma unroll
            for (int q = 0; q < Q; ++q) acc[d][q] = f32x4{0.f, 0.f, 0.f, 0.f};
        if ((w0 | w1) == 0) {
            sweep<false>(0, SPAN, R, acc);
        } else {
            const bool few = kFewSequences > 0 && few_sequences(w0, w1);
            if (!few) {
                uint32_t m0, m1;
#pragma nounroll
                for (int c = 0; c < NCX; c += 4) {
                    MfmaRaw<Q> raw;
                    MfmaChunk<Q> dy;
                    read_dy(c, raw);
                    mfma_pack(raw, dy);
                    row_masks(4 * c, 4 * n, TP::FRONT, TP::FRONT + nrow, m0, m1);
                    mask(dy, m0, m1);
                    add_db(dy);
                }
            }
            if (few) {
                int a = sequence_of(w0, w1, TP::FRONT);
                do {
                    const int b = next_sequence(w0, w1, a > TP::FRONT ? a : TP::FRONT);
                    sweep<true>(a, b < SPAN ? b : SPAN, nrow, acc);
                    a = b;
                } while (a < TP::FRONT + nrow);
            } else {
                passes<false>(w0, w1, nrow, acc);
            }
        }
        float chk = 0.f;
#pragma unroll
        for (int d = 0; d < ND; ++d)
#pragma unroll
            for (int q = 0; q < Q; ++q) chk = __builtin_fmaf(acc[d][q][0], 0.f, chk);
        if (__builtin_amdgcn_ballot_w64(active && !__builtin_isfinite(chk)) != 0) {
#pragma unroll
            for (int d = 0; d < ND; ++d)
#pragma unroll
                for (int q = 0; q < Q; ++q) acc[d][q] = f32x4{0.f, 0.f, 0.f, 0.f};
            passes<true>(w0, w1, nrow, acc);
            int a = sequence_of(w0, w1, TP::FRONT), b = next_sequence(w0, w1, a);
#pragma nounroll
            for (int t = 0; t < nrow; ++t) {
                if (t + TP::FRONT >= b) { a = b; b = next_sequence(w0, w1, a); }
                RowVec<true, Q> xr, gr;
                float xv[Q], gv[Q];
                auto row_of = [&](RowVec<true, Q>& v, uint32_t at) __attribute__((always_inline)) {
                    const u32x2 t2 = mfma_lds(at);
                    v.d[0] = t2.x; v.d[1] = t2.y;
                };
                // the lane's slice of row 0 of a tile, its pieces in order, and the permutation of the row at hand
                const uint32_t x0 = (ax[0] + n * ROWB) ^ mfma_place(-n & 3), g0 = (ady[0] - 4 * n * ROWB) ^ mfma_place(n);
                row_of(xr, (x0 + t * ROWB) ^ mfma_place(t & 3));
                xr.to_f32(xv);
#pragma unroll
                for (int d = 0; d < ND; ++d)
#pragma unroll
                    for (int i = 0; i < 4; ++i) {
                        const int r = t + 16 * d + 4 * n + i;
                        if (r >= a && r < b && r < SPAN) {
                            row_of(gr, (g0 + r * ROWB) ^ mfma_place((r >> 2) & 3));
                            gr.to_f32(gv);
#pragma unroll
                            for (int q = 0; q < Q; ++q)
                                if (!__builtin_isfinite(xv[q]) || !__builtin_isfinite(gv[q])) acc[d][q][i] = __builtin_fmaf(xv[q], gv[q], acc[d][q][i]);
                        }
                    }
            }
        }
#pragma unroll
        for (int d = 0; d < ND; ++d)
#pragma unroll
            for (int q = 0; q < Q; ++q)
#pragma unroll
                for (int i = 0; i < 4; ++i) tot[d][q][i] += acc[d][q][i];
    }
    // first staged row of the sequence that holds row `at` (0: it began before), at < 128
    __device__ __forceinline__ static int sequence_of(uint64_t w0, uint64_t w1, int at) {
        if (at >= 64) {
            const uint64_t m = w1 & (~0ull >> (127 - at));
            if (m) return 127 - (int)__builtin_clzll(m);
            at = 63;
        }
        const uint64_t m = w0 & (~0ull >> (63 - at));
        return m ? 63 - (int)__builtin_clzll(m) : 0;
    }
    // first staged row of the sequence after the one that holds row `at` (128: none)
    __device__ __forceinline__ static int next_sequence(uint64_t w0, uint64_t w1, int at) {
        if (at < 63) {
            const uint64_t m = w0 & (~0ull << (at + 1));
            if (m) return (int)__builtin_ctzll(m);
            return w1 ? 64 + (int)__builtin_ctzll(w1) : 128;
        }
        const uint64_t m = at < 127 ? w1 & (~0ull << (at - 63)) : 0;
        return m ? 64 + (int)__builtin_ctzll(m) : 128;
    }
    // the block's sums to its slab: rows of taps (the weight's order), then db
    __device__ __forceinline__ void finish(float* __restrict__ slab, int C, int lane) const {
        float db[Q];
#pragma unroll
        for (int q = 0; q < Q; ++q) {                        // the four columns hold rows 0 .. 3, 4 .. 7, ... of every 16
            float v = dbs[q];
            v += __int_as_float(__builtin_amdgcn_ds_bpermute((lane ^ 1) * 4, __float_as_int(v)));
            v += __int_as_float(__builtin_amdgcn_ds_bpermute((lane ^ 2) * 4, __float_as_int(v)));
            db[q] = v;
        }
        if (!active) return;
#pragma unroll
        for (int d = 0; d < ND; ++d)
#pragma unroll
            for (int i = 0; i < 4; ++i) {
                const int m = 4 * TP::CK0 + 16 * d + 4 * n + i - (TP::PP - TP::P);
                if (m >= 0 && m < KT) *reinterpret_cast<float4*>(slab + (size_t)(KT - 1 - m) * C + c0) = make_float4(tot[d][0][i], tot[d][1][i], tot[d][2][i], tot[d][3][i]);
            }
        if (n == 0) *reinterpret_cast<float4*>(slab + (size_t)KT * C + c0) = make_float4(db[0], db[1], db[2], db[3]);
    }
};

// Backward: 64-row tiles (a dy tile with its halo rows, an x tile without), 4 wave-columns; waves of three kinds: dx
// (MfmaConv over dy), dw and db, loaders and boundaries.
// T=131072, C=2048, 31 taps: 272 us on one sequence (the role-split kernel of the vector ALU 479; a copy of the bytes takes 313),
// 340 on log-normal lengths (511). A SIMD has one wave of dx and one of dw, each of which issues an instruction every 5 cycles or
// so: what tiles with boundaries cost goes with the instructions they run (without the sweeps over single sequences 356 us;
// sequences of 320 rows 303 against 353). Tried for dw, all slower: one sweep of unrolled chunks that branches at each, one sweep and
// a left-over per boundary (spills), bit masks per chunk in place of the compares of sweep() (spills).
template <int KT>
struct MfmaBwdShape {
    using TP = MfmaTaps<KT>;
    static constexpr int NDX = kMfmaCh / (16 * kMfmaQ), NDW = NDX, NWC = NDX + NDW, NWL = 3;
    static constexpr int NT = (NWC + NWL + 1) * 64;
    static constexpr int R = 64, NROWS = R + TP::HALO;
    static constexpr int X_AT = NROWS * kMfmaCb, BUF_BYTES = X_AT + R * kMfmaCb;
    // lanes read up to four rows behind an x tile (masked); the boundary bits lie there behind the second one
    static constexpr int LDS_BYTES = 2 * BUF_BYTES + 4 * kMfmaCb;
    static_assert(2 * kMfmaWords * 4 <= 4 * kMfmaCb, "room for the boundary bits");
    static_assert(LDS_BYTES <= kLdsBytes, "two pairs of tiles fit the LDS");
    using W = MfmaWeights<KT, kMfmaCh, NWC>;
    static_assert(W::BYTES <= BUF_BYTES, "the weight table lies in the second buffer until its tiles come");
    static_assert((NROWS + 31) / 32 + 2 <= kMfmaWords && NROWS <= 96, "boundary bits");
};

template <int KT, bool RES, bool LINES>
__global__ void __launch_bounds__(MfmaBwdShape<KT>::NT)
dwconv_bwd_mfma_kernel(const void* __restrict__ x, const void* __restrict__ dy, const int32_t* __restrict__ cu,
                       const void* __restrict__ w, void* __restrict__ dx, float* __restrict__ partial, const LdsGeo g) {
    using SH = MfmaBwdShape<KT>;
    using TP = MfmaTaps<KT>;
    constexpr int R = SH::R;
    extern __shared__ __attribute__((aligned(16))) char lds_raw[];
    uint32_t* words = reinterpret_cast<uint32_t*>(lds_raw + 2 * SH::BUF_BYTES);
    uint32_t* tab = reinterpret_cast<uint32_t*>(lds_raw + SH::BUF_BYTES);
    const int lane = (int)(threadIdx.x & 63);
    const int wv = wave_id();
    int cb, tb;
    lds_block_coords(g, cb, tb);
    const int T = g.T, S = g.S, C = g.C;
    const int rowb = C * 2;
    const int col_byte0 = cb * kMfmaCb;
    const int valid_bytes = rowb - col_byte0 < kMfmaCb ? rowb - col_byte0 : kMfmaCb;
    const int nch = valid_bytes / 2;
    const int ntl = (g.ntiles + g.nbt - 1) / g.nbt;
    int q = tb;

    if (wv >= SH::NWC) {
        __builtin_amdgcn_s_setprio(3);
        const int lw = wv - SH::NWC;
        auto prepare = [&](int par, int t0) __attribute__((always_inline)) {
            char* buf = lds_raw + par * SH::BUF_BYTES;
            if (lw < SH::NWL) {
                mfma_stage<SH::NROWS, SH::NWL, SWZ_QUAD, kLoadAuxOnceBwd>(dy, buf, t0 - TP::FRONT, T, (size_t)rowb, col_byte0, valid_bytes, lw, lane, TP::HALO);
                mfma_stage<R, SH::NWL, SWZ_ROW, kLoadAuxOnceBwdX>(x, buf + SH::X_AT, t0, T, (size_t)rowb, col_byte0, valid_bytes, lw, lane, 0);
            } else {
                mfma_bounds(cu, S, T, t0 - TP::FRONT, SH::NROWS, words + par * kMfmaWords, lane);
            }
        };
        prepare(0, tb * R);
        lds_barrier();                       // the weight table is written
        lds_barrier();                       // and has been read
        for (int it = 0; it < ntl; ++it) {
            if (lw < SH::NWL) wait_vmem_all();
            lds_barrier();                   // tile `it` has landed, the buffer of the tile before is free
            q = lds_next_slot(g, q);
            const int t0 = it + 1 < ntl ? lds_tile_row0(g, it + 1, q, R) : T;
            if (t0 < T) prepare((it + 1) & 1, t0);
        }
        return;
    }
    SH::W::template fill<true>(tab, w, g.w_flags, cb * kMfmaCh, nch, (int)threadIdx.x);
    lds_barrier();
    if (wv < SH::NDX) {
        MfmaConv<KT, R / 16, true, RES, LINES> conv;
        conv.init(tab, SH::W::odd(tab), w, g.w_flags, nullptr, wv, lane, cb * kMfmaCh, nch, rowb);
        lds_barrier();
        for (int it = 0; it < ntl; ++it) {
            lds_barrier();
            const int t0 = lds_tile_row0(g, it, q, R);
            if (t0 < T)
                conv.rows(lds_raw + (it & 1) * SH::BUF_BYTES, words + (it & 1) * kMfmaWords, 0, mfma_out_rsrc(dx, t0, T - t0 < R ? T - t0 : R, rowb), rowb);
            q = lds_next_slot(g, q);
        }
    } else {
        MfmaDw<KT> dw;
        dw.init(lds_raw, wv - SH::NDX, lane, cb * kMfmaCh, nch, SH::X_AT);
        lds_barrier();
        for (int it = 0; it < ntl; ++it) {
            lds_barrier();
            const int t0 = lds_tile_row0(g, it, q, R);
            if (t0 < T) dw.tile(words + (it & 1) * kMfmaWords, T - t0 < R ? T - t0 : R);
            dw.next_buffer(it & 1 ? -SH::BUF_BYTES : SH::BUF_BYTES);
            q = lds_next_slot(g, q);
        }
        dw.finish(partial + (size_t)tb * (KT + 1) * C, C, lane);
    }
}

// ---- gated backward --------------------------------------------------------------------------------------------------
// z = [u | g] [T, 2C], the conv ran over h = u * silu(g). dz is MfmaConv over dy with the gate in its stores. dw needs h in
// fp32, which the matrix cores take only as three bf16 terms: three instructions of 10.7 cycles per 1024 products, what the
// vector ALU's FMAs take too, and the terms to be made (built and measured that way: 726 us, no gain). So dw stays on the
// vector ALU: a wave has 128 channels (two per lane) of 8 rows of the tile, with KT sums per channel and 8 rows of h in
// registers, and reads its KT + 7 rows of dy one after the other. What the role-split kernel spends on dx's FMAs is gone.
// Bound by the dz waves (one per SIMD: 555 us without the dw waves, loads alone 276). T=131072, C=2048, 31 taps, before and
// now: log-normal lengths 721 and 673 us, one sequence 674 to 729 and 619, 20 to 512 residues 737 and 705; T=8192, C=512 38 and
// 27. Two dz and one dw wave of 16 rows per SIMD: 1028 us.
// a[-i] += h[i] * d for the i < N whose bit of `in` is set (all lanes of the wave are on). Rows of another sequence are left out
// by the execution mask, not multiplied by zero (their product may be with an Inf). In one instruction block: sums that two
// branches of compiled code change come to lie in two sets of registers (56 spilled). The masked form lies behind the section's
// other code, so that the usual one runs on without a jump (T=131072, C=2048, 31 taps, one sequence: 699 us with one, 627).
#define NPLM_ROW_FMAC(i) "v_fmac_f32 %[a" #i "], %[h" #i "], %[d0]\n\tv_fmac_f32 %[b" #i "], %[g" #i "], %[d1]\n\t"
#define NPLM_ROW_SOME(i) "s_bitcmp1_b32 %[in], " #i "\n\ts_cselect_b64 exec, -1, 0\n\t" NPLM_ROW_FMAC(i)
#define NPLM_ROW_OUT(i) [a##i] "+v"(a[-i][0]), [b##i] "+v"(a[-i][1])
#define NPLM_ROW_IN(i) [h##i] "v"(h[i][0]), [g##i] "v"(h[i][1])
#define NPLM_FMAC_ROWS(ALL, FMAC, SOME, OUT, ...)                                                                              \
    asm volatile("s_and_b32 %[t], %[in], " #ALL "\n\ts_cmp_eq_u32 %[t], " #ALL "\n\ts_cbranch_scc0 .Lsome%=\n\t" FMAC          \
                 ".Ldone%=:\n\t.subsection 1\n.Lsome%=:\n\t" SOME "s_mov_b64 exec, -1\n\ts_branch .Ldone%=\n\t.subsection 0"   \
                 : [t] "=&s"(t), OUT : [in] "s"(in), __VA_ARGS__, [d0] "v"(d0), [d1] "v"(d1) : "scc")
#define NPLM_COMMA ,
template <int N>
__device__ __forceinline__ void fmac_rows(float (*a)[2], const float (*h)[2], float d0, float d1, uint32_t in) {
    static_assert(N >= 1 && N <= 4, "rows of a block");
    uint32_t t;
    if constexpr (N == 1)
        NPLM_FMAC_ROWS(1, NPLM_ROW_FMAC(0), NPLM_ROW_SOME(0), NPLM_ROW_OUT(0), NPLM_ROW_IN(0));
    else if constexpr (N == 2)
        NPLM_FMAC_ROWS(3, NPLM_ROW_FMAC(0) NPLM_ROW_FMAC(1), NPLM_ROW_SOME(0) NPLM_ROW_SOME(1), NPLM_ROW_OUT(0) NPLM_COMMA NPLM_ROW_OUT(1),
                       NPLM_ROW_IN(0), NPLM_ROW_IN(1));
    else if constexpr (N == 3)
        NPLM_FMAC_ROWS(7, NPLM_ROW_FMAC(0) NPLM_ROW_FMAC(1) NPLM_ROW_FMAC(2), NPLM_ROW_SOME(0) NPLM_ROW_SOME(1) NPLM_ROW_SOME(2),
                       NPLM_ROW_OUT(0) NPLM_COMMA NPLM_ROW_OUT(1) NPLM_COMMA NPLM_ROW_OUT(2), NPLM_ROW_IN(0), NPLM_ROW_IN(1), NPLM_ROW_IN(2));
    else
        NPLM_FMAC_ROWS(15, NPLM_ROW_FMAC(0) NPLM_ROW_FMAC(1) NPLM_ROW_FMAC(2) NPLM_ROW_FMAC(3),
                       NPLM_ROW_SOME(0) NPLM_ROW_SOME(1) NPLM_ROW_SOME(2) NPLM_ROW_SOME(3),
                       NPLM_ROW_OUT(0) NPLM_COMMA NPLM_ROW_OUT(1) NPLM_COMMA NPLM_ROW_OUT(2) NPLM_COMMA NPLM_ROW_OUT(3),
                       NPLM_ROW_IN(0), NPLM_ROW_IN(1), NPLM_ROW_IN(2), NPLM_ROW_IN(3));
}
#undef NPLM_ROW_FMAC
#undef NPLM_ROW_SOME
#undef NPLM_ROW_OUT
#undef NPLM_ROW_IN
#undef NPLM_FMAC_ROWS
#undef NPLM_COMMA
template <int KT>
struct GatedDw {
    using TP = MfmaTaps<KT>;
    static constexpr int RW = 8, CB = kMfmaGatedCb, NJ = RW + KT - 1;
    static constexpr int OFS = TP::PP - TP::P - 4 * TP::CK0; // staged row of tap 0 of output row 0 (below 4)
    float acc[KT][2], db[2];
    uint32_t ady[4], au;       // LDS addresses of the lane's slice of the wave's first staged row of dy (by the row's permutation) and of u

    // lds: the first buffer; wr: the wave's first row
    __device__ __forceinline__ void init(const char* lds, int wr, int lane, int x_at) {
        const uint32_t base = (uint32_t)(uintptr_t)(const __attribute__((address_space(3))) char*)lds + wr * CB;
#pragma unroll
        for (int f = 0; f < 4; ++f) ady[f] = base + ((lane * 4) ^ mfma_place((f + (wr >> 2)) & 3));
        au = base + x_at + ((lane * 4) ^ mfma_place((wr >> 2) & 3));
#pragma unroll
        for (int m = 0; m < KT; ++m) acc[m][0] = acc[m][1] = 0.f;
        db[0] = db[1] = 0.f;
    }
    __device__ __forceinline__ void next_buffer(int by) {
#pragma unroll
        for (int f = 0; f < 4; ++f) ady[f] += by;
        au += by;
    }
    __device__ __forceinline__ static uint32_t lds32(uint32_t at) { return *(const __attribute__((address_space(3))) uint32_t*)(uintptr_t)at; }
    template <int j>
    __device__ __forceinline__ uint32_t read_dy() const {
        constexpr int r = j + OFS;
        return lds32(ady[(r + (r >> 2)) & 3] + r * CB);
    }
    // bits: boundaries of the wave's staged rows (bit p: a sequence begins at staged row p of the wave, p > 0)
    __device__ __forceinline__ void sums(uint64_t bits) {
        // the wave's rows of the sequence that staged row j + OFS belongs to, as bits; four to a register
        uint32_t own[(NJ + 3) / 4];
#pragma unroll
        for (int i = 0; i < (NJ + 3) / 4; ++i) own[i] = ~0u;
        if (bits != 0) {
            static_for<NJ>([&](auto j_c) __attribute__((always_inline)) {
                constexpr int j = decltype(j_c)::value, r = j + OFS, F = TP::FRONT;
                int lo = 0;
                if constexpr (r > 0) lo = 63 - (int)__builtin_clzll((bits & (~0ull >> (63 - r))) | 1ull);
                int hi = (int)__builtin_ctzll((bits & (~0ull << (r + 1))) | 1ull << 63);
                lo = lo > F ? lo - F : 0;
                hi = hi - F < RW ? hi - F : RW;
                const uint32_t in = hi > lo ? (1u << hi) - (1u << lo) : 0u;
                own[j / 4] = (own[j / 4] & ~(255u << j % 4 * 8)) | in << j % 4 * 8;
            });
        }
#pragma unroll
        for (int i = 0; i < (NJ + 3) / 4; ++i) own[i] = (uint32_t)__builtin_amdgcn_readfirstlane((int)own[i]);
        float h[RW][2];
#pragma unroll
        for (int u = 0; u < RW; ++u) {
            const uint32_t at = u < 4 ? au : au ^ mfma_place(1);        // rows 4 .. 7 have the next permutation
            const uint32_t xu = lds32(at + u * CB), xg = lds32(at + (u + kMfmaGatedRows) * CB);
            h[u][0] = gate_mul(bf16_lo(xu), bf16_lo(xg));
            h[u][1] = gate_mul(bf16_hi(xu), bf16_hi(xg));
        }
        uint32_t nxt[2] = {read_dy<0>(), read_dy<1>()};
        static_for<NJ>([&](auto j_c) __attribute__((always_inline)) {
            constexpr int j = decltype(j_c)::value;
            const float d0 = bf16_lo(nxt[j & 1]), d1 = bf16_hi(nxt[j & 1]);
            if constexpr (j + 2 < NJ) nxt[j & 1] = read_dy<j + 2>();
            if constexpr (j >= TP::P && j < TP::P + RW) { db[0] += d0; db[1] += d1; }         // (rows from T on are staged as zeros)
            const uint32_t in = own[j / 4] >> j % 4 * 8;
            constexpr int u0 = j >= KT ? j - KT + 1 : 0, nu = (j < RW ? j + 1 : RW) - u0;
            fmac_rows<(nu < 4 ? nu : 4)>(&acc[j - u0], &h[u0], d0, d1, in >> u0);
            if constexpr (nu > 4) fmac_rows<nu - 4>(&acc[j - u0 - 4], &h[u0 + 4], d0, d1, in >> (u0 + 4));
            __builtin_amdgcn_sched_barrier(0);
        });
    }
    // words: the tile's boundary bits; wr: the wave's first row, in front of T
    __device__ __forceinline__ void tile(const uint32_t* words, int wr) {
        static_assert(NJ + OFS <= 62, "one word of bits");
        uint32_t v[3];
        const uint32_t* wp = words + (wr >> 5);
#pragma unroll
        for (int i = 0; i < 3; ++i) v[i] = (uint32_t)__builtin_amdgcn_readfirstlane((int)wp[i]);
        const int sh = wr & 31;
        const uint64_t lo = ((uint64_t)v[0] | (uint64_t)v[1] << 32) >> sh;
        const uint64_t bits = (lo | (sh ? (uint64_t)v[2] << (64 - sh) : 0)) & ~1ull & ((1ull << (NJ + OFS)) - 1ull);
        sums(bits);
    }
    // the sums by way of LDS, [2 KT + 2][64] floats a wave
    static constexpr int BOX = (2 * KT + 2) * 64;
    __device__ __forceinline__ void give(float* box, int lane) const {
#pragma unroll
        for (int c = 0; c < 2; ++c) {
            box[c * 64 + lane] = db[c];
#pragma unroll
            for (int m = 0; m < KT; ++m) box[(2 + 2 * m + c) * 64 + lane] = acc[m][c];
        }
    }
    __device__ __forceinline__ void take(const float* box, int lane) {
#pragma unroll
        for (int c = 0; c < 2; ++c) {
            db[c] += box[c * 64 + lane];
#pragma unroll
            for (int m = 0; m < KT; ++m) acc[m][c] += box[(2 + 2 * m + c) * 64 + lane];
        }
    }
    // the block's sums to its slab: rows of taps (the weight's order), then db
    __device__ __forceinline__ void finish(float* __restrict__ slab, int C, int c0) const {
#pragma unroll
        for (int m = 0; m < KT; ++m) *reinterpret_cast<float2*>(slab + (size_t)(KT - 1 - m) * C + c0) = make_float2(acc[m][0], acc[m][1]);
        *reinterpret_cast<float2*>(slab + (size_t)KT * C + c0) = make_float2(db[0], db[1]);
    }
};

// 64-row tiles of dy (with its halo rows), u and g; waves of four kinds: dz (4 x 32 channels), dw and db (8 x 8 rows), loaders and
// boundaries.
template <int KT>
struct MfmaGatedBwdShape {
    using TP = MfmaTaps<KT>;
    static constexpr int CB = kMfmaGatedCb, CH = CB / 2, R = kMfmaGatedRows, NROWS = R + TP::HALO;
    static constexpr int NCW = 4, NDZ = NCW, NDW = R / GatedDw<KT>::RW, NWC = NDZ + NDW, NWL = 3;
    static constexpr int NT = (NWC + NWL + 1) * 64;
    static constexpr int X_AT = NROWS * CB, BUF_BYTES = X_AT + 2 * R * CB;
    static constexpr int WORDS_AT = 2 * BUF_BYTES;
    static constexpr int LDS_BYTES = WORDS_AT + 2 * kMfmaWords * 4;
    static_assert(CH == 128, "a dw wave has two channels per lane");
    static_assert(NDW == 8 && NDW / 2 * GatedDw<KT>::BOX * 4 <= WORDS_AT, "half of the sums in the buffers");
    static_assert(LDS_BYTES <= kLdsBytes, "two buffers of three tiles fit the LDS");
    using W = MfmaWeights<KT, CH, NWC>;
    static_assert(W::BYTES <= BUF_BYTES, "the weight table lies in the second buffer until its tiles come");
    static_assert((NROWS + 31) / 32 + 2 <= kMfmaWords && NROWS <= 96, "boundary bits");
};

template <int KT, bool RES>
__global__ void __launch_bounds__(MfmaGatedBwdShape<KT>::NT)
dwconv_bwd_gated_mfma_kernel(const void* __restrict__ z, const void* __restrict__ dy, const int32_t* __restrict__ cu,
                             const void* __restrict__ w, void* __restrict__ dz, float* __restrict__ partial, const LdsGeo g) {
    using SH = MfmaGatedBwdShape<KT>;
    using TP = MfmaTaps<KT>;
    constexpr int R = SH::R;
    extern __shared__ __attribute__((aligned(16))) char lds_raw[];
    uint32_t* words = reinterpret_cast<uint32_t*>(lds_raw + SH::WORDS_AT);
    uint32_t* tab = reinterpret_cast<uint32_t*>(lds_raw + SH::BUF_BYTES);
    const int lane = (int)(threadIdx.x & 63);
    const int wv = wave_id();
    int cb, tb;
    lds_block_coords(g, cb, tb);
    const int T = g.T, S = g.S, C = g.C;
    const int rowb = C * 2;
    const int col_byte0 = cb * SH::CB;
    const int valid_bytes = rowb - col_byte0 < SH::CB ? rowb - col_byte0 : SH::CB;
    const int nch = valid_bytes / 2;
    const int ntl = (g.ntiles + g.nbt - 1) / g.nbt;
    int q = tb;

    if (wv >= SH::NWC) {
        __builtin_amdgcn_s_setprio(3);
        const int lw = wv - SH::NWC;
        auto prepare = [&](int par, int t0) __attribute__((always_inline)) {
            char* buf = lds_raw + par * SH::BUF_BYTES;
            if (lw < SH::NWL) {
                mfma_stage<SH::NROWS, SH::NWL, SWZ_BOTH, kLoadAuxOnceBwd, SH::CB>(dy, buf, t0 - TP::FRONT, T, (size_t)rowb, col_byte0, valid_bytes, lw, lane, TP::HALO);
                mfma_stage<R, SH::NWL, SWZ_QUAD, kLoadAuxOnceBwdX, SH::CB>(z, buf + SH::X_AT, t0, T, 2 * (size_t)rowb, col_byte0, valid_bytes, lw, lane, 0);
                mfma_stage<R, SH::NWL, SWZ_QUAD, kLoadAuxOnceBwdX, SH::CB>(z, buf + SH::X_AT + R * SH::CB, t0, T, 2 * (size_t)rowb, rowb + col_byte0, valid_bytes, lw, lane, 0);
            } else {
                mfma_bounds(cu, S, T, t0 - TP::FRONT, SH::NROWS, words + par * kMfmaWords, lane);
            }
        };
        prepare(0, tb * R);
        lds_barrier();                       // the weight table is written
        lds_barrier();                       // and has been read
        for (int it = 0; it < ntl; ++it) {
            if (lw < SH::NWL) wait_vmem_all();
            lds_barrier();                   // tile `it` has landed, the buffer of the tile before is free
            q = lds_next_slot(g, q);
            const int t0 = it + 1 < ntl ? lds_tile_row0(g, it + 1, q, R) : T;
            if (t0 < T) prepare((it + 1) & 1, t0);
        }
        for (int k = 0; k < 6; ++k) lds_barrier();      // (the dw waves join their sums)
        return;
    }
    SH::W::template fill<true>(tab, w, g.w_flags, cb * SH::CH, nch, (int)threadIdx.x);
    lds_barrier();
    if (wv < SH::NDZ) {
        __builtin_amdgcn_s_setprio(2);       // a dz wave has the longest way through a tile (log-normal lengths: 682 us without, 673 with)
        MfmaConv<KT, R / 16, true, RES, true, true> conv;
        conv.init(tab, SH::W::odd(tab), w, g.w_flags, nullptr, wv, lane, cb * SH::CH, nch, rowb);
        lds_barrier();
        for (int it = 0; it < ntl; ++it) {
            lds_barrier();
            const int t0 = lds_tile_row0(g, it, q, R);
            const char* buf = lds_raw + (it & 1) * SH::BUF_BYTES;
            if (t0 < T)
                conv.rows(buf, words + (it & 1) * kMfmaWords, 0, mfma_out_rsrc(dz, t0, T - t0 < R ? T - t0 : R, 2 * rowb), rowb, buf + SH::X_AT);
            q = lds_next_slot(g, q);
        }
        for (int k = 0; k < 6; ++k) lds_barrier();
    } else {
        using DW = GatedDw<KT>;
        DW dw;
        const int dv = wv - SH::NDZ, wr = dv * DW::RW;
        dw.init(lds_raw, wr, lane, SH::X_AT);
        lds_barrier();
        for (int it = 0; it < ntl; ++it) {
            lds_barrier();
            if (lds_tile_row0(g, it, q, R) + wr < T) dw.tile(words + (it & 1) * kMfmaWords, wr);
            dw.next_buffer(it & 1 ? -SH::BUF_BYTES : SH::BUF_BYTES);
            q = lds_next_slot(g, q);
        }
        // the eight waves' sums in a fixed order: 0 + 4, 1 + 5, ...; then 0 + 2, 1 + 3; then 0 + 1
        float* box = reinterpret_cast<float*>(lds_raw);
#pragma nounroll
        for (int half = SH::NDW / 2; half > 0; half /= 2) {
            lds_barrier();
            if (dv >= half && dv < 2 * half) dw.give(box + (dv - half) * DW::BOX, lane);
            lds_barrier();
            if (dv < half) dw.take(box + dv * DW::BOX, lane);
        }
        if (dv == 0 && 2 * lane < nch) dw.finish(partial + (size_t)tb * (KT + 1) * C, C, cb * SH::CH + 2 * lane);
    }
}

// ---- gated forward ---------------------------------------------------------------------------------------------------
// y = conv(h), h = u * silu(g) of z = [u | g] [T, 2C]. h is fp32 and stays it: the producers split it into three bf16 terms that add
// up to it exactly (8 significant bits each, by truncation), and the consumers take the products of all three with the taps, which are
// exact as well. So the sums differ from the vector ALU's by their order alone.
// bf16 ends at 2^-133 and fp32 at 2^-149, so the producers form 2^16 h (the factor rides in the sigmoid's sum and costs nothing) and the
// weights are taken 2^-16 times: the same products, and terms that end where fp32 does. What that leaves out at the other ends, an h of
// 2^112 on and weights below 2^-110, goes the way of values that are not finite. (Marking the chunks whose terms lack bits, for the
// consumers to add them from z, took 366 us of the 359 without and 394 of 389 at 300 rows a sequence, T=131072, C=2048, 31 taps.)
// What bounds it: on the vector ALU the 31 FMAs an element (0.8 of all issue slots); here the gate and the split, 14
// instructions an element of which two are quarter-rate, each evaluated once: a block walks down a run of steps of 64 rows, and a
// step's window takes over the halo rows from the step before in the ring. The producers alone take 201 us, the consumers alone 257
// with one of 64 rows per SIMD (boundaries then cost twice what they do with two of 32: 430 and 395 us on log-normal lengths).
// T=131072, C=2048, 31 taps, before and now: one sequence 393 to 413 and 357 to 369 us, log-normal lengths 415 to 444 and 387 to 406;
// T=32768, C=768, 300 rows a sequence 57 and 43; T=8192, C=512 24 and 16. Outputs that are not the correctly rounded value
// 6.3e-5 (7.8e-5). Waves: 8 consumers (32 channels x 32 rows of a step; no packing, no gate), 8 producers (a chunk of 4 rows x 128 channels at a time, z straight into registers two phases ahead). The boundary bits of all the block's runs are
// found before the first.
template <int KT>
struct MfmaGatedFwdShape {
    using TP = MfmaTaps<KT>;
    using RG = MfmaRing<KT>;
    static constexpr int NCW = 4, NCONS = 8, RW = RG::R * NCW / NCONS, NPROD = 8, UNITS = RG::R / 4 / NPROD, NW = NCONS + NPROD, NT = NW * 64;
    static constexpr int WORDS = (kMfmaGatedSteps * RG::R + TP::HALO + 31) / 32 + 2;     // boundary bits of a run (lanes read two words further)
    static_assert(WORDS <= 64, "a wave clears them in one go");
    using W = MfmaWeights<KT, RG::CH, NCONS, true>;
    static_assert(W::BYTES <= RG::BYTES, "the weight table lies in the ring until it is written");
    static_assert(RG::BYTES + 64 * WORDS * 4 <= kLdsBytes, "fits the LDS");
    // LDS of a call whose blocks have up to this many runs; the words begin behind the ring
    static constexpr long long lds_bytes(long long runs) { return RG::BYTES + runs * WORDS * 4; }
};

template <int KT, bool RES>
__global__ void __launch_bounds__(MfmaGatedFwdShape<KT>::NT)
dwconv_fwd_gated_mfma_kernel(const void* __restrict__ z, const int32_t* __restrict__ cu, const void* __restrict__ w,
                             const void* __restrict__ bias, void* __restrict__ y, const LdsGeo g, const int steps) {
    using SH = MfmaGatedFwdShape<KT>;
    using TP = MfmaTaps<KT>;
    using RG = MfmaRing<KT>;
    constexpr int R = RG::R;
    extern __shared__ __attribute__((aligned(16))) char lds_raw[];
    uint32_t* words = reinterpret_cast<uint32_t*>(lds_raw + RG::BYTES);
    uint32_t* tab = reinterpret_cast<uint32_t*>(lds_raw);
    const int lane = (int)(threadIdx.x & 63);
    const int wv = wave_id();
    int cb, tb;
    lds_block_coords(g, cb, tb);
    const int T = g.T, C = g.C;
    const int rowb = C * 2;
    const int col_byte0 = cb * kMfmaGatedCb;
    const int valid_bytes = rowb - col_byte0 < kMfmaGatedCb ? rowb - col_byte0 : kMfmaGatedCb;
    const int nch = valid_bytes / 2;
    // the block's runs: one a round, none in the last round where the slot lies past the last run
    const int rounds = (g.ntiles + g.nbt - 1) / g.nbt;
    const int last = (int)((tb + (long long)(rounds - 1) * g.rot_step) % g.nbt);
    const int runs = lds_tile_row0(g, rounds - 1, last, R * steps) < T ? rounds : rounds - 1;
    const int phases = runs > 0 ? runs * (steps + 1) + 1 : 0;
    auto bounds = [&]() __attribute__((always_inline)) {
        int q = tb;
        for (int it = 0; it < runs; ++it) {
            if (it % SH::NW == wv)
                mfma_bounds<SH::WORDS>(cu, g.S, T, lds_tile_row0(g, it, q, R * steps) - TP::FRONT, R * steps + TP::HALO, words + it * SH::WORDS, lane);
            q = lds_next_slot(g, q);
        }
    };

    if (wv < SH::NCONS) {
        __builtin_amdgcn_s_setprio(1);       // (the longer way through a phase)
        SH::W::template fill<false>(tab, w, g.w_flags, cb * RG::CH, nch, (int)threadIdx.x);
        bounds();
        lds_barrier();
        const int rg = wv / SH::NCW, r0 = rg * SH::RW;
        MfmaConv<KT, SH::RW / 16, false, RES, false, false, 3> conv;      // (stores without `nt`: 64 bytes of a row at a time)
        conv.init(tab, SH::W::odd(tab), w, g.w_flags, bias, wv % SH::NCW, lane, cb * RG::CH, nch, rowb);
        lds_barrier();                       // the table has been read
        int slot = 0, it = 0, s = 0, q = tb, row0 = lds_tile_row0(g, 0, q, R * steps);
        for (int p = 0; p < phases; ++p) {
            if (p >= 2) {
                const int t0 = row0 + s * R + r0;
                if (s < steps && t0 < T)
                    conv.rows(conv.slice + (slot + r0 / 4) * RG::REC, words + it * SH::WORDS, s * R + r0,
                              mfma_out_rsrc(y, t0, T - t0 < SH::RW ? T - t0 : SH::RW, rowb), rowb, nullptr, {z, t0, T});
                slot = RG::next(slot);
                if (++s > steps) {           // (the phase between two runs has no step)
                    s = 0;
                    q = lds_next_slot(g, q);
                    row0 = lds_tile_row0(g, ++it, q, R * steps);
                }
            }
            lds_barrier();
        }
    } else {
        const int pw = wv - SH::NCONS;
        struct Unit { uint32_t u[4], g[4]; };
        struct Step { Unit a[SH::UNITS]; };
        const int zrow = 2 * rowb, at_lane = lane * 4 < valid_bytes ? col_byte0 + lane * 4 : (int)0xc0000000;
        int it = 0, j = 0, q = tb, row0 = runs > 0 ? lds_tile_row0(g, 0, q, R * steps) : T;
        // the loads of the next phase in the order of phases; rows that do not exist land as zeros (or, in front of row 0 of a
        // tensor beyond 4 GiB, as other rows: what becomes of them is never used)
        auto fetch = [&](Step& o) __attribute__((always_inline)) {
            const int first = row0 - TP::FRONT, rb = first > 0 ? first : 0;
            const bool live = it < runs;
            const rsrc_t rs = live ? rows_rsrc(z, rb, T, (size_t)zrow) : make_rsrc(z, 0);
#pragma unroll
            for (int i = 0; i < SH::UNITS; ++i) {
                const int k = 16 * j - RG::PRE + pw + i * SH::NPROD;         // chunk of the run (below 0: none)
                const int at = k >= 0 ? (first - rb + 4 * k) * zrow + at_lane : (int)0xc0000000;
#pragma unroll
                for (int r = 0; r < 4; ++r) {
                    o.a[i].u[r] = __builtin_amdgcn_raw_buffer_load_b32(rs, at + r * zrow, 0, 0);
                    o.a[i].g[r] = __builtin_amdgcn_raw_buffer_load_b32(rs, at + r * zrow + rowb, 0, 0);
                }
            }
            if (++j > steps) {
                j = 0;
                q = lds_next_slot(g, q);
                row0 = ++it < runs ? lds_tile_row0(g, it, q, R * steps) : 0;
            }
        };
        auto make = [&](const Step& v, int slot) __attribute__((always_inline)) {
#pragma unroll
            for (int i = 0; i < SH::UNITS; ++i) {
                int rec = slot + pw + i * SH::NPROD;
                rec = rec < RG::LEN ? rec : rec - RG::LEN;
                float h[2][4];
#pragma unroll
                for (int r = 0; r < 4; ++r) {
                    h[0][r] = gate_mul_up(bf16_lo(v.a[i].u[r]), bf16_lo(v.a[i].g[r]));
                    h[1][r] = gate_mul_up(bf16_hi(v.a[i].u[r]), bf16_hi(v.a[i].g[r]));
                }
#pragma unroll
                for (int r = 0; r < 4; ++r) asm volatile("" : "+v"(h[0][r]), "+v"(h[1][r]));     // (h rounded: no product is contracted into the differences)
                const uint32_t at = rec * RG::REC + lane * 16;
#pragma unroll
                for (int t = 0; t < 3; ++t) {
                    u32x4 o;
#pragma unroll
                    for (int c = 0; c < 2; ++c) {
                        o[2 * c] = __builtin_amdgcn_perm(__float_as_uint(h[c][1]), __float_as_uint(h[c][0]), 0x07060302);
                        o[2 * c + 1] = __builtin_amdgcn_perm(__float_as_uint(h[c][3]), __float_as_uint(h[c][2]), 0x07060302);
                        if (t < 2) {
#pragma unroll
                            for (int r = 0; r < 4; ++r) h[c][r] -= bf16_hi(__float_as_uint(h[c][r]));
                        }
                    }
                    *(__attribute__((address_space(3))) u32x4*)(uintptr_t)(at + t * RG::TERM) = o;
                }
            }
        };
        Step a, b;
        fetch(a);
        fetch(b);
        bounds();
        lds_barrier();
        lds_barrier();
        int slot = (RG::LEN - RG::PRE) % RG::LEN;
        // (the way out in the middle of the body keeps "all but the other step's loads have landed" a wait for a count)
        for (int p = 0; p < phases; ++p) {
            make(a, slot);
            slot = RG::next(slot);
            fetch(a);
            lds_barrier();
            if (++p == phases) break;
            make(b, slot);
            slot = RG::next(slot);
            fetch(b);
            lds_barrier();
        }
    }
}

}  // namespace nplm
