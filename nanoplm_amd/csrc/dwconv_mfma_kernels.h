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
// would reach it. Every sum that holds such a product is itself not finite; the kernels test their sums and form the rows
// of a wave's group again, one product at a time and only the ones that belong, when one is not.
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
struct MfmaChunk {
    u32x2 b[kMfmaQ];
    __device__ __forceinline__ s16x4 op(int q) const { return __builtin_bit_cast(s16x4, b[q]); }
};
struct MfmaRaw { uint32_t r[4][kMfmaQ / 2]; };

// (lds_u32x2 loads: one ds_read_b64 per row, rows 512 bytes apart)
typedef const __attribute__((address_space(3))) u32x2* lds_u32x2;
__device__ __forceinline__ u32x2 mfma_lds(uint32_t at) { return *(lds_u32x2)(uintptr_t)at; }
template <int ROWS = 4>
__device__ __forceinline__ void mfma_read(const char* p, MfmaRaw& o) {
#pragma unroll
    for (int r = 0; r < 4; ++r) {
        u32x2 t = {0, 0};
        if (r < ROWS) t = *(lds_u32x2)(p + r * kMfmaCb);
        o.r[r][0] = t.x; o.r[r][1] = t.y;
    }
}
__device__ __forceinline__ void mfma_pack(const MfmaRaw& r, MfmaChunk& c) {
#pragma unroll
    for (int h = 0; h < kMfmaQ / 2; ++h) {
        c.b[2 * h].x = __builtin_amdgcn_perm(r.r[1][h], r.r[0][h], 0x05040100);
        c.b[2 * h].y = __builtin_amdgcn_perm(r.r[3][h], r.r[2][h], 0x05040100);
        c.b[2 * h + 1].x = __builtin_amdgcn_perm(r.r[1][h], r.r[0][h], 0x07060302);
        c.b[2 * h + 1].y = __builtin_amdgcn_perm(r.r[3][h], r.r[2][h], 0x07060302);
    }
}
__device__ __forceinline__ f32x4 mfma4(s16x4 a, s16x4 b, f32x4 c) { return __builtin_amdgcn_mfma_f32_4x4x4bf16_1k(a, b, c, 0, 0, 0); }

// Staging: rows of a 512-byte column block, two per 1 KiB direct load. The 16-byte pieces of a row are permuted (by the
// lanes' global addresses, inside the row) so that lanes which read four rows at once read different banks: piece p of row
// r lies at p ^ (swz(r) << 2). ROWSWZ: swz = r & 3 (readers at distance 1 row), else (r >> 2) & 3 (distance 4 rows).
template <bool ROWSWZ>
__device__ __forceinline__ int mfma_swz(int row) { return ROWSWZ ? row & 3 : (row >> 2) & 3; }
// Every one of the NLW loader waves issues the same number of loads (a surplus one repeats the last rows), so that "all but
// the newest tile's have landed" is a compile-time wait.
template <int NROWS, int NLW, bool ROWSWZ, int ONCE_AUX>
__device__ __forceinline__ void mfma_stage(const void* __restrict__ src, char* dst, int first_row, int T, size_t row_bytes,
                                           int col_byte0, int valid_bytes, int lw, int lane, int edge) {
    constexpr int RPL = 1024 / kMfmaCb, NL = (NROWS + RPL - 1) / RPL, CNT = (NL + NLW - 1) / NLW;
    const int rb = first_row > 0 ? first_row : 0;
    const rsrc_t rs = rows_rsrc(src, rb, T, row_bytes);
    const int rowb = (int)row_bytes;
    const int lrow = lane / (kMfmaCb / 16), lpiece = lane % (kMfmaCb / 16);
    // rows outside [0, T) are not clamped: their offsets fall outside the descriptor (or, on a tensor beyond 4 GiB, on other
    // rows of it), and what lands in LDS for them is never used
#pragma unroll
    for (int i = 0; i < CNT; ++i) {
        const int gi = lw + i * NLW < NL ? lw + i * NLW : NL - 1;
        const int row = RPL * gi + lrow;
        const int piece = lpiece ^ (mfma_swz<ROWSWZ>(row) << 2);
        const bool once = gi * RPL >= edge && gi * RPL + RPL <= NROWS - edge;
        if ((NROWS % RPL == 0 || row < NROWS) && piece * 16 < valid_bytes)
            load_to_lds<ONCE_AUX>(rs, dst + gi * 1024, (first_row - rb + row) * rowb + col_byte0 + piece * 16, 0, once);
    }
}

// Boundary bits of the rows [a, a + n): bit p of `words` is set iff a sequence begins at row a + p (0 < p < n); the tensor's
// first and one-past-last row count. One whole wave; a search with 64 probes a step finds the first entry of cu beyond row
// a, then entries are taken 64 at a time. Indices stay in [0, S] whatever cu holds.
__device__ __forceinline__ void mfma_bounds(const int32_t* __restrict__ cu, int S, int T, int a, int n, uint32_t* words, int lane) {
    if (lane < kMfmaWords) words[lane] = 0;
    auto mark = [&](int row) __attribute__((always_inline)) {
        const uint32_t p = (uint32_t)row - (uint32_t)a;      // (unsigned: cu may hold anything)
        if (row > a && p < (uint32_t)n) __hip_atomic_fetch_or(words + (p >> 5), 1u << (p & 31), __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
    };
    if (lane == 0) mark(0);
    if (lane == 1) mark(T);
    int lo = 0, hi = S + 1;              // the first i in [lo, hi) with cu[i] > a, else hi
    while (hi - lo > 64) {
        const int step = (hi - lo + 63) >> 6;
        const int i = lo + (lane + 1) * step - 1;
        const uint64_t m = __builtin_amdgcn_ballot_w64(cu[i < hi ? i : hi - 1] > a);
        if (m == 0) { lo = hi; break; }
        const int f = (int)__builtin_ctzll(m);
        const int nhi = lo + (f + 1) * step;
        lo += f * step;
        hi = nhi < hi ? nhi : hi;
    }
    for (; lo <= S; lo += 64) {
        const int i = lo + lane <= S ? lo + lane : S;
        const int v = cu[i];
        mark(v);
        if (__builtin_amdgcn_readlane(v, 63) >= a + n) break;
    }
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

// The caller's weight of channel c at tap m of the plan (0 .. KP-1), as the conv takes it (FLIP: the transposed conv of dx).
template <int KP, bool FLIP>
__device__ __forceinline__ float mfma_weight(const void* __restrict__ w, int w_flags, int c, int m, bool res) {
    const int off = w_tap_off(w_flags), kw = KP - 2 * off;
    const int r = (FLIP ? KP - 1 - m : m) - off;
    float v = 0.f;
    if (r >= 0 && r < kw) {
        const size_t i = (size_t)c * kw + r;
        v = (w_flags & W_BF16) ? bf16_to_f32(reinterpret_cast<const uint16_t*>(w)[i]) : reinterpret_cast<const float*>(w)[i];
    }
    return v + (res && m == (KP - 1) / 2 ? 1.f : 0.f);
}

// Weight table of a column block in LDS, [channel][WSTR] dwords of two bf16: entry e of a channel is plan tap e - 4 + 4 CK0.
template <int KT, bool FLIP>
__device__ __forceinline__ void mfma_fill_weights(uint32_t* tab, const void* __restrict__ w, int w_flags, int ch0, int nch, int tid, int nthreads) {
    using TP = MfmaTaps<KT>;
    for (int i = tid; i < kMfmaCh * TP::WSTR; i += nthreads) {
        const int c = i / TP::WSTR, p = i - c * TP::WSTR;
        uint32_t t = 0;
        if (c < nch) {
#pragma unroll
            for (int h = 0; h < 2; ++h) {
                const int m = 2 * p + h - 4 + 4 * TP::CK0;
                if (m >= 0 && m < TP::KP) t |= (__float_as_uint(mfma_weight<TP::KP, FLIP>(w, w_flags, ch0 + c, m, false)) >> 16) << (16 * h);
            }
        }
        tab[i] = t;
    }
}

// One wave's conv over staged rows: 16 Q channels, groups of 16 NSTEP output rows. FLIP: dx from dy. RES: the identity is one
// more band (a single 1 per row), since a bf16 weight plus one is not one in bf16.
template <int KT, int NSTEP, bool FLIP, bool RES>
struct MfmaConv {
    using TP = MfmaTaps<KT>;
    static constexpr int Q = kMfmaQ, NCK = TP::NCK;
    static constexpr int ROWS = 16 * NSTEP;                  // output rows of a group
    static_assert(ROWS % 32 == 0, "a group's boundary bits start at a word");
    static constexpr int NCHUNK = 4 * (NSTEP - 1) + NCK;     // chunks that the steps of a group read (per lane)
    static constexpr int IDC = (TP::FRONT + 0) / 4;          // chunk of the identity's first row
    static constexpr int IDN = (TP::FRONT + 3) / 4 - IDC + 1;
    s16x4 A[NCK][Q];
    s16x4 I[RES ? IDN : 1];
    f32x4 bias;            // where the sums start (dx: 0)
    int off[4];            // LDS offset of the lane's slice of chunk c, by c & 3 (without c * 4 rows)
    int n;                 // the lane's column: output rows 4 n .. 4 n + 3 of a step
    int c0;                // its first channel
    int swap;              // stores: the lane whose output goes out through this one (x 4)
    int out_at;            // byte offset of that lane's slice of output row 4 n, or kMfmaNoStore
    bool active;
    const void* w;
    int w_flags;

    __device__ __forceinline__ void init(const uint32_t* tab, const void* w_, int w_flags_, const void* b, int wc, int lane, int ch0, int nch, int rowb) {
        n = lane & 3;
        const int blk = lane >> 2;
        const int lc = (wc * 16 + blk) * Q;
        active = lc < nch;
        const int lcc = active ? lc : nch - Q;
        c0 = ch0 + lcc;
        swap = ((lane >> 4) + 4 * (lane & 15)) * 4;
        const int lcs = (wc * 16 + (lane & 15)) * Q;
        out_at = lcs < nch ? 4 * (lane >> 4) * rowb + (ch0 + lcs) * 2 : kMfmaNoStore;
        w = w_;
        w_flags = w_flags_;
#pragma unroll
        for (int k = 0; k < 4; ++k) off[k] = 4 * n * kMfmaCb + ((lcc * 2) ^ (((n + k) & 3) << 6));
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
                for (int e = 0; e < 4; ++e) I[k][e] = (4 * (IDC + k) + e == TP::FRONT + n) ? (short)0x3f80 : (short)0;
        }
#pragma unroll
        for (int q = 0; q < Q; ++q) {
            bias[q] = 0.f;
            if (b) bias[q] = (w_flags & W_BF16) ? bf16_to_f32(reinterpret_cast<const uint16_t*>(b)[c0 + q]) : reinterpret_cast<const float*>(b)[c0 + q];
        }
    }

    __device__ __forceinline__ f32x4 start(int q) const {
        if constexpr (FLIP) return f32x4{0.f, 0.f, 0.f, 0.f};
        float b = bias[q];
        asm volatile("" : "+v"(b));                          // (else four copies of it stay in registers)
        return f32x4{b, b, b, b};
    }
    // acc += the products of window chunk k
    template <int k>
    __device__ __forceinline__ void taps(f32x4 (&acc)[Q], const MfmaChunk& x) const {
#pragma unroll
        for (int q = 0; q < Q; ++q) acc[q] = mfma4(A[k][q], x.op(q), acc[q]);
        if constexpr (RES && k >= IDC && k < IDC + IDN) {
#pragma unroll
            for (int q = 0; q < Q; ++q) acc[q] = mfma4(I[k - IDC], x.op(q), acc[q]);
        }
    }
    // Adjacent lanes of a sum are rows 0, 4, 8, 12; they trade places first, so that 16 adjacent lanes store the 32 Q bytes
    // of one row (as 4-row pieces of 8 bytes the memory pipeline takes four times the requests: T=131072, C=2048, 31 taps
    // 223 us against 200).
    __device__ __forceinline__ void store(rsrc_t ro, int at, int rowb, int row, const float (&v)[Q]) const {
        RowVec<true, Q> o;
        o.from_f32(v);
#pragma unroll
        for (int h = 0; h < Q / 2; ++h) o.d[h] = (uint32_t)__builtin_amdgcn_ds_bpermute(swap, (int)o.d[h]);
        o.bstore(ro, at, row * rowb);
    }

    // boundary bits of this lane's window in step s (rows 16 s + 4 n on) of a group whose bits start at wp
    __device__ __forceinline__ MfmaBits window_bits(const uint32_t* wp, int s) const {
        const int at = 16 * s + 4 * n;
        const uint32_t* d = wp + (at >> 5);
        const uint32_t d0 = d[0], d1 = d[1], d2 = d[2];
        return MfmaBits{__builtin_amdgcn_alignbit(d1, d0, at & 31), __builtin_amdgcn_alignbit(d2, d1, at & 31)};
    }

    // One group of output rows: lp = the group's first window row in LDS, words = the tile's boundary bits, p0 = the window row's
    // place among them; ro = descriptor of the group's output rows (those in front of T).
    __device__ __forceinline__ void rows(const char* lp, const uint32_t* words, int p0, rsrc_t ro, int rowb) const {
        constexpr int SPAN = 16 * NSTEP + TP::HALO;          // window rows of the group
        const uint32_t* wp = words + (p0 >> 5);              // p0 is a multiple of 32
        bool open;                                           // no boundary inside the window (a bit at its first row is none)
        {
            uint32_t any = 0;
#pragma unroll
            for (int i = 0; i * 32 < SPAN; ++i) any |= wp[i] & (i == 0 ? ~1u : SPAN - i * 32 >= 32 ? ~0u : (1u << (SPAN & 31)) - 1u);
            open = __builtin_amdgcn_readfirstlane((int)any) == 0;
        }
        uint32_t redo = 0;                                   // steps whose sums are not all finite
        if (open) {
            float chk = 0.f;
            f32x4 acc[(NCK + 3) / 4][Q];
            MfmaRaw raw;
            mfma_read(lp + off[0], raw);
            static_for<NCHUNK>([&](auto c_c) __attribute__((always_inline)) {
                constexpr int c = decltype(c_c)::value;
                MfmaChunk x;
                mfma_pack(raw, x);
                if constexpr (c + 1 < NCHUNK)
                    mfma_read<(c + 1 == NCHUNK - 1 ? TP::LASTROWS : 4)>(lp + off[(c + 1) & 3] + (c + 1) * 4 * kMfmaCb, raw);
                static_for<NSTEP>([&](auto s_c) __attribute__((always_inline)) {
                    constexpr int s = decltype(s_c)::value;
                    constexpr int k = c - 4 * s;
                    if constexpr (k >= 0 && k < NCK) {
                        f32x4 (&a)[Q] = acc[s % ((NCK + 3) / 4)];
                        if constexpr (k == 0) {
#pragma unroll
                            for (int q = 0; q < Q; ++q) a[q] = start(q);
                        }
                        taps<k>(a, x);
                        if constexpr (k == NCK - 1) {
#pragma unroll
                            for (int q = 0; q < Q; ++q) chk = __builtin_fmaf(a[q][0], 0.f, chk);
#pragma unroll
                            for (int i = 0; i < 4; ++i) {
                                float v[Q];
#pragma unroll
                                for (int q = 0; q < Q; ++q) v[q] = a[q][i];
                                store(ro, out_at, rowb, 16 * s + i, v);
                            }
                        }
                    }
                });
                __builtin_amdgcn_sched_barrier(0);
            });
            if (__builtin_amdgcn_ballot_w64(active && !__builtin_isfinite(chk)) != 0) redo = (1u << NSTEP) - 1;
        } else {
#pragma nounroll
            for (int s = 0; s < NSTEP; ++s) {
                const MfmaBits bits = window_bits(wp, s);
                const char* sp = lp + 16 * s * kMfmaCb;
                int i0 = 0;
                do {
                    int lo, hi;
                    mfma_row_bounds(bits, TP::FRONT + (i0 < 4 ? i0 : 3), lo, hi);
                    const MfmaBits in = mfma_row_mask(lo, hi);
                    // window rows that some lane's pass takes, and those that every lane's takes (lanes of a column hold the same):
                    // a chunk that none takes is skipped, one that all take whole needs no mask
                    uint64_t some, every;
                    mfma_columns(in, some, every);
                    f32x4 acc[Q];
#pragma unroll
                    for (int q = 0; q < Q; ++q) acc[q] = start(q);
                    MfmaRaw raw;
                    mfma_read(sp + off[0], raw);
                    static_for<NCK>([&](auto k_c) __attribute__((always_inline)) {
                        constexpr int k = decltype(k_c)::value;
                        const MfmaRaw cur = raw;
                        if constexpr (k + 1 < NCK)
                            mfma_read<(k + 1 == NCK - 1 ? TP::LASTROWS : 4)>(sp + off[(k + 1) & 3] + (k + 1) * 4 * kMfmaCb, raw);
                        if ((some >> (4 * k)) & 15) {
                            MfmaChunk x;
                            mfma_pack(cur, x);
                            if (((every >> (4 * k)) & 15) != 15) {
                                const uint32_t b4 = 4 * k < 32 ? in.lo >> (4 * k & 31) : in.hi >> (4 * k & 31);
                                const uint32_t m0 = __builtin_amdgcn_perm((uint32_t)((int)(b4 << 30) >> 31), (uint32_t)((int)(b4 << 31) >> 31), 0x05040100);
                                const uint32_t m1 = __builtin_amdgcn_perm((uint32_t)((int)(b4 << 28) >> 31), (uint32_t)((int)(b4 << 29) >> 31), 0x05040100);
#pragma unroll
                                for (int q = 0; q < Q; ++q) { x.b[q].x &= m0; x.b[q].y &= m1; }
                            }
                            taps<k>(acc, x);
                        }
                        __builtin_amdgcn_sched_barrier(0);
                    });
                    const int i1 = hi - TP::FRONT < 4 ? hi - TP::FRONT : 4;
                    float chk = 0.f;
#pragma unroll
                    for (int q = 0; q < Q; ++q) chk = __builtin_fmaf(acc[q][0], 0.f, chk);
                    if (__builtin_amdgcn_ballot_w64(active && !__builtin_isfinite(chk)) != 0) { redo |= 1u << s; break; }
                    const int range = __builtin_amdgcn_ds_bpermute(swap, i0 | i1 << 8);     // rows of the pass in the lane that stores them
#pragma unroll
                    for (int i = 0; i < 4; ++i) {
                        float v[Q];
#pragma unroll
                        for (int q = 0; q < Q; ++q) v[q] = acc[q][i];
                        store(ro, i >= (range & 255) && i < (range >> 8) ? out_at : kMfmaNoStore, rowb, 16 * s + i, v);
                    }
                    i0 = i0 < 4 ? i1 : 4;
                } while (__builtin_amdgcn_ballot_w64(i0 < 4) != 0);
            }
        }
        // one product at a time, only the products that belong to the row
#pragma nounroll
        for (; redo != 0; redo &= redo - 1) {
            const int s = __builtin_ctz(redo);
            exact_step(lp + 16 * s * kMfmaCb, window_bits(wp, s), ro, rowb, s);
        }
    }

    // The 16 output rows of a step one product at a time, only the products that belong to them.
    __device__ __forceinline__ void exact_step(const char* sp, MfmaBits bits, rsrc_t ro, int rowb, int s) const {
        const int koff = w_tap_off(w_flags), kw = TP::KP - 2 * koff;
        const bool res = (w_flags & W_RESIDUAL) != 0;
#pragma nounroll
        for (int i = 0; i < 4; ++i) {
            int lo, hi;
            mfma_row_bounds(bits, TP::FRONT + i, lo, hi);
            float v[Q];
#pragma unroll
            for (int q = 0; q < Q; ++q) v[q] = bias[q];
#pragma nounroll
            for (int m = koff; m < koff + kw; ++m) {
                const int p = TP::FRONT + i - TP::PP + m;       // window row of tap m
                if (p < lo || p >= hi || !active) continue;
                // (the lane's row 4 n + p of the step: its piece is where the chunk of that row has it)
                const char* a = sp + (off[0] ^ (((((p >> 2) + n) & 3) ^ (n & 3)) << 6)) + p * kMfmaCb;
                RowVec<true, Q> x;
                float f[Q];
                x.load(a);
                x.to_f32(f);
#pragma unroll
                for (int q = 0; q < Q; ++q)
                    v[q] = __builtin_fmaf(mfma_weight<TP::KP, FLIP>(w, w_flags, c0 + q, m, res), f[q], v[q]);
            }
            store(ro, out_at, rowb, 16 * s + i, v);
        }
    }
};

// Forward: 64-row tiles, 8 compute waves (4 wave-columns x 2 groups of 32 rows), 3 loader waves and one that finds the
// boundaries of the next tile; two tile buffers.
// Bound by HBM from 64 row tiles on: T=131072, C=2048, 31 taps, one sequence 184 us (5.8 TB/s), 248 on the vector ALU. More rows
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
    static constexpr int LDS_BYTES = TAB_AT + kMfmaCh * TP::WSTR * 4;
    static_assert(LDS_BYTES <= kLdsBytes, "fits the LDS");
    static_assert((NROWS + 31) / 32 + 2 <= kMfmaWords, "lanes read two words past the one of their window's first row");
};

template <int KT, bool RES>
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
                mfma_stage<SH::NROWS, SH::NWL, false, kLoadAuxOnceFwd>(x, lds_raw + par * SH::BUF_BYTES, t0 - TP::FRONT, T, (size_t)rowb,
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
    mfma_fill_weights<KT, false>(tab, w, g.w_flags, cb * kMfmaCh, nch, (int)threadIdx.x, SH::NWC * 64);
    lds_barrier();
    MfmaConv<KT, SH::RW / 16, false, RES> conv;
    conv.init(tab, w, g.w_flags, bias, wc, lane, cb * kMfmaCh, nch, rowb);
    for (int it = 0; it < ntl; ++it) {
        lds_barrier();
        const int tf = lds_tile_row0(g, it, q, R) + r0;
        if (tf < T)
            conv.rows(lds_raw + (it & 1) * SH::BUF_BYTES + r0 * kMfmaCb, words + (it & 1) * kMfmaWords, r0,
                      mfma_out_rsrc(y, tf, T - tf < SH::RW ? T - tf : SH::RW, rowb), rowb);
        q = lds_next_slot(g, q);
    }
}

}  // namespace nplm
