// C ABI of libnplm_dwconv (see include/nplm_dwconv.h): argument checks, launch planning and
// dispatch to the per-K launchers. Host code only; the kernels live in dwconv_kernels.h and
// dwconv_lds_kernels.h.
//
// The entry points stand where a conv module's forward/backward would sit on the reference's
// packed path (src/nanoplm/pretraining/models/modern_bert/modeling.py:421-439; backward driven by
// src/nanoplm/pretraining/pure_pipeline.py:739-742). The reference holds no such op to replace.
#include <hip/hip_runtime.h>

#include <limits.h>
#include <stdlib.h>

#include <atomic>
#include <vector>

#include "../../include/nplm_dwconv.h"
#include "dwconv_internal.h"

// Scratch of nplm_dwconv_bwd_static: the dw/db partial-sum slabs of one backward call, for callers that
// cannot hand in a workspace they allocated. One copy per GPU, held until the process ends. Host code
// never uses this name as an address: static_scratch_for_current_device() asks the runtime where the
// current device's copy lives and the kernels are given that pointer.
static __device__ __align__(256) unsigned char scratch[NPLM_DWCONV_STATIC_SCRATCH_BYTES];

namespace nplm {
namespace {

constexpr int kVersion = 102;   // 0.1.2: odd kernel sizes up to 31 without kernels of their own run as the next built size

// MI355X: 256 CUs in 8 XCDs. Geometry is a pure function of the problem size so that the
// reduction order (and with it every output bit) is reproducible.
constexpr int kNumCU = 256;
constexpr int kNumXCD = 8;
constexpr long long kMaxRows = (long long)INT_MAX - (1 << 20);   // row arithmetic is int32 with tile-sized slack
constexpr int kMaxTileRows = 1 << 16;
constexpr size_t kSlabBudgetBytes = 16u << 20;   // cap on dw/db partials (written once, read once)

constexpr bool specialised_k(int K) { return K == 3 || K == 5 || K == 7 || K == 9 || K == 15 || K == 31; }
// The kernel size a plain conv of K taps runs as: an odd K below 31 without kernels of its own takes the next size that
// has them, with (exec - K) / 2 zero taps on either side (W_TAP_OFF_SHIFT); the caller's weight and dw rows stay K long.
// Runtime-K kernels (one wave per row) remain for K > 31.
constexpr int exec_kernel_size(int K) { return K > 31 || specialised_k(K) ? K : K < 3 ? 3 : K < 15 ? 15 : 31; }

// The number of taps the LDS-staged and role-split kernels run such a size with: they are built for 11 and 21 taps as well,
// so K = 11 and K = 17 .. 21 leave out zero taps (and halo rows) of the 15 and 31 that plans and workspaces are made for.
// The role-split kernels' tiles and token blocks and the order of every sum are those of exec_kernel_size(K); a slab holds
// lds_taps(K) + 1 rows and fits its place.
// Measured at C=2048, T=65536, log-normal lengths, bf16, whole calls, running as 15 / 31 -> this (us): K=11 forward 111 -> 93,
// with backward 304 -> 262; K=17 130 -> 104, 379 -> 313; K=21 133 -> 108, 379 -> 318; gated K=11 191 -> 185, 457 -> 427, K=21
// 226 -> 199, 588 -> 504; fp32 forward and backward 455 -> 446 (K=11), 544 -> 492 (K=21). Forms of 13 and 25 taps, which are not
// built, would give (forward / backward alone, same sizes): K=13 107 / 170 -> 93 / 163, gated 185 / 264 -> 180 / 258, fp32 179 / 271
// -> 173 / 269; K=23 and 25 136 / 249 -> 118 / 221, gated 229 / 361 -> 210 / 327, fp32 205 / 340 -> 207 / 305.
constexpr int lds_taps(int K) { return K == 11 ? 11 : K >= 17 && K <= 21 ? 21 : exec_kernel_size(K); }

// A role-split call is planned (tiles, column blocks) with the shape of exec_kernel_size(K) and launched with the kernel's own
// shape at lds_taps(K): they have to be one shape for every K, else rows would be left out or computed twice.
constexpr bool split_plans_fit_their_kernels() {
    for (int K = 1; K <= 31; K += 2)
        for (int v = 0; v < 4; ++v) {
            const bool fwd = v & 1, bf16 = v & 2;
            const int plan = exec_kernel_size(K), run = lds_taps(K);
            if (!lds_split_kernel_size(plan)) continue;
            if (lds_split_shape(fwd, bf16, plan) != lds_split_shape(fwd, bf16, run)) return false;
            if (lds_split_gated_shape(bf16, plan) != lds_split_gated_shape(bf16, run)) return false;
            if (lds_split_gated_fwd_shape(bf16, plan) != lds_split_gated_fwd_shape(bf16, run)) return false;
        }
    return true;
}
static_assert(split_plans_fit_their_kernels(), "a role-split plan and the kernel it launches differ in shape");

int pow2_floor(int v) { int p = 1; while (p * 2 <= v) p *= 2; return p; }
int ceil_div(long long a, long long b) { return (int)((a + b - 1) / b); }

struct Plan {
    bool generic;
    int vec, unroll, maxt;
    int R, ntiles, ncols, nwc, bw, bt, ncb, nbt, remap;
};

int default_vec(bool bwd, bool bf16, int K) { return max_vec(bwd, bf16, K); }

// Largest VEC <= cap that divides C, keeps every row slice aligned, and still spreads a row over a
// whole wave (C / VEC >= 64) unless nothing smaller is left.
int pick_vec(bool bf16, int C, int cap, uintptr_t align_bits) {
    const int E = bf16 ? 2 : 4;
    const int vmax = bf16 ? 8 : 4;
    for (int v = (cap < vmax ? cap : vmax); v > 1; v >>= 1) {
        if (C % v) continue;
        if (align_bits % (uintptr_t)(v * E)) continue;
        if (C / v < 64) continue;
        return v;
    }
    return 1;
}

// tune may be null. Returns 0 or a negative argument error.
int make_plan(bool bwd, bool bf16, long long T, int C, int K, uintptr_t align_bits,
              const nplm_dwconv_tuning* tune, Plan* out) {
    Plan p{};
    nplm_dwconv_tuning z{};
    if (!tune) tune = &z;
    p.generic = !specialised_k(K);
    const int vcap = tune->vec > 0 ? tune->vec : default_vec(bwd, bf16, K);
    p.vec = p.generic ? 1 : pick_vec(bf16, C, vcap, align_bits);
    if (tune->vec > 0 && p.vec != tune->vec) return -NPLM_DWCONV_ETUNING;
    p.unroll = tune->unroll > 0 ? tune->unroll : default_unroll(bwd, K, p.vec);
    p.maxt = tune->maxt > 0 ? tune->maxt : default_maxt(bwd, K, p.vec);
    if (p.maxt < 64 || p.maxt > 1024 || p.maxt % 64) return -NPLM_DWCONV_ETUNING;
    // long kernels re-read K-1 halo rows per tile: longer tiles (measured at K=31: 256 rows beat 64 by 25 %)
    int R = tune->tile_rows > 0 ? tune->tile_rows : (K >= 15 ? 256 : (bwd ? 32 : 64));
    if (R > kMaxTileRows || p.unroll > 64) return -NPLM_DWCONV_ETUNING;
    R = ceil_div(R, p.unroll) * p.unroll;
    // row offsets inside a tile are 32-bit byte offsets
    const long long row_bytes = (long long)C * (bf16 ? 2 : 4);
    while ((long long)(R + K) * row_bytes >= INT_MAX && R > p.unroll) R = ceil_div(R / 2, p.unroll) * p.unroll;
    if ((long long)(R + K) * row_bytes >= INT_MAX) return -NPLM_DWCONV_ESHAPE;
    p.R = R;
    p.ntiles = ceil_div(T, R);
    p.ncols = C / p.vec;
    p.nwc = ceil_div(p.ncols, 64);
    const int wpb_max = p.maxt / 64;
    p.bt = tune->bt > 0 ? tune->bt : (bwd ? 4 : 2);
    if (p.bt > wpb_max) p.bt = wpb_max;
    p.bw = tune->bw > 0 ? tune->bw : pow2_floor(p.nwc);
    if (p.bw > wpb_max / p.bt) p.bw = wpb_max / p.bt;
    if (p.bw < 1 || (p.bw & (p.bw - 1))) return -NPLM_DWCONV_ETUNING;
    p.ncb = ceil_div(p.nwc, p.bw);
    // waves the grid is sized for: 2 per SIMD keep the HBM-bound kernels streaming; the long kernels
    // are ALU-bound and want every wave their registers allow (K=31 backward at C=2048: 848 -> 657 us)
    const int waves_per_cu = K >= 15 ? 32 : 8;
    int nbt = tune->nbt > 0 ? tune->nbt : (kNumCU * waves_per_cu) / (p.ncb * p.bw * p.bt);
    const int nbt_useful = ceil_div(p.ntiles, p.bt);
    if (nbt > nbt_useful) nbt = nbt_useful;
    if (bwd) {
        const size_t slab = (size_t)(K + 1) * C * sizeof(float);
        const long long cap = (long long)(kSlabBudgetBytes / slab);
        if (tune->nbt <= 0 && nbt > cap) nbt = (int)cap;
    }
    if (nbt < 1) nbt = 1;
    // keep the grid a multiple of the XCD count when it is large enough: every XCD gets equal work
    if (tune->nbt <= 0 && nbt >= kNumXCD) nbt -= nbt % kNumXCD;
    p.nbt = nbt;
    p.remap = (tune->xcd_remap == 1) && ((long long)p.ncb * p.nbt) % kNumXCD == 0;
    *out = p;
    return 0;
}

Geo make_geo(const Plan& p, long long T, int C, int S, int w_flags) {
    Geo g{};
    g.T = (int32_t)T; g.C = C; g.S = S; g.w_flags = w_flags;
    g.R = p.R; g.ntiles = p.ntiles; g.ncols = p.ncols; g.nwc = p.nwc;
    g.bw = p.bw; g.bt = p.bt; g.ncb = p.ncb; g.nbt = p.nbt; g.xcd_remap = p.remap;
    return g;
}

int check_common(long long T, int C, int K, int S, int act_dtype, int w_dtype) {
    if (T < 0 || T > kMaxRows || C < 1 || S < 0) return -NPLM_DWCONV_ESHAPE;
    if ((long long)C * K > INT_MAX / 8) return -NPLM_DWCONV_ESHAPE;
    if (K < 1 || K > NPLM_DWCONV_MAX_K || (K % 2) == 0) return -NPLM_DWCONV_EKSIZE;
    if ((act_dtype != NPLM_DWCONV_F32 && act_dtype != NPLM_DWCONV_BF16) ||
        (w_dtype != NPLM_DWCONV_F32 && w_dtype != NPLM_DWCONV_BF16))
        return -NPLM_DWCONV_EDTYPE;
    return 0;
}

hipError_t launch_fwd(int K, bool bf16, const Plan& p, const ConvPtrs& a, const Geo& g, hipStream_t s) {
    const dim3 grid(p.ncb * p.nbt), block(p.bw * p.bt * 64);
    switch (K) {
        case 3: return launch_fwd_k3(bf16, p.vec, p.unroll, p.maxt, a, g, grid, block, s);
        case 5: return launch_fwd_k5(bf16, p.vec, p.unroll, p.maxt, a, g, grid, block, s);
        case 7: return launch_fwd_k7(bf16, p.vec, p.unroll, p.maxt, a, g, grid, block, s);
        case 9: return launch_fwd_k9(bf16, p.vec, p.unroll, p.maxt, a, g, grid, block, s);
        case 15: return launch_fwd_k15(bf16, p.vec, p.unroll, p.maxt, a, g, grid, block, s);
        case 31: return launch_fwd_k31(bf16, p.vec, p.unroll, p.maxt, a, g, grid, block, s);
    }
    return hipErrorInvalidConfiguration;
}
hipError_t launch_bwd(int K, bool bf16, const Plan& p, bool wdx, bool wdw, const ConvPtrs& a, const Geo& g,
                      hipStream_t s) {
    const dim3 grid(p.ncb * p.nbt), block(p.bw * p.bt * 64);
    const size_t shmem = (size_t)p.bw * p.bt * p.vec * 64 * sizeof(float);
    switch (K) {
        case 3: return launch_bwd_k3(bf16, p.vec, p.unroll, p.maxt, wdx, wdw, a, g, grid, block, shmem, s);
        case 5: return launch_bwd_k5(bf16, p.vec, p.unroll, p.maxt, wdx, wdw, a, g, grid, block, shmem, s);
        case 7: return launch_bwd_k7(bf16, p.vec, p.unroll, p.maxt, wdx, wdw, a, g, grid, block, shmem, s);
        case 9: return launch_bwd_k9(bf16, p.vec, p.unroll, p.maxt, wdx, wdw, a, g, grid, block, shmem, s);
        case 15: return launch_bwd_k15(bf16, p.vec, p.unroll, p.maxt, wdx, wdw, a, g, grid, block, shmem, s);
        case 31: return launch_bwd_k31(bf16, p.vec, p.unroll, p.maxt, wdx, wdw, a, g, grid, block, shmem, s);
    }
    return hipErrorInvalidConfiguration;
}

// ---- LDS-staged pipelined kernels ---------------------------------------------------------------
constexpr size_t kLdsBytesPerCU = 160u << 10;

struct LdsPlan {
    LdsShapeSel sh;
    int R, ntiles, ncb, nbt, xcd_group, rot_step;
};

// Whether the LDS kernels can take this problem at all (16-byte row granularity, built kernel size).
bool lds_eligible(bool bf16, long long T, int C, int K, uintptr_t align_bits) {
    const int E = bf16 ? 2 : 4;
    if (!lds_kernel_size(K) || T < 1) return false;
    if (((long long)C * E) % 16 || align_bits % 16) return false;
    return (long long)C * E >= 1024;
}

// Whether they are also the faster choice. A block owns one column block of its rows (1 KiB by default,
// see lds_shape_for) and the grid's time follows the number of column blocks, so a row that fills its
// column blocks poorly wastes lanes and loader slots. Measured on MI355X (T=131072, K=7, bf16 rows of
// 1024 .. 10240 bytes and fp32 rows of 1024 .. 8192 bytes): LDS-staged wins for a single column block
// filled to 5/8 or more; for several, the backward needs them filled to 4/5 on average, the forward only
// to 11/20; the sliding-window kernels win otherwise.
bool lds_preferred(bool bwd, bool bf16, long long T, int C, int K, uintptr_t align_bits) {
    if (!lds_eligible(bf16, T, C, K, align_bits)) return false;
    if (K > 9 && bwd) return false;        // K = 15, 31: no single-role LDS backward (it does not fit the registers); see split_eligible
    const long long E = bf16 ? 2 : 4;
    const long long row_bytes = (long long)C * E;
    const LdsShapeSel sh = lds_shape_for(bwd, bf16, K, row_bytes);
    const long long cb_bytes = (long long)sh.ncw * 64 * sh.vec * E;
    const long long ncb = ceil_div(row_bytes, cb_bytes);
    if (ncb == 1) return row_bytes * 8 >= cb_bytes * 5;
    return bwd ? row_bytes * 5 >= ncb * cb_bytes * 4 : row_bytes * 20 >= ncb * cb_bytes * 11;
}

int make_lds_plan(bool bwd, bool bf16, long long T, int C, int K, const nplm_dwconv_tuning* tune, LdsPlan* out,
                  bool gated = false) {
    LdsPlan p{};
    nplm_dwconv_tuning z{};
    if (!tune) tune = &z;
    const int E = bf16 ? 2 : 4;
    p.sh = gated ? lds_gated_shape(bwd, bf16, lds_gated_narrow((long long)C * E, K), K) : lds_shape_for(bwd, bf16, K, (long long)C * E);
    if (tune->vec > 0) p.sh.vec = tune->vec;
    if (tune->unroll > 0) p.sh.rw = tune->unroll;
    if (tune->bt > 0) p.sh.nrg = tune->bt;
    if (tune->bw > 0) p.sh.ncw = tune->bw;
    if (tune->nwl > 0) p.sh.nwl = tune->nwl;
    if (tune->nbuf > 0 && !bwd) p.sh.nbuf = tune->nbuf;
    const long long cb_bytes = (long long)p.sh.ncw * 64 * p.sh.vec * E;
    const long long row_bytes = (long long)C * E;
    p.R = p.sh.rw * p.sh.nrg;
    const size_t tile_rows = gated ? (bwd ? (size_t)(p.R + K - 1) + 2 * (size_t)p.R : 2 * (size_t)(p.R + K - 1))
                                   : (size_t)(p.R + K - 1) + (bwd ? p.R : 0);
    const size_t shmem = (size_t)p.sh.nbuf * tile_rows * cb_bytes;
    if (shmem > kLdsBytesPerCU || cb_bytes % 256) return -NPLM_DWCONV_ETUNING;
    if ((long long)(p.R + K) * row_bytes * (gated ? 2 : 1) + 2 * row_bytes >= INT_MAX) return -NPLM_DWCONV_ESHAPE;
    p.ncb = ceil_div(row_bytes, cb_bytes);
    p.ntiles = ceil_div(T, p.R);
    int nbt = tune->nbt > 0 ? tune->nbt : kNumCU / p.ncb;
    if (nbt < 1) nbt = 1;
    if (nbt > p.ntiles) nbt = p.ntiles;
    if (bwd && tune->nbt <= 0) {
        const size_t slab = (size_t)(K + 1) * C * sizeof(float);
        const long long cap = (long long)(kSlabBudgetBytes / slab);
        if (nbt > cap && cap >= 1) nbt = (int)cap;
    }
    p.nbt = nbt;
    // adjacent tiles share an XCD in runs of G (tune->xcd_remap: 0 = default 8, > 0 = G, < 0 = off)
    int G = tune->xcd_remap == 0 ? 8 : (tune->xcd_remap > 0 ? tune->xcd_remap : 0);
    const long long nblocks = (long long)p.ncb * p.nbt;
    if (G > 0 && !(nblocks % kNumXCD == 0 && (nblocks / kNumXCD) % G == 0 && p.nbt % G == 0)) G = 0;
    p.xcd_group = G;
    // per-round rotation of the tile slots: an odd step near nbt / golden ratio, so that no short period of
    // sequence boundaries keeps landing on the same token-blocks
    p.rot_step = nbt > 2 ? (int)((long long)nbt * 618 / 1000) | 1 : 0;
    if (p.rot_step >= nbt) p.rot_step = nbt - 1;
    *out = p;
    return 0;
}

LdsGeo make_lds_geo(const LdsPlan& p, long long T, int C, int S, int w_flags) {
    LdsGeo g{};
    g.T = (int32_t)T; g.C = C; g.S = S; g.w_flags = w_flags;
    g.ntiles = p.ntiles; g.ncb = p.ncb; g.nbt = p.nbt; g.xcd_group = p.xcd_group; g.rot_step = p.rot_step;
    return g;
}

hipError_t launch_fwd_lds(int K, const LdsPlan& p, const ConvPtrs& a, const LdsGeo& g, hipStream_t s) {
    const dim3 grid(p.ncb * p.nbt);
    switch (K) {
        case 3: return launch_fwd_lds_k3(p.sh, a, g, grid, s);
        case 5: return launch_fwd_lds_k5(p.sh, a, g, grid, s);
        case 7: return launch_fwd_lds_k7(p.sh, a, g, grid, s);
        case 9: return launch_fwd_lds_k9(p.sh, a, g, grid, s);
        case 11: return launch_fwd_lds_k11(p.sh, a, g, grid, s);
        case 15: return launch_fwd_lds_k15(p.sh, a, g, grid, s);
        case 31: return launch_fwd_lds_k31(p.sh, a, g, grid, s);
    }
    return hipErrorInvalidConfiguration;
}
hipError_t launch_bwd_lds(int K, const LdsPlan& p, bool wdx, bool wdw, const ConvPtrs& a, const LdsGeo& g,
                          hipStream_t s) {
    const dim3 grid(p.ncb * p.nbt);
    switch (K) {
        case 3: return launch_bwd_lds_k3(p.sh, wdx, wdw, a, g, grid, s);
        case 5: return launch_bwd_lds_k5(p.sh, wdx, wdw, a, g, grid, s);
        case 7: return launch_bwd_lds_k7(p.sh, wdx, wdw, a, g, grid, s);
        case 9: return launch_bwd_lds_k9(p.sh, wdx, wdw, a, g, grid, s);
        case 15: return launch_bwd_lds_k15(p.sh, wdx, wdw, a, g, grid, s);
        case 31: return launch_bwd_lds_k31(p.sh, wdx, wdw, a, g, grid, s);
    }
    return hipErrorInvalidConfiguration;
}

// ---- role-split LDS-staged kernels at K = 31 and 15 (dwconv_lds_split_kernels.h), run with lds_taps() taps ---
#define NPLM_LAUNCH_SPLIT(NAME)                                                                          \
    hipError_t NAME(int taps, bool bf16, const ConvPtrs& a, const LdsGeo& g, dim3 grid, hipStream_t s) { \
        switch (taps) {                                                                                  \
            case 11: return NAME##_k11(bf16, a, g, grid, s);                                             \
            case 15: return NAME##_k15(bf16, a, g, grid, s);                                             \
            case 21: return NAME##_k21(bf16, a, g, grid, s);                                             \
            case 31: return NAME##_k31(bf16, a, g, grid, s);                                             \
        }                                                                                                \
        return hipErrorInvalidConfiguration;                                                             \
    }
NPLM_LAUNCH_SPLIT(launch_bwd_split)
NPLM_LAUNCH_SPLIT(launch_fwd_split_gated)
NPLM_LAUNCH_SPLIT(launch_bwd_split_gated)
#undef NPLM_LAUNCH_SPLIT
// The library takes a plain forward of up to 15 taps to the matrix cores or to the kernels with loader waves (choose_algo());
// of the role-split ones only the size that shape overrides may name is built, and calls of 11 taps run there with 15.
hipError_t launch_fwd_split(int taps, bool bf16, const ConvPtrs& a, const LdsGeo& g, dim3 grid, hipStream_t s) {
    switch (taps) {
        case 15: return launch_fwd_split_k15(bf16, a, g, grid, s);
        case 21: return launch_fwd_split_k21(bf16, a, g, grid, s);
        case 31: return launch_fwd_split_k31(bf16, a, g, grid, s);
    }
    return hipErrorInvalidConfiguration;
}

#define NPLM_LAUNCH_MFMA(NAME)                                                                \
    hipError_t NAME(int taps, const ConvPtrs& a, const LdsGeo& g, dim3 grid, hipStream_t s) { \
        switch (taps) {                                                                       \
            case 11: return NAME##_k11(a, g, grid, s);                                        \
            case 15: return NAME##_k15(a, g, grid, s);                                        \
            case 21: return NAME##_k21(a, g, grid, s);                                        \
            case 31: return NAME##_k31(a, g, grid, s);                                        \
        }                                                                                     \
        return hipErrorInvalidConfiguration;                                                  \
    }
NPLM_LAUNCH_MFMA(launch_fwd_mfma)
NPLM_LAUNCH_MFMA(launch_bwd_mfma)
#undef NPLM_LAUNCH_MFMA

bool split_eligible(bool bf16, long long T, int C, int K, uintptr_t align_bits) {
    const int E = bf16 ? 2 : 4;
    if (!lds_split_kernel_size(K) || T < 1) return false;
    if (((long long)C * E) % 16 || align_bits % 16) return false;
    const SplitShapeSel sh = lds_split_shape(false, bf16, K);      // the column block is the same in both passes
    return (long long)C * E >= (long long)sh.ncw * 64 * sh.vec * E;
}
// The matrix-core kernels (dwconv_mfma_kernels.h) have the column blocks of the role-split ones in bf16.
bool mfma_eligible(bool bf16, bool w_bf16, long long T, int C, int K, uintptr_t align_bits) {
    return bf16 && w_bf16 && split_eligible(bf16, T, C, K, align_bits);
}
constexpr long long kMfmaMinRows = 4096;
// The library's own choice of them: their tiles of 64 rows reach make_split_plan()'s limit on a tile's bytes in rows that the
// shorter tiles of other kernels still take (C beyond 13 million, gated 5.5 million, bf16); those rows keep the others.
bool mfma_tile_fits(int C, int K, bool gated) {
    const int tile_rows = gated ? kMfmaGatedRows : kMfmaFwdRows;
    return ((long long)(tile_rows + K) * (gated ? 2 : 1) + 2) * C * 2 < INT_MAX;
}
// Output rows that do not begin on whole cache lines (128 bytes). A wave of the matrix-core kernels stores 128 bytes of a row
// (gated 64) at a time where the others store 256 or 512; off the lines' grid each piece is two parts of lines, which other waves
// complete later. mfma_lines() lets them meet in the L2; in outputs too large for it and the Infinity Cache many reach HBM as parts all
// the same, and up to 15 taps the others are faster there. Measured with lengths of 20 to 512 (backward at 11 and 21 taps: 700) residues, us,
// matrix cores / the best of the others, by MiB of output:
//   forward, 11 taps: T=131072 C=1000 (250 MiB) 125 / 103, C=1160 (290) 152 / 147, C=2008 (502) 243 / 216; T=65536 C=1800 (225) 110 / 107,
//     C=1160 (145) 69 / 80, C=1000 (125) 56 / 61; T=131072 C=648 (162) 83 / 98; 15 taps the same to 3 %. Rows that fill the others'
//     1 KiB column blocks to less than 3/5 stay: C=584 (0.57) T=131072 77 / 96.
//   backward, 11 / 15 taps: T=131072 C=2008 (502) 424 / 359, 427 / 369; C=1160 (290) 235 / 212, 242 / 227; C=1032 (258) 200 / 213, 210 / 219;
//     C=648 (162) 118 / 129, 129 / 139; T=16384 C=1000 (31) 34 / 38, 37 / 41.
//   gated backward, 31 taps (stores with `nt` always): T=131072 C=2008 (502) 1015 / 778, C=1000 507 / 384; T=65536 C=584 (73) 151 / 145;
//     T=16384 C=1000 (31) 64 / 69, C=648 (20) 51 / 52, C=520 (16) 45 / 51.
// 31 taps save more FMAs than that costs (T=131072 C=2040 forward 254 / 331, backward 430 / 509), and so do 21 forward (259 / 303); 21
// backward come out even (C=2008 423 / 394, C=1160 257 / 247, C=1800 378 / 383, T=98304 C=1160 179 / 190) and stay.
bool mfma_lines_ok(bool bwd, bool gated, long long T, int C, int K, int taps, uintptr_t out_bits) {
    const long long row_bytes = 2LL * C;
    if (((uintptr_t)row_bytes | out_bits) % 128 == 0) return true;
    const long long mib = T * row_bytes >> 20;
    if (gated) return mib < 30;
    if (taps > 15) return true;
    if (bwd) return mib < 270;
    return mib < 200 || !lds_preferred(false, true, T, C, K, 0) ||
           row_bytes * 5 < ceil_div(row_bytes, kLdsDefaultCb) * 3LL * kLdsDefaultCb;
}
// A backward tile with sequence boundaries makes one pass over its rows per sequence for dw, so the gain goes with the length
// of the sequences. Measured at T=131072, us, matrix cores against role-split, for lengths of 20 to 128 residues (mean 75), 20
// to 512 (mean 263), log-normal (mean 333), one sequence:
//   K=31, C=1024   257/279   198/257   188/251   139/240      (C=2048: 488/541, 346/488, -, 274/467; T=16384, C=512: 33/39, 31/37,
//                                                              32/38, 24/35)
//   K=15, C=1024   200/193   156/171   152/172   132/162      (T=16384, C=512: 25/28, 24/25, 23/25, 20/23; T=4096: 17/20, 16/18, 16/18, 16/16)
//   K=21, C=1024   245/224   180/202   183/205   135/188      (T=65536, C=512: 77/73, 64/63, 58/61, 46/57)
//   K=11, C=1024   198/175   159/157   159/149   136/146
// About 24 rows a sequence: K=31 671/628, 32: 613/608 (C=2048). 21 taps pay for the 32 lags of the plan, which short
// sequences do not leave room for (from 200 rows on they would gain where C = 1024, not where C = 512); 11 taps are bound by HBM on the
// vector ALU too. Sequences of 522, 705, 1928 rows on average: K=21 164/195, 157/191, 144/189; K=11 151/150, 151/149, 142/145.
// S counts empty sequences too, which the device alone could tell apart: a cu with a long tail of them is taken for shorter ones.
bool mfma_bwd_preferred(long long T, int taps, int S) {
    const int rows = taps == 31 ? 32 : taps == 15 ? 64 : 512;
    return T >= (long long)S * rows;
}
// Steps (backward: tiles) of 64 rows that a block of the gated matrix-core kernels gets.
long long mfma_gated_steps_of_a_block(long long T, int C) {
    const int ncb = ceil_div(2LL * C, kMfmaGatedCb), nbt = ncb < kNumCU ? kNumCU / ncb : 1;
    return ceil_div(ceil_div(T, kMfmaGatedRows), nbt);
}
// The gated backward with dz on the matrix cores: 31 taps. Measured, us, against role-split, for lengths of 20 to 128 residues
// (mean 75), 20 to 512 (263), log-normal (333), short and long mixed (193), one sequence:
//   T=131072, C=2048   793/793   683/737   676/737   698/750   624/705         T=32768, C=1024   112/114   96/106   96/104   -   88/103
//   T=16384, C=1024    62/70     53/68     -         -         51/64           T=8192, C=512     26/37     25/35     -        -        23/33
// A wave of dw makes one pass over its rows whatever begins there, but masked row by row: short sequences cost it more than the
// role-split kernel's roles, which share the loss, once a call is longer than its first tiles. 15 taps (T=131072, C=1024: 302/264,
// T=4096: 19/22) and 21 (306/299) have too few FMAs to save. Calls of up to 16384 rows take it whatever begins in them (C=1024):
//   T=16384   1 row 143/226   4 94/108   16 86/81   32 76/78   75 62/70       T=4096   1 row 45/79   8 32/42   32 29/38   75 26/36
// and so do the shortest: T=2048, C=768 1 row 28/47, 16 22/29, 75 19/27, 300 18/26, one sequence 17/24; T=20, C=512 15/20. Below 4096 rows
// only where a block has up to four tiles of 64 rows, which goes by C; with more of them short sequences cost what they do in long calls:
//   rows a sequence   4         8        16       24       32       48       75       300
//   T=2048, C=4096 (4 tiles)    58/74    54/63    53/57    55/57    47/54    44/55    41/51    38/49
//   T=4000, C=2560 (6)          -        70/61    70/57    67/57    61/56    55/53    -        -
//   T=4000, C=4096 (8)          97/108   91/88    94/81    85/79    76/78    71/76    64/74    57/69
//   T=4000, C=8192 (16)         -        168/145  163/132  154/131  144/131  123/124  -        -
bool mfma_gated_bwd_preferred(long long T, int C, int taps, int S) {
    if (taps != 31) return false;
    if (T >= kMfmaMinRows) return T <= 16384 || T >= 192ll * S;
    return mfma_gated_steps_of_a_block(T, C) <= 4 || T < 5ll * S || T >= 64ll * S;
}
// The gated forward on the matrix cores: steps of 64 rows in a run, which a block walks down without staging or gating a halo again.
// All of a block's runs are of one length, the longest that deals the call out evenly (T=65536, C=1152, 15 taps: runs of 16 steps,
// three rounds for two and a bit, 115 us, of 13 95).
int mfma_gated_fwd_steps(long long T, int C) {
    const long long per_block = mfma_gated_steps_of_a_block(T, C);
    return ceil_div(per_block, ceil_div(per_block, kMfmaGatedSteps));
}
// Which gated forwards take it, measured by the mean rows of a sequence, us, role-split / matrix cores:
//   31 taps              16 rows      32           75           300          one sequence
//   T=131072, C=2048     639 / 692    581 / 561    488 / 476    432 / 387    405 / 361
//   T=131072, C=1152     377 / 410    344 / 334    280 / 278    255 / 225    239 / 208
//   T=32768, C=768       86 / 83      82 / 68      69 / 58      57 / 43      54 / 38
//   T=16384, C=1024      59 / 56      -            49 / 40      44 / 33      40 / 31
//   T=8192, C=512        27 / 22      -            26 / 18      24 / 16      23 / 14
//   T=2048, C=768        26 / 15      -            26 / 13      24 / 12      23 / 12     (one of the role-split tiles of 128 rows takes 22)
//   T=20, C=512          22 / 12      -            -            -            21 / 12
//   15 taps, T=16384, C=768 44 / 40, -, 34 / 32, 31 / 25, 30 / 22; T=65536, C=1024 139 / 148, 122 / 123, 100 / 105, 90 / 96, 83 / 93
//   (C=768 115 / 120, 96 / 99, 83 / 81, 75 / 68, 68 / 63; T=131072, C=2048 517 / 551, 441 / 457, 376 / 384, 358 / 335, 353 / 333)
//   21 taps as 31, 11 as 15: T=2048, C=768 (21 taps) 26 / 15, -, 20 / 13, 19 / 13, 19 / 12;
//   T=4000, C=2048 31 / 34, -, 27 / 26, 25 / 23, 24 / 21; T=16384, C=1152 58 / 66, 54 / 55, 45 / 46, 40 / 37, 39 / 32;
//   C=1024 41 / 45, 37 / 40, 32 / 34, 31 / 28, 29 / 25.
// A boundary costs the consumers a sweep of their own; short calls gain on every mix because a run begins without a full tile of halo.
// Where 11 taps break even (between 75 and 300 rows) 15 would still gain a tenth, but 11 taps and the same taps padded to 15 have to
// give the same bits, so both go by the one line.
// Up to 2048 rows what counts is how many steps a block gets, which goes by C too. With one (two at 21 taps) a block is done before the
// role-split one has staged its tile; with more it is not, but for sequences so short that the others' masked passes take over:
//   rows a sequence       4            8            16           24           75           150          300          one
//   11 taps, 2 steps: T=2048, C=1536    18.1 / 17.1  16.4 / 16.8  15.0 / 16.7  14.8 / 16.7  13.4 / 14.2  13.2 / 14.1  12.7 / 12.8  11.7 / 11.8
//   3: T=2048, C=3072     29.3 / 26.5  24.8 / 26.1  23.1 / 26.0  21.3 / 25.4  18.8 / 21.3  17.9 / 19.2  17.6 / 18.5  16.4 / 16.5
//   4: T=2048, C=4096     30.8 / 27.9  25.7 / 28.1  23.5 / 28.4  22.5 / 26.7  20.2 / 22.5  19.9 / 21.3  19.2 / 19.9  18.4 / 19.1
//   15 taps, 2: T=2048, C=1536          20.5 / 16.9  18.5 / 16.8  17.5 / 16.7  16.8 / 16.4  15.6 / 14.2  15.4 / 13.2  15.1 / 13.0  13.9 / 11.8
//   4: T=2048, C=4096     34.4 / 29.4  28.7 / 28.9  26.8 / 28.9  25.7 / 26.4  23.1 / 23.7  22.5 / 21.4  22.2 / 21.0  20.9 / 19.4
//   21 taps, 2: T=1536, C=2048          25.3 / 20.1  22.8 / 20.0  21.3 / 20.7  21.3 / 19.9  19.8 / 16.5  19.1 / 16.2  18.7 / 14.6  17.8 / 13.5
//   4: T=2048, C=4096     40.0 / 34.6  33.8 / 33.6  30.8 / 36.2  30.0 / 33.1  27.1 / 27.5  26.8 / 25.3  26.0 / 24.9  24.7 / 22.5
// 31 taps of up to 16384 rows gain everywhere but at 16 rows a sequence (T=16384, C=4096 4 rows 263 / 170, 8 203 / 171, 16 173 / 184, 24 164 / 163).
// Rows of partial cache lines change none of this: a wave stores 64 bytes of a row without `nt`, and the pieces meet in the L2. 31 taps,
// T=131072, 75 rows, 300 rows, one sequence: C=1000 253 / 251, 234 / 214, 226 / 208; C=1160 315 / 313, 287 / 262, 277 / 245; C=2008 489 / 496,
// 450 / 418, 436 / 407; T=16384, C=520 40 / 33, 38 / 28, 34 / 25; C=1160 62 / 52, 58 / 43, 55 / 40; 15 taps, T=16384, 300 rows, one sequence C=1000
// 39 / 33, 37 / 31; C=2008 63 / 57, 61 / 57; 11 taps C=2008 60 / 57, 59 / 56.
bool mfma_gated_fwd_preferred(long long T, int C, int taps, int S) {
    if (taps == 31) return T <= 16384 || T >= 32ll * S;
    if (T > 2048) return T <= 16384 && T >= 192ll * S;
    const long long steps = mfma_gated_steps_of_a_block(T, C);
    return steps <= (taps == 21 ? 2 : 1) || T < 6ll * S || (T >= 192ll * S && (taps == 21 || steps == 2));
}
int make_split_plan(bool fwd, bool bf16, long long T, int C, int K, const nplm_dwconv_tuning* tune, LdsPlan* out,
                    bool gated = false, int tile_rows = 0, int block_bytes = 0) {
    LdsPlan p{};
    nplm_dwconv_tuning z{};
    if (!tune) tune = &z;
    const int E = bf16 ? 2 : 4;
    const SplitShapeSel sh = !gated ? lds_split_shape(fwd, bf16, K) : fwd ? lds_split_gated_fwd_shape(bf16, K) : lds_split_gated_shape(bf16, K);
    const long long cb_bytes = block_bytes ? block_bytes : (long long)sh.ncw * 64 * sh.vec * E;
    const long long row_bytes = (long long)C * E;
    p.R = tile_rows ? tile_rows : sh.rw * sh.nrg;
    if ((long long)(p.R + K) * row_bytes * (gated ? 2 : 1) + 2 * row_bytes >= INT_MAX) return -NPLM_DWCONV_ESHAPE;
    p.ncb = ceil_div(row_bytes, cb_bytes);
    p.ntiles = ceil_div(T, p.R);
    int nbt = tune->nbt > 0 ? tune->nbt : kNumCU / p.ncb;     // one block of 16 waves per CU
    if (nbt < 1) nbt = 1;
    if (nbt > p.ntiles) nbt = p.ntiles;
    if (tune->nbt <= 0 && !fwd) {
        const long long cap = (long long)(kSlabBudgetBytes / ((size_t)(K + 1) * C * sizeof(float)));
        if (nbt > cap && cap >= 1) nbt = (int)cap;
    }
    p.nbt = nbt;
    int G = tune->xcd_remap == 0 ? 8 : (tune->xcd_remap > 0 ? tune->xcd_remap : 0);
    const long long nblocks = (long long)p.ncb * p.nbt;
    if (G > 0 && !(nblocks % kNumXCD == 0 && (nblocks / kNumXCD) % G == 0 && p.nbt % G == 0)) G = 0;
    p.xcd_group = G;
    p.rot_step = nbt > 2 ? (int)((long long)nbt * 618 / 1000) | 1 : 0;
    if (p.rot_step >= nbt) p.rot_step = nbt - 1;
    *out = p;
    return 0;
}

// algo requested by the caller (0 = library's choice) -> 1 sliding-window, 2 LDS-staged, 3 role-split LDS-staged, 4 matrix
// cores. Measured on MI355X, bf16, T=131072:
//   K=7, C=1024: both passes are fastest LDS-staged (the chip sweeps one compact window of rows with every load of a
//     tile issued at once).
//   11 to 31 taps, bf16 weights too, forward: matrix cores. On the vector ALU these sizes are bound by their FMAs (K=31, one
//     sequence: 248 us where a copy of the same bytes takes 208); in us, matrix cores against the best of the others:
//     K=31 C=2048: 189 against 256 (log-normal lengths), 184 / 247 (one sequence), 232 / 293 (20 to 128 residues);
//     K=21 C=1024: 88 / 107; K=15: 182 / 191 at C=2048, 85 / 91 at C=1024; K=11 C=1024: 85 / 93;
//     T=16384 C=1024: 21.2 / 31.4 at K=31, 16.0 / 20.0 at K=11. From kMfmaMinRows rows on: below, every block has a tile
//     or two and what is measured is the launch (2048 rows, C=1024: K=31 11.8 / 12.5, K=15 10.0 / 10.2; 600 rows, C=512:
//     12.2 / 11.8), while the others' sums are those of the sliding-window kernels bit for bit.
//     Whatever the length of the sequences (lengths spread by half around the mean, T=65536, C=1024, K=31: 4 rows 92 / 211, 16 92 / 115, 24
//     87 / 108, 48 72 / 101; K=21: 16 81 / 99, 32 71 / 89; K=11: 16 69 / 94, 75 54 / 71) and also where rows fill their column blocks poorly (T=32768, K=31: C=264
//     25 / 35, C=520 33 / 44; K=11: 18 / 22, 25 / 29).
//     fp32 weights would take three bf16 terms each: 280 us against 265 (K=31, C=2048), so they stay on the vector ALU.
//   the same calls backward: matrix cores where a sequence has enough rows (mfma_bwd_preferred()).
//   Very large outputs whose rows are not whole cache lines keep the other kernels (mfma_lines_ok()).
//   K=31 and K=15 backward of fp32 weights (ALU-bound; one wave cannot hold the fused backward's registers): the role-split
//     kernel, when every output is asked for - C=2048, K=31: 510 us against 720 sliding-window on the log-normal length mix;
//     K=15: 345 against 385 (C=1024: 177 against 205). A backward asked for dx alone or dw/db alone takes the
//     sliding-window kernel, like everything the LDS kernels are not built for (other sizes, narrow or unaligned rows).
//   K=31 forward of fp32 weights: the role-split kernel's dx role on every wave, 262 us against 299 LDS-staged with loader
//     waves (C=2048); K=15: LDS-staged with loader waves, 190 us against 203 role-split and 227 sliding-window (C=2048).
int choose_algo(bool bwd, const nplm_dwconv_tuning* tune, bool bf16, bool w_bf16, long long T, int C, int K, int taps, int S, uintptr_t align_bits,
                uintptr_t out_bits) {
    if (tune && tune->algo == 4) return mfma_eligible(bf16, w_bf16, T, C, K, align_bits) ? 4 : -NPLM_DWCONV_ETUNING;
    if (tune && tune->algo == 3) return split_eligible(bf16, T, C, K, align_bits) ? 3 : -NPLM_DWCONV_ETUNING;
    if (tune && tune->algo == 2) return lds_eligible(bf16, T, C, K, align_bits) ? 2 : -NPLM_DWCONV_ETUNING;
    if (tune && tune->algo == 1) return 1;
    if (mfma_eligible(bf16, w_bf16, T, C, K, align_bits) && T >= kMfmaMinRows && mfma_tile_fits(C, K, false) &&
        mfma_lines_ok(bwd, false, T, C, K, taps, out_bits) && (!bwd || mfma_bwd_preferred(T, taps, S))) return 4;
    if (split_eligible(bf16, T, C, K, align_bits) && (bwd || K == 31)) return 3;
    return lds_preferred(bwd, bf16, T, C, K, align_bits) ? 2 : 1;
}

// 256 threads x 4 x 16 B = one contiguous 16 KiB chunk per block
__global__ void __launch_bounds__(256) copy_chunks_kernel(const u32x4* __restrict__ src, u32x4* __restrict__ dst, size_t nvec) {
    const size_t base = (size_t)blockIdx.x * 1024 + threadIdx.x;
    u32x4 v[4];
#pragma unroll
    for (int u = 0; u < 4; ++u)
        if (base + u * 256 < nvec) v[u] = src[base + u * 256];
#pragma unroll
    for (int u = 0; u < 4; ++u)
        if (base + u * 256 < nvec) dst[base + u * 256] = v[u];
}

__global__ void fill_zero_kernel(float* p, long long n) {
    const long long i = (long long)blockIdx.x * blockDim.x + threadIdx.x;
    if (i < n) p[i] = 0.f;
}
__global__ void fill_zero16_kernel(uint16_t* p, long long n) {
    const long long i = (long long)blockIdx.x * blockDim.x + threadIdx.x;
    if (i < n) p[i] = 0;
}
hipError_t fill_zero16(void* p, long long n, hipStream_t s) {
    if (!p || n <= 0) return hipSuccess;
    hipLaunchKernelGGL(fill_zero16_kernel, dim3((unsigned)((n + 255) / 256)), dim3(256), 0, s, (uint16_t*)p, n);
    return hipGetLastError();
}
hipError_t fill_zero(float* p, long long n, hipStream_t s) {
    if (!p || n <= 0) return hipSuccess;
    hipLaunchKernelGGL(fill_zero_kernel, dim3((unsigned)((n + 255) / 256)), dim3(256), 0, s, p, n);
    return hipGetLastError();
}

// cu_seqlens [2B+1] of a right-padded mask [B, L] over the flat rows: G threads sum a row of the mask (a bool counts as one
// whatever its byte if that is not zero, any other value is taken as int32, sums wrap in 32 bits) and write b * L and
// b * L + that sum; the last entry is B * L. It takes the place of eight elementwise and reduction launches (sum, arange, mul,
// add, stack, full, cat and a copy): a padded call of 32 x 512 rows at C=768 goes from 65 to 25 us, of which the conv kernel is
// 13. Short rows are bound by the launch and by how many blocks it starts, so several rows share a block; a long row is bound by
// the loads that its threads have in flight, so G grows with L and a thread issues eight loads at once. Time on the device,
// elementwise / 256 threads per row and one load at a time / this (us, int64): B=32, L=512 17.6 / 2.5 / 2.3; B=65536, L=8
// 24.7 / 24.8 / 2.5; B=2^20, L=8 77 / 399 / 18; B=1, L=16384 20.4 / 9.8 / 3.8; B=1, L=65536 26.7 / 34.7 / 9.5; B=1024, L=16384
// 63 / 23.1 / 20.3.
template <typename V, bool BOOL, int G>
__global__ void __launch_bounds__(G > 256 ? G : 256) mask_cu_kernel(const V* __restrict__ mask, long long row_stride, int L, unsigned B,
                                                                   int32_t* __restrict__ cu) {
    constexpr int NT = G > 256 ? G : 256;
    const unsigned b = blockIdx.x * (NT / G) + threadIdx.x / G;
    const int lane = threadIdx.x % G;
    unsigned n = 0;
    if (b < B) {
        const V* row = mask + (size_t)b * (size_t)row_stride;
        auto count = [](V v) { return BOOL ? (unsigned)(v != 0) : (unsigned)(int32_t)v; };
        int i = lane;
        for (; i + 7 * G < L; i += 8 * G) {
            V v[8];
#pragma unroll
            for (int u = 0; u < 8; ++u) v[u] = row[i + u * G];
#pragma unroll
            for (int u = 0; u < 8; ++u) n += count(v[u]);
        }
        for (; i < L; i += G) n += count(row[i]);
    }
#pragma unroll
    for (int d = (G < 64 ? G : 64) / 2; d > 0; d >>= 1) n += (unsigned)__shfl_xor((int)n, d, 64);
    if constexpr (G > 64) {
        __shared__ unsigned part[G / 64];
        if (threadIdx.x % 64 == 0) part[threadIdx.x / 64] = n;
        __syncthreads();
        n = 0;
#pragma unroll
        for (int i = 0; i < G / 64; ++i) n += part[i];
    }
    if (lane == 0 && b < B) {
        const unsigned start = b * (unsigned)L;
        cu[2 * (size_t)b] = (int32_t)start;
        cu[2 * (size_t)b + 1] = (int32_t)(start + n);
        if (b + 1 == B) cu[2 * (size_t)B] = (int32_t)(B * (unsigned)L);
    }
}
template <typename V, bool BOOL, int G>
hipError_t launch_mask_cu_g(const void* mask, long long row_stride, int L, unsigned B, int32_t* cu, hipStream_t s) {
    constexpr unsigned NT = G > 256 ? G : 256, rows = NT / G;
    hipLaunchKernelGGL((mask_cu_kernel<V, BOOL, G>), dim3((B + rows - 1) / rows), dim3(NT), 0, s, (const V*)mask, row_stride, L, B, cu);
    return hipGetLastError();
}
// Threads per row by its length. Measured with 8 / 64 / 256 / 1024 (us, int64): 65536 rows of 64 6.0 / 10.2 / 28.9 / 120, of 128
// 11.2 / 14.1 / 31.3 / 122, of 256 20.6 / 22.0 / 34.3 / 120 (1024 rows of 256 3.8 / 2.5 / 2.5 / 3.7); 16384 rows of 1024 33.5 /
// 20.1 / 21.6 / 40.1; 32 rows of 2048 16.1 / 3.0 / 2.5 / 2.6, of 8192 58.7 / 6.0 / 3.5 / 3.3; one row of 16384 37 / 7.2 / 4.4 / 3.8,
// of 65536 - / 24.1 / 12.4 / 9.5.
template <typename V, bool BOOL>
hipError_t launch_mask_cu(const void* mask, long long row_stride, int L, unsigned B, int32_t* cu, hipStream_t s) {
    if (L <= 128) return launch_mask_cu_g<V, BOOL, 8>(mask, row_stride, L, B, cu, s);
    if (L <= 1024) return launch_mask_cu_g<V, BOOL, 64>(mask, row_stride, L, B, cu, s);
    if (L <= 8192) return launch_mask_cu_g<V, BOOL, 256>(mask, row_stride, L, B, cu, s);
    return launch_mask_cu_g<V, BOOL, 1024>(mask, row_stride, L, B, cu, s);
}

// Shapes the gated (z = [u | g]) kernels are built for.
bool gated_supported(bool bwd, bool bf16, long long T, int C, int K, uintptr_t align_bits) {
    const int E = bf16 ? 2 : 4;
    if (!lds_gated_kernel_size(K, bwd) || T < 1) return false;
    if (((long long)C * E) % 16 || align_bits % 16) return false;
    return (long long)C * E >= 1024;
}

// Long gated backward (K = 15, 31), role-split (dwconv_lds_split_kernels.h, GATED): rows of whole 16-byte chunks that fill
// at least one 512-byte column block, 16-byte aligned tensors. Measured at T=131072, C=2048, bf16, backward + finalize
// against the sliding-window kernel below (log-normal length mix / one long sequence): K=31 728 / 685 against 949 / 808 us,
// K=15 584 / 535 against 613 / 593 us; dz is the same bit for bit (same tap order).
bool split_gated_eligible(bool bf16, long long T, int C, int K, uintptr_t align_bits) {
    return split_eligible(bf16, T, C, K, align_bits);
}
// Otherwise: the sliding-window kernel with one channel per lane; same shapes as the gated forward.
bool long_gated_bwd_supported(bool bf16, long long T, int C, int K, uintptr_t align_bits) {
    return long_gated_kernel_size(K) && gated_supported(false, bf16, T, C, K, align_bits);
}
int make_long_gated_plan(bool bf16, long long T, int C, int K, Plan* out) {
    nplm_dwconv_tuning t{};
    t.vec = 1;
    return make_plan(true, bf16, T, C, K, 0, &t, out);
}

// algo of a gated call: 4 matrix cores, 3 role-split, 2 LDS-staged, 1 sliding-window; align_bits: of z, dy and the output, out_bits: of dz.
int choose_gated_algo(bool bwd, bool bf16, bool w_bf16, long long T, int C, int K, int taps, int S, uintptr_t align_bits, uintptr_t out_bits) {
    const bool supported = gated_supported(false, bf16, T, C, K, align_bits);
    const bool role_split = long_gated_kernel_size(K) && split_gated_eligible(bf16, T, C, K, align_bits);
    if (!supported && !(bwd && role_split)) return -NPLM_DWCONV_EUNSUPPORTED;
    if (!role_split) return bwd && long_gated_kernel_size(K) ? 1 : 2;
    if (!bf16 || !w_bf16) return 3;
    if (bwd) return mfma_tile_fits(C, K, true) && mfma_lines_ok(true, true, T, C, K, taps, out_bits) && mfma_gated_bwd_preferred(T, C, taps, S) ? 4 : 3;
    LdsPlan lp;
    return mfma_gated_fwd_preferred(T, C, taps, S) &&
           make_split_plan(true, bf16, T, C, K, nullptr, &lp, true, mfma_gated_fwd_steps(T, C) * kMfmaGatedRows, kMfmaGatedCb) == 0 &&
           MfmaGatedFwdShape<31>::lds_bytes(ceil_div(lp.ntiles, lp.nbt)) <= kLdsBytes ? 4 : 3;
}

// launch flags of the kernels (W_BF16 | W_RESIDUAL) from the ABI's weight dtype and flags
int kernel_w_flags(int32_t w_dtype, uint32_t flags) {
    return (w_dtype == NPLM_DWCONV_BF16 ? W_BF16 : 0) | ((flags & NPLM_DWCONV_RESIDUAL) ? W_RESIDUAL : 0);
}

int fwd_impl(const void* x, const int32_t* cu, const void* w, const void* b, void* y, int64_t T, int32_t C,
             int32_t K, int32_t S, int32_t act_dtype, int32_t w_dtype, uint32_t flags, void* stream,
             const nplm_dwconv_tuning* tune) {
    int rc = check_common(T, C, K, S, act_dtype, w_dtype);
    if (rc) return rc;
    if (flags & ~(uint32_t)NPLM_DWCONV_RESIDUAL) return -NPLM_DWCONV_EFLAGS;
    if (T == 0) return 0;
    if (!x || !cu || !w || !y) return -NPLM_DWCONV_ENULL;
    const int taps = lds_taps(K), tap_off = (exec_kernel_size(K) - K) / 2;
    const int lds_w_flags = kernel_w_flags(w_dtype, flags) | ((taps - K) / 2 << W_TAP_OFF_SHIFT);
    K = exec_kernel_size(K);        // from here on the kernel size that runs
    const int w_flags = kernel_w_flags(w_dtype, flags) | (tap_off << W_TAP_OFF_SHIFT);
    const bool bf16 = act_dtype == NPLM_DWCONV_BF16;
    const uintptr_t E = bf16 ? 2 : 4;
    const uintptr_t bits = (uintptr_t)x | (uintptr_t)y;
    if (bits % E) return -NPLM_DWCONV_EALIGN;
    const uintptr_t WE = (w_dtype == NPLM_DWCONV_BF16) ? 2 : 4;
    if (((uintptr_t)w | (uintptr_t)b) % WE || (uintptr_t)cu % 4) return -NPLM_DWCONV_EALIGN;
    hipStream_t s = (hipStream_t)stream;
    const int algo = choose_algo(false, tune, bf16, w_dtype == NPLM_DWCONV_BF16, T, C, K, taps, S, bits, (uintptr_t)y);
    if (algo < 0) return algo;
    if (algo == 3 || algo == 4) {
        LdsPlan lp;
        rc = make_split_plan(true, bf16, T, C, K, tune, &lp, false, algo == 4 ? kMfmaFwdRows : 0);
        if (rc) return rc;
        const ConvPtrs la{x, nullptr, cu, w, b, y, nullptr};
        if (algo == 4) return (int)launch_fwd_mfma(taps, la, make_lds_geo(lp, T, C, S, w_flags), dim3(lp.ncb * lp.nbt), s);
        const int run = K == 31 ? taps : K;
        const LdsGeo lg = make_lds_geo(lp, T, C, S, run == K ? w_flags : lds_w_flags);
        return (int)launch_fwd_split(run, bf16, la, lg, dim3(lp.ncb * lp.nbt), s);
    }
    if (algo == 2) {
        // of the shorter forms the loader-wave forward has the one of 11 taps; shape overrides name shapes of K
        const int lds_k = (taps == 11 && !tune) ? taps : K;
        LdsPlan lp;
        rc = make_lds_plan(false, bf16, T, C, lds_k, tune, &lp);
        if (rc) return rc;
        const ConvPtrs la{x, nullptr, cu, w, b, y, nullptr};
        const hipError_t e = launch_fwd_lds(lds_k, lp, la, make_lds_geo(lp, T, C, S, lds_k == K ? w_flags : lds_w_flags), s);
        if (e == hipErrorInvalidConfiguration && tune) return -NPLM_DWCONV_ETUNING;
        return (int)e;
    }
    Plan p;
    rc = make_plan(false, bf16, T, C, K, bits, tune, &p);
    if (rc) return rc;
    if (p.generic) {
        const int wpb = 4;
        int blocks = ceil_div(T, wpb);
        if (blocks > kNumCU * 16) blocks = kNumCU * 16;
        if (bf16)
            hipLaunchKernelGGL(dwconv_generic_rows_kernel<true>, dim3(blocks), dim3(wpb * 64), 0, s, x, cu, w, b, y,
                               (int)T, C, S, K, w_flags, 0);
        else
            hipLaunchKernelGGL(dwconv_generic_rows_kernel<false>, dim3(blocks), dim3(wpb * 64), 0, s, x, cu, w, b, y,
                               (int)T, C, S, K, w_flags, 0);
        return (int)hipGetLastError();
    }
    const ConvPtrs a{x, nullptr, cu, w, b, y, nullptr};
    const hipError_t e = launch_fwd(K, bf16, p, a, make_geo(p, T, C, S, w_flags), s);
    if (e == hipErrorInvalidConfiguration && tune) return -NPLM_DWCONV_ETUNING;
    return (int)e;
}

int bwd_impl(const void* x, const void* dy, const int32_t* cu, const void* w, void* dx, float* dw, float* db,
             void* workspace, size_t workspace_bytes, int64_t T, int32_t C, int32_t K, int32_t S,
             int32_t act_dtype, int32_t w_dtype, uint32_t flags, void* stream, const nplm_dwconv_tuning* tune) {
    int rc = check_common(T, C, K, S, act_dtype, w_dtype);
    if (rc) return rc;
    if (flags & ~(uint32_t)(NPLM_DWCONV_RESIDUAL | NPLM_DWCONV_GRADS_BF16)) return -NPLM_DWCONV_EFLAGS;
    const int out_bf16 = (flags & NPLM_DWCONV_GRADS_BF16) ? 1 : 0;      // dw, db are bf16 buffers
    hipStream_t s = (hipStream_t)stream;
    const bool want_red = dw || db;
    if (T == 0) {
        hipError_t e = out_bf16 ? fill_zero16(dw, (long long)C * K, s) : fill_zero(dw, (long long)C * K, s);
        if (e == hipSuccess) e = out_bf16 ? fill_zero16(db, C, s) : fill_zero(db, C, s);
        return (int)e;
    }
    const int taps = lds_taps(K), lds_tap_off = (taps - K) / 2, tap_off = (exec_kernel_size(K) - K) / 2;
    K = exec_kernel_size(K);        // from here on the kernel size that runs (workspace for slabs of K + 1 rows; dw rows stay the caller's)
    const int w_flags = kernel_w_flags(w_dtype, flags) | (tap_off << W_TAP_OFF_SHIFT);
    if (!dx && !want_red) return 0;
    if (!dy || !cu || !w || (want_red && !x)) return -NPLM_DWCONV_ENULL;
    const bool bf16 = act_dtype == NPLM_DWCONV_BF16;
    const uintptr_t E = bf16 ? 2 : 4;
    const uintptr_t bits = (uintptr_t)x | (uintptr_t)dy | (uintptr_t)dx;
    if (bits % E) return -NPLM_DWCONV_EALIGN;
    const uintptr_t WE = (w_dtype == NPLM_DWCONV_BF16) ? 2 : 4;
    if ((uintptr_t)w % WE || (uintptr_t)cu % 4 || ((uintptr_t)dw | (uintptr_t)db) % (out_bf16 ? 2 : 4)) return -NPLM_DWCONV_EALIGN;

    int algo = choose_algo(true, tune, bf16, w_dtype == NPLM_DWCONV_BF16, T, C, K, taps, S, bits, (uintptr_t)dx);
    if (algo < 0) return algo;
    if (algo >= 3 && !(dx && want_red)) {     // these kernels are fused only: a partial request takes the others
        if (tune && tune->algo >= 3) return -NPLM_DWCONV_ETUNING;
        algo = 1;
    }
    if (algo == 3 || algo == 4) {
        LdsPlan lp;
        rc = make_split_plan(false, bf16, T, C, K, tune, &lp);
        if (rc) return rc;
        const size_t slab_bytes = (size_t)(K + 1) * C * sizeof(float);
        if (!workspace || (uintptr_t)workspace % 256 || workspace_bytes < slab_bytes * (size_t)lp.nbt)
            return -NPLM_DWCONV_EWORKSPACE;
        float* part = reinterpret_cast<float*>(workspace);
        const ConvPtrs la{x, dy, cu, w, nullptr, dx, part};
        // (the matrix-core kernels place the caller's taps among those of K, the role-split ones among the taps that run)
        const LdsGeo lg = make_lds_geo(lp, T, C, S, algo == 4 ? w_flags : kernel_w_flags(w_dtype, flags) | (lds_tap_off << W_TAP_OFF_SHIFT));
        const dim3 grid(lp.ncb * lp.nbt);
        hipError_t e = algo == 4 ? launch_bwd_mfma(taps, la, lg, grid, s) : launch_bwd_split(taps, bf16, la, lg, grid, s);
        if (e != hipSuccess) return (int)e;
        if (tune && tune->mid_event) {
            e = hipEventRecord((hipEvent_t)tune->mid_event, s);
            if (e != hipSuccess) return (int)e;
        }
        const long long n_out = (long long)(taps + 1) * C;
        hipLaunchKernelGGL(dwconv_finalize_kernel<FIN_SPLIT>, dim3((unsigned)((n_out + 63) / 64)), dim3(64 * FIN_SPLIT), 0,
                           s, (const float*)part, lp.nbt, C, taps, dw, db, out_bf16, lds_tap_off);
        return (int)hipGetLastError();
    }
    if (algo == 2) {
        LdsPlan lp;
        rc = make_lds_plan(true, bf16, T, C, K, tune, &lp);
        if (rc) return rc;
        const size_t slab_bytes = (size_t)(K + 1) * C * sizeof(float);
        float* part = nullptr;
        if (want_red) {
            if (!workspace || (uintptr_t)workspace % 256 || workspace_bytes < slab_bytes * (size_t)lp.nbt)
                return -NPLM_DWCONV_EWORKSPACE;
            part = reinterpret_cast<float*>(workspace);
        }
        const ConvPtrs la{x, dy, cu, w, nullptr, dx, part};
        hipError_t e = launch_bwd_lds(K, lp, dx != nullptr, want_red, la,
                                      make_lds_geo(lp, T, C, S, w_flags), s);
        if (e == hipErrorInvalidConfiguration && tune) return -NPLM_DWCONV_ETUNING;
        if (e != hipSuccess) return (int)e;
        if (tune && tune->mid_event) {
            e = hipEventRecord((hipEvent_t)tune->mid_event, s);
            if (e != hipSuccess) return (int)e;
        }
        if (want_red) {
            const long long n_out = (long long)(K + 1) * C;
            hipLaunchKernelGGL(dwconv_finalize_kernel<FIN_SPLIT>, dim3((unsigned)((n_out + 63) / 64)),
                               dim3(64 * FIN_SPLIT), 0, s, (const float*)part, lp.nbt, C, K, dw, db, out_bf16, tap_off);
            e = hipGetLastError();
        }
        return (int)e;
    }
    Plan p;
    rc = make_plan(true, bf16, T, C, K, bits, tune, &p);
    if (rc) return rc;
    if (!tune) {
        // never use more slabs than nplm_dwconv_bwd_workspace_bytes() promised for aligned inputs
        Plan nominal;
        rc = make_plan(true, bf16, T, C, K, 0, nullptr, &nominal);
        if (rc) return rc;
        if (p.nbt > nominal.nbt) {
            p.nbt = nominal.nbt;
            p.remap = p.remap && ((long long)p.ncb * p.nbt) % kNumXCD == 0;
        }
    }
    const size_t slab = (size_t)(K + 1) * C * sizeof(float);
    float* partial = nullptr;
    if (want_red) {
        if (!workspace || (uintptr_t)workspace % 256 || workspace_bytes < slab * (size_t)p.nbt)
            return -NPLM_DWCONV_EWORKSPACE;
        partial = reinterpret_cast<float*>(workspace);
    }

    if (p.generic) {
        if (dx) {
            const int wpb = 4;
            int blocks = ceil_div(T, wpb);
            if (blocks > kNumCU * 16) blocks = kNumCU * 16;
            if (bf16)
                hipLaunchKernelGGL(dwconv_generic_rows_kernel<true>, dim3(blocks), dim3(wpb * 64), 0, s, dy, cu, w,
                                   (const void*)nullptr, dx, (int)T, C, S, K, w_flags, 1);
            else
                hipLaunchKernelGGL(dwconv_generic_rows_kernel<false>, dim3(blocks), dim3(wpb * 64), 0, s, dy, cu, w,
                                   (const void*)nullptr, dx, (int)T, C, S, K, w_flags, 1);
            const hipError_t e = hipGetLastError();
            if (e != hipSuccess) return (int)e;
        }
        if (want_red) {
            const int rows = ceil_div(T, p.nbt);
            const dim3 grid(p.nbt, ceil_div(C, 256));
            if (bf16)
                hipLaunchKernelGGL(dwconv_generic_dw_kernel<true>, grid, dim3(256), 0, s, x, dy, cu, partial, (int)T, C,
                                   S, K, rows);
            else
                hipLaunchKernelGGL(dwconv_generic_dw_kernel<false>, grid, dim3(256), 0, s, x, dy, cu, partial, (int)T,
                                   C, S, K, rows);
            const hipError_t e = hipGetLastError();
            if (e != hipSuccess) return (int)e;
        }
    } else {
        const ConvPtrs a{x, dy, cu, w, nullptr, dx, partial};
        const hipError_t e = launch_bwd(K, bf16, p, dx != nullptr, want_red, a, make_geo(p, T, C, S, w_flags), s);
        if (e == hipErrorInvalidConfiguration && tune) return -NPLM_DWCONV_ETUNING;
        if (e != hipSuccess) return (int)e;
    }
    if (tune && tune->mid_event) {
        const hipError_t e = hipEventRecord((hipEvent_t)tune->mid_event, s);
        if (e != hipSuccess) return (int)e;
    }
    if (want_red) {
        const long long n_out = (long long)(K + 1) * C;
        hipLaunchKernelGGL(dwconv_finalize_kernel<FIN_SPLIT>, dim3((unsigned)((n_out + 63) / 64)), dim3(64 * FIN_SPLIT), 0, s,
                           (const float*)partial, p.nbt, C, K, dw, db, out_bf16, tap_off);
        const hipError_t e = hipGetLastError();
        if (e != hipSuccess) return (int)e;
    }
    return 0;
}

// Device address of `scratch` on the current device, looked up once per device and kept.
constexpr int kMaxDevices = 64;
std::atomic<void*> g_scratch_ptr[kMaxDevices];

hipError_t static_scratch_for_current_device(void** out) {
    int dev = -1;
    hipError_t e = hipGetDevice(&dev);
    if (e != hipSuccess) return e;
    if (dev < 0 || dev >= kMaxDevices) return hipErrorInvalidDevice;
    void* p = g_scratch_ptr[dev].load(std::memory_order_acquire);
    if (!p) {
        e = hipGetSymbolAddress(&p, HIP_SYMBOL(scratch));
        if (e != hipSuccess) return e;
        if (!p) return hipErrorInvalidSymbol;
        g_scratch_ptr[dev].store(p, std::memory_order_release);   // every thread finds the same address
    }
    *out = p;
    return hipSuccess;
}

}  // namespace
}  // namespace nplm

// ---- LayerNorm-fused conv: shapes, geometry and the one-wave-per-row kernels' launchers ----------------------------
namespace nplm {
namespace {
// rows of one 2 KiB column block: one forward kernel that takes the statistics from the tile it has staged
bool ln_whole_rows(bool bf16, int C, int K, uintptr_t align_bits) {
    const long long row_bytes = (long long)C * (bf16 ? 2 : 4);
    return lds_ln_kernel_size(K) && row_bytes % 16 == 0 && row_bytes <= kLnCbBytes && align_bits % 16 == 0;
}
// forward, fp32 rows of up to 4 KiB: the same kernel with 6 or 8 wave-columns and shorter tiles, see lds_ln_3k_shape()
// and lds_ln_4k_shape()
bool ln_fwd_whole_4k(bool bf16, int C, int K, uintptr_t align_bits) {
    const long long row_bytes = (long long)C * 4;
    return !bf16 && lds_ln_kernel_size(K) && row_bytes % 16 == 0 && row_bytes > kLnCbBytes && row_bytes <= 2 * kLnCbBytes &&
           align_bits % 16 == 0;
}
// backward: rows of up to 4 KiB also fit a block, see lds_ln_bwd_wide_shape() and lds_ln_bwd_3k_shape()
bool ln_bwd_whole_4k(bool bf16, int C, int K, uintptr_t align_bits) {
    const long long row_bytes = (long long)C * (bf16 ? 2 : 4);
    return lds_ln_bwd_wide_kernel_size(K) && row_bytes % 16 == 0 && row_bytes > kLnCbBytes && row_bytes <= 4096 &&
           align_bits % 16 == 0;
}
// other rows of up to 8 KiB: a row-statistics kernel, then the conv forward that normalises as it reads (the forward
// asks ln_fwd_whole_4k first)
bool ln_wide_rows(bool bf16, int C, int K, uintptr_t align_bits) {
    const long long row_bytes = (long long)C * (bf16 ? 2 : 4);
    return lds_ln_kernel_size(K) && row_bytes % 16 == 0 && row_bytes > kLnCbBytes && row_bytes <= 8192 && align_bits % 16 == 0;
}
// 16-byte chunks per lane of the one-wave-per-row kernels: rows of at most 2, 4, 8 KiB
int ln_row_chunks(long long row_bytes) { return row_bytes <= 2048 ? 2 : row_bytes <= 4096 ? 4 : 8; }
int ln_row_blocks(long long T) {
    const int blocks = ceil_div(T, 4);
    return blocks > kNumCU * 8 ? kNumCU * 8 : blocks;
}
// the default shape of a pass as an explicit geometry, whatever lds_shape_for() would pick for the width
int make_default_lds_plan(bool bwd, bool bf16, long long T, int C, int K, LdsPlan* out) {
    nplm_dwconv_tuning t{};
    const LdsShapeSel sh = lds_default_shape(bwd, bf16, K);
    t.vec = sh.vec; t.unroll = sh.rw; t.bt = sh.nrg; t.bw = sh.ncw; t.nwl = sh.nwl; t.nbuf = sh.nbuf;
    return make_lds_plan(bwd, bf16, T, C, K, &t, out);
}
template <bool BF16>
hipError_t launch_ln_stats(int nch, const void* x, float* stats, float eps, long long T, int C, hipStream_t s) {
    const dim3 grid(ln_row_blocks(T)), block(256);
    if (nch == 2) hipLaunchKernelGGL((ln_stats_kernel<BF16, 2>), grid, block, 0, s, x, stats, eps, (int)T, C);
    else if (nch == 4) hipLaunchKernelGGL((ln_stats_kernel<BF16, 4>), grid, block, 0, s, x, stats, eps, (int)T, C);
    else hipLaunchKernelGGL((ln_stats_kernel<BF16, 8>), grid, block, 0, s, x, stats, eps, (int)T, C);
    return hipGetLastError();
}
template <bool BF16>
hipError_t launch_ln_bwd_dx(int nch, const void* x, const float* stats, const void* gamma, int w_flags, const float* dn,
                            const void* dy, void* dx, long long T, int C, hipStream_t s) {
    const dim3 grid(ln_row_blocks(T)), block(256);
    if (nch == 2) hipLaunchKernelGGL((ln_bwd_dx_kernel<BF16, 2>), grid, block, 0, s, x, stats, gamma, w_flags, dn, dy, dx, (int)T, C);
    else if (nch == 4) hipLaunchKernelGGL((ln_bwd_dx_kernel<BF16, 4>), grid, block, 0, s, x, stats, gamma, w_flags, dn, dy, dx, (int)T, C);
    else hipLaunchKernelGGL((ln_bwd_dx_kernel<BF16, 8>), grid, block, 0, s, x, stats, gamma, w_flags, dn, dy, dx, (int)T, C);
    return hipGetLastError();
}
}  // namespace
}  // namespace nplm

using namespace nplm;

extern "C" {

int nplm_dwconv_version(void) { return kVersion; }

int nplm_dwconv_gated_fwd(const void* z, const int32_t* cu, const void* w, const void* b, void* y, int64_t T,
                          int32_t C, int32_t K, int32_t S, int32_t act_dtype, int32_t w_dtype, uint32_t flags,
                          void* stream) {
    int rc = check_common(T, C, K, S, act_dtype, w_dtype);
    if (rc) return rc;
    if (flags & ~(uint32_t)NPLM_DWCONV_RESIDUAL) return -NPLM_DWCONV_EFLAGS;
    if (T == 0) return 0;
    if (!z || !cu || !w || !y) return -NPLM_DWCONV_ENULL;
    const int taps = lds_taps(K), lds_tap_flags = (taps - K) / 2 << W_TAP_OFF_SHIFT;
    const int tap_flags = ((exec_kernel_size(K) - K) / 2) << W_TAP_OFF_SHIFT;
    K = exec_kernel_size(K);        // from here on the kernel size that runs
    const bool bf16 = act_dtype == NPLM_DWCONV_BF16;
    const uintptr_t WE = (w_dtype == NPLM_DWCONV_BF16) ? 2 : 4;
    if (((uintptr_t)w | (uintptr_t)b) % WE || (uintptr_t)cu % 4) return -NPLM_DWCONV_EALIGN;
    const int algo = choose_gated_algo(false, bf16, w_dtype == NPLM_DWCONV_BF16, T, C, K, taps, S, (uintptr_t)z | (uintptr_t)y, 0);
    if (algo < 0) return algo;
    LdsPlan lp;
    if (algo == 4) {
        const int steps = mfma_gated_fwd_steps(T, C);
        rc = make_split_plan(true, bf16, T, C, K, nullptr, &lp, true, steps * kMfmaGatedRows, kMfmaGatedCb);
        if (rc) return rc;
        const ConvPtrs la{z, nullptr, cu, w, b, y, nullptr};
        const LdsGeo lg = make_lds_geo(lp, T, C, S, kernel_w_flags(w_dtype, flags) | tap_flags);
        const dim3 grid(lp.ncb * lp.nbt);
        return (int)(K == 15 ? launch_fwd_gated_mfma_k15(la, lg, steps, grid, (hipStream_t)stream)
                             : launch_fwd_gated_mfma_k31(la, lg, steps, grid, (hipStream_t)stream));
    }
    if (algo == 3) {
        rc = make_split_plan(true, bf16, T, C, K, nullptr, &lp, true);
        if (rc) return rc;
        const ConvPtrs la{z, nullptr, cu, w, b, y, nullptr};
        const LdsGeo lg = make_lds_geo(lp, T, C, S, kernel_w_flags(w_dtype, flags) | lds_tap_flags);
        const dim3 grid(lp.ncb * lp.nbt);
        return (int)launch_fwd_split_gated(taps, bf16, la, lg, grid, (hipStream_t)stream);
    }
    rc = make_lds_plan(false, bf16, T, C, K, nullptr, &lp, true);
    if (rc) return rc == -NPLM_DWCONV_ETUNING ? -NPLM_DWCONV_EUNSUPPORTED : rc;
    const ConvPtrs la{z, nullptr, cu, w, b, y, nullptr};
    const bool narrow = lds_gated_narrow((long long)C * (bf16 ? 2 : 4), K);
    const LdsGeo g = make_lds_geo(lp, T, C, S, kernel_w_flags(w_dtype, flags) | tap_flags);
    const dim3 grid(lp.ncb * lp.nbt);
    hipStream_t s = (hipStream_t)stream;
    switch (K) {
        case 15: return (int)launch_fwd_lds_gated_k15(bf16, narrow, la, g, grid, s);
        case 31: return (int)launch_fwd_lds_gated_k31(bf16, narrow, la, g, grid, s);
        case 3: return (int)launch_fwd_lds_gated_k3(bf16, narrow, la, g, grid, s);
        case 5: return (int)launch_fwd_lds_gated_k5(bf16, narrow, la, g, grid, s);
        case 7: return (int)launch_fwd_lds_gated_k7(bf16, narrow, la, g, grid, s);
        case 9: return (int)launch_fwd_lds_gated_k9(bf16, narrow, la, g, grid, s);
    }
    return -NPLM_DWCONV_EUNSUPPORTED;
}

// ---- LayerNorm-fused conv (dwconv_ln_kernels.h and the NORM variants of the LDS-staged kernels) ----------------------
int nplm_dwconv_ln_fwd(const void* x, const int32_t* cu, const void* ln_weight, const void* ln_bias, float eps,
                       const void* w, const void* b, void* y, float* stats, int64_t T, int32_t C, int32_t K, int32_t S,
                       int32_t act_dtype, int32_t w_dtype, uint32_t flags, void* stream) {
    int rc = check_common(T, C, K, S, act_dtype, w_dtype);
    if (rc) return rc;
    if (flags & ~(uint32_t)NPLM_DWCONV_RESIDUAL) return -NPLM_DWCONV_EFLAGS;
    if (T == 0) return 0;
    if (!x || !cu || !w || !y || !ln_weight) return -NPLM_DWCONV_ENULL;
    const bool bf16 = act_dtype == NPLM_DWCONV_BF16;
    const uintptr_t E = bf16 ? 2 : 4;
    const uintptr_t WE = (w_dtype == NPLM_DWCONV_BF16) ? 2 : 4;
    if (((uintptr_t)w | (uintptr_t)b | (uintptr_t)ln_weight | (uintptr_t)ln_bias) % WE || (uintptr_t)cu % 4 ||
        (uintptr_t)stats % 4 || ((uintptr_t)x | (uintptr_t)y) % E)
        return -NPLM_DWCONV_EALIGN;
    const uintptr_t bits = (uintptr_t)x | (uintptr_t)y;
    hipStream_t s = (hipStream_t)stream;
    const ConvPtrs la{x, nullptr, cu, w, b, y, nullptr};
    const bool rows4k = ln_fwd_whole_4k(bf16, C, K, bits);
    if (!rows4k && ln_wide_rows(bf16, C, K, bits)) {
        if (!stats) return -NPLM_DWCONV_ENULL;      // the statistics pass between the two kernels through it
        LdsPlan lp;
        rc = make_default_lds_plan(false, bf16, T, C, K, &lp);
        if (rc) return rc == -NPLM_DWCONV_ETUNING ? -NPLM_DWCONV_EUNSUPPORTED : rc;
        const int nch = ln_row_chunks((long long)C * (long long)E);
        hipError_t e = bf16 ? launch_ln_stats<true>(nch, x, stats, eps, T, C, s) : launch_ln_stats<false>(nch, x, stats, eps, T, C, s);
        if (e != hipSuccess) return (int)e;
        const LnSide side{stats, ln_weight, ln_bias, nullptr};
        const LdsGeo g = make_lds_geo(lp, T, C, S, kernel_w_flags(w_dtype, flags));
        const dim3 grid(lp.ncb * lp.nbt);
        switch (K) {
            case 3: return (int)launch_ln_fwd_wide_k3(bf16, la, side, g, grid, s);
            case 5: return (int)launch_ln_fwd_wide_k5(bf16, la, side, g, grid, s);
            case 7: return (int)launch_ln_fwd_wide_k7(bf16, la, side, g, grid, s);
            case 9: return (int)launch_ln_fwd_wide_k9(bf16, la, side, g, grid, s);
        }
        return -NPLM_DWCONV_EUNSUPPORTED;
    }
    if (!rows4k && !ln_whole_rows(bf16, C, K, bits)) return -NPLM_DWCONV_EUNSUPPORTED;
    LdsPlan lp{};
    lp.sh = !rows4k ? lds_ln_shape(bf16) : lds_ln_rows3k(bf16, C) ? lds_ln_3k_shape(K) : lds_ln_4k_shape(bf16, K);
    lp.R = lp.sh.rw * lp.sh.nrg;
    lp.ncb = 1;
    lp.ntiles = ceil_div(T, lp.R);
    lp.nbt = lp.ntiles < kNumCU ? lp.ntiles : kNumCU;          // one block of 16 waves and three tiles per CU
    lp.xcd_group = (lp.nbt % (kNumXCD * 8) == 0) ? 8 : 0;
    // fp32 rows of 4 KiB: 6 of a tile's 13 staged rows are a neighbour's, and a neighbour on another XCD means reading them
    // from HBM again; 32 consecutive tiles per XCD instead of 8 (T=131072, C=1024, K=7: 217 against 222 us per call; the
    // other whole-row kernels, with longer tiles, measure the same either way)
    if (rows4k && lp.nbt % (kNumXCD * 32) == 0) lp.xcd_group = 32;
    lp.rot_step = lp.nbt > 2 ? (int)((long long)lp.nbt * 618 / 1000) | 1 : 0;
    if (lp.rot_step >= lp.nbt) lp.rot_step = lp.nbt - 1;
    const LnArgs ln{ln_weight, ln_bias, stats, eps};
    const LdsGeo g = make_lds_geo(lp, T, C, S, kernel_w_flags(w_dtype, flags));
    const dim3 grid(lp.nbt);
    if (rows4k) {
        switch (K) {
            case 3: return (int)launch_ln_fwd_4k_k3(bf16, la, ln, g, grid, s);
            case 5: return (int)launch_ln_fwd_4k_k5(bf16, la, ln, g, grid, s);
            case 7: return (int)launch_ln_fwd_4k_k7(bf16, la, ln, g, grid, s);
            case 9: return (int)launch_ln_fwd_4k_k9(bf16, la, ln, g, grid, s);
        }
        return -NPLM_DWCONV_EUNSUPPORTED;
    }
    switch (K) {
        case 3: return (int)launch_ln_fwd_k3(bf16, la, ln, g, grid, s);
        case 5: return (int)launch_ln_fwd_k5(bf16, la, ln, g, grid, s);
        case 7: return (int)launch_ln_fwd_k7(bf16, la, ln, g, grid, s);
        case 9: return (int)launch_ln_fwd_k9(bf16, la, ln, g, grid, s);
    }
    return -NPLM_DWCONV_EUNSUPPORTED;
}

// ---- backward of the LayerNorm-fused forward: conv backward over the re-normalised x (NORM variant of
// dwconv_bwd_lds_kernel: dn, dw, db and the LayerNorm parameter sums), then the LayerNorm input gradient ---------------
namespace {
bool ln_supported(bool bf16, int C, int K, uintptr_t align_bits) {
    return ln_whole_rows(bf16, C, K, align_bits) || ln_wide_rows(bf16, C, K, align_bits);
}
// workspace: [conv slabs: nbt x (K+1) x C][LayerNorm slabs: nbt x 2 x C][dn: T x C fp32], each part 256-byte aligned;
// rows of one 2 KiB column block finish dx inside the conv backward (the WHOLE variant) and need no dn
struct LnBwdLayout {
    LdsPlan lp;
    bool whole, whole4k;      // dx inside the conv backward: rows of one 2 KiB column block; rows of one 4 KiB block
    size_t conv_slabs, ln_slabs, dn, total;
};
int ln_bwd_layout(bool bf16, long long T, int C, int K, LnBwdLayout* out) {
    LnBwdLayout l{};
    l.whole4k = ln_bwd_whole_4k(bf16, C, K, 0);
    l.whole = l.whole4k || ln_whole_rows(bf16, C, K, 0);
    if (l.whole) {
        l.lp.sh = !l.whole4k ? lds_ln_bwd_shape(bf16, K) : lds_ln_bwd_rows3k(bf16, C) ? lds_ln_bwd_3k_shape(K) : lds_ln_bwd_wide_shape(bf16, K);
        l.lp.R = l.lp.sh.rw * l.lp.sh.nrg;
        l.lp.ncb = 1;
        l.lp.ntiles = ceil_div(T, l.lp.R);
        l.lp.nbt = l.lp.ntiles < kNumCU ? l.lp.ntiles : kNumCU;
        l.lp.xcd_group = (l.lp.nbt % (kNumXCD * 8) == 0) ? 8 : 0;
        // rows of 2 to 4 KiB: a tile is 5 to 10 rows behind K-1 halo rows of dy, and a neighbour on another XCD means reading
        // those from HBM again (fp32 C=1024, K=7: 6-row tiles, HBM-side reads 1.066 of x + dy with 8 consecutive tiles per
        // XCD); 32 consecutive tiles per XCD, as in the forward of these rows
        if (l.whole4k && l.lp.nbt % (kNumXCD * 32) == 0) l.lp.xcd_group = 32;
        l.lp.rot_step = l.lp.nbt > 2 ? (int)((long long)l.lp.nbt * 618 / 1000) | 1 : 0;
        if (l.lp.rot_step >= l.lp.nbt) l.lp.rot_step = l.lp.nbt - 1;
    } else {
        int rc = make_default_lds_plan(true, bf16, T, C, K, &l.lp);
        if (rc) return rc;
    }
    auto up = [](size_t v) { return (v + 255) & ~(size_t)255; };
    l.conv_slabs = up((size_t)l.lp.nbt * (K + 1) * C * sizeof(float));
    l.ln_slabs = up((size_t)l.lp.nbt * 2 * C * sizeof(float));
    l.dn = l.whole ? 0 : up((size_t)T * C * sizeof(float));
    l.total = l.conv_slabs + l.ln_slabs + l.dn;
    *out = l;
    return 0;
}
}  // namespace

size_t nplm_dwconv_ln_bwd_workspace_bytes(int64_t T, int32_t C, int32_t K, int32_t act_dtype) {
    if (check_common(T, C, K, 0, act_dtype, NPLM_DWCONV_F32) || T == 0) return 0;
    const bool bf16 = act_dtype == NPLM_DWCONV_BF16;
    if (!ln_supported(bf16, C, K, 0)) return 0;
    LnBwdLayout l;
    if (ln_bwd_layout(bf16, T, C, K, &l)) return 0;
    return l.total;
}

int nplm_dwconv_ln_bwd(const void* x, const void* dy, const int32_t* cu, const float* stats, const void* ln_weight,
                       const void* ln_bias, const void* w, void* dx, float* dw, float* db, float* dln_weight,
                       float* dln_bias, void* workspace, size_t workspace_bytes, int64_t T, int32_t C, int32_t K,
                       int32_t S, int32_t act_dtype, int32_t w_dtype, uint32_t flags, void* stream) {
    int rc = check_common(T, C, K, S, act_dtype, w_dtype);
    if (rc) return rc;
    if (flags & ~(uint32_t)(NPLM_DWCONV_RESIDUAL | NPLM_DWCONV_GRADS_BF16)) return -NPLM_DWCONV_EFLAGS;
    const int out_bf16 = (flags & NPLM_DWCONV_GRADS_BF16) ? 1 : 0;      // dw, db, dln_weight, dln_bias are bf16 buffers
    hipStream_t s = (hipStream_t)stream;
    if (!dw || !db || !dln_weight) return -NPLM_DWCONV_ENULL;
    if (T == 0) {
        auto zero = [&](float* p, long long n) { return out_bf16 ? fill_zero16(p, n, s) : fill_zero(p, n, s); };
        hipError_t e = zero(dw, (long long)C * K);
        if (e == hipSuccess) e = zero(db, C);
        if (e == hipSuccess) e = zero(dln_weight, C);
        if (e == hipSuccess) e = zero(dln_bias, C);
        return (int)e;
    }
    if (!x || !dy || !cu || !stats || !ln_weight || !w || !dx) return -NPLM_DWCONV_ENULL;
    const bool bf16 = act_dtype == NPLM_DWCONV_BF16;
    const uintptr_t E = bf16 ? 2 : 4;
    const uintptr_t WE = (w_dtype == NPLM_DWCONV_BF16) ? 2 : 4;
    if (((uintptr_t)w | (uintptr_t)ln_weight | (uintptr_t)ln_bias) % WE || ((uintptr_t)cu | (uintptr_t)stats) % 4 ||
        ((uintptr_t)dw | (uintptr_t)db | (uintptr_t)dln_weight | (uintptr_t)dln_bias) % (out_bf16 ? 2 : 4) ||
        ((uintptr_t)x | (uintptr_t)dy | (uintptr_t)dx) % E)
        return -NPLM_DWCONV_EALIGN;
    if (!ln_supported(bf16, C, K, (uintptr_t)x | (uintptr_t)dy | (uintptr_t)dx)) return -NPLM_DWCONV_EUNSUPPORTED;
    LnBwdLayout l;
    rc = ln_bwd_layout(bf16, T, C, K, &l);
    if (rc) return rc == -NPLM_DWCONV_ETUNING ? -NPLM_DWCONV_EUNSUPPORTED : rc;
    if (!workspace || (uintptr_t)workspace % 256 || workspace_bytes < l.total) return -NPLM_DWCONV_EWORKSPACE;
    char* ws = reinterpret_cast<char*>(workspace);
    float* part = reinterpret_cast<float*>(ws);
    float* part_ln = reinterpret_cast<float*>(ws + l.conv_slabs);
    float* dn = reinterpret_cast<float*>(ws + l.conv_slabs + l.ln_slabs);
    // the conv's own residual flag stays off: the identity branch bypasses the LayerNorm and joins where dx is formed
    // (the WHOLE variant takes the flag to mean exactly that)
    const int w_flags = kernel_w_flags(w_dtype, l.whole ? (flags & NPLM_DWCONV_RESIDUAL) : 0);
    const ConvPtrs la{x, dy, cu, w, nullptr, l.whole ? dx : (void*)dn, part};
    const LnSide ln{stats, ln_weight, ln_bias, part_ln};
    const LdsGeo g = make_lds_geo(l.lp, T, C, S, w_flags);
    const dim3 grid(l.lp.ncb * l.lp.nbt);
    hipError_t e = hipErrorInvalidConfiguration;
    if (l.whole4k) {
        switch (K) {
            case 3: e = launch_ln_bwd_whole4k_k3(bf16, la, ln, g, grid, s); break;
            case 5: e = launch_ln_bwd_whole4k_k5(bf16, la, ln, g, grid, s); break;
            case 7: e = launch_ln_bwd_whole4k_k7(bf16, la, ln, g, grid, s); break;
            case 9: e = launch_ln_bwd_whole4k_k9(bf16, la, ln, g, grid, s); break;
        }
    } else if (l.whole) {
        switch (K) {
            case 3: e = launch_ln_bwd_whole_k3(bf16, la, ln, g, grid, s); break;
            case 5: e = launch_ln_bwd_whole_k5(bf16, la, ln, g, grid, s); break;
            case 7: e = launch_ln_bwd_whole_k7(bf16, la, ln, g, grid, s); break;
            case 9: e = launch_ln_bwd_whole_k9(bf16, la, ln, g, grid, s); break;
        }
    } else {
        switch (K) {
            case 3: e = launch_ln_bwd_k3(bf16, la, ln, g, grid, s); break;
            case 5: e = launch_ln_bwd_k5(bf16, la, ln, g, grid, s); break;
            case 7: e = launch_ln_bwd_k7(bf16, la, ln, g, grid, s); break;
            case 9: e = launch_ln_bwd_k9(bf16, la, ln, g, grid, s); break;
        }
    }
    if (e != hipSuccess) return (int)e;
    // both slab sets in one launch; the LayerNorm slabs read as a conv of one tap: "dw" = d ln_weight, "db" = d ln_bias
    const int blocks_a = (int)(((long long)(K + 1) * C + 63) / 64), blocks_b = (int)((2LL * C + 63) / 64);
    hipLaunchKernelGGL(dwconv_finalize2_kernel<FIN_SPLIT>, dim3((unsigned)(blocks_a + blocks_b)), dim3(64 * FIN_SPLIT), 0, s,
                       (const float*)part, (int)K, dw, db, blocks_a, (const float*)part_ln, 1, dln_weight, dln_bias, l.lp.nbt, (int)C,
                       out_bf16);
    if (l.whole) return (int)hipGetLastError();
    const void* res = (flags & NPLM_DWCONV_RESIDUAL) ? dy : nullptr;
    const int nch = ln_row_chunks((long long)C * (long long)E);
    return (int)(bf16 ? launch_ln_bwd_dx<true>(nch, x, stats, ln_weight, w_flags, dn, res, dx, T, C, s)
                      : launch_ln_bwd_dx<false>(nch, x, stats, ln_weight, w_flags, dn, res, dx, T, C, s));
}

size_t nplm_dwconv_gated_bwd_workspace_bytes(int64_t T, int32_t C, int32_t K, int32_t act_dtype) {
    if (check_common(T, C, K, 0, act_dtype, NPLM_DWCONV_F32) || T == 0) return 0;
    K = exec_kernel_size(K);        // the slabs have the rows of the kernel size that runs
    const bool bf16 = act_dtype == NPLM_DWCONV_BF16;
    if (long_gated_bwd_supported(bf16, T, C, K, 0)) {
        // enough for either kernel: which one runs also depends on pointer alignment, not known here
        Plan p;
        if (make_long_gated_plan(bf16, T, C, K, &p)) return 0;
        int slabs = p.nbt;
        LdsPlan lp;
        if (split_gated_eligible(bf16, T, C, K, 0) && make_split_plan(false, bf16, T, C, K, nullptr, &lp, true) == 0 && lp.nbt > slabs)
            slabs = lp.nbt;
        const size_t bytes = (size_t)slabs * (K + 1) * C * sizeof(float);
        return (bytes + 255) & ~(size_t)255;
    }
    if (!gated_supported(true, bf16, T, C, K, 0)) return 0;
    LdsPlan lp;
    if (make_lds_plan(true, bf16, T, C, K, nullptr, &lp, true)) return 0;
    const size_t bytes = (size_t)lp.nbt * (K + 1) * C * sizeof(float);
    return (bytes + 255) & ~(size_t)255;
}

int nplm_dwconv_gated_bwd(const void* z, const void* dy, const int32_t* cu, const void* w, void* dz, float* dw,
                          float* db, void* workspace, size_t workspace_bytes, int64_t T, int32_t C, int32_t K,
                          int32_t S, int32_t act_dtype, int32_t w_dtype, uint32_t flags, void* stream) {
    int rc = check_common(T, C, K, S, act_dtype, w_dtype);
    if (rc) return rc;
    if (flags & ~(uint32_t)(NPLM_DWCONV_RESIDUAL | NPLM_DWCONV_GRADS_BF16)) return -NPLM_DWCONV_EFLAGS;
    const int out_bf16 = (flags & NPLM_DWCONV_GRADS_BF16) ? 1 : 0;      // dw, db are bf16 buffers
    hipStream_t s = (hipStream_t)stream;
    if (!dw || !db) return -NPLM_DWCONV_ENULL;
    if (T == 0) {
        hipError_t e = out_bf16 ? fill_zero16(dw, (long long)C * K, s) : fill_zero(dw, (long long)C * K, s);
        if (e == hipSuccess) e = out_bf16 ? fill_zero16(db, C, s) : fill_zero(db, C, s);
        return (int)e;
    }
    if (!z || !dy || !cu || !w || !dz) return -NPLM_DWCONV_ENULL;
    const int taps = lds_taps(K), lds_tap_off = (taps - K) / 2;
    const int tap_off = (exec_kernel_size(K) - K) / 2, tap_flags = tap_off << W_TAP_OFF_SHIFT;
    K = exec_kernel_size(K);        // from here on the kernel size that runs (workspace for slabs of K + 1 rows; dw rows stay the caller's)
    const bool bf16 = act_dtype == NPLM_DWCONV_BF16;
    const uintptr_t WE = (w_dtype == NPLM_DWCONV_BF16) ? 2 : 4;
    if ((uintptr_t)w % WE || (uintptr_t)cu % 4 || ((uintptr_t)dw | (uintptr_t)db) % (out_bf16 ? 2 : 4)) return -NPLM_DWCONV_EALIGN;
    const int algo = choose_gated_algo(true, bf16, w_dtype == NPLM_DWCONV_BF16, T, C, K, taps, S, (uintptr_t)z | (uintptr_t)dy | (uintptr_t)dz,
                                       (uintptr_t)dz);
    if (algo < 0) return algo;
    if (algo >= 3) {
        LdsPlan lp;
        const bool mfma = algo == 4;
        rc = mfma ? make_split_plan(false, bf16, T, C, K, nullptr, &lp, true, kMfmaGatedRows, kMfmaGatedCb)
                  : make_split_plan(false, bf16, T, C, K, nullptr, &lp, true);
        if (rc) return rc;
        const size_t slab = (size_t)(K + 1) * C * sizeof(float);
        if (!workspace || (uintptr_t)workspace % 256 || workspace_bytes < slab * (size_t)lp.nbt) return -NPLM_DWCONV_EWORKSPACE;
        float* part = reinterpret_cast<float*>(workspace);
        const ConvPtrs la{z, dy, cu, w, nullptr, dz, part};
        const LdsGeo lg = make_lds_geo(lp, T, C, S, kernel_w_flags(w_dtype, flags) | (mfma ? tap_flags : lds_tap_off << W_TAP_OFF_SHIFT));
        const dim3 grid(lp.ncb * lp.nbt);
        hipError_t e = mfma ? launch_bwd_gated_mfma_k31(la, lg, grid, s) : launch_bwd_split_gated(taps, bf16, la, lg, grid, s);
        if (e != hipSuccess) return (int)e;
        const long long n_out = (long long)(taps + 1) * C;
        hipLaunchKernelGGL(dwconv_finalize_kernel<FIN_SPLIT>, dim3((unsigned)((n_out + 63) / 64)), dim3(64 * FIN_SPLIT), 0, s,
                           (const float*)part, lp.nbt, C, taps, dw, db, out_bf16, lds_tap_off);
        return (int)hipGetLastError();
    }
    if (algo == 1) {
        Plan p;
        rc = make_long_gated_plan(bf16, T, C, K, &p);
        if (rc) return rc;
        const size_t slab = (size_t)(K + 1) * C * sizeof(float);
        if (!workspace || (uintptr_t)workspace % 256 || workspace_bytes < slab * (size_t)p.nbt) return -NPLM_DWCONV_EWORKSPACE;
        float* part = reinterpret_cast<float*>(workspace);
        const ConvPtrs a{z, dy, cu, w, nullptr, dz, part};
        const Geo g = make_geo(p, T, C, S, kernel_w_flags(w_dtype, flags) | tap_flags);
        const dim3 grid(p.ncb * p.nbt), block(p.bw * p.bt * 64);
        const size_t shmem = (size_t)p.bw * p.bt * p.vec * 64 * sizeof(float);
        hipError_t e = K == 15 ? launch_bwd_gated_k15(bf16, p.unroll, p.maxt, a, g, grid, block, shmem, s)
                               : launch_bwd_gated_k31(bf16, p.unroll, p.maxt, a, g, grid, block, shmem, s);
        if (e != hipSuccess) return (int)e;
        const long long n_out = (long long)(K + 1) * C;
        hipLaunchKernelGGL(dwconv_finalize_kernel<FIN_SPLIT>, dim3((unsigned)((n_out + 63) / 64)), dim3(64 * FIN_SPLIT), 0, s,
                           (const float*)part, p.nbt, C, K, dw, db, out_bf16, tap_off);
        return (int)hipGetLastError();
    }
    LdsPlan lp;
    rc = make_lds_plan(true, bf16, T, C, K, nullptr, &lp, true);
    if (rc) return rc == -NPLM_DWCONV_ETUNING ? -NPLM_DWCONV_EUNSUPPORTED : rc;
    const size_t slab_bytes = (size_t)(K + 1) * C * sizeof(float);
    if (!workspace || (uintptr_t)workspace % 256 || workspace_bytes < slab_bytes * (size_t)lp.nbt)
        return -NPLM_DWCONV_EWORKSPACE;
    float* part = reinterpret_cast<float*>(workspace);
    const ConvPtrs la{z, dy, cu, w, nullptr, dz, part};
    const bool narrow = lds_gated_narrow((long long)C * (bf16 ? 2 : 4), K);
    const LdsGeo g = make_lds_geo(lp, T, C, S, kernel_w_flags(w_dtype, flags) | tap_flags);
    const dim3 grid(lp.ncb * lp.nbt);
    hipError_t e = hipErrorInvalidConfiguration;
    switch (K) {
        case 3: e = launch_bwd_lds_gated_k3(bf16, narrow, la, g, grid, s); break;
        case 5: e = launch_bwd_lds_gated_k5(bf16, narrow, la, g, grid, s); break;
        case 7: e = launch_bwd_lds_gated_k7(bf16, narrow, la, g, grid, s); break;
        case 9: e = launch_bwd_lds_gated_k9(bf16, narrow, la, g, grid, s); break;
    }
    if (e != hipSuccess) return (int)e;
    const long long n_out = (long long)(K + 1) * C;
    hipLaunchKernelGGL(dwconv_finalize_kernel<FIN_SPLIT>, dim3((unsigned)((n_out + 63) / 64)), dim3(64 * FIN_SPLIT), 0, s,
                       (const float*)part, lp.nbt, C, K, dw, db, out_bf16, tap_off);
    return (int)hipGetLastError();
}

const char* nplm_dwconv_strerror(int code) {
    if (code == 0) return "success";
    if (code > 0) return hipGetErrorString((hipError_t)code);
    switch (-code) {
        case NPLM_DWCONV_ENULL: return "nplm_dwconv: a required pointer is NULL";
        case NPLM_DWCONV_ESHAPE: return "nplm_dwconv: invalid sizes (need 0 <= T <= 2^31 - 2^20 - 1, C >= 1, S >= 0, C*K < 2^28)";
        case NPLM_DWCONV_EKSIZE: return "nplm_dwconv: kernel size must be odd and in [1, 255]";
        case NPLM_DWCONV_EDTYPE: return "nplm_dwconv: unknown element type (0 = fp32, 1 = bf16)";
        case NPLM_DWCONV_EALIGN: return "nplm_dwconv: pointer not aligned to its element size";
        case NPLM_DWCONV_EWORKSPACE: return "nplm_dwconv: workspace NULL, not 256-byte aligned, or too small";
        case NPLM_DWCONV_ECU: return "nplm_dwconv: cu_seqlens must start at 0, be non-decreasing and end at T";
        case NPLM_DWCONV_EFLAGS: return "nplm_dwconv: unknown bits set in flags";
        case NPLM_DWCONV_EUNSUPPORTED: return "nplm_dwconv: shape not supported by the fused (gated, LayerNorm) kernels";
        case NPLM_DWCONV_ESCRATCH: return "nplm_dwconv: the dw/db partial sums of this shape do not fit the library's static scratch (16 MiB); use nplm_dwconv_bwd_ex with a caller-owned workspace";
        case NPLM_DWCONV_ETUNING: return "nplm_dwconv: geometry override not available in this build";
    }
    return "nplm_dwconv: unknown error code";
}

int nplm_dwconv_fwd(const void* x, const int32_t* cu, const void* w, const void* b, void* y, int64_t T, int32_t C,
                    int32_t K, int32_t S, int32_t act_dtype, int32_t w_dtype, void* stream) {
    return fwd_impl(x, cu, w, b, y, T, C, K, S, act_dtype, w_dtype, 0, stream, nullptr);
}

int nplm_dwconv_fwd_ex(const void* x, const int32_t* cu, const void* w, const void* b, void* y, int64_t T, int32_t C,
                       int32_t K, int32_t S, int32_t act_dtype, int32_t w_dtype, uint32_t flags, void* stream) {
    return fwd_impl(x, cu, w, b, y, T, C, K, S, act_dtype, w_dtype, flags, stream, nullptr);
}

int nplm_dwconv_fwd_tuned(const void* x, const int32_t* cu, const void* w, const void* b, void* y, int64_t T,
                          int32_t C, int32_t K, int32_t S, int32_t act_dtype, int32_t w_dtype, void* stream,
                          const nplm_dwconv_tuning* tune) {
    return fwd_impl(x, cu, w, b, y, T, C, K, S, act_dtype, w_dtype, tune ? tune->flags : 0u, stream, tune);
}

size_t nplm_dwconv_bwd_workspace_bytes(int64_t T, int32_t C, int32_t K, int32_t act_dtype) {
    if (check_common(T, C, K, 0, act_dtype, NPLM_DWCONV_F32) || T == 0) return 0;
    K = exec_kernel_size(K);        // the slabs have the rows of the kernel size that runs
    const bool bf16 = act_dtype == NPLM_DWCONV_BF16;
    // enough for whichever kernel family the library picks for these sizes (the choice also depends
    // on pointer alignment, which is not known here)
    Plan p;
    if (make_plan(true, bf16, T, C, K, 0, nullptr, &p)) return 0;
    int slabs = p.nbt;
    if (choose_algo(true, nullptr, bf16, true, T, C, K, K, 1, 0, 0) == 2) {
        LdsPlan lp;
        if (make_lds_plan(true, bf16, T, C, K, nullptr, &lp) == 0 && lp.nbt > slabs) slabs = lp.nbt;
    }
    if (split_eligible(bf16, T, C, K, 0)) {
        LdsPlan lp;
        if (make_split_plan(false, bf16, T, C, K, nullptr, &lp) == 0 && lp.nbt > slabs) slabs = lp.nbt;
    }
    const size_t bytes = (size_t)slabs * (K + 1) * C * sizeof(float);
    return (bytes + 255) & ~(size_t)255;
}

int nplm_dwconv_mask_cu(const void* mask, int32_t kind, int64_t row_stride, int64_t B, int64_t L, int32_t* cu, void* stream) {
    if (B < 1 || B > 1 << 28 || L < 1 || L > kMaxRows / B || row_stride < 0) return -NPLM_DWCONV_ESHAPE;    // a grid has fewer than 2^32 threads
    if (!mask || !cu) return -NPLM_DWCONV_ENULL;
    hipStream_t s = (hipStream_t)stream;
    switch (kind) {
        case 0: return (int)launch_mask_cu<uint8_t, true>(mask, row_stride, (int)L, (unsigned)B, cu, s);
        case 1: return (int)launch_mask_cu<int32_t, false>(mask, row_stride, (int)L, (unsigned)B, cu, s);
        case 2: return (int)launch_mask_cu<int64_t, false>(mask, row_stride, (int)L, (unsigned)B, cu, s);
        case 3: return (int)launch_mask_cu<uint8_t, false>(mask, row_stride, (int)L, (unsigned)B, cu, s);
    }
    return -NPLM_DWCONV_EDTYPE;
}

int32_t nplm_dwconv_exec_kernel_size(int32_t K) { return exec_kernel_size(K); }

int32_t nplm_dwconv_debug_algo(int32_t bwd, int64_t T, int32_t C, int32_t K, int32_t S, int32_t act_dtype, int32_t w_dtype) {
    const int rc = check_common(T, C, K, S, act_dtype, w_dtype);
    if (rc) return rc;
    return choose_algo(bwd != 0, nullptr, act_dtype == NPLM_DWCONV_BF16, w_dtype == NPLM_DWCONV_BF16, T, C, exec_kernel_size(K), lds_taps(K), S, 0, 0);
}

int32_t nplm_dwconv_debug_gated_algo(int32_t bwd, int64_t T, int32_t C, int32_t K, int32_t S, int32_t act_dtype, int32_t w_dtype) {
    const int rc = check_common(T, C, K, S, act_dtype, w_dtype);
    if (rc) return rc;
    return choose_gated_algo(bwd != 0, act_dtype == NPLM_DWCONV_BF16, w_dtype == NPLM_DWCONV_BF16, T, C, exec_kernel_size(K), lds_taps(K), S, 0, 0);
}

int32_t nplm_dwconv_bwd_slabs(int64_t T, int32_t C, int32_t K, int32_t act_dtype, const nplm_dwconv_tuning* tune) {
    if (check_common(T, C, K, 0, act_dtype, NPLM_DWCONV_F32) || T == 0) return 0;
    K = exec_kernel_size(K);
    const bool bf16 = act_dtype == NPLM_DWCONV_BF16;
    const int algo = choose_algo(true, tune, bf16, true, T, C, K, K, 1, 0, 0);
    if (algo < 0) return 0;
    if (algo >= 3) {
        LdsPlan lp;
        if (make_split_plan(false, bf16, T, C, K, tune, &lp)) return 0;
        return lp.nbt;
    }
    if (algo == 2) {
        LdsPlan lp;
        if (make_lds_plan(true, bf16, T, C, K, tune, &lp)) return 0;
        return lp.nbt;
    }
    Plan p;
    if (make_plan(true, bf16, T, C, K, 0, tune, &p)) return 0;
    return p.nbt;
}

int nplm_dwconv_bwd(const void* x, const void* dy, const int32_t* cu, const void* w, void* dx, float* dw, float* db,
                    void* workspace, size_t workspace_bytes, int64_t T, int32_t C, int32_t K, int32_t S,
                    int32_t act_dtype, int32_t w_dtype, void* stream) {
    return bwd_impl(x, dy, cu, w, dx, dw, db, workspace, workspace_bytes, T, C, K, S, act_dtype, w_dtype, 0, stream,
                    nullptr);
}

int nplm_dwconv_bwd_ex(const void* x, const void* dy, const int32_t* cu, const void* w, void* dx, float* dw, float* db,
                       void* workspace, size_t workspace_bytes, int64_t T, int32_t C, int32_t K, int32_t S,
                       int32_t act_dtype, int32_t w_dtype, uint32_t flags, void* stream) {
    return bwd_impl(x, dy, cu, w, dx, dw, db, workspace, workspace_bytes, T, C, K, S, act_dtype, w_dtype, flags,
                    stream, nullptr);
}

int nplm_dwconv_bwd_static(const void* x, const void* dy, const int32_t* cu, const void* w, void* dx, float* dw,
                           float* db, int64_t T, int32_t C, int32_t K, int32_t S, int32_t act_dtype, int32_t w_dtype,
                           uint32_t flags, void* stream) {
    const int rc = check_common(T, C, K, S, act_dtype, w_dtype);
    if (rc) return rc;
    void* ws = nullptr;
    size_t ws_bytes = 0;
    if (T > 0 && (dw || db)) {
        // the same number of slabs nplm_dwconv_bwd_ex would ask its caller for
        ws_bytes = nplm_dwconv_bwd_workspace_bytes(T, C, K, act_dtype);
        if (ws_bytes == 0 || ws_bytes > (size_t)NPLM_DWCONV_STATIC_SCRATCH_BYTES) return -NPLM_DWCONV_ESCRATCH;
        const hipError_t e = static_scratch_for_current_device(&ws);
        if (e != hipSuccess) return (int)e;
    }
    return bwd_impl(x, dy, cu, w, dx, dw, db, ws, ws_bytes, T, C, K, S, act_dtype, w_dtype, flags, stream, nullptr);
}

int nplm_dwconv_bwd_tuned(const void* x, const void* dy, const int32_t* cu, const void* w, void* dx, float* dw,
                          float* db, void* workspace, size_t workspace_bytes, int64_t T, int32_t C, int32_t K,
                          int32_t S, int32_t act_dtype, int32_t w_dtype, void* stream,
                          const nplm_dwconv_tuning* tune) {
    return bwd_impl(x, dy, cu, w, dx, dw, db, workspace, workspace_bytes, T, C, K, S, act_dtype, w_dtype,
                    tune ? tune->flags : 0u, stream, tune);
}

int nplm_dwconv_debug_copy(const void* src, void* dst, size_t bytes, void* stream) {
    if (!src || !dst) return -NPLM_DWCONV_ENULL;
    if (bytes % 16 || ((uintptr_t)src | (uintptr_t)dst) % 16) return -NPLM_DWCONV_EALIGN;
    if (bytes == 0) return 0;
    const size_t nvec = bytes / 16;
    hipLaunchKernelGGL(copy_chunks_kernel, dim3((unsigned)((nvec + 1023) / 1024)), dim3(256), 0, (hipStream_t)stream,
                       (const u32x4*)src, (u32x4*)dst, nvec);
    return (int)hipGetLastError();
}

int64_t nplm_dwconv_debug_intervals(const int32_t* cu_host, int32_t S, int64_t T, int64_t start, int64_t step,
                                    int64_t relocate_every, int32_t* cs_out, int32_t* ce_out) {
    if (!cu_host || !cs_out || !ce_out || S < 0 || T < 0 || T > kMaxRows || start < 0 || step < 1) return -1;
    SeqCursor sc;
    sc.seq = 0; sc.cs = 0; sc.ce = 0;
    int64_t n = 0;
    for (int64_t t = start; t < T; t += step, ++n) {
        if (n == 0 || (relocate_every > 0 && n % relocate_every == 0))
            sc.locate(cu_host, S, (int)T, (int)t, sc.seq);
        else
            sc.advance(cu_host, S, (int)T, (int)t);
        cs_out[n] = sc.cs;
        ce_out[n] = sc.ce;
    }
    return n;
}

int64_t nplm_dwconv_debug_starts(const int32_t* cu_host, int32_t S, int64_t T, int32_t a, int32_t n, uint32_t* marks_out) {
    if (!cu_host || !marks_out || S < 0 || T < 0 || T > kMaxRows || n < 1 || n > 256) return -1;
    struct Lanes {
        const int32_t* cu;
        uint32_t* words;
        int a, n;
        int64_t reads;
        void mark(int row) {
            const uint32_t p = (uint32_t)row - (uint32_t)a;
            if (row > a && p < (uint32_t)n) words[(p - 1) >> 5] |= 1u << ((p - 1) & 31);
        }
        uint64_t above(uint32_t lo, uint32_t step, uint32_t end, int row) {
            ++reads;
            uint64_t m = 0;
            for (uint32_t l = 0; l < 64; ++l) {
                const uint32_t i = lo + (l + 1) * step - 1;
                m |= (uint64_t)(cu[i < end ? i : end] > row) << l;
            }
            return m;
        }
        int take(uint32_t lo, uint32_t end, int& first) {
            ++reads;
            for (uint32_t l = 0; l < 64; ++l) mark(cu[lo + l < end ? lo + l : end]);
            first = cu[lo < end ? lo : end];
            return cu[lo + 63 < end ? lo + 63 : end];
        }
    } lanes{cu_host, marks_out, a, n, 0};
    for (int i = 0; i < (n + 31) / 32; ++i) marks_out[i] = 0;
    lanes.mark((int)T);
    walk_starts(lanes, S, (int)T, a, n);
    return lanes.reads;
}

int nplm_dwconv_check_cu(const int32_t* cu, int32_t S, int64_t T, void* stream) {
    if (!cu) return -NPLM_DWCONV_ENULL;
    if (S < 0 || T < 0 || T > kMaxRows) return -NPLM_DWCONV_ESHAPE;
    std::vector<int32_t> h((size_t)S + 1);
    hipError_t e = hipMemcpyAsync(h.data(), cu, h.size() * sizeof(int32_t), hipMemcpyDeviceToHost, (hipStream_t)stream);
    if (e == hipSuccess) e = hipStreamSynchronize((hipStream_t)stream);
    if (e != hipSuccess) return (int)e;
    if (h[0] != 0 || h[S] != (int32_t)T) return -NPLM_DWCONV_ECU;
    for (int32_t i = 0; i < S; ++i)
        if (h[i + 1] < h[i]) return -NPLM_DWCONV_ECU;
    return 0;
}

}  // extern "C"
