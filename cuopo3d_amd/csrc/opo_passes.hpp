// opo_passes.hpp -- the two passes of a z-slice as device functions, shared
// by the single-solve kernels and the batched (many-solve) kernels.
//
//   nl_time_tile  one tile of the fused pass: pointwise RK4 half step(s) of
//                 the three fields, then the along-t line operator
//                 (dispersion/walk-off/absorption, or GDD at a trip's end);
//   nl_time_reg   the same for long lines, fields in registers;
//   nl_plane_slices  all slices of a plane wave.
#pragma once
#include "opo_device.hpp"
#include "opo_kernels.hpp"
#include "opo_mfma.hpp"
#include "opo_rk4.hpp"

namespace opo {

// Whether a solve has stopped (its status word is set).  Kernels read the word
// first and look at it once their field loads are out: returning at once would put a
// read from memory ahead of the first field load of every launch.
__device__ __forceinline__ int stop_flag(const int *status) { return status ? *status : 0; }

// Blocks are handed to the 8 XCDs round-robin (block b runs on XCD b % 8).
// Remap so that neighbouring tiles, which share cache lines at the tile
// edges, are processed on the same XCD and hit its L2.
__device__ __forceinline__ int xcd_local_tile(int b, int nb) {
    if (nb % 8 != 0) return b;
    return (b % 8) * (nb / 8) + b / 8;
}

// LDS budget of the fused pass: three tiles of NT x TX <= 48 KiB (two or
// more workgroups per CU), at least 4 pixels wide.
template <typename T, int NT> constexpr int tline3_tx() {
    constexpr int per_px = 3 * NT * (int)sizeof(cplx<T>);
    constexpr int tx = (per_px * 4 > 49152) ? 98304 / per_px : 49152 / per_px;
    return tx >= 16 ? 16 : (tx >= 8 ? 8 : (tx >= 4 ? 4 : (tx >= 2 ? 2 : 1)));
}

// LDS layout of one field's tile in the fused pass: time row t (TX
// pixels) starts at t*TX + (t / G)*PAD, G the innermost group length of
// the line operator (N2 of the two-level split, N3 of the three-level one).
// Narrow tiles pad every G rows by TX elements so the rows that the
// innermost phase walks in parallel fall in different banks.
// Rows between two pads of a narrow tile: the innermost group of the line
// operator.  (Padding 2-pixel 2048-sample tiles every 16 rows instead,
// conflict-free in a 64-bank model of the LDS, measured no faster.)
// One-pixel tiles of lines that are three-level in any case (FP64 2048, FP32
// 4096) are the same in USE_ONE and USE_T.
template <int TX> constexpr int tile_use() { return TX == 1 ? USE_ONE : USE_T; }
template <typename T, int NT, int TX> constexpr int pad_group() { return inner_len<T, NT, tile_use<TX>()>(); }
template <typename T, int NT, int TX> struct TimeTile {
    static constexpr int G = pad_group<T, NT, TX>();
    static constexpr int PAD = (G > 1 && TX < 16) ? TX : 0;
    static constexpr int FT = NT * TX + (NT / G) * PAD;   // elements per field
    __device__ static __forceinline__ int at(int i) { return i + (i / (G * TX)) * PAD; }
};

// Tasks of a line-operator phase per line (of the phase with the fewest).
template <typename T, int NT> constexpr int phase_tasks() {
    if constexpr (three_level<T, NT>()) return NT / (Split3<NT>::N1 > Split3<NT>::N2 ? Split3<NT>::N1 : Split3<NT>::N2);
    else return NT / (Split<NT>::N1 > Split<NT>::N2 ? Split<NT>::N1 : Split<NT>::N2);
}

// Points of the outer register DFT of a three-level time line (two-level lines
// have no register form: 1), and the threads of a tile that each hold that many
// samples of one pixel.
template <typename T, int NT> constexpr int outer_radix() {
    if constexpr (three_level<T, NT>()) return Split3<NT>::N1;
    else return 1;
}
template <typename T, int NT, int TX> constexpr int reg_threads() { return TX * NT / outer_radix<T, NT>(); }
// Waves per SIMD the register form is compiled for.
template <typename T, int NT, int TX> constexpr int reg_waves() {
    return reg_threads<T, NT, TX>() < 512 ? 3 : (outer_radix<T, NT>() == 8 ? 4 : 2);
}

// Elements a persistent workgroup of the fused pass stages in LDS: the
// rotation table, then three line tables of (hi, lo) pairs.
template <typename T, int NT, int TX> constexpr int time_stage_elems() {
    return tw_elems<T, NT, tile_use<TX>()>() + 6 * NT;
}

// Launch variants of the fused pass for one NT (chosen by the autotuner).
// V < 9: one tile per workgroup, V = 3 m + b with tile width m = 0: TXd,
// 1: TXd/2, 2: 2 TXd pixels and b = 0: 256, 1: 512, 2: 384 or 768 threads
// (as many as a line-operator phase of the three fields has tasks).  V >= 9: persistent workgroups (k + 1 per CU), each walking a
// contiguous run of tiles with the next tile prefetched into registers;
// V - 9 = 2 (3 m + b) + k with b = 0: 256, 1: 384, 2: 512 threads.
// FP64 has the one-tile variants only; NT < 64 only variant 0; a variant whose three
// tiles exceed 112 KiB of LDS (persistent: tiles plus staged tables beyond
// 144 KiB) does not exist, nor persistent variants of lines longer than 256
// samples.  (Not offered, measured slower or no faster on every grid: a form
// that keeps whole t-lines in one wave's registers, exchanging through
// wave-private LDS, 15-40 % slower; 1024 threads per tile; persistent workgroups on 512- to
// 2048-sample lines, 23-90 % slower, their prefetch registers spilling
// beside 32- and 64-point register DFTs, also with only the twiddles
// staged so that 4-pixel tiles fit; the register form of 64- to 256-sample lines,
// at most equal and on 32 x 32 x 128 21 against 14.5 us per slice, of 2-pixel
// 2048-sample tiles, 1650 against 1290, and of 4096 samples, spilling 292 bytes,
// 1575 against 886.)
constexpr int kTimeClassic = 9;
constexpr int kTimeVariants = kTimeClassic + 18;
template <typename T, int NT, int V> struct TimeVariant {
    static constexpr int txd = tline3_tx<T, NT>();
    static constexpr bool persistent = V >= kTimeClassic;
    static constexpr int idx = persistent ? V - kTimeClassic : V;
    static constexpr int m = persistent ? idx / 6 : idx / 3;
    static constexpr int b = persistent ? (idx / 2) % 3 : idx % 3;
    static constexpr int per_cu = persistent ? idx % 2 + 1 : 0;
    static constexpr int tx = m == 0 ? txd : (m == 1 ? txd / 2 : txd * 2);
    // threads of b = 2: one task each in the phases of the three fields
    static constexpr int wide = 3 * phase_tasks<T, NT>() * tx >= 768 ? 768 : 384;
    // the register form (nl_time_reg): b = 0 of FP32 lines of 512 and 1024
    // samples and the 4-pixel tile of 2048 (shorter lines: at most equal, 60 %
    // slower on small grids; 2-pixel tiles of 2048 28 % slower than the classic)
    static constexpr bool reg =
        sizeof(T) == 4 && !persistent && b == 0 && (NT == 512 || NT == 1024 || (NT == 2048 && m == 2));
    static constexpr int bs = reg ? reg_threads<T, NT, (tx > 0 ? tx : 1)>() : persistent ? (b == 0 ? 256 : (b == 1 ? 384 : 512)) : (b == 0 ? 256 : (b == 1 ? 512 : wide));
    // one-pixel tiles only where nothing wider fits (FP64 2048-sample lines:
    // there they give the 384- and 512-thread blocks)
    static constexpr int min_tx = ((sizeof(T) == 8 && NT >= 2048) || NT >= 4096) ? 1 : 2;
    static constexpr int data_bytes = 3 * TimeTile<T, NT, (tx > 0 ? tx : 1)>::FT * (int)sizeof(cplx<T>);
    static constexpr int table_bytes = time_stage_elems<T, NT, 2>() * (int)sizeof(cplx<T>);
    static constexpr bool valid =
        (V == 0 || reg) ? (V == 0 || (tx >= min_tx && tx <= 32 && bs >= 64 && bs <= 512)) : ((sizeof(T) == 4 || !persistent) && NT >= 64 && tx >= min_tx && tx <= 32 && data_bytes <= 114688 &&
                   (!persistent || (NT <= 256 && data_bytes + table_bytes <= 147456)));
};
// Untuned choice for `pixels` pixels of an NT class (0: many), from tuner runs
// on square grids; us per slice, both passes, chosen against the next best or
// the plain default (tile TXd, 512 threads):
//  * FP32 2048: 4-pixel register tiles, 128^2 1130 against 1290, 32^2 58 / 71
//    (16^2, 64 tiles: 49 / 40);
//  * FP32 1024: register tiles of 8 pixels from 128^2 (484 / 510), of 4 from
//    64^2 (99 / 109), below 768 threads (32^2 34.4 / 35.7, register 44);
//  * FP32 512: 8-pixel register tiles from 64^2 (47.6 / 49.8, 128^2 180 /
//    191), below 768 threads (32^2 26.6 / 26.9, register 29.4);
//  * lines of 64 to 1024 samples on fewer than 1024 pixels, and of up to 256
//    on fewer than 4096, half the tile, so that more CUs have one (16^2 x 1024
//    22.0 / 25.5, 32^2 x 128 12.9 / 14.5, 32^2 x 256 17.0 / 17.9);
//  * FP64: 512 threads (64^2 x 256 55.9 / 58.8 on 256), 128 samples half the
//    tile on 256 threads (96^2 69 / 73), 64 samples half the tile on 512
//    below 256^2 (64^2 25.5 / 26.6, 512^2 1469 / 1283), 2048 one pixel on 384 (64^2 607 / 618).
// A number of pixels from every range that the rule tells apart.
constexpr long long kPixelSteps[] = {1, 1024, 4096, 16384, 65536};
constexpr int time_default_variant(bool fp64, int nt, long long pixels) {
    if (nt < 64) return 0;
    const bool few = pixels > 0 && pixels < 4096, least = pixels > 0 && pixels < 1024;
    if (fp64) {
        if (nt >= 2048) return 2;
        if (nt == 128) return 3;
        if (nt == 64) return pixels > 0 && pixels < 65536 ? 4 : 1;
        return least && nt == 256 ? 4 : 1;
    }
    if (nt >= 4096) return 1;
    if (nt >= 2048) return least ? 1 : 6;
    if (nt >= 512) return least ? 4 : (few ? 2 : (nt == 512 || pixels == 0 || pixels >= 16384 ? 6 : 0));
    return few ? 4 : 1;
}

// Variants of the xy pass.  16 <= NX <= 32: V < 3 one plane per workgroup, V = 3
// + b groups of 256 / NX planes (xy_group) on 256, 512 or 1024 threads.  FP64 256:
// the band shapes of xy_split_launch.  The other sizes have one launch shape,
// and every number that stood for a block size or for persistent workgroups of
// lines in LDS is taken for it (saved choices stay valid): xy_variant_shape is the
// number that the tuner times for V.  (Persistent workgroups walking a run of
// matrix-core planes, one or two per CU, are slower: batched 64-point planes 311
// and 221 against 201 us per launch, 96 566 and 456 against 442, 128 675 and 610
// against 552.)
constexpr int kXyVariants = 9;
constexpr bool xy_variant_numbered(bool fp64, int nx, int v) {
    if (v < 0 || v >= kXyVariants) return false;
    if (nx < 16 || nx == 512) return v == 0;
    if (nx == 256 || (fp64 && nx == 128)) return v < 3;
    if (nx <= 32) return v < 6;
    return v < 3 || (!fp64 && nx * nx / (256 << ((v - 3) / 2)) <= 16);
}
constexpr int xy_variant_shape(bool fp64, int nx, int v) {
    if (fp64 && nx == 256) return v;
    return nx <= 32 && v >= 3 ? v : 0;
}
// Threads per workgroup.
constexpr int xy_variant_bs(bool fp64, int nx, int v) {
    if (nx == 256) return fp64 && v == 1 ? 512 : 256;
    if (nx == 512) return fp64 ? 256 : 512;
    if (nx < 16) return 256;
    return nx <= 32 && v >= 3 ? 256 << (v - 3) : 4 * nx;
}
// Untuned choice: one plane per workgroup; FP64 256-point planes in bands of
// 16 (256 x 256 x 64 242 us per slice).
constexpr int xy_default_variant(bool fp64, int nx) { return fp64 && nx == 256 ? 2 : 0; }

template <typename T> struct alignas(4 * sizeof(T)) cpair {
    cplx<T> a, b;
};

// Values move component-wise: a cpair<double> or cplx<double> copied as a
// struct between memory spaces goes through a private-memory temporary
// (scratch) in the fused-pass kernels.
template <typename T> __device__ __forceinline__ cplx<T> ld_c(const cplx<T> *p) { return cplx<T>{p->x, p->y}; }
template <typename T> __device__ __forceinline__ void st_c(cplx<T> *p, cplx<T> v) {
    p->x = v.x;
    p->y = v.y;
}
// Two consecutive cells of a field in global memory (p 4 sizeof(T)-byte
// aligned: an even cell index), to registers and back from LDS (q).
template <typename T> __device__ __forceinline__ cpair<T> load_pair(const cplx<T> *p) {
    const OPO_GLOBAL cpair<T> *g = (const OPO_GLOBAL cpair<T> *)p;
    return cpair<T>{cplx<T>{g->a.x, g->a.y}, cplx<T>{g->b.x, g->b.y}};
}
template <typename T> __device__ __forceinline__ void store_pair(cplx<T> *p, const cplx<T> *q) {
    OPO_GLOBAL cpair<T> *g = (OPO_GLOBAL cpair<T> *)p;
    const cplx<T> a = ld_c(q), b = ld_c(q + 1);
    g->a.x = a.x;
    g->a.y = a.y;
    g->b.x = b.x;
    g->b.y = b.y;
}

// Pointwise part of the fused pass for two cells: RK4 half step(s), then
// the mirror factors on s and i when the pass closes a round trip.
template <typename T, bool PHASE>
__device__ __forceinline__ void nl_point_pair(const Rk4Args<T> &rk, int t, Tri<T> &A0, Tri<T> &A1) {
    if (rk.nsteps > 0) {
        rk4_half_step<T, PHASE>(rk, 0, A0);
        rk4_half_step<T, PHASE>(rk, 0, A1);
        if (rk.nsteps > 1) {
            rk4_half_step<T, PHASE>(rk, 1, A0);
            rk4_half_step<T, PHASE>(rk, 1, A1);
        }
    }
    if (rk.out_scale) {
        if (rk.eom) {
            const cplx<T> e = rk.eom[2 * t], el = rk.eom[2 * t + 1];
            A0.s = cmul_hl(A0.s, e, el);
            A1.s = cmul_hl(A1.s, e, el);
            A0.i = cmul_hl(A0.i, e, el);
            A1.i = cmul_hl(A1.i, e, el);
        }
        const cplx<T> ms = {rk.ms_re, rk.ms_im}, msl = {rk.ms_lo_re, rk.ms_lo_im};
        const cplx<T> mi = {rk.mi_re, rk.mi_im}, mil = {rk.mi_lo_re, rk.mi_lo_im};
        A0.s = cmul_hl(A0.s, ms, msl);
        A1.s = cmul_hl(A1.s, ms, msl);
        A0.i = cmul_hl(A0.i, mi, mil);
        A1.i = cmul_hl(A1.i, mi, mil);
    }
}

// Pointwise part of the fused pass for one cell at time sample t (the same
// operations as nl_point_pair applies to each of its two cells).
template <typename T, bool PHASE>
__device__ __forceinline__ void nl_point(const Rk4Args<T> &rk, int t, Tri<T> &A) {
    if (rk.nsteps > 0) rk4_half_step<T, PHASE>(rk, 0, A);
    if (rk.nsteps > 1) rk4_half_step<T, PHASE>(rk, 1, A);
    if (rk.out_scale) {
        if (rk.eom) {
            const cplx<T> e = rk.eom[2 * t], el = rk.eom[2 * t + 1];
            A.s = cmul_hl(A.s, e, el);
            A.i = cmul_hl(A.i, e, el);
        }
        A.s = cmul_hl(A.s, cplx<T>{rk.ms_re, rk.ms_im}, cplx<T>{rk.ms_lo_re, rk.ms_lo_im});
        A.i = cmul_hl(A.i, cplx<T>{rk.mi_re, rk.mi_im}, cplx<T>{rk.mi_lo_re, rk.mi_lo_im});
    }
}

// Whether a one-tile workgroup of the fused pass copies the rotation table
// into LDS: both outer phases of the line operator then read it there
// instead of every lane fetching its pairs through the vector memory path,
// whose latency the reverse phase has nothing to hide behind.  For lines of
// 64 (256 x 256 x 64 cavity 1.6 % faster, 512 x 512 x 64 3.5 %, grids below
// 1 MB within 1 %) to 1024 samples, where the copy fits beside the tile;
// 2048-sample lines measured no faster (145.8 against 145.5 ms per
// 128 x 128 x 2048 trip), copying the line tables as well 0.1-1.3 % slower.
template <typename T, int NT, int TX> constexpr bool time_stage_twiddles() {
    return NT >= 64 && NT <= 1024 &&
           (3 * TimeTile<T, NT, TX>::FT + tw_elems<T, NT, tile_use<TX>()>()) * (int)sizeof(cplx<T>) <= 150 * 1024;
}

// One tile of the fused pass: TX consecutive pixels of row y, all NT time
// samples, all three fields.  lds holds 3 * NT * TX elements; twl holds the
// staged rotation table where time_stage_twiddles() (else unused).
template <typename T, int NT, int TX, int BS, bool PHASE>
__device__ __forceinline__ void nl_time_tile(const TLine3Args<T> &a, int nx, int ny, int tile,
                                             const cplx<T> *__restrict__ tw, cplx<T> *lds, cplx<T> *twl, int stop) {
    using L = TimeTile<T, NT, TX>;
    constexpr int TILE = NT * TX, FT = L::FT;
    constexpr bool STW = time_stage_twiddles<T, NT, TX>();
    constexpr int TWN = tw_elems<T, NT, tile_use<TX>()>(), TWP = STW ? (TWN + BS - 1) / BS : 1;
    const int tid = threadIdx.x;
    // twiddle copy: loads issued now, stored to LDS after the pointwise step
    cplx<T> twr[TWP];
    if constexpr (STW) {
#pragma unroll
        for (int j = 0; j < TWP; ++j)
            if (tid + j * BS < TWN) twr[j] = gld_c(tw + tid + j * BS);
    }
    // FP64 lines of 16: looked at late, the word cost 20 VGPRs and 3 % of a
    // 512 x 512 x 16 trip.
    constexpr bool STOP_FIRST = sizeof(T) == 8 && NT == 16;
    if (STOP_FIRST && stop) return;
    const int tiles_x = nx / TX;
    const int y = tile / tiles_x, x0 = (tile % tiles_x) * TX;
    const size_t plane = (size_t)nx * ny;
    const size_t base = (size_t)y * nx + x0;
    const Rk4Args<T> &rk = a.rk;
    // pointwise step in registers, two pixels per thread per iteration
    // (versions that issued the loads of one or of four iterations ahead of
    // the arithmetic were measured no faster: more registers, no latency
    // gained)
    if constexpr (TX % 2 == 0) {
        for (int i = 2 * tid; i < TILE; i += 2 * BS) {
            const int t = i / TX, xl = i % TX;
            const size_t gi = (size_t)t * plane + base + xl;
            cpair<T> p = load_pair(a.psrc + gi);
            cpair<T> s = load_pair(a.f[1] + gi);
            cpair<T> q = load_pair(a.f[2] + gi);
            Tri<T> A0 = {p.a, s.a, q.a}, A1 = {p.b, s.b, q.b};
            nl_point_pair<T, PHASE>(rk, t, A0, A1);
            const int li = L::at(i);
            lds[li] = A0.p;
            lds[li + 1] = A1.p;
            lds[FT + li] = A0.s;
            lds[FT + li + 1] = A1.s;
            lds[2 * FT + li] = A0.i;
            lds[2 * FT + li + 1] = A1.i;
        }
    } else {
        for (int i = tid; i < TILE; i += BS) {
            const int t = i / TX, xl = i % TX;
            const size_t gi = (size_t)t * plane + base + xl;
            Tri<T> A = {gld_c(a.psrc + gi), gld_c(a.f[1] + gi), gld_c(a.f[2] + gi)};
            nl_point<T, PHASE>(rk, t, A);
            const int li = L::at(i);
            lds[li] = A.p;
            lds[FT + li] = A.s;
            lds[2 * FT + li] = A.i;
        }
    }
    if constexpr (STW) {
#pragma unroll
        for (int j = 0; j < TWP; ++j)
            if (tid + j * BS < TWN) st_c(twl + tid + j * BS, twr[j]);
    }
    __syncthreads();
    if (!STOP_FIRST && stop) return;
    const LineSet<T> ls{lds + a.first_field * FT, FT, a.tab0, a.tab_stride, 3 - a.first_field};
    // the line tables are in global memory (measured: the batched 512-sample
    // t pass 0.5 % faster than with generic reads; the xy planes were slower)
    line_op_any<T, NT, +1, 1, TX, L::PAD, false, L::G, true, TwShear, tile_use<TX>()>(ls, TX, STW ? twl : tw, tid, BS);
    if constexpr (TX % 2 == 0) {
        for (int i = 2 * tid; i < TILE; i += 2 * BS) {
            const int t = i / TX, xl = i % TX;
            const size_t gi = (size_t)t * plane + base + xl;
            const int li = L::at(i);
            store_pair(a.f[0] + gi, lds + li);
            store_pair(a.f[1] + gi, lds + FT + li);
            store_pair(a.f[2] + gi, lds + 2 * FT + li);
        }
    } else {
        for (int i = tid; i < TILE; i += BS) {
            const int t = i / TX, xl = i % TX;
            const size_t gi = (size_t)t * plane + base + xl;
            for (int f = 0; f < 3; ++f) gst_c(a.f[f] + gi, ld_c(lds + f * FT + L::at(i)));
        }
    }
}



// Copy the rotation table and the line tables of fields first..2
// (each 2NT elements, tab_stride apart) into stab.
template <typename T, int NT, int TX>
__device__ __forceinline__ void stage_time_tables(const cplx<T> *__restrict__ tw, const TLine3Args<T> &a,
                                                  cplx<T> *stab, int tid, int nthr) {
    // the four arrays' loads of an index go out together (one memory
    // latency per index instead of one per array)
    constexpr int TWN = tw_elems<T, NT, tile_use<TX>()>();
    static_assert(TWN <= 2 * NT, "one index range covers the rotations and the tables");
    const int nf = 3 - a.first_field;
    for (int i = tid; i < 2 * NT; i += nthr) {
        cplx<T> v[4];
        if (i < TWN) v[0] = gld_c(tw + i);
#pragma unroll
        for (int f = 0; f < 3; ++f)
            if (f < nf) v[1 + f] = gld_c(a.tab0 + (size_t)f * a.tab_stride + i);
        if (i < TWN) stab[i] = v[0];
#pragma unroll
        for (int f = 0; f < 3; ++f)
            if (f < nf) stab[TWN + 2 * NT * f + i] = v[1 + f];
    }
}

// All slices of a plane-wave solve (1 x 1 pixel, no transverse step) in one
// launch: the line stays in LDS from slice to slice, with the rotations and
// the tables staged beside it where they fit.  One workgroup per solve, so
// nothing but latency bounds it: a launch per slice spent 4.4 us on
// 256 samples (the kernel boundary, the field and constant reads from L2),
// the loop 2.0 us
// (2048 samples 18.4 -> 8.1 us).  The operations are those of the launches it replaces.
// Threads: enough for one cell each in the pointwise step and one task each
// in the phases, within the registers of the long lines.
template <typename T, int NT> constexpr int plane_threads() {
    if constexpr (sizeof(T) == 8) return NT >= 512 ? 512 : 256;
    else return NT >= 1024 ? 768 : (NT >= 512 ? 512 : 256);
}
// Elements staged beside the line: rotations and tables where 156 KiB of LDS
// hold them (FP32 to 1024 samples, FP64 to 512), else in FP32 the rotations
// (4096 samples 16.9 -> 14.8 us per slice), in FP64 nothing (with the
// rotations 2048 samples went 11.2 -> 11.9 us).
template <typename T, int NT> constexpr int plane_stage_elems() {
    constexpr int all = time_stage_elems<T, NT, 1>();
    return (3 * TimeTile<T, NT, 1>::FT + all) * (int)sizeof(cplx<T>) <= 156 * 1024 ? all
           : sizeof(T) == 4                                                         ? tw_elems<T, NT, USE_ONE>()
                                                                                    : 0;
}
template <typename T, int NT, int BS>
__device__ __forceinline__ void nl_plane_slices(const TLine3Args<T> &a, int slices, const cplx<T> *__restrict__ tw,
                                                cplx<T> *lds, cplx<T> *stab) {
    using L = TimeTile<T, NT, 1>;
    constexpr int FT = L::FT;
    constexpr int TWN = tw_elems<T, NT, USE_ONE>();
    constexpr int SE = plane_stage_elems<T, NT>();
    constexpr bool ST = SE > TWN;
    const int tid = threadIdx.x;
    if constexpr (ST) {
        stage_time_tables<T, NT, 1>(tw, a, stab, tid, BS);
    } else {
        for (int i = tid; i < SE; i += BS) stab[i] = gld_c(tw + i);
    }
    const cplx<T> *rot = SE > 0 ? stab : tw;
    const LineSet<T> ls{lds, FT, ST ? stab + TWN : a.tab0, ST ? 2 * NT : a.tab_stride, 3};
    for (int k = 0; k < slices; ++k) {
        for (int i = tid; i < NT; i += BS) {
            const int li = L::at(i);
            Tri<T> A;
            if (k == 0) A = {gld_c(a.psrc + i), gld_c(a.f[1] + i), gld_c(a.f[2] + i)};
            else A = {lds[li], lds[FT + li], lds[2 * FT + li]};
            rk4_half_step<T, false>(a.rk, 0, A);
            if (k > 0) rk4_half_step<T, false>(a.rk, 0, A);
            lds[li] = A.p;
            lds[FT + li] = A.s;
            lds[2 * FT + li] = A.i;
        }
        __syncthreads();
        line_op_any<T, NT, +1, 1, 1, L::PAD, false, L::G, false, TwShear, USE_ONE>(ls, 1, rot, tid, BS);
    }
    for (int i = tid; i < NT; i += BS)
        for (int f = 0; f < 3; ++f) gst_c(a.f[f] + i, ld_c(lds + f * FT + L::at(i)));
}

// The fused pass with the fields in registers (FP32, b = 0 of TimeVariant).
// A thread holds the N1 samples of its pixel and sub-index m (t = M n1 + m)
// of all three fields: it loads them, takes the pointwise step and the outer
// register DFTs, and only the inner phases go through LDS, one field after
// the other.  The classic tile fills a CU's LDS with three fields of a narrow
// tile, and its phases follow each other.  With one field in LDS a 2048-sample
// tile has four pixels (32-byte runs in HBM) instead of two: 72 KiB and 17 of
// rotations, 96 VGPRs of field, one workgroup of 8 waves per CU; of the shorter
// lines several workgroups share a CU, so that one's HBM traffic runs behind the
// arithmetic of the others (1024 samples: three of four pixels, one of eight;
// 512 samples: three of four pixels, two of eight).  us per slice, both passes:
// 128 x 128 x 2048 1290 -> 1130, 64 x 64 x 1024 109 -> 99, 64 x 64 x 512 49.8 -> 47.6.
// The same operations per element as the classic tile.
// Rotations staged in LDS where that costs no workgroup of the CU.
template <typename T, int NT, int TX> constexpr bool reg_stage() {
    constexpr int wgs = reg_waves<T, NT, TX>() * 256 / reg_threads<T, NT, TX>();
    return (TimeTile<T, NT, TX>::FT + tw_elems<T, NT>()) * (int)sizeof(cplx<T>) <= 163840 / wgs;
}
template <typename T, int NT, int TX, bool PHASE>
__device__ __forceinline__ void nl_time_reg(const TLine3Args<T> &a, int nx, int ny, int tile,
                                            const cplx<T> *__restrict__ tw, cplx<T> *lds, cplx<T> *twl, int stop) {
    static_assert(three_level<T, NT>(), "the outer radix is that of the three-level split");
    using L = TimeTile<T, NT, TX>;
    constexpr int N1 = outer_radix<T, NT>(), M = NT / N1, BS = reg_threads<T, NT, TX>();
    constexpr bool STW = reg_stage<T, NT, TX>();
    const int tid = threadIdx.x, l = tid % TX, m = tid / TX;
    const int tiles_x = nx / TX;
    const size_t plane = (size_t)nx * ny;
    const size_t base = (size_t)(tile / tiles_x) * nx + (tile % tiles_x) * TX + l + (size_t)m * plane;
    cplx<T> v[3][N1];
#pragma unroll
    for (int n = 0; n < N1; ++n) {
        const size_t gi = base + (size_t)(M * n) * plane;
        v[0][n] = gld_c(a.psrc + gi);
        v[1][n] = gld_c(a.f[1] + gi);
        v[2][n] = gld_c(a.f[2] + gi);
    }
    if constexpr (STW)
        for (int i = tid; i < tw_elems<T, NT>(); i += BS) twl[i] = gld_c(tw + i);
#pragma unroll
    for (int n = 0; n < N1; ++n) {
        Tri<T> A = {v[0][n], v[1][n], v[2][n]};
        nl_point<T, PHASE>(a.rk, M * n + m, A);
        v[0][n] = A.p;
        v[1][n] = A.s;
        v[2][n] = A.i;
    }
    if constexpr (STW) __syncthreads();
    if (stop) return;
    const cplx<T> *rot = STW ? twl : tw;
#pragma unroll
    for (int f = 0; f < 3; ++f) {
        if (f >= a.first_field) {
            dft_twiddle<TwShear, T, N1, M, +1, 1, false>(v[f], m, rot);
#pragma unroll
            for (int k = 0; k < N1; ++k) lds[L::at((M * k + m) * TX) + l] = v[f][k];
            __syncthreads();
            const LineSet<T> ls{lds, 0, a.tab0 + (f - a.first_field) * a.tab_stride, 0, 1};
            line_inner3<T, NT, 1, TX, L::PAD, L::G, +1, true, TwShear>(ls, TX, rot, tid, BS);
            // a thread reads back, and for the next field overwrites, only
            // the slots that it wrote
#pragma unroll
            for (int k = 0; k < N1; ++k) v[f][k] = lds[L::at((M * k + m) * TX) + l];
            twiddle_idft<TwShear, T, N1, M, +1, 1, false>(v[f], m, rot);
        }
#pragma unroll
        for (int n = 0; n < N1; ++n) gst_c(a.f[f] + base + (size_t)(M * n) * plane, v[f][n]);
        __builtin_amdgcn_sched_barrier(0);
    }
}

// Contiguous run [u0, u1) of the work units of this workgroup.
__device__ __forceinline__ void unit_run(int units, int &u0, int &u1) {
    const long long G = gridDim.x, b = blockIdx.x;
    u0 = (int)(b * units / G);
    u1 = (int)((b + 1) * units / G);
}

// Persistent form of the fused pass: the workgroup walks a run of tiles.
// The raw fields of tile u+1 are loaded into registers as soon as tile u
// is in LDS, so their HBM latency hides behind the line operator of tile
// u; twiddles and tables are staged in LDS (stab, time_stage_elems) whenever
// the tile belongs to another solve than the staged tables, so the
// prefetch is the only global load in flight inside the loop.
//
// Src supplies the work units: units(), skip(u), key(u) (identity of the
// tables a unit needs), args(u) (pointers, step weights, first field),
// nx(u), ny(u), tile(u), and stage(u, stab, tid, nthr) (copy the rotations to
// stab and the line tables of fields first..2 after them).
template <typename T, int NT, int TX, int BS, typename Src>
__device__ __forceinline__ void nl_time_run(const Src &src, cplx<T> *lds, cplx<T> *stab) {
    static_assert(TX % 2 == 0, "pairs of pixels");
    using L = TimeTile<T, NT, TX>;
    constexpr int TILE = NT * TX, FT = L::FT;
    constexpr int PT = (TILE + 2 * BS - 1) / (2 * BS);
    constexpr bool EVEN = TILE % (2 * BS) == 0;
    const int tid = threadIdx.x;
    int u0, u1;
    unit_run(src.units(), u0, u1);
    cpair<T> rp[PT], rs[PT], ri[PT];
    auto offset = [&](int u, int i) {
        const int nx = src.nx(u), tiles_x = nx / TX, tile = src.tile(u);
        const size_t base = (size_t)(tile / tiles_x) * nx + (tile % tiles_x) * TX;
        return (size_t)(i / TX) * ((size_t)nx * src.ny(u)) + base + i % TX;
    };
    auto load = [&](int u) {
        if (src.skip(u)) return;
        const TLine3Args<T> a = src.args(u);
#pragma unroll
        for (int j = 0; j < PT; ++j) {
            const int i = 2 * tid + j * 2 * BS;
            if (EVEN || i < TILE) {
                const size_t gi = offset(u, i);
                rp[j] = load_pair(a.psrc + gi);
                rs[j] = load_pair(a.f[1] + gi);
                ri[j] = load_pair(a.f[2] + gi);
            }
        }
    };
    int staged = -1;
    if (u0 < u1) load(u0);
    for (int u = u0; u < u1; ++u) {
        if (src.skip(u)) {
            if (u + 1 < u1) load(u + 1);
            continue;
        }
        const TLine3Args<T> a = src.args(u);
        if (src.key(u) != staged) {   // the barrier below publishes the tables
            src.stage(u, stab, tid, BS);
            staged = src.key(u);
        }
#pragma unroll
        for (int j = 0; j < PT; ++j) {
            const int i = 2 * tid + j * 2 * BS;
            if (EVEN || i < TILE) {
                Tri<T> A0 = {rp[j].a, rs[j].a, ri[j].a}, A1 = {rp[j].b, rs[j].b, ri[j].b};
                nl_point_pair<T, false>(a.rk, i / TX, A0, A1);
                const int li = L::at(i);
                lds[li] = A0.p;
                lds[li + 1] = A1.p;
                lds[FT + li] = A0.s;
                lds[FT + li + 1] = A1.s;
                lds[2 * FT + li] = A0.i;
                lds[2 * FT + li + 1] = A1.i;
            }
        }
        __syncthreads();
        if (u + 1 < u1) load(u + 1);
        const LineSet<T> ls{lds + a.first_field * FT, FT, stab + tw_elems<T, NT>(), 2 * NT, 3 - a.first_field};
        line_op_any<T, NT, +1, 1, TX, L::PAD, false, L::G>(ls, TX, stab, tid, BS);
        for (int i = 2 * tid; i < TILE; i += 2 * BS) {
            const size_t gi = offset(u, i);
            const int li = L::at(i);
            store_pair(a.f[0] + gi, lds + li);
            store_pair(a.f[1] + gi, lds + FT + li);
            store_pair(a.f[2] + gi, lds + 2 * FT + li);
        }
        __syncthreads();
    }
}

// Work units of the fused pass of one solve: its tiles.
template <typename T, int NT, int TX> struct TimeSolo {
    const TLine3Args<T> &a;
    int nx_, ny_;
    const cplx<T> *tw;
    __device__ int units() const { return (nx_ / TX) * ny_; }
    __device__ bool skip(int) const { return false; }
    __device__ int key(int) const { return 0; }
    __device__ const TLine3Args<T> &args(int) const { return a; }
    __device__ int nx(int) const { return nx_; }
    __device__ int ny(int) const { return ny_; }
    __device__ int tile(int u) const { return u; }
    __device__ void stage(int, cplx<T> *stab, int tid, int nthr) const {
        stage_time_tables<T, NT, TX>(tw, a, stab, tid, nthr);
    }
};

}  // namespace opo
