// opo_kernels.hip -- CDNA4 kernels of the split-step Fourier path.
//
// Per z-slice the reference applies N(dz/2) D(dz) Q(dz) N(dz/2)
// (Solver3D.cuh:949-957).  D is diagonal in omega (a line operator along t),
// Q is diagonal in (kx, ky) and its table factorises exactly into an x
// factor and a y factor, so Q = Q_y Q_x is two line operators on each
// t-plane.  The kernels here:
//   k_rk4      pointwise RK4 half step(s) of all three fields, optionally
//              reading the pump from the injection buffer and applying the
//              mirror factors to s and i on the way out;
//   k_tline    along-t operator on tiles of TX consecutive x pixels x NT,
//              staged in LDS (coalesced TX*8-byte rows);
//   k_tline3   the fused pass of a slice (opo_passes.hpp), k_plane all slices
//              of a plane wave;
//   k_xydense  Q_x then Q_y on whole t-planes of up to 128 points, lines in
//              registers, one crossing through LDS (opo_mfma.hpp);
//   k_xyband   Q_x or Q_y on bands of longer planes, likewise; k_xrows and
//              k_ycols where lines do not fit the registers;
//   k_power_*  compensated power sums with a fixed reduction order.
#include <atomic>

#include "opo_device.hpp"
#include "opo_kernels.hpp"
#include "opo_rk4.hpp"
#include "opo_passes.hpp"
#include "opo_power.hpp"

namespace opo {

template <typename T, bool PHASE>
__global__ void __launch_bounds__(256) k_rk4(const cplx<T> *__restrict__ psrc, cplx<T> *ap,
                                             cplx<T> *as, cplx<T> *ai, size_t n, size_t plane, Rk4Args<T> a,
                                             const int *status) {
    if (status && *status) return;
    const size_t stride = (size_t)gridDim.x * blockDim.x;
    for (size_t i = (size_t)blockIdx.x * blockDim.x + threadIdx.x; i < n; i += stride) {
        Tri<T> A = {psrc[i], as[i], ai[i]};
        rk4_half_step<T, PHASE>(a, 0, A);
        if (a.nsteps > 1) rk4_half_step<T, PHASE>(a, 1, A);
        if (a.out_scale) {
            if (a.eom) {  // KernelEOM (Solver1D.cuh:62-72) at time sample i / plane
                const size_t t = i / plane;
                A.s = cmul_hl(A.s, a.eom[2 * t], a.eom[2 * t + 1]);
                A.i = cmul_hl(A.i, a.eom[2 * t], a.eom[2 * t + 1]);
            }
            // roundTripChange (Cavity3D.cuh:12-28): (sqrt(R) e^{i phi}) * A
            A.s = cmul_hl(A.s, cplx<T>{a.ms_re, a.ms_im}, cplx<T>{a.ms_lo_re, a.ms_lo_im});
            A.i = cmul_hl(A.i, cplx<T>{a.mi_re, a.mi_im}, cplx<T>{a.mi_lo_re, a.mi_lo_im});
        }
        ap[i] = A.p;
        as[i] = A.s;
        ai[i] = A.i;
    }
}

template <typename T>
hipError_t launch_rk4(hipStream_t st, const cplx<T> *psrc, cplx<T> *ap, cplx<T> *as, cplx<T> *ai,
                      size_t n, size_t plane, const Rk4Args<T> &a, const int *status) {
    const int bs = 256;
    size_t want = (n + bs - 1) / bs;
    int grid = (int)(want < 8192 ? want : 8192);
    if (grid < 1) grid = 1;
    if (a.has_phase)
        hipLaunchKernelGGL((k_rk4<T, true>), dim3(grid), dim3(bs), 0, st, psrc, ap, as, ai, n, plane, a, status);
    else
        hipLaunchKernelGGL((k_rk4<T, false>), dim3(grid), dim3(bs), 0, st, psrc, ap, as, ai, n, plane, a, status);
    return hipGetLastError();
}

// ---------------------------------------------------------- t operator
// Tile width (pixels along x) per time length and precision: keep the tile
// at <= 64 KiB so two or more workgroups share a CU.
template <typename T, int NT> constexpr int tline_tx() {
    constexpr int bytes = NT * (int)sizeof(cplx<T>);
    return bytes <= 4096 ? 16 : (65536 / bytes >= 16 ? 16 : 65536 / bytes);
}

template <typename T, int NT, int TX, int BS>
__global__ void __launch_bounds__(BS) k_tline(FieldOps<T> ops, int nx, int ny, const cplx<T> *__restrict__ tw,
                                              const int *status) {
    if (status && *status) return;
    __shared__ cplx<T> lds[NT * TX];
    const int tid = threadIdx.x;
    const int tiles_x = nx / TX;
    const int y = blockIdx.x / tiles_x, x0 = (blockIdx.x % tiles_x) * TX;
    const int f = blockIdx.y;
    cplx<T> *A = ops.f[f];
    const size_t plane = (size_t)nx * ny;
    const size_t base = (size_t)y * nx + x0;
    chunked_copy<T, NT * TX, BS>(tid, [&](int i) { return A[(size_t)(i / TX) * plane + base + i % TX]; },
                                 [&](int i, cplx<T> v) { lds[i] = v; });
    __syncthreads();
    line_op<T, NT, +1, 1, TX, false, TwShear, tile_use<TX>()>(lds, TX, tw, ops.tab[f], tid, BS);
    chunked_copy<T, NT * TX, BS>(tid, [&](int i) { return lds[i]; },
                                 [&](int i, cplx<T> v) { A[(size_t)(i / TX) * plane + base + i % TX] = v; });
}

template <typename T, int NT>
static hipError_t tline_dispatch(hipStream_t st, const Geometry &g, const FieldOps<T> &ops, int nf,
                                 const cplx<T> *tw, const int *status) {
    constexpr int TXmax = tline_tx<T, NT>();
    if (g.nx % TXmax == 0) {
        dim3 grid((unsigned)((g.nx / TXmax) * g.ny), (unsigned)nf);
        hipLaunchKernelGGL((k_tline<T, NT, TXmax, 256>), grid, dim3(256), 0, st, ops, g.nx, g.ny, tw, status);
    } else if (g.nx == 1) {
        dim3 grid((unsigned)g.ny, (unsigned)nf);
        hipLaunchKernelGGL((k_tline<T, NT, 1, 256>), grid, dim3(256), 0, st, ops, g.nx, g.ny, tw, status);
    } else {
        return hipErrorInvalidValue;
    }
    return hipGetLastError();
}

bool tline_supported(int nt, bool fp64) {
    switch (nt) {
        case 1: case 16: case 32: case 64: case 128: case 256: case 512: case 1024: case 2048: return true;
        case 4096: return !fp64;   // three fields of a 4096-sample line fill 102 KiB of LDS in FP32
        default: return false;
    }
}

template <typename T>
hipError_t launch_tline(hipStream_t st, const Geometry &g, const FieldOps<T> &ops, int nf,
                        const cplx<T> *tw, const int *status) {
    switch (g.nt) {
        case 1: return tline_dispatch<T, 1>(st, g, ops, nf, tw, status);
        case 16: return tline_dispatch<T, 16>(st, g, ops, nf, tw, status);
        case 32: return tline_dispatch<T, 32>(st, g, ops, nf, tw, status);
        case 64: return tline_dispatch<T, 64>(st, g, ops, nf, tw, status);
        case 128: return tline_dispatch<T, 128>(st, g, ops, nf, tw, status);
        case 256: return tline_dispatch<T, 256>(st, g, ops, nf, tw, status);
        case 512: return tline_dispatch<T, 512>(st, g, ops, nf, tw, status);
        case 1024: return tline_dispatch<T, 1024>(st, g, ops, nf, tw, status);
        case 2048: return tline_dispatch<T, 2048>(st, g, ops, nf, tw, status);
        case 4096:
            if constexpr (sizeof(T) == 4) return tline_dispatch<T, 4096>(st, g, ops, nf, tw, status);
            else return hipErrorInvalidValue;
        default: return hipErrorInvalidValue;
    }
}

template <typename T, int NT, int TX, int BS, bool PHASE>
__global__ void __launch_bounds__(BS) k_tline3(TLine3Args<T> a, int nx, int ny,
                                               const cplx<T> *__restrict__ tw, const int *status) {
    const int stop = stop_flag(status);
    __shared__ cplx<T> lds[3 * TimeTile<T, NT, TX>::FT];
    __shared__ cplx<T> twl[time_stage_twiddles<T, NT, TX>() ? tw_elems<T, NT, tile_use<TX>()>() : 1];
    nl_time_tile<T, NT, TX, BS, PHASE>(a, nx, ny, xcd_local_tile(blockIdx.x, gridDim.x), tw, lds, twl, stop);
}

template <typename T, int NT, int TX, bool PHASE>
__global__ void __launch_bounds__((reg_threads<T, NT, TX>()), (reg_waves<T, NT, TX>())) k_tline3r(TLine3Args<T> a, int nx, int ny,
                                                                         const cplx<T> *__restrict__ tw,
                                                                         const int *status) {
    const int stop = stop_flag(status);
    __shared__ cplx<T> lds[TimeTile<T, NT, TX>::FT];
    __shared__ cplx<T> twl[reg_stage<T, NT, TX>() ? tw_elems<T, NT>() : 1];
    nl_time_reg<T, NT, TX, PHASE>(a, nx, ny, xcd_local_tile(blockIdx.x, gridDim.x), tw, lds, twl, stop);
}

template <typename T, int NT, int TX, int BS>
__global__ void __launch_bounds__(BS) k_tline3p(TLine3Args<T> a, int nx, int ny,
                                                const cplx<T> *__restrict__ tw, const int *status) {
    if (status && *status) return;
    __shared__ cplx<T> lds[3 * TimeTile<T, NT, TX>::FT];
    __shared__ cplx<T> stab[time_stage_elems<T, NT, TX>()];
    nl_time_run<T, NT, TX, BS>(TimeSolo<T, NT, TX>{a, nx, ny, tw}, lds, stab);
}

template <typename T, int NT, int BS>
__global__ void __launch_bounds__(BS) k_plane(TLine3Args<T> a, int slices, const cplx<T> *__restrict__ tw,
                                              const int *status) {
    if (status && *status) return;
    __shared__ cplx<T> lds[3 * TimeTile<T, NT, 1>::FT];
    __shared__ cplx<T> stab[plane_stage_elems<T, NT>() + 1];
    nl_plane_slices<T, NT, BS>(a, slices, tw, lds, stab);
}

// Compute units of the current device (persistent grids are sized by it).
static int cu_count() {
    static std::atomic<int> cached[64];
    int dev = 0;
    if (hipGetDevice(&dev) != hipSuccess || dev < 0 || dev >= 64) return 256;
    int n = cached[dev].load(std::memory_order_relaxed);
    if (n <= 0) {
        if (hipDeviceGetAttribute(&n, hipDeviceAttributeMultiprocessorCount, dev) != hipSuccess || n <= 0)
            n = 256;
        cached[dev].store(n, std::memory_order_relaxed);
    }
    return n;
}

unsigned persistent_grid(int units, int per_cu) {
    const long long g = (long long)per_cu * cu_count();
    return (unsigned)(units < g ? units : g);
}

// ----------------------------------------------------- variant tables
// Chosen variant per (precision, size): process-wide, read at every launch
// and written by the tuner, so the entries are atomics (a launch sees either
// the old or the new choice, both of which give the same results).
struct TuneTables {
    std::atomic<int> time[2][13];   // [fp64][log2 NT]
    std::atomic<int> xy[2][8];      // [fp64][NX index]
    TuneTables() {
        for (int f = 0; f < 2; ++f) {   // -1: untuned, the default for the work at hand
            for (int k = 0; k < 13; ++k) time[f][k].store(-1);
            for (int k = 0; k < 8; ++k) xy[f][k].store(-1);
        }
    }
};
static TuneTables &tune_tables() {
    static TuneTables tt;   // initialised once, thread-safe
    return tt;
}

static int log2i(int n) {
    int l = 0;
    while ((1 << l) < n) ++l;
    return (1 << l) == n ? l : -1;
}
static int nx_index(int nx) {
    switch (nx) {
        case 1: return 0; case 16: return 1; case 32: return 2; case 64: return 3;
        case 96: return 4; case 128: return 5; case 256: return 6; case 512: return 7; default: return -1;
    }
}

template <typename T, int NT>
static void time_variant_info(int v, bool &valid, int &tx, int &bs, int &per_cu) {
    valid = false;
    static_for<0, kTimeVariants>([&](auto vv) {
        constexpr int V = decltype(vv)::value;
        using Vr = TimeVariant<T, NT, V>;
        if (V == v) {
            valid = Vr::valid;
            tx = Vr::tx;
            bs = Vr::bs;
            per_cu = Vr::per_cu;
        }
    });
}

template <typename T>
static bool time_info(int nt, int v, int &tx, int &bs, int &per_cu) {
    bool valid = false;
    switch (nt) {
#define TI(N) case N: time_variant_info<T, N>(v, valid, tx, bs, per_cu); break;
        TI(1) TI(16) TI(32) TI(64) TI(128) TI(256) TI(512) TI(1024) TI(2048)
        case 4096:
            if constexpr (sizeof(T) == 4) time_variant_info<T, 4096>(v, valid, tx, bs, per_cu);
            break;
#undef TI
        default: return false;
    }
    return valid;
}

template <typename T>
static bool time_info(int nt, int v, int &tx, int &bs) {
    int per_cu = 0;
    return time_info<T>(nt, v, tx, bs, per_cu);
}



int tune_variant_count(int axis) { return axis == 0 ? kTimeVariants : kXyVariants; }

bool tune_variant_valid(bool fp64, int axis, int n, int v) {
    if (axis == 0) {
        if (v < 0 || v >= kTimeVariants) return false;
        int tx = 0, bs = 0;
        return fp64 ? time_info<double>(n, v, tx, bs) : time_info<float>(n, v, tx, bs);
    }
    return nx_index(n) >= 0 && xy_variant_numbered(fp64, n, v);
}

bool tune_variant_timed(bool fp64, int axis, int n, int v) {
    return tune_variant_valid(fp64, axis, n, v) && (axis == 0 || xy_variant_shape(fp64, n, v) == v);
}

static std::atomic<int> *tune_entry(bool fp64, int axis, int n) {
    TuneTables &tt = tune_tables();
    if (axis == 0) {
        const int l = log2i(n);
        return (l >= 0 && l < 13) ? &tt.time[fp64][l] : nullptr;
    }
    const int k = nx_index(n);
    return k >= 0 ? &tt.xy[fp64][k] : nullptr;
}

int tune_stored(bool fp64, int axis, int n) {
    const std::atomic<int> *e = tune_entry(fp64, axis, n);
    return e ? e->load(std::memory_order_relaxed) : 0;
}

void tune_restore(bool fp64, int axis, int n, int stored) {
    if (std::atomic<int> *e = tune_entry(fp64, axis, n)) e->store(stored, std::memory_order_relaxed);
}

int tune_report(bool fp64, int axis, int n) {
    const int v = tune_stored(fp64, axis, n), many = tune_get(fp64, axis, n);
    if (v < 0 && axis == 0)
        for (long long px : kPixelSteps)
            if (time_default_variant(fp64, n, px) != many) return -1;
    return many;
}

int tune_get(bool fp64, int axis, int n, long long pixels) {
    const int v = tune_stored(fp64, axis, n);
    if (v >= 0) return v;
    return axis == 0 ? time_default_variant(fp64, n, pixels) : xy_default_variant(fp64, n);
}

bool tune_set(bool fp64, int axis, int n, int v) {
    if (!tune_variant_valid(fp64, axis, n, v < 0 ? 0 : v) || v < -1) return false;
    TuneTables &tt = tune_tables();
    if (axis == 0) tt.time[fp64][log2i(n)].store(v, std::memory_order_relaxed);
    else tt.xy[fp64][nx_index(n)].store(v, std::memory_order_relaxed);
    return true;
}

int tune_tile_px(bool fp64, int nt, int v) {
    int tx = 0, bs = 0;
    const bool ok = fp64 ? time_info<double>(nt, v, tx, bs) : time_info<float>(nt, v, tx, bs);
    return ok ? tx : 0;
}

int time_variant_for(bool fp64, int nt, int nx, long long pixels) {
    const int v = tune_get(fp64, 0, nt, pixels);
    const int tx = tune_tile_px(fp64, nt, v);
    return (tx > 0 && nx % tx == 0) ? v : 0;
}

int tune_per_cu(bool fp64, int axis, int n, int v) {
    if (axis == 1) return 0;
    int tx = 0, bs = 0, per_cu = 0;
    const bool ok = fp64 ? time_info<double>(n, v, tx, bs, per_cu) : time_info<float>(n, v, tx, bs, per_cu);
    return ok ? per_cu : 0;
}

int tune_block(bool fp64, int axis, int n, int v) {
    if (axis == 1) return xy_variant_bs(fp64, n, v);
    int tx = 0, bs = 0;
    const bool ok = fp64 ? time_info<double>(n, v, tx, bs) : time_info<float>(n, v, tx, bs);
    return ok ? bs : 0;
}

template <typename T, int NT, int V>
static hipError_t tline3_launch_v(hipStream_t st, const Geometry &g, const TLine3Args<T> &a,
                                  const cplx<T> *tw, const int *status) {
    using Vr = TimeVariant<T, NT, V>;
    if constexpr (!Vr::valid) {
        return hipErrorInvalidValue;
    } else {
        if (g.nx % Vr::tx != 0) return hipErrorInvalidValue;
        const int units = (g.nx / Vr::tx) * g.ny;
        if constexpr (Vr::persistent) {
            if (a.rk.has_phase) return hipErrorInvalidValue;
            hipLaunchKernelGGL((k_tline3p<T, NT, Vr::tx, Vr::bs>), dim3(persistent_grid(units, Vr::per_cu)),
                               dim3(Vr::bs), 0, st, a, g.nx, g.ny, tw, status);
            return hipGetLastError();
        }
        dim3 grid((unsigned)units);
        if constexpr (Vr::reg) {
            if (a.rk.has_phase && V != 0) return hipErrorInvalidValue;
            if (a.rk.has_phase)
                hipLaunchKernelGGL((k_tline3r<T, NT, Vr::tx, V == 0>), grid, dim3(Vr::bs), 0, st, a, g.nx, g.ny, tw,
                                   status);
            else
                hipLaunchKernelGGL((k_tline3r<T, NT, Vr::tx, false>), grid, dim3(Vr::bs), 0, st, a, g.nx, g.ny, tw,
                                   status);
        } else if (a.rk.has_phase) {
            if constexpr (V == 0)
                hipLaunchKernelGGL((k_tline3<T, NT, Vr::tx, Vr::bs, true>), grid, dim3(Vr::bs), 0, st, a,
                                   g.nx, g.ny, tw, status);
            else
                return hipErrorInvalidValue;
        } else {
            hipLaunchKernelGGL((k_tline3<T, NT, Vr::tx, Vr::bs, false>), grid, dim3(Vr::bs), 0, st, a, g.nx,
                               g.ny, tw, status);
        }
        return hipGetLastError();
    }
}

template <typename T, int NT>
static hipError_t tline3_dispatch(hipStream_t st, const Geometry &g, const TLine3Args<T> &a,
                                  const cplx<T> *tw, const int *status) {
    if (g.nx == 1) {
        dim3 grid((unsigned)g.ny);
        if (a.rk.has_phase)
            hipLaunchKernelGGL((k_tline3<T, NT, 1, 256, true>), grid, dim3(256), 0, st, a, g.nx, g.ny, tw, status);
        else
            hipLaunchKernelGGL((k_tline3<T, NT, 1, 256, false>), grid, dim3(256), 0, st, a, g.nx, g.ny, tw, status);
        return hipGetLastError();
    }
    const int v = a.rk.has_phase ? 0 : time_variant_for(sizeof(T) == 8, NT, g.nx, (long long)g.nx * g.ny);
    hipError_t e = hipErrorInvalidValue;
    static_for<0, kTimeVariants>([&](auto vv) {
        constexpr int V = decltype(vv)::value;
        if (V == v) e = tline3_launch_v<T, NT, V>(st, g, a, tw, status);
    });
    return e;
}

template <typename T>
hipError_t launch_tline3(hipStream_t st, const Geometry &g, const TLine3Args<T> &a,
                         const cplx<T> *tw, const int *status) {
    switch (g.nt) {
        case 1: return tline3_dispatch<T, 1>(st, g, a, tw, status);
        case 16: return tline3_dispatch<T, 16>(st, g, a, tw, status);
        case 32: return tline3_dispatch<T, 32>(st, g, a, tw, status);
        case 64: return tline3_dispatch<T, 64>(st, g, a, tw, status);
        case 128: return tline3_dispatch<T, 128>(st, g, a, tw, status);
        case 256: return tline3_dispatch<T, 256>(st, g, a, tw, status);
        case 512: return tline3_dispatch<T, 512>(st, g, a, tw, status);
        case 1024: return tline3_dispatch<T, 1024>(st, g, a, tw, status);
        case 2048: return tline3_dispatch<T, 2048>(st, g, a, tw, status);
        case 4096:
            if constexpr (sizeof(T) == 4) return tline3_dispatch<T, 4096>(st, g, a, tw, status);
            else return hipErrorInvalidValue;
        default: return hipErrorInvalidValue;
    }
}

template <typename T, int NT>
static hipError_t plane_launch(hipStream_t st, const TLine3Args<T> &a, int slices, const cplx<T> *tw,
                               const int *status) {
    constexpr int BS = plane_threads<T, NT>();
    hipLaunchKernelGGL((k_plane<T, NT, BS>), dim3(1), dim3(BS), 0, st, a, slices, tw, status);
    return hipGetLastError();
}

template <typename T>
hipError_t launch_plane_slices(hipStream_t st, int nt, const TLine3Args<T> &a, int slices, const cplx<T> *tw,
                               const int *status) {
    switch (nt) {
        case 1: return plane_launch<T, 1>(st, a, slices, tw, status);
        case 16: return plane_launch<T, 16>(st, a, slices, tw, status);
        case 32: return plane_launch<T, 32>(st, a, slices, tw, status);
        case 64: return plane_launch<T, 64>(st, a, slices, tw, status);
        case 128: return plane_launch<T, 128>(st, a, slices, tw, status);
        case 256: return plane_launch<T, 256>(st, a, slices, tw, status);
        case 512: return plane_launch<T, 512>(st, a, slices, tw, status);
        case 1024: return plane_launch<T, 1024>(st, a, slices, tw, status);
        case 2048: return plane_launch<T, 2048>(st, a, slices, tw, status);
        case 4096:
            if constexpr (sizeof(T) == 4) return plane_launch<T, 4096>(st, a, slices, tw, status);
            else return hipErrorInvalidValue;
        default: return hipErrorInvalidValue;
    }
}

// --------------------------------------------------------- xy operator
// NX = NY = 1: the two one-entry tables, a sample per thread.
template <typename T>
__global__ void __launch_bounds__(256) k_xypixel(FieldOps<T> ops, int nt, const int *status) {
    if (stop_flag(status)) return;
    const int t = blockIdx.x * 256 + threadIdx.x, f = blockIdx.y;
    if (t >= nt) return;
    const cplx<T> v = cmul_hl(ld_c(ops.f[f] + t), ld_c(ops.tab[f]), ld_c(ops.tab[f] + 1));
    st_c(ops.f[f] + t, cmul_hl(v, ld_c(ops.taby[f]), ld_c(ops.taby[f] + 1)));
}

// Planes of 16 to 128 points (opo_mfma.hpp): P consecutive planes by PC sets
// of waves.
template <typename T, int NX, int NY, int PC, int P>
__global__ void __launch_bounds__((PC * dense_threads<NX, NY>()), (dense_waves<T, (NX > NY ? NX : NY)>()))
    k_xydense(FieldOps<T> ops, const int *status) {
    const int stop = stop_flag(status);
    __shared__ DensePlane<T, NX, NY> S[PC];
    __shared__ DenseTabs<T, NX, NY> Tb;
    const int f = blockIdx.y;
    dense_group<T, NX, NY, PC, P>(ops.f[f] + (size_t)blockIdx.x * P * NX * NY, ops.tab[f], ops.taby[f], S, Tb,
                                  threadIdx.x, stop);
}
// Lines of planes beyond that, a band of 16 rows or columns per wave.
template <typename T, int N, bool ROWS>
__global__ void __launch_bounds__(64 * kDenseBandWaves) k_xyband(FieldOps<T> ops, int nx, int ny, int units,
                                                                const int *status) {
    const int stop = stop_flag(status);
    __shared__ DenseTab<T, N> Tb;
    const int f = blockIdx.y, w = __builtin_amdgcn_readfirstlane(threadIdx.x / 64);
    stage_dense<N>(ROWS ? ops.tab[f] : ops.taby[f], Tb, threadIdx.x, 64 * kDenseBandWaves);
    const int u = blockIdx.x * kDenseBandWaves + w, bands = (ROWS ? ny : nx) / 16;
    const int t = u / bands, b = u % bands;
    dense_band<T, N, ROWS>(ops.f[f] + (size_t)t * nx * ny + (ROWS ? (size_t)b * 16 * nx : (size_t)b * 16), nx, Tb,
                           threadIdx.x % 64, u < units, stop);
}

// Lines that do not fit a wave's registers (FP64 256 points, 512 points in
// either precision), and few lines (dense_axis), run in LDS: Q_x on bands of RB
// consecutive rows, then Q_y on bands of CB consecutive columns (rows of the
// band are CB elements contiguous in HBM).
template <typename T, int NX, int RB, int BS>
__global__ void __launch_bounds__(BS) k_xrows(FieldOps<T> ops, int ny, const cplx<T> *__restrict__ tw,
                                              const int *status) {
    const int stop = stop_flag(status);
    constexpr int NXP = NX + 1;
    __shared__ cplx<T> lds[RB * NXP];
    constexpr bool STW = band_rotations_in_lds<T, NX>();
    __shared__ cplx<T> twl[STW ? tw_elems<T, NX, USE_BAND>() : 1];
    if constexpr (STW) stage_rotations<T, NX>(tw, twl, threadIdx.x, BS);
    const int bands = ny / RB;
    const int t = blockIdx.x / bands, r0 = (blockIdx.x % bands) * RB, f = blockIdx.y;
    cplx<T> *A = ops.f[f] + ((size_t)t * ny + r0) * NX;
    chunked_copy<T, RB * NX, BS>(threadIdx.x, [&](int i) { return A[i]; },
                                 [&](int i, cplx<T> v) { lds[(i / NX) * NXP + (i % NX)] = v; });
    __syncthreads();
    if (stop) return;
    band_line_op<T, NX, -1, NXP, 1, TwShear>(lds, RB, STW ? twl : tw, ops.tab[f], threadIdx.x, BS);
    chunked_copy<T, RB * NX, BS>(threadIdx.x, [&](int i) { return lds[(i / NX) * NXP + (i % NX)]; },
                                 [&](int i, cplx<T> v) { A[i] = v; });
}

template <typename T, int NY, int CB, int BS>
__global__ void __launch_bounds__(BS) k_ycols(FieldOps<T> ops, int nx, const cplx<T> *__restrict__ tw,
                                              const int *status) {
    const int stop = stop_flag(status);
    constexpr int CBP = CB + 1;
    __shared__ cplx<T> lds[NY * CBP];
    constexpr bool STW = band_rotations_in_lds<T, NY>();
    __shared__ cplx<T> twl[STW ? tw_elems<T, NY, USE_BAND>() : 1];
    if constexpr (STW) stage_rotations<T, NY>(tw, twl, threadIdx.x, BS);
    const int bands = nx / CB;
    const int t = blockIdx.x / bands, c0 = (blockIdx.x % bands) * CB, f = blockIdx.y;
    cplx<T> *A = ops.f[f] + (size_t)t * NY * nx + c0;
    chunked_copy<T, NY * CB, BS>(threadIdx.x, [&](int i) { return A[(size_t)(i / CB) * nx + (i % CB)]; },
                                 [&](int i, cplx<T> v) { lds[(i / CB) * CBP + (i % CB)] = v; });
    __syncthreads();
    if (stop) return;
    // lines are the CB columns (line c starts at c, its elements CBP apart)
    band_line_op<T, NY, -1, 1, CBP, TwShear>(lds, CB, STW ? twl : tw, ops.taby[f], threadIdx.x, BS);
    chunked_copy<T, NY * CB, BS>(threadIdx.x, [&](int i) { return lds[(i / CB) * CBP + (i % CB)]; },
                                 [&](int i, cplx<T> v) { A[(size_t)(i / CB) * nx + (i % CB)] = v; });
}

constexpr int kSplitBand = 32;   // rows or columns: 131 KiB of LDS at FP64 256 points

template <typename T, int NX, int B, int BS>
static hipError_t xy_split_launch_b(hipStream_t st, const Geometry &g, const FieldOps<T> &ops, int nf,
                                    const cplx<T> *tw, const int *status) {
    if (g.ny != NX || NX % B != 0) return hipErrorInvalidValue;
    hipLaunchKernelGGL((k_xrows<T, NX, B, BS>), dim3((unsigned)(g.nt * (NX / B)), (unsigned)nf), dim3(BS), 0, st,
                       ops, g.ny, tw, status);
    hipError_t e = hipGetLastError();
    if (e != hipSuccess) return e;
    hipLaunchKernelGGL((k_ycols<T, NX, B, BS>), dim3((unsigned)(g.nt * (NX / B)), (unsigned)nf), dim3(BS), 0, st,
                       ops, g.nx, tw, status);
    return hipGetLastError();
}
// Variants of the FP64 256 x 256 planes: v = 0 bands of 32 with 256 threads,
// 1 bands of 32 with 512, 2 bands of 16 with 256.
template <typename T, int NX>
static hipError_t xy_split_launch(hipStream_t st, const Geometry &g, const FieldOps<T> &ops, int nf,
                                  const cplx<T> *tw, const int *status, int v = 0) {
    if (v == 1) return xy_split_launch_b<T, NX, kSplitBand, 512>(st, g, ops, nf, tw, status);
    if (v == 2) return xy_split_launch_b<T, NX, 16, 256>(st, g, ops, nf, tw, status);
    return xy_split_launch_b<T, NX, kSplitBand, 256>(st, g, ops, nf, tw, status);
}

// Bands: Q_x on bands of 16 rows or Q_y on bands of 16 columns.
template <typename T, int N, bool ROWS>
static hipError_t xy_band_launch(hipStream_t st, const Geometry &g, const FieldOps<T> &ops, int nf,
                                 const int *status) {
    const int units = g.nt * ((ROWS ? g.ny : g.nx) / 16);
    hipLaunchKernelGGL((k_xyband<T, N, ROWS>),
                       dim3((unsigned)((units + kDenseBandWaves - 1) / kDenseBandWaves), (unsigned)nf),
                       dim3(64 * kDenseBandWaves), 0, st, ops, g.nx, g.ny, units, status);
    return hipGetLastError();
}

// The launch shapes of square planes on the matrix cores, 4 NX threads per
// plane (a wave per 16 lines): one plane per workgroup, or for NX <= 32 (v >= 3)
// groups of 256 / NX planes on 256, 512 or 1024 threads.
template <typename T, int NX>
static hipError_t xy_dense_launch(hipStream_t st, const Geometry &g, const FieldOps<T> &ops, int nf,
                                  const int *status) {
    // Few FP64 128-point planes, one workgroup of a CU each, leave CUs idle:
    // the same lines as bands of four waves (128 x 128 x 16: 43.7 -> 42.3 us per
    // slice).
    if constexpr (sizeof(T) == 8 && NX == 128) {
        if (g.nt * nf < 64) {
            const hipError_t e = xy_band_launch<T, NX, true>(st, g, ops, nf, status);
            return e != hipSuccess ? e : xy_band_launch<T, NX, false>(st, g, ops, nf, status);
        }
    }
    if constexpr (NX <= 32) {
        constexpr int P = xy_group(NX, 3), PC = 256 / (4 * NX);   // planes at once on 256 threads
        const int v = tune_get(sizeof(T) == 8, 1, NX);
        if (xy_group(NX, v) > 1) {
            if (g.nt % P != 0) return hipErrorInvalidValue;
            const dim3 grid((unsigned)(g.nt / P), (unsigned)nf);
            const int bs = xy_variant_bs(sizeof(T) == 8, NX, v);
            if (bs == 256) hipLaunchKernelGGL((k_xydense<T, NX, NX, PC, P>), grid, dim3(256), 0, st, ops, status);
            else if (bs == 512) hipLaunchKernelGGL((k_xydense<T, NX, NX, 2 * PC, P>), grid, dim3(512), 0, st, ops, status);
            else hipLaunchKernelGGL((k_xydense<T, NX, NX, 4 * PC, P>), grid, dim3(1024), 0, st, ops, status);
            return hipGetLastError();
        }
    }
    hipLaunchKernelGGL((k_xydense<T, NX, NX, 1, 1>), dim3((unsigned)g.nt, (unsigned)nf), dim3(4 * NX), 0, st, ops, status);
    return hipGetLastError();
}

// NX != NY planes of up to 128 points in one pass: the plane is read and written
// once instead of twice (FP32 64 x 32 x 128 cavity, 375 slices: 8.5 ms as two
// band passes, 6.3 here, 10.4 with lines in LDS).
template <typename T, int NX, int NY>
static hipError_t xy_dense_rect(hipStream_t st, const Geometry &g, const FieldOps<T> &ops, int nf, const int *status) {
    if constexpr (NX == NY) {
        return hipErrorInvalidValue;   // xy_dense_launch
    } else {
        hipLaunchKernelGGL((k_xydense<T, NX, NY, 1, 1>), dim3((unsigned)g.nt, (unsigned)nf),
                           dim3((unsigned)dense_threads<NX, NY>()), 0, st, ops, status);
        return hipGetLastError();
    }
}
template <typename T, int NX>
static hipError_t xy_dense_rect_y(hipStream_t st, const Geometry &g, const FieldOps<T> &ops, int nf, const int *status) {
    switch (g.ny) {
        case 16: return xy_dense_rect<T, NX, 16>(st, g, ops, nf, status);
        case 32: return xy_dense_rect<T, NX, 32>(st, g, ops, nf, status);
        case 64: return xy_dense_rect<T, NX, 64>(st, g, ops, nf, status);
        case 96: return xy_dense_rect<T, NX, 96>(st, g, ops, nf, status);
        default: return xy_dense_rect<T, NX, 128>(st, g, ops, nf, status);
    }
}

static bool line_len_supported(int n) {
    switch (n) {
        case 16: case 32: case 64: case 96: case 128: case 256: case 512: return true;
        default: return false;
    }
}

// NX = 1: the identity transform with its table (absorption).
template <typename T>
static hipError_t xy_pixel_launch(hipStream_t st, const Geometry &g, const FieldOps<T> &ops, int nf,
                                  const int *status) {
    hipLaunchKernelGGL((k_xypixel<T>), dim3((unsigned)((g.nt + 255) / 256), (unsigned)nf), dim3(256), 0, st, ops, g.nt,
                       status);
    return hipGetLastError();
}

bool xyplane_supported(int nx, int ny, bool fp64) {
    if (nx != ny) return line_len_supported(nx) && line_len_supported(ny);
    return nx == 1 || line_len_supported(nx);
}

// Planes with an axis beyond 128 points, and planes of few lines (dense_axis):
// Q_x on bands of rows, then Q_y on bands of columns.  Lines that fit a wave's
// registers take 16 per wave (k_xyband; FP32 256 x 256 x 64, rows + cols: 100 us
// in LDS, 73 here), the others bands in LDS (k_xrows, k_ycols) of 32 rows or
// columns where the other dimension allows, else 16 (every supported length is a
// multiple of 16).  256- and 512-point lines there:
// FP32 bands of 32 on 512 threads (256: one 16-point DFT per thread and
// phase; 512: 131 KiB of LDS, as fast as bands of 16 on 256 threads), FP64
// bands of 16 (256: 64 KiB of LDS, two workgroups per CU; 512: 131 KiB).
template <typename T, int N> constexpr int max_band() {
    return (sizeof(T) == 8 && N >= 256) ? 16 : 32;
}
template <typename T, int N> constexpr int band32_threads() { return (sizeof(T) == 4 && N >= 256) ? 512 : 256; }

template <typename T, int NX>
static hipError_t rows_launch(hipStream_t st, const Geometry &g, const FieldOps<T> &ops, int nf,
                              const cplx<T> *tw, const int *status) {
    if constexpr (dense_line<T>(NX)) {
        if (dense_axis<T>(NX, g.ny, g.nt, true)) return xy_band_launch<T, NX, true>(st, g, ops, nf, status);
    }
    if constexpr (band_line<T>(NX) && max_band<T, NX>() == 32) {
        constexpr int B32 = band32_threads<T, NX>();
        if (g.ny % 32 == 0) {
            hipLaunchKernelGGL((k_xrows<T, NX, 32, B32>), dim3((unsigned)(g.nt * (g.ny / 32)), (unsigned)nf),
                               dim3(B32), 0, st, ops, g.ny, tw, status);
            return hipGetLastError();
        }
    }
    if constexpr (band_line<T>(NX) && !(sizeof(T) == 8 && dense_line<T>(NX))) {   // those only beside 64 or more
        hipLaunchKernelGGL((k_xrows<T, NX, 16, 256>), dim3((unsigned)(g.nt * (g.ny / 16)), (unsigned)nf), dim3(256),
                           0, st, ops, g.ny, tw, status);
        return hipGetLastError();
    }
    return hipErrorInvalidValue;   // not reached: every other line is dense
}
template <typename T, int NY>
static hipError_t cols_launch(hipStream_t st, const Geometry &g, const FieldOps<T> &ops, int nf,
                              const cplx<T> *tw, const int *status) {
    if constexpr (dense_line<T>(NY)) {
        if (dense_axis<T>(NY, g.nx, g.nt, false)) return xy_band_launch<T, NY, false>(st, g, ops, nf, status);
    }
    if constexpr (band_line<T>(NY) && max_band<T, NY>() == 32) {
        constexpr int B32 = band32_threads<T, NY>();
        if (g.nx % 32 == 0) {
            hipLaunchKernelGGL((k_ycols<T, NY, 32, B32>), dim3((unsigned)(g.nt * (g.nx / 32)), (unsigned)nf),
                               dim3(B32), 0, st, ops, g.nx, tw, status);
            return hipGetLastError();
        }
    }
    if constexpr (band_line<T>(NY) && !(sizeof(T) == 8 && dense_line<T>(NY))) {   // those only beside 64 or more
        hipLaunchKernelGGL((k_ycols<T, NY, 16, 256>), dim3((unsigned)(g.nt * (g.nx / 16)), (unsigned)nf), dim3(256),
                           0, st, ops, g.nx, tw, status);
        return hipGetLastError();
    }
    return hipErrorInvalidValue;   // not reached: every other line is dense
}
// Planes whose lines both run on the matrix cores, in one launch.
template <typename T> static bool dense_plane_grid(const Geometry &g) {
    return g.nx <= 128 && g.ny <= 128 && dense_axis<T>(g.nx, g.ny, g.nt, true) && dense_axis<T>(g.ny, g.nx, g.nt, false);
}
template <typename T>
static hipError_t xy_rect_launch(hipStream_t st, const Geometry &g, const FieldOps<T> &ops, int nf,
                                 const cplx<T> *tw_x, const cplx<T> *tw_y, const int *status) {
    if (!line_len_supported(g.nx) || !line_len_supported(g.ny) || g.nx % 16 || g.ny % 16)
        return hipErrorInvalidValue;
    if (g.nx != g.ny && dense_plane_grid<T>(g)) {
        switch (g.nx) {
            case 16: return xy_dense_rect_y<T, 16>(st, g, ops, nf, status);
            case 32: return xy_dense_rect_y<T, 32>(st, g, ops, nf, status);
            case 64: return xy_dense_rect_y<T, 64>(st, g, ops, nf, status);
            case 96: return xy_dense_rect_y<T, 96>(st, g, ops, nf, status);
            default: return xy_dense_rect_y<T, 128>(st, g, ops, nf, status);
        }
    }
    hipError_t e = hipErrorInvalidValue;
    switch (g.nx) {
        case 16: e = rows_launch<T, 16>(st, g, ops, nf, tw_x, status); break;
        case 32: e = rows_launch<T, 32>(st, g, ops, nf, tw_x, status); break;
        case 64: e = rows_launch<T, 64>(st, g, ops, nf, tw_x, status); break;
        case 96: e = rows_launch<T, 96>(st, g, ops, nf, tw_x, status); break;
        case 128: e = rows_launch<T, 128>(st, g, ops, nf, tw_x, status); break;
        case 256: e = rows_launch<T, 256>(st, g, ops, nf, tw_x, status); break;
        case 512: e = rows_launch<T, 512>(st, g, ops, nf, tw_x, status); break;
    }
    if (e != hipSuccess) return e;
    switch (g.ny) {
        case 16: return cols_launch<T, 16>(st, g, ops, nf, tw_y, status);
        case 32: return cols_launch<T, 32>(st, g, ops, nf, tw_y, status);
        case 64: return cols_launch<T, 64>(st, g, ops, nf, tw_y, status);
        case 96: return cols_launch<T, 96>(st, g, ops, nf, tw_y, status);
        case 128: return cols_launch<T, 128>(st, g, ops, nf, tw_y, status);
        case 256: return cols_launch<T, 256>(st, g, ops, nf, tw_y, status);
        case 512: return cols_launch<T, 512>(st, g, ops, nf, tw_y, status);
        default: return hipErrorInvalidValue;
    }
}

template <typename T>
hipError_t launch_xyplane(hipStream_t st, const Geometry &g, const FieldOps<T> &ops, int nf,
                          const cplx<T> *tw, const cplx<T> *tw_y, const int *status) {
    if (g.nx != g.ny || (g.nx == 128 && !dense_plane_grid<T>(g))) return xy_rect_launch<T>(st, g, ops, nf, tw, tw_y, status);
    switch (g.nx) {
        case 1: return xy_pixel_launch<T>(st, g, ops, nf, status);
        case 16: return xy_dense_launch<T, 16>(st, g, ops, nf, status);
        case 32: return xy_dense_launch<T, 32>(st, g, ops, nf, status);
        case 64: return xy_dense_launch<T, 64>(st, g, ops, nf, status);
        case 96: return xy_dense_launch<T, 96>(st, g, ops, nf, status);
        case 128: return xy_dense_launch<T, 128>(st, g, ops, nf, status);
        case 256:
            if constexpr (sizeof(T) == 4) return xy_rect_launch<T>(st, g, ops, nf, tw, tw_y, status);
            else return xy_split_launch<T, 256>(st, g, ops, nf, tw, status, tune_get(true, 1, 256));
        case 512: return xy_rect_launch<T>(st, g, ops, nf, tw, tw_y, status);   // bands of 16, one shape
        default: return hipErrorInvalidValue;
    }
}

// --------------------------------------------------------------- power
template <typename T>
__global__ void __launch_bounds__(256) k_power_partial(const cplx<T> *f0, const cplx<T> *f1,
                                                       const cplx<T> *f2, size_t n, double *partial,
                                                       const int *status) {
    if (status && *status) return;
    __shared__ double red[3][256];
    power_partial_block<T>(f0, f1, f2, n, blockIdx.x, gridDim.x, red, partial + blockIdx.x, gridDim.x);
}

__global__ void __launch_bounds__(256) k_power_final(const double *partial, int nblk, double pref0,
                                                     double pref1, double pref2, double *series,
                                                     int *trip, int *status, int check_nan,
                                                     int series_cap) {
    if (status && *status) return;
    __shared__ double red[3][256];
    power_final_sum(partial, nblk, nblk, red);
    if (threadIdx.x == 0) {
        double pw[3] = {pref0 * red[0][0], pref1 * red[1][0], pref2 * red[2][0]};
        int k = 0;
        if (trip) {
            k = *trip;
            *trip = k + 1;
        }
        if (k < series_cap)
            for (int f = 0; f < 3; ++f) series[3 * (size_t)k + f] = pw[f];
        if (check_nan && status && !isfinite(pw[1])) *status = k + 1;
    }
}

template <typename T>
hipError_t launch_power_partial(hipStream_t st, const cplx<T> *f0, const cplx<T> *f1,
                                const cplx<T> *f2, size_t n, int nblk, double *partial,
                                const int *status) {
    hipLaunchKernelGGL((k_power_partial<T>), dim3(nblk), dim3(256), 0, st, f0, f1, f2, n, partial, status);
    return hipGetLastError();
}

hipError_t launch_power_final(hipStream_t st, const double *partial, int nblk, double pref0,
                              double pref1, double pref2, double *series, int *trip, int *status,
                              int check_nan, int series_cap) {
    hipLaunchKernelGGL(k_power_final, dim3(1), dim3(256), 0, st, partial, nblk, pref0, pref1, pref2,
                       series, trip, status, check_nan, series_cap);
    return hipGetLastError();
}

// Power of one pixel's time series: pref * sum_t |A(x, y, t)|^2, one
// workgroup, Neumaier-compensated per thread and reduced in a fixed tree
// order (averagePowerTime, Solver3D.cuh:509-523).
template <typename T>
__global__ void __launch_bounds__(256) k_power_pixel(const cplx<T> *f, size_t plane, int nt,
                                                     double pref, double *out) {
    __shared__ double red[256];
    const int tid = threadIdx.x;
    double s = 0.0, c = 0.0;
    for (int t = tid; t < nt; t += 256) {
        const cplx<T> a = f[(size_t)t * plane];
        const double re = (double)a.x, im = (double)a.y;
        neumaier_add(s, c, fma(re, re, im * im));
    }
    red[tid] = s + c;
    __syncthreads();
    for (int w = 128; w > 0; w >>= 1) {
        if (tid < w) red[tid] += red[tid + w];
        __syncthreads();
    }
    if (tid == 0) out[0] = pref * red[0];
}

template <typename T>
hipError_t launch_power_pixel(hipStream_t st, const cplx<T> *f, size_t plane, int nt, double pref,
                              double *out) {
    hipLaunchKernelGGL((k_power_pixel<T>), dim3(1), dim3(256), 0, st, f, plane, nt, pref, out);
    return hipGetLastError();
}

// ------------------------------------------------------- instantiation
#define OPO_INST(T)                                                                               \
    template hipError_t launch_rk4<T>(hipStream_t, const cplx<T> *, cplx<T> *, cplx<T> *,          \
                                      cplx<T> *, size_t, size_t, const Rk4Args<T> &, const int *); \
    template hipError_t launch_tline<T>(hipStream_t, const Geometry &, const FieldOps<T> &, int,   \
                                        const cplx<T> *, const int *);                            \
    template hipError_t launch_tline3<T>(hipStream_t, const Geometry &, const TLine3Args<T> &,      \
                                         const cplx<T> *, const int *);                           \
    template hipError_t launch_plane_slices<T>(hipStream_t, int, const TLine3Args<T> &, int,       \
                                               const cplx<T> *, const int *);                     \
    template hipError_t launch_xyplane<T>(hipStream_t, const Geometry &, const FieldOps<T> &, int, \
                                          const cplx<T> *, const cplx<T> *, const int *);         \
    template hipError_t launch_power_partial<T>(hipStream_t, const cplx<T> *, const cplx<T> *,     \
                                                const cplx<T> *, size_t, int, double *, const int *); \
    template hipError_t launch_power_pixel<T>(hipStream_t, const cplx<T> *, size_t, int, double,   \
                                              double *);
OPO_INST(float)
OPO_INST(double)

}  // namespace opo
