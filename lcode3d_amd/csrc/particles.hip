// Particle kernels: field-free estimate, fused interpolation + pusher,
// coarse->fine interpolation + TSC deposition, and the device-side plasma
// set-up.  Particle positions and momenta are FP64 in every form; the
// deposition's arithmetic and LDS sums are FP64 too (its output grids are
// FP32 in the mixed form).

#include "common.hpp"

#include <algorithm>

namespace lcode {

namespace {

constexpr int kBlock = 256;
// Blocks of the grid-wide spill deposition (build option).
#ifndef LCODE_SPILL_BLOCKS
#define LCODE_SPILL_BLOCKS 256
#endif
constexpr int kSpillBlocks = LCODE_SPILL_BLOCKS;

// A value that every lane of the wave holds alike, in a scalar register.
__device__ __forceinline__ int scalar(int v) { return __builtin_amdgcn_readfirstlane(v); }

__device__ __forceinline__ double scalar(double v) {
    return __hiloint2double(scalar(__double2hiint(v)), scalar(__double2loint(v)));
}

__device__ __forceinline__ int clampi(int v, int n) {
    return v < 0 ? 0 : (v >= n ? n - 1 : v);
}

// Field-free half-step estimate with coordinate-only reflection using >= and
// <= (lcode.py:369-391).  Returns the estimated offsets.
__device__ __forceinline__ void estimate_one(double m, double xi0, double yi0,
                                             double xo, double yo, double px,
                                             double py, double pz, double dxi,
                                             double r, double& ex,
                                             double& ey) {
    double x = xi0 + xo, y = yi0 + yo;
    const double gamma_m = sqrt(m * m + pz * pz + px * px + py * py);
    x += px / (gamma_m - pz) * dxi;
    y += py / (gamma_m - pz) * dxi;
    if (x >= +r) x = +2 * r - x;
    if (x <= -r) x = -2 * r - x;
    if (y >= +r) y = +2 * r - y;
    if (y <= -r) y = -2 * r - y;
    ex = x - xi0;
    ey = y - yi0;
}

__global__ void __launch_bounds__(kBlock)
estimate_kernel(EstimateArgs a) {
    const int k = blockIdx.x * blockDim.x + threadIdx.x;
    if (k >= a.n) return;
    double ex, ey;
    estimate_one(a.m[k], a.x_init[k], a.y_init[k], a.prev_x_offt[k],
                 a.prev_y_offt[k], a.px[k], a.py[k], a.pz[k], a.dxi,
                 a.reflect, ex, ey);
    a.out_x[k] = ex;
    a.out_y[k] = ey;
}

// move_smart_kernel (lcode.py:704-793): midpoint position, 6-field TSC
// gather, two fixed-point iterations of the half-step momentum, offset and
// momentum update, reflection with strict > / < flipping the momentum.
// One-wave blocks spread the (few) coarse particles over all CUs.
#ifndef LCODE_PUSH_BLOCK
#define LCODE_PUSH_BLOCK 64
#endif
constexpr int kPushBlock = LCODE_PUSH_BLOCK;
// Deposition tiles per row that the push's per-tile bound table holds
// (more: each particle raises its tile's slot with a device atomic).
constexpr int kRegionRowMax = 128;
// A launch has about one wave per SIMD, so occupancy buys nothing: with a
// low waves-per-EU target the compiler issues the 54 field gathers of a
// particle together instead of one round trip at a time.
#ifndef LCODE_PUSH_WAVES
#define LCODE_PUSH_WAVES 2
#endif
#if LCODE_PUSH_WAVES > 0
#define LCODE_PUSH_ATTR __attribute__((amdgpu_waves_per_eu(1, LCODE_PUSH_WAVES)))
#else
#define LCODE_PUSH_ATTR
#endif

#ifndef LCODE_PUSH_BOUND_READ
#define LCODE_PUSH_BOUND_READ 1
#endif

// One coarse particle's push; returns max(|x_offt|, |y_offt|) after it and
// the particle's initial position in xi0, yi0.
// G: storage type of the field grids (the momentum update is FP64 in both).
template <typename G>
__device__ __forceinline__ double push_one(const PushArgs& a, int k, double& xi0,
                                           double& yi0) {
    const double m = a.m[k], q = a.q[k];
    const double opx = a.px[k], opy = a.py[k], opz = a.pz[k];
    xi0 = a.x_init[k];
    yi0 = a.y_init[k];
    double x_offt = a.prev_x_offt[k], y_offt = a.prev_y_offt[k];
    double ex, ey;
    if (a.est_x) {
        ex = a.est_x[k];
        ey = a.est_y[k];
    } else {
        estimate_one(m, xi0, yi0, x_offt, y_offt, opx, opy, opz, a.dxi,
                     a.reflect, ex, ey);
    }
    const double x_half = xi0 + (x_offt + ex) / 2;
    const double y_half = yi0 + (y_offt + ey) / 2;
    Tsc t;
    tsc_weights(x_half, y_half, a.N, a.h, t, a.fault);
    const double Ex = interp9(gp<G>(a.F[0]), a.N, t);
    const double Ey = interp9(gp<G>(a.F[1]), a.N, t);
    const double Ez = interp9(gp<G>(a.F[2]), a.N, t);
    const double Bx = interp9(gp<G>(a.F[3]), a.N, t);
    const double By = interp9(gp<G>(a.F[4]), a.N, t);
    const double Bz = interp9(gp<G>(a.F[5]), a.N, t);

    double px = opx, py = opy, pz = opz;
    double dpx = 0, dpy = 0, dpz = 0;
#pragma unroll
    for (int it = 0; it < 2; ++it) {
        const double gamma_m = sqrt(m * m + pz * pz + px * px + py * py);
        const double vx = px / gamma_m, vy = py / gamma_m, vz = pz / gamma_m;
        const double factor_1 = q * a.dxi / (1 - pz / gamma_m);
        dpx = factor_1 * (Ex + vy * Bz - vz * By);
        dpy = factor_1 * (Ey - vx * Bz + vz * Bx);
        dpz = factor_1 * (Ez + vx * By - vy * Bx);
        px = opx + dpx / 2;
        py = opy + dpy / 2;
        pz = opz + dpz / 2;
    }
    const double gamma_m = sqrt(m * m + pz * pz + px * px + py * py);
    x_offt += px / (gamma_m - pz) * a.dxi;
    y_offt += py / (gamma_m - pz) * a.dxi;
    px = opx + dpx;
    py = opy + dpy;
    pz = opz + dpz;

    const double r = a.reflect;
    double x = xi0 + x_offt, y = yi0 + y_offt;
    if (x > +r) { x = +2 * r - x; x_offt = x - xi0; px = -px; }
    if (x < -r) { x = -2 * r - x; x_offt = x - xi0; px = -px; }
    if (y > +r) { y = +2 * r - y; y_offt = y - yi0; py = -py; }
    if (y < -r) { y = -2 * r - y; y_offt = y - yi0; py = -py; }

    a.out_x[k] = x_offt;
    a.out_y[k] = y_offt;
    a.out_px[k] = px;
    a.out_py[k] = py;
    a.out_pz[k] = pz;
    // infinity marks a non-finite particle (fmax alone would drop a NaN)
    const bool finite = isfinite(x_offt) && isfinite(y_offt) && isfinite(px) &&
                        isfinite(py) && isfinite(pz);
    return finite ? fmax(fabs(x_offt), fabs(y_offt)) : __builtin_inf();
}

template <typename G>
__global__ void __launch_bounds__(kPushBlock) LCODE_PUSH_ATTR
push_kernel(PushArgs a) {
    const int k = blockIdx.x * blockDim.x + threadIdx.x;
    const int k0 = blockIdx.x * blockDim.x;
    // the block's first initial row, for the per-tile bound table: loaded
    // with the particle data, not after the stores (which may alias it)
    const double x_first = a.region_max ? a.x_init[k0] : 0.;
    double d = 0., xi0 = 0., yi0 = 0.;
    if (k < a.n && gate_open(a.gate)) d = push_one<G>(a, k, xi0, yi0);
    if (a.max_cells) {
        // cells the particles moved from their initial positions, at most
        // (the deposition sizes its tile halo by it); a non-finite state,
        // or one beyond kFarCells cells, is the kNonFinite mark, on which
        // the deposition writes NaN instead of depositing
        const double c = ceil(d / a.h);
        int cells = c <= kFarCells ? (int)c : kNonFinite;
        if (a.region_max) {
            // the bound of the deposition tile that holds the particle's
            // initial cell: the block's particles (consecutive, fewer than
            // a coarse row) lie in at most two rows of tiles, max-reduced
            // in an LDS table first (one LDS atomic per particle), then one
            // device atomic per tile touched (a slot takes those of the ~10
            // blocks over its particles); a shuffle loop over the wave's
            // tiles instead cost the push ~3 us of dependent latency
            __shared__ int rtab[2 * kRegionRowMax];
            const int nr = a.region_n, rn = nr - 1;
            const int ri0 = min(max(cell_of(x_first, a.N, a.h) / a.region_t, 0), rn);
            for (int e = threadIdx.x; e < 2 * kRegionRowMax; e += blockDim.x) rtab[e] = 0;
            __syncthreads();
            if (cells > 0) {   // (a particle that moved exists: k < n)
                const int ri = min(max(cell_of(xi0, a.N, a.h) / a.region_t, 0), rn);
                const int rj = min(max(cell_of(yi0, a.N, a.h) / a.region_t, 0), rn);
                const int dr = ri - ri0;
                if (dr >= 0 && dr < 2 && nr <= kRegionRowMax)
                    atomicMax(&rtab[dr * kRegionRowMax + rj], cells);
                else
                    atomicMax(a.region_max + ri * nr + rj, cells);
            }
            __syncthreads();
            if (nr <= kRegionRowMax) {
                for (int e = threadIdx.x; e < 2 * nr; e += blockDim.x) {
                    const int dr = e / nr, rj = e - dr * nr;
                    const int v = rtab[dr * kRegionRowMax + rj];
                    if (v > 0 && ri0 + dr <= rn) atomicMax(a.region_max + (ri0 + dr) * nr + rj, v);
                }
            }
        }
#pragma unroll
        for (int off = 32; off > 0; off >>= 1) cells = max(cells, __shfl_xor(cells, off, 64));
        // one atomic per wave, and (LCODE_PUSH_BOUND_READ) only when it raises
        // the bound: after the first waves the bound is reached and the rest
        // only read it (an atomic from every wave to the one address took the
        // push at 641^2 from 9.0 to 13.7 us)
        if ((threadIdx.x & 63) == 0) {
            if (!LCODE_PUSH_BOUND_READ ||
                cells > __hip_atomic_load(a.max_cells, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT))
                atomicMax(a.max_cells, cells);
            if (cells == kNonFinite) {
                if (a.host_flag)
                    __hip_atomic_store(a.host_flag, 1, __ATOMIC_RELAXED,
                                       __HIP_MEMORY_SCOPE_SYSTEM);
            }
        }
    }
}

// Coarse->fine interpolation of fine particle (fi, fj) (lcode.py:591-621)
// and its deposition values (lcode.py:651-655): dro = q / (1 - pz / gamma), dj
// = p dro / gamma, evaluated with one division as dro = q gamma r, dj = q p r,
// r = 1 / (gamma - pz) (the same quantities, rounded differently).  Reads
// everything from global memory.
struct FineParticle {
    double x, y;         // position
    double v[4];         // dro, djx, djy, djz
};

__device__ __forceinline__ void fine_particle(const DepositArgs& a, int fi, int fj,
                                              FineParticle& p) {
    const double ipi = a.ip[fi], ini = a.in[fi];
    const double ipj = a.ip[fj], inj = a.in[fj];
    const double A = ipi * ipj, B = ipi * inj, C = ini * ipj, D = ini * inj;
    const int nc = a.nc;
    // neighbour indices come from the caller: clamp so that bad ones cannot
    // read outside the coarse arrays
    const int pi = clampi((int)a.P[fi], nc), ni = clampi((int)a.Nn[fi], nc);
    const int pj = clampi((int)a.P[fj], nc), nj = clampi((int)a.Nn[fj], nc);
    const int pp = pi * nc + pj, pn = pi * nc + nj;
    const int np = ni * nc + pj, nn = ni * nc + nj;
#define LCODE_MIX(arr) (A * arr[pp] + B * arr[pn] + C * arr[np] + D * arr[nn])
    p.x = a.fg[fi] + LCODE_MIX(a.x_offt);
    p.y = a.fg[fj] + LCODE_MIX(a.y_offt);
    const double s = a.smallness;
    const double m = s * LCODE_MIX(a.m), q = s * LCODE_MIX(a.q), px = s * LCODE_MIX(a.px),
                 py = s * LCODE_MIX(a.py), pz = s * LCODE_MIX(a.pz);
#undef LCODE_MIX
    const double gamma = sqrt(m * m + px * px + py * py + pz * pz);
    const double qr = q / (gamma - pz);
    p.v[0] = gamma * qr;
    p.v[1] = px * qr;
    p.v[2] = py * qr;
    p.v[3] = pz * qr;
}


constexpr int kDepBlock = 256;   // threads of a deposition tile's block

// x / h + .5, its product rounded before the sum as the reference rounds its
// quotient (lcode.py:404): far from the axis a product left unrounded moves the
// weights by 1e-14 against it.
__device__ __forceinline__ double in_cells(double x, double inv_h) {
#pragma clang fp contract(off)
    const double q = x * inv_h;
    return q + .5;
}

// The cell of a fine particle, at its initial position or displaced: one rule for both,
// or a particle at rest on a cell's edge would seem to have moved.
__device__ __forceinline__ int dep_cell(double x, int N, double inv_h) {
    return (int)floor(in_cells(x, inv_h)) + N / 2;
}

// First fine index whose initial cell is >= c (fg is increasing).
__device__ int first_fine_at_or_after(const double* fg, int nf, int c, int N,
                                      double inv_h) {
    int lo = 0, hi = nf;
    while (lo < hi) {
        const int mid = (lo + hi) >> 1;
        if (dep_cell(fg[mid], N, inv_h) < c) lo = mid + 1; else hi = mid;
    }
    return lo;
}

template <typename G>
__device__ __forceinline__ void deposit_spill_one(const DepositArgs& a, int fk, int N) {
    FineParticle fp;
    fine_particle(a, fk / a.nf, fk % a.nf, fp);
    Tsc t;
    tsc_weights<double>(fp.x, fp.y, N, a.h, t, nullptr, 1. / a.h);
#pragma unroll
    for (int k = 0; k < 9; ++k) {
        const size_t idx = (size_t)(t.i + stencil_di(k)) * N + (t.j + stencil_dj(k));
        unsafeAtomicAdd(gp<G>(a.ro) + idx, (G)(fp.v[0] * t.w[k]));
        unsafeAtomicAdd(gp<G>(a.jx) + idx, (G)(fp.v[1] * t.w[k]));
        unsafeAtomicAdd(gp<G>(a.jy) + idx, (G)(fp.v[2] * t.w[k]));
        unsafeAtomicAdd(gp<G>(a.jz) + idx, (G)(fp.v[3] * t.w[k]));
    }
}

// deposit_kernel (lcode.py:626-663) as owner-computes tiles: each block
// accumulates its T^2 cells of ro, jx, jy, jz in LDS (FP64 LDS atomics,
// ds_add_f64), then stores them once, adding the ion background last
// (lcode.py:687).  Every cell of the grid is written by exactly one block, so
// the outputs need no zeroing.  A block visits the fine particles whose initial
// cell lies within halo + 1 cells of its tile; their per-index interpolation
// data and, when they fit, the coarse particles they interpolate from are
// staged in LDS first.  A particle displaced by more than a.halo cells from its
// initial cell is appended to the spill list by its home tile (the tile owning
// its initial cell), and deposit_spill_kernel, launched next, adds the list with
// device atomics across the whole grid.  A non-finite particle deposits nothing:
// the tile (or, when the pushes reported one, every tile) is written as NaN.  A
// split tile is deposited by two blocks, each over half of the strips; the
// second block to finish adds the first one's sums (published in global memory)
// and stores the tile.
//
// One thread takes a group of fine particles (fineness x fineness, one initial
// cell) and sums their 3 x 3 x 4 stencil values in registers while they share a
// stencil centre; the sums go to LDS when the centre changes and after the group
// (43.8 us per launch at 641^2 against 57.7 with one thread per particle).  The
// group's second particle is the one that more likely stays in the first one's
// cell.  Adjacent lanes hold adjacent cells, so the atomics of one instruction
// fall on distinct addresses.
//
// What bounds it at 641^2: a tile's start and end take 10 us (three dependent
// rounds of loads - bounds and the ends of the fine ranges, tables and coarse
// rectangle, then the stores - and the launch), the rest is the chain of a
// particle: two rounds of LDS reads and about 60 dependent FP64 operations, with
// three waves per SIMD to overlap it (VALU issue 62 % of that time, LDS 40 %).
// us per launch with 24-cell tiles everywhere and a longer start / now: 129^2 25.3 /
// 12.3, 361^2 28.8 / 20.0, 641^2 39.9 / 33.6, 1281^2 with fineness 3 231 / 167 (VALU issue
// 70 % there).  Tried at 641^2 and slower: strips of
// particles along j whose sums slide with the centre (61 us: the lanes leave
// their columns at different steps), 5 waves per block (44 - 65), 32-cell tiles
// with 8 waves (35 - 52).
template <int T>
struct DepTile {
    static constexpr int kPitch = T;                // LDS row of the sums
    static constexpr int kComp = T * kPitch;        // one component
    static constexpr int kExtMax = T + 14;          // initial cells per side: T + 2 halo + 2, halo <= 6
};

// LDS of a tile block: the sums, the fine-index tables of both axes (a.fine_max
// entries each) and the staged coarse rectangle (a.coarse_max squared, or 0).
// The staged particles lie in 16-byte pairs, so that one read brings two of a
// corner's values: (x_offt, y_offt), (m, q), (px, py), pz.
struct DepLds {
    double2 *wi, *wj;          // interpolation weights (ip, in)
    double2 *cpos, *cmq, *cpxy;
    int4 *xi, *xj;             // coarse neighbours (P, Nn), initial cell, -
    double *acc, *fi, *fj, *cpz;
    __device__ DepLds(unsigned char* p, int acc_len, int fine_max, int coarse_max) {
        auto take = [&](size_t bytes) {
            unsigned char* q = p;
            p += bytes;
            return q;
        };
        const size_t f = fine_max, c = (size_t)coarse_max * coarse_max;
        wi = (double2*)take(16 * f);
        wj = (double2*)take(16 * f);
        xi = (int4*)take(16 * f);
        xj = (int4*)take(16 * f);
        cpos = (double2*)take(16 * c);
        cmq = (double2*)take(16 * c);
        cpxy = (double2*)take(16 * c);
        acc = (double*)take(8 * (size_t)acc_len);
        fi = (double*)take(8 * f);
        fj = (double*)take(8 * f);
        cpz = (double*)take(8 * c);
    }
};

inline size_t deposit_lds_bytes(int T, int fine_max, int coarse_max) {
    return 8 * (size_t)(4 * T * T) + 80 * (size_t)fine_max +
           56 * (size_t)coarse_max * coarse_max;
}

// First fine index whose initial cell is >= c (fg is increasing), from this
// lane's sample of a 64-entry window at w0 (the cell of entry w0 + lane), else
// by search.  Every lane of the wave calls it.
__device__ __forceinline__ int wave_first_fine(const double* fg, int nf, int c, int N, double inv_h,
                                               int w0, int sample) {
    const int lane = threadIdx.x & 63;
    const int n = __popcll(__ballot(w0 + lane < nf && sample < c));
    const bool open_left = n > 0 || w0 == 0, open_right = n < 64 || w0 + 64 >= nf;
    if (open_left && open_right) return min(w0 + n, nf);
    return first_fine_at_or_after(fg, nf, c, N, inv_h);
}

// gamma = sqrt(s) and q / (gamma - pz), both rounded as the operations are: the
// hardware's estimates (25 bits) refined by one step of Goldschmidt's coupled iteration
// for sqrt(s) and 1 / (2 sqrt(s)) and one of Newton's for the reciprocal, then root and
// quotient corrected by their exact remainders (Markstein); the fixup gives
// division's infinities and NaN where gamma = pz.  Left out is the compiler's
// rescaling of tiny and huge arguments (gamma is a particle's energy).  Worst of 2^20
// random arguments 0.5 ulp for both; q times a reciprocal of two Newton steps,
// which costs as much (1281^2, fineness 3: 981 us a step with either), 1.4.
__device__ __forceinline__ void gamma_and_quotient(double s, double pz, double q, double& gamma,
                                                   double& qr) {
    const double r0 = __builtin_amdgcn_rsq(s);
    double g = s * r0, hh = .5 * r0;
    double e = fma(-hh, g, .5);
    g = fma(g, e, g);
    hh = fma(hh, e, hh);
    e = fma(-g, g, s);
    gamma = fma(e, hh, g);
    const double d = gamma - pz;
    double r = __builtin_amdgcn_rcp(d);
    r = fma(fma(-d, r, 1.), r, r);
    const double t = q * r;
    qr = __builtin_amdgcn_div_fixup(fma(fma(-d, t, q), r, t), d, q);
}

// G: storage type of the output grids (float: the mixed form).  The arithmetic
// and the sums are FP64 in both: at 641^2 FP32 LDS atomics (ds_add_f32) kept the
// LDS pipeline 8x longer busy than FP64 ones, and FP32 arithmetic left the
// density response of a small beam (amplitude 0.01) with relative errors up to
// 4e-4 in Ez.
template <int T, int W, bool STAGED, typename G>
__global__ void __launch_bounds__(kDepBlock) __attribute__((amdgpu_waves_per_eu(W)))
deposit_tile_kernel(DepositArgs a) {
    // the count slot of the next call is zeroed here (also when gated off)
    // unless a spill kernel follows, which does it
    if (a.spill_in_tiles && blockIdx.x == 0 && threadIdx.x == 0) *a.spill_next = 0;
    if (!gate_open(a.gate)) return;   // block-uniform: before any barrier
    using D = DepTile<T>;
    // W = 3: the values ahead of the checks, where their latency overlaps the
    // position's (151 registers); W = 4: after them (127)
    constexpr bool kEarly = W < 4;
    constexpr int kAcc = 4 * D::kComp;
    extern __shared__ __align__(16) unsigned char lds_raw[];
    const DepLds l(lds_raw, kAcc, a.fine_max, STAGED ? a.coarse_max : 0);
    __shared__ int last_block, split_last, tile_nan;
    __shared__ int range[4], corner[4];
    const int N = a.N;
    const double inv_h = scalar(1. / a.h);
    const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63;
    // tile of this block: row-major, or from the host's table (which keeps
    // neighbouring tiles on one XCD and gives each CU a mix of the wake's heavy
    // tiles and light ones; its last nsplit entries are the second parts of the
    // split tiles)
    const int ntx = a.ntx, lin = blockIdx.x;
    const unsigned word = scalar(a.tile_order ? (int)a.tile_order[lin] : 0);
    const DepBlock blk = dep_block(a.tile_order, word, lin);
    const int tile = blk.tile, slot = blk.slot, part = blk.part;
    const int nparts = slot >= 0 ? 2 : 1;
    const int ty = tile / ntx, tx = tile - ty * ntx;
    const int ci0 = ty * T, cj0 = tx * T;
    // the fine grid around this wave's end of a range (waves 0, 1: first and
    // last row, 2, 3: column): a window of 64 about where an even grid of
    // a.group points per cell has it, with the coarse neighbour there (the
    // corners of the coarse rectangle), loaded while the bounds below arrive
    static_assert(kDepBlock >= 256, "one wave per end of the two ranges");
    const bool last_end = wave & 1;
    const int end_cell = (wave < 2 ? ci0 : cj0) + (last_end ? T : -1);   // about
    const int guess = (int)floor(((double)(end_cell - N / 2) - .5) * a.group + .5 * (a.nf - 1));
    const int w0 = scalar(min(max(guess - 32, 0), max(a.nf - 64, 0)));
    const int64_t* const neighbour = last_end ? a.Nn : a.P;
    int sample = 0, sample_c = 0;
    if (a.nf > 0) {
        const int k = min(w0 + lane, a.nf - 1);
        sample_c = (int)neighbour[k];
        sample = dep_cell(a.fg[k], N, inv_h);
    }
    // halo: the displacement bound of the last pushes when one is given.
    // A fine particle's offset is a convex mix of coarse offsets, so its
    // cell moved at most `bound` cells: with bound <= a.halo no particle
    // can leave the halo, and every block (all read the same bound) skips
    // the spill list.  Otherwise particles beyond the halo take the exact
    // spill path.
    // With per-tile bounds the tile takes the largest of its 3 x 3 tile
    // neighbourhood: the fine particles it visits (initial cells within
    // halo + 1 of it) interpolate from coarse particles whose initial cells
    // lie within coarseness + 1 more cells, inside that neighbourhood (the
    // host enables the per-tile bounds only when that holds), and every tile
    // a particle's stencil reaches has the particle's home tile in its
    // neighbourhood, so all of them visit it, or (beyond a.halo) none does
    // and its home tile lists it.
    const int global = scalar(a.halo_cells ? max(*a.halo_cells, 0) : a.halo + 1);
    // the pushes met a non-finite (or absurdly far) particle: the whole
    // deposition is NaN, with no particle visited (already reported)
    const bool nonfinite = global >= kNonFinite;
    int bound = global;
    if (a.halo_regions && !nonfinite) {
        bound = 0;
        for (int di = -1; di <= 1; ++di)
            for (int dj = -1; dj <= 1; ++dj) {
                const int r = ty + di, c = tx + dj;
                if (r >= 0 && r < ntx && c >= 0 && c < ntx)
                    bound = max(bound, a.halo_regions[r * ntx + c]);
            }
    }
    const int halo = scalar(min(bound, a.halo));
    const bool may_spill = scalar(bound) > a.halo;
    if (threadIdx.x == 0 && part == 0) {
        // zero the slots the next pushes raise; nothing reads them here
        if (a.halo_next && tile == 0) *a.halo_next = 0;
        if (a.halo_regions_next) a.halo_regions_next[tile] = 0;
    }
    if (threadIdx.x == 0) tile_nan = 0;
    for (int k = threadIdx.x; k < kAcc; k += kDepBlock) l.acc[k] = 0;
    const int ext = T + 2 * halo + 2;
    if (wave < 4) {
        const int lo = (wave < 2 ? ci0 : cj0) - 1 - halo;
        const int r = wave_first_fine(a.fg, a.nf, lo + (last_end ? ext : 0), N, inv_h, w0, sample);
        // the coarse neighbour of the range's first (last) fine index
        const int at = min(max(last_end ? r - 1 : r, 0), max(a.nf - 1, 0));
        int c = __shfl(sample_c, at - w0, 64);
        if (at < w0 || at >= w0 + 64) c = (int)neighbour[at];
        if (lane == 0) {
            range[wave] = r;
            corner[wave] = clampi(c, a.nc);
        }
    }
    __syncthreads();
    const int fi_a = scalar(range[0]), ni = scalar(range[1]) - fi_a;
    const int fj_a = scalar(range[2]), nj = scalar(range[3]) - fj_a;
    const bool overfull = ni > a.fine_max || nj > a.fine_max || ext > D::kExtMax;
    if (overfull) {
        // denser fine grid than the host-checked fineness allows: flag the
        // tile as faulted and fill it with NaN rather than drop particles
        if (threadIdx.x == 0 && part == 0) atomicAdd(a.fault, 1);
    } else if (!nonfinite && ni > 0 && nj > 0) {
        // coarse rectangle referenced by this block's fine particles:
        // indices_prev/next grow with the fine index, so it is [P[first],
        // Nn[last]] on each axis; the host checked the fit
        int cI0 = 0, cJ0 = 0, cH = a.nc, cW = a.nc;
        if constexpr (STAGED) {
            cI0 = scalar(corner[0]);
            cJ0 = scalar(corner[2]);
            cH = scalar(corner[1]) - cI0 + 1;
            cW = scalar(corner[3]) - cJ0 + 1;
            if (cH > a.coarse_max || cW > a.coarse_max || cH < 0 || cW < 0) {
                if (threadIdx.x == 0 && part == 0) atomicAdd(a.fault, 1);
                cH = cH < 0 ? 0 : (cH > a.coarse_max ? a.coarse_max : cH);
                cW = cW < 0 ? 0 : (cW > a.coarse_max ? a.coarse_max : cW);
            }
        }
        // the tables, their neighbour indices as offsets in the rectangle:
        // rows scaled by its width, each clamped into it, so that a row part
        // plus a column part is an in-bounds index
        const int hmax = max(cH - 1, 0), wmax = max(cW - 1, 0);
        // staged as shares of a fine particle (`sm` first: a plasma of coarseness^2
        // masses then has an exact 1 / fineness^2, and a particle at rest exactly its
        // charge); `same`: every particle has the first one's mass and charge
        const double sm = a.smallness;
        bool same = STAGED;
        double m0 = 0., q0 = 0.;
        struct Coarse {
            double x, y, m, q, px, py, pz;
        };
        struct Fine {
            double ip, in, fg;
            int P, Nn;
        };
        auto coarse_load = [&](int r, int c) {
            const size_t g = (size_t)(cI0 + r) * a.nc + cJ0 + c;
            return Coarse{a.x_offt[g], a.y_offt[g], a.m[g], a.q[g], a.px[g], a.py[g], a.pz[g]};
        };
        auto coarse_store = [&](int r, int c, const Coarse& v) {
            const int k = r * cW + c;
            l.cpos[k] = make_double2(v.x, v.y);
            l.cmq[k] = make_double2(sm * v.m, sm * v.q);
            l.cpxy[k] = make_double2(sm * v.px, sm * v.py);
            l.cpz[k] = sm * v.pz;
            same = same && v.m == m0 && v.q == q0;
        };
        auto fine_load = [&](int k) {
            const int f = k >= ni ? fj_a + k - ni : fi_a + k;
            return Fine{a.ip[f], a.in[f], a.fg[f], clampi((int)a.P[f], a.nc),
                        clampi((int)a.Nn[f], a.nc)};
        };
        auto fine_store = [&](int k, const Fine& v) {
            const bool isj = k >= ni;
            // (the j tables follow the i tables)
            const int s = isj ? k - ni + a.fine_max : k, lo = isj ? cJ0 : cI0,
                      hi = isj ? wmax : hmax, scale = isj ? 1 : cW;
            l.wi[s] = make_double2(v.ip, v.in);
            l.fi[s] = v.fg;
            l.xi[s] = make_int4(min(max(v.P - lo, 0), hi) * scale,
                                min(max(v.Nn - lo, 0), hi) * scale,
                                dep_cell(v.fg, N, inv_h), 0);
        };
        // 16 x 16 threads over the rectangle; every thread's first entries of both
        // tables on their way together, the rest (large ranges) in turn
        const int tr = threadIdx.x >> 4, tc = threadIdx.x & 15;
        const bool have_c = STAGED && tr < cH && tc < cW, have_f = (int)threadIdx.x < ni + nj;
        Coarse first_c{};
        Fine first_f{};
        if (have_f) first_f = fine_load(threadIdx.x);
        if constexpr (STAGED) {
            if (have_c) first_c = coarse_load(tr, tc);
            if (cH > 0 && cW > 0) {
                const size_t first = (size_t)cI0 * a.nc + cJ0;
                m0 = a.m[first];
                q0 = a.q[first];
            }
        }
        if (have_f) fine_store(threadIdx.x, first_f);
        for (int k = threadIdx.x + kDepBlock; k < ni + nj; k += kDepBlock)
            fine_store(k, fine_load(k));
        if constexpr (STAGED) {
            if (have_c) coarse_store(tr, tc, first_c);
            for (int r = tr; r < cH; r += kDepBlock / 16)
                for (int c = r == tr ? tc + 16 : tc; c < cW; c += 16)
                    coarse_store(r, c, coarse_load(r, c));
        }
        const bool uniform = __syncthreads_and(same);
        m0 = scalar(sm * m0);
        q0 = scalar(sm * q0);
        // can a particle's stencil centre lie outside [1, N - 2]?
        const bool edge = ci0 < 2 * halo + 2 || ci0 + T + 2 * halo + 1 > N - 2 ||
                          cj0 < 2 * halo + 2 || cj0 + T + 2 * halo + 1 > N - 2;
        const int gs = a.group > 0 ? a.group : 1, gs2 = gs * gs;
        const int ngi = (ni + gs - 1) / gs, ngj = (nj + gs - 1) / gs, ng = ngi * ngj;
        const float per_row = 1.f / ngj;
        // a particle at this offset in its cell (or above) is followed by one in
        // the next cell within its group
        const double roomy = scalar(.5 - (double)(gs - 1) / gs);
        const int ih = N / 2;
        constexpr int kNoCentre = -(1 << 20);
        double pat[4][9];
#pragma unroll
        for (int k = 0; k < 36; ++k) (&pat[0][0])[k] = 0.;
        // The last round of groups is rarely full, and wave w of every block sits
        // on SIMD w: the blocks of a CU (256 apart in launch order) start the
        // rounds at different waves, so that the extra ones spread over its SIMDs
        const int start = (wave + (lin >> 8)) % (kDepBlock / 64) * 64 + lane + part * kDepBlock;
#pragma unroll 1
        for (int L = start; L < ng; L += nparts * kDepBlock) {
            const int gi = (int)((L + .5f) * per_row), gj = L - gi * ngj;
            int ai = kNoCentre, aj = kNoCentre;   // centre of the sums in pat
            int qa = 0, qb = 0;     // particle of the group
            bool swap = false;      // its rows first, then its columns
            // the sums to the cells that are the tile's (none about kNoCentre)
            auto flush = [&]() {
                const int si = ai - 1 - ci0, sj = aj - 1 - cj0;
                double* const p0 = l.acc + si * D::kPitch + sj;
                bool in_i[3], in_j[3];
#pragma unroll
                for (int r = 0; r < 3; ++r) {
                    in_i[r] = (unsigned)(si + r) < (unsigned)T;
                    in_j[r] = (unsigned)(sj + r) < (unsigned)T;
                }
#pragma unroll
                for (int k = 0; k < 9; ++k) {
                    const int r = stencil_di(k) + 1, c = stencil_dj(k) + 1;
                    if (in_i[r] & in_j[c]) {
#pragma unroll
                        for (int n = 0; n < 4; ++n)
                            atomicAdd(p0 + r * D::kPitch + c + n * D::kComp, pat[n][k]);
                    }
                }
#pragma unroll
                for (int k = 0; k < 36; ++k) (&pat[0][0])[k] = 0.;
            };
#pragma unroll 1
            for (int q = 0; q < gs2; ++q) {
                // (opaque in the loop, or the compiler makes a copy of the whole
                // loop for each value of the block's flags, with more registers)
                int is_uniform = scalar(uniform), is_edge = scalar(edge);
                asm volatile("" : "+s"(is_uniform), "+s"(is_edge));
                const int li = gi * gs + (swap ? qb : qa), lj = gj * gs + (swap ? qa : qb);
                if (++qb == gs) {
                    qb = 0;
                    ++qa;
                }
                if (li >= ni || lj >= nj) continue;
                // coarse->fine interpolation (lcode.py:591-621), then TSC centre and
                // offset in the cell (lcode.py:404-407)
                const double2 wi = l.wi[li], wj = l.wj[lj];
                const int4 xi = l.xi[li], xj = l.xj[lj];
                const double wA = wi.x * wj.x, wB = wi.x * wj.y, wC = wi.y * wj.x,
                             wD = wi.y * wj.y;
                const int pp = xi.x + xj.x, pn = xi.x + xj.y;
                const int np = xi.y + xj.x, nn = xi.y + xj.y;
                double x, y;
                if constexpr (STAGED) {
                    const double2 cA = l.cpos[pp], cB = l.cpos[pn], cC = l.cpos[np],
                                  cD = l.cpos[nn];
                    x = l.fi[li] + (wA * cA.x + wB * cB.x + wC * cC.x + wD * cD.x);
                    y = l.fj[lj] + (wA * cA.y + wB * cB.y + wC * cC.y + wD * cD.y);
                } else {
#define LCODE_MIX(arr) (wA * arr[pp] + wB * arr[pn] + wC * arr[np] + wD * arr[nn])
                    x = l.fi[li] + LCODE_MIX(a.x_offt);
                    y = l.fj[lj] + LCODE_MIX(a.y_offt);
                }
                // the deposition values (lcode.py:651-655) from the mixed mass,
                // charge and momentum: dro = q gamma r, dj = q p r with r = 1 /
                // (gamma - pz)
                double v[4];
                auto values = [&]() {
                    double m, qq, px, py, pz;
                    if (STAGED && is_uniform) {
                        const double w = (wA + wB) + (wC + wD);
                        m = w * m0;
                        qq = w * q0;
                    } else if constexpr (STAGED) {
                        const double2 mA = l.cmq[pp], mB = l.cmq[pn], mC = l.cmq[np], mD = l.cmq[nn];
                        m = wA * mA.x + wB * mB.x + wC * mC.x + wD * mD.x;
                        qq = wA * mA.y + wB * mB.y + wC * mC.y + wD * mD.y;
                    } else {
                        m = sm * LCODE_MIX(a.m);
                        qq = sm * LCODE_MIX(a.q);
                    }
                    if constexpr (STAGED) {
                        const double2 pA = l.cpxy[pp], pB = l.cpxy[pn], pC = l.cpxy[np],
                                      pD = l.cpxy[nn];
                        px = wA * pA.x + wB * pB.x + wC * pC.x + wD * pD.x;
                        py = wA * pA.y + wB * pB.y + wC * pC.y + wD * pD.y;
                        pz = wA * l.cpz[pp] + wB * l.cpz[pn] + wC * l.cpz[np] + wD * l.cpz[nn];
                    } else {
                        px = sm * LCODE_MIX(a.px);
                        py = sm * LCODE_MIX(a.py);
                        pz = sm * LCODE_MIX(a.pz);
#undef LCODE_MIX
                    }
                    double gamma, qr;
                    gamma_and_quotient(m * m + px * px + py * py + pz * pz, pz, qq, gamma, qr);
                    v[0] = gamma * qr;
                    v[1] = px * qr;
                    v[2] = py * qr;
                    v[3] = pz * qr;
                };
                if constexpr (kEarly) values();
                const double xh = in_cells(x, inv_h), yh = in_cells(y, inv_h);
                const double fx = floor(xh), fy = floor(yh);
                const double xl = xh - fx - .5, yl = yh - fy - .5;
                // (.5 + x)^2 / 2, (.5 - x)^2 / 2 and .75 - x^2
                const double wxP = fma(xl, fma(xl, .5, .5), .125), wxM = fma(xl, fma(xl, .5, -.5), .125);
                const double wyP = fma(yl, fma(yl, .5, .5), .125), wyM = fma(yl, fma(yl, .5, -.5), .125);
                const double wx[3] = {wxM, fma(-xl, xl, .75), wxP};
                const double wy[3] = {wyP, fma(-yl, yl, .75), wyM};   // stencil order
                int ti = (int)fx + ih, tj = (int)fy + ih;
                const int ci = xi.z, cj = xj.z;   // initial cell
                const bool home = ((unsigned)(ci - ci0) < (unsigned)T) &
                                  ((unsigned)(cj - cj0) < (unsigned)T);
                // (NaN where the position is not finite)
                const bool odd = __builtin_isunordered(xl, yl);
                if (is_edge && !odd && !(ti >= 1 && ti <= N - 2 && tj >= 1 && tj <= N - 2)) {
                    // (a centre further than kFarCells stays as it is: beyond the halo)
                    constexpr int kFar = (int)kFarCells;
                    if ((unsigned)ti - ih + kFar < 2u * kFar &&
                        (unsigned)tj - ih + kFar < 2u * kFar) {
                        if (home) atomicAdd(a.fault, 1);
                        ti = min(max(ti, 1), N - 2);
                        tj = min(max(tj, 1), N - 2);
                    }
                }
                if (q == 0) swap = yl >= roomy;
                if (odd | ((unsigned)(ti - ci + halo) > 2u * halo) |
                    ((unsigned)(tj - cj + halo) > 2u * halo)) {
                    if (home) {
                        if (odd || !(fabs(xh) <= kFarCells && fabs(yh) <= kFarCells)) {
                            // non-finite or absurdly far particle (a deposition
                            // called without the pushes' bound): its home tile
                            // becomes NaN
                            tile_nan = 1;
                            if (a.host_flag)
                                __hip_atomic_store(a.host_flag, 1, __ATOMIC_RELAXED,
                                                   __HIP_MEMORY_SCOPE_SYSTEM);
                        } else {
                            // moved more than the halo: its home tile lists it
                            // (beyond a bound the pushes reported: cannot happen;
                            // counted as a fault rather than listed for a pass
                            // that does not run)
                            if (!is_edge && !(ti >= 1 && ti <= N - 2 && tj >= 1 && tj <= N - 2))
                                atomicAdd(a.fault, 1);
                            if (may_spill) {
                                a.spill[atomicAdd(a.spill_count, 1)] =
                                    (fi_a + li) * a.nf + fj_a + lj;
                                if (a.host_spill)
                                    __hip_atomic_store(a.host_spill, 1, __ATOMIC_RELAXED,
                                                       __HIP_MEMORY_SCOPE_SYSTEM);
                            } else {
                                atomicAdd(a.fault, 1);
                            }
                        }
                    }
                    continue;
                }
                // does the 3 x 3 stencil reach this tile?
                if (((unsigned)(ti + 1 - ci0) >= (unsigned)(T + 2)) |
                    ((unsigned)(tj + 1 - cj0) >= (unsigned)(T + 2)))
                    continue;
                if ((ti != ai) | (tj != aj)) {
                    if (ai != kNoCentre) flush();   // another centre
                    ai = ti;
                    aj = tj;
                }
                if constexpr (!kEarly) values();
#pragma unroll
                for (int k = 0; k < 9; ++k) {
                    const double w = wx[k % 3] * wy[k / 3];
#pragma unroll
                    for (int n = 0; n < 4; ++n) pat[n][k] += v[n] * w;
                }
            }
            flush();
        }
    }
    // the ion background of this thread's cells, on its way while the block's
    // other waves finish
    constexpr int kOut = (T * T + kDepBlock - 1) / kDepBlock;
    double base[kOut];
#pragma unroll
    for (int u = 0; u < kOut; ++u) {
        const int k = threadIdx.x + u * kDepBlock;
        const int i = ci0 + k / T, j = cj0 + k % T;
        base[u] = 0.;
        if (k < T * T && i < N && j < N && a.ro_initial)
            base[u] = a.ro_initial[(size_t)i * N + j];
    }
    __syncthreads();
    // a split tile: both parts publish their sums (all NaN from a part that
    // met a non-finite particle of the tile, so that the total is NaN); the
    // second to finish adds the other's sums to its own and stores the tile
    bool store = true;
    if (nparts == 2) {
        double* const mine = a.split_part + ((size_t)slot * 2 + part) * kAcc;
        const double* const other = a.split_part + ((size_t)slot * 2 + 1 - part) * kAcc;
        // The sums travel as device-scope atomic stores and loads (written
        // through to, and read from, the device-coherent level), and every
        // wave waits for its stores to complete before the barrier that
        // precedes the count (the barrier alone does not wait for global
        // stores).  A device-scope fence instead writes back and invalidates
        // the whole L2 of the XCD, under every other block there (measured:
        // 40.7 -> 58.6 us per launch with 39 split tiles).
        for (int k = threadIdx.x; k < kAcc; k += kDepBlock)
            __hip_atomic_store(mine + k, tile_nan ? __builtin_nan("") : l.acc[k],
                               __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        __builtin_amdgcn_s_waitcnt(0);   // vmcnt, expcnt and lgkmcnt all zero
        __syncthreads();
        if (threadIdx.x == 0) split_last = atomicAdd(a.split_count + slot, 1) == 1;
        __syncthreads();
        store = split_last;
        if (store) {
            for (int k = threadIdx.x; k < kAcc; k += kDepBlock)
                l.acc[k] += __hip_atomic_load(other + k, __ATOMIC_RELAXED,
                                              __HIP_MEMORY_SCOPE_AGENT);
            if (threadIdx.x == 0) a.split_count[slot] = 0;
            __syncthreads();
        }
    }
    // store the tile, adding the ion background to ro last (lcode.py:687)
    if (store) {
#pragma unroll
        for (int u = 0; u < kOut; ++u) {
            const int k = threadIdx.x + u * kDepBlock;
            const int r = k / T, c = k % T;
            const int i = ci0 + r, j = cj0 + c;
            if (k >= T * T || i >= N || j >= N) continue;
            const size_t idx = (size_t)i * N + j;
            G* const ro = gp<G>(a.ro);
            G* const jx = gp<G>(a.jx);
            G* const jy = gp<G>(a.jy);
            G* const jz = gp<G>(a.jz);
            const bool bad = overfull || nonfinite || tile_nan;
            const double nan = __builtin_nan("");
            const double* s = l.acc + r * D::kPitch + c;
            // the FP64 ion background is added in FP64, then rounded once
            ro[idx] = (G)(bad ? nan : a.ro_initial ? s[0] + base[u] : s[0]);
            jx[idx] = (G)(bad ? nan : s[D::kComp]);
            jy[idx] = (G)(bad ? nan : s[2 * D::kComp]);
            jz[idx] = (G)(bad ? nan : s[3 * D::kComp]);
        }
    }
    // a particle may have spilled somewhere (the bound every block read exceeds the
    // largest halo) and no spill kernel follows: the last block to finish, after every
    // block's stores are visible, deposits the list.  One thread makes the block's
    // stores visible (they are complete at the barrier): a fence in every wave, which
    // also drops the XCD's L2, took lcode_deposit at 193^2 with offsets just beyond the
    // halo 71 us instead of 28.5, a step there with spills 282 instead of 146.
    // (Device-scope atomic stores without a fence: 25.4 and 119, but 0.2 us more in
    // every launch with 8- and 16-cell tiles, which take them by a branch.)
    if (a.spill_in_tiles && global > a.halo && !nonfinite) {
        __builtin_amdgcn_s_waitcnt(0);   // this wave's stores are complete
        __syncthreads();
        if (threadIdx.x == 0) {
            __builtin_amdgcn_fence(__ATOMIC_RELEASE, "agent");
            last_block = atomicAdd(a.done, 1) == (int)gridDim.x - 1;
        }
        __syncthreads();
        if (last_block) {
            __threadfence();
            const int count = __hip_atomic_load(a.spill_count, __ATOMIC_RELAXED,
                                                __HIP_MEMORY_SCOPE_AGENT);
            for (int p = threadIdx.x; p < count; p += kDepBlock)
                deposit_spill_one<G>(a, a.spill[p], N);
            if (threadIdx.x == 0) *a.done = 0;
        }
    }
}

// Deposits the particles the tile kernel listed as displaced beyond its
// halo, with device-scope atomics over the whole grid (after the tile
// kernel's stores, which it follows on the stream), and zeroes the count
// slot of the next call.  An empty list costs one load per block.
template <typename G>
__global__ void __launch_bounds__(kBlock)
deposit_spill_kernel(DepositArgs a) {
    if (blockIdx.x == 0 && threadIdx.x == 0) *a.spill_next = 0;
    if (!gate_open(a.gate)) return;
    const int count = *a.spill_count;
    for (int p = blockIdx.x * blockDim.x + threadIdx.x; p < count;
         p += gridDim.x * blockDim.x)
        deposit_spill_one<G>(a, a.spill[p], a.N);
}

// The displacement bound of a deposition without a push before it: raises
// *bound to the cells that the coarse offsets move a particle at most, or to
// halo + 1 (which sends the deposition to its largest halo and the spill list)
// when an offset is not finite or larger, or when an interpolation weight would
// let a fine particle move further than its coarse ones.  At 641^2 it takes 7 of
// lcode_deposit's 39 us, which took 122 with the largest halo's three times as many
// particles per tile and a fence in every wave; with particles beyond that halo it is
// what it costs (58 -> 63).
__global__ void __launch_bounds__(kBlock)
deposit_bound_kernel(DepositArgs a, int* bound) {
    const int k = blockIdx.x * blockDim.x + threadIdx.x;
    int cells = 0;
    if (k < a.nc * a.nc) {
        // (rounded up by more than the interpolation's rounding)
        const double d = fmax(fabs(a.x_offt[k]), fabs(a.y_offt[k])) * (1. + 1e-9) / a.h;
        const bool finite = isfinite(a.x_offt[k]) && isfinite(a.y_offt[k]);
        cells = finite && d <= a.halo ? (int)ceil(d) : a.halo + 1;
    }
    if (k < a.nf) {
        const double p = a.ip[k], n = a.in[k];
        if (!(p >= 0. && n >= 0. && p + n <= 1. + 1e-10)) cells = a.halo + 1;
    }
#pragma unroll
    for (int off = 32; off > 0; off >>= 1) cells = max(cells, __shfl_xor(cells, off, 64));
    if ((threadIdx.x & 63) == 0 &&
        cells > __hip_atomic_load(bound, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT))
        atomicMax(bound, cells);
}

__global__ void __launch_bounds__(64) zero_ints_kernel(int* p, int n) {
    for (int k = threadIdx.x; k < n; k += blockDim.x) p[k] = 0;
}

// ---------------------------------------------------------------------------
// Plasma set-up (make_plasma, lcode.py:452-573) on the device, in the
// reference's FP64 arithmetic (integer counters converted exactly)
// ---------------------------------------------------------------------------

// Coarse grid point i of 2 hc - 1: -(hc - 1 - i) s for the left half,
// (i - hc + 1) s for the right one (lcode.py:452-465).
__device__ __forceinline__ double coarse_at(int i, int hc, double s) {
#pragma clang fp contract(off)
    const int k = i - (hc - 1);
    return k < 0 ? -((double)(-k) * s) : (double)k * s;
}

// Fine grid point i (lcode.py:468-487): odd fineness, 2 hf - 1 points on
// k s; even fineness, 2 hf points on (.5 + k) s.
__device__ __forceinline__ double fine_at(int i, int hf, int odd, double s) {
#pragma clang fp contract(off)
    if (odd) {
        const int k = i - (hf - 1);
        return k < 0 ? -((double)(-k) * s) : (double)k * s;
    }
    return i < hf ? -((.5 + (double)(hf - 1 - i)) * s) : (.5 + (double)(i - hf)) * s;
}

__global__ void __launch_bounds__(kBlock)
plasma_coarse_kernel(PlasmaArgs a) {
#pragma clang fp contract(off)
    const int k = blockIdx.x * blockDim.x + threadIdx.x;
    if (k >= a.nc * a.nc) return;
    const int i = k / a.nc, j = k % a.nc;
    const double s = a.cell * a.coarseness;
    a.x_init[k] = coarse_at(i, a.hc, s);
    a.y_init[k] = coarse_at(j, a.hc, s);
    const double c2 = (double)(a.coarseness * a.coarseness);
    a.m[k] = 1. * kElectronMass * c2;        // ones * ELECTRON_MASS * c**2
    a.q[k] = 1. * kElectronCharge * c2;
}

// virt_params (lcode.py:526-570): searchsorted of each fine point in the
// coarse grid (first index with coarse >= fine), the clipped neighbour
// indices and the interpolation weights with the boundary fixes.
__global__ void __launch_bounds__(kBlock)
plasma_fine_kernel(PlasmaArgs a) {
    // no fused multiply-adds: every operation rounds as NumPy's does
#pragma clang fp contract(off)
    const int f = blockIdx.x * blockDim.x + threadIdx.x;
    if (f >= a.nf) return;
    const double sc = a.cell * a.coarseness;
    const double sf = a.cell / a.fineness;
    const double x = fine_at(f, a.hf, a.fineness % 2, sf);
    int lo = 0, hi = a.nc;
    while (lo < hi) {
        const int mid = (lo + hi) >> 1;
        if (coarse_at(mid, a.hc, sc) < x) lo = mid + 1; else hi = mid;
    }
    const int nxt = lo < 0 ? 0 : (lo > a.nc - 1 ? a.nc - 1 : lo);
    const int prv = lo - 1 < 0 ? 0 : (lo - 1 > a.nc - 1 ? a.nc - 1 : lo - 1);
    double wp = (coarse_at(nxt, a.hc, sc) - x) / sc;
    double wn = (x - coarse_at(prv, a.hc, sc)) / sc;
    if (nxt == 0) { wp = 0.; wn = 1.; }
    if (prv == a.nc - 1) { wn = 0.; wp = 1.; }
    a.fg[f] = x;
    a.ip[f] = wp;
    a.in[f] = wn;
    a.P[f] = prv;
    a.Nn[f] = nxt;
}

inline int blocks_for(long n) { return (int)((n + kBlock - 1) / kBlock); }

}  // namespace

int launch_estimate(const EstimateArgs& a, hipStream_t s, Profiler* prof) {
    if (a.n == 0) return LCODE_OK;
    ProfScope ps(prof, "estimate", s);
    estimate_kernel<<<blocks_for(a.n), kBlock, 0, s>>>(a);
    LCODE_HIP(hipGetLastError());
    return LCODE_OK;
}

int launch_push(const PushArgs& a, hipStream_t s, Profiler* prof) {
    if (a.n == 0) return LCODE_OK;
    ProfScope ps(prof, "push", s, true);
    const dim3 blocks((a.n + kPushBlock - 1) / kPushBlock);
    if (a.grid32)
        launch_timed(ps, push_kernel<float>, blocks, dim3(kPushBlock), 0, s, a);
    else
        launch_timed(ps, push_kernel<double>, blocks, dim3(kPushBlock), 0, s, a);
    LCODE_HIP(hipGetLastError());
    return LCODE_OK;
}

int launch_make_plasma(const PlasmaArgs& a, hipStream_t s) {
    if (a.nc > 0) {
        plasma_coarse_kernel<<<blocks_for((long)a.nc * a.nc), kBlock, 0, s>>>(a);
        LCODE_HIP(hipGetLastError());
    }
    if (a.nf > 0) {
        plasma_fine_kernel<<<blocks_for(a.nf), kBlock, 0, s>>>(a);
        LCODE_HIP(hipGetLastError());
    }
    return LCODE_OK;
}

int launch_deposit_bound(const DepositArgs& a, int* bound, hipStream_t s, Profiler* prof) {
    ProfScope ps(prof, "deposit_bound", s, true);
    const int n = std::max(a.nc * a.nc, a.nf);
    if (n > 0)
        launch_timed(ps, deposit_bound_kernel, dim3(blocks_for(n)), dim3(kBlock), 0, s, a, bound);
    LCODE_HIP(hipGetLastError());
    return LCODE_OK;
}

int launch_zero_ints(int* p, int n, hipStream_t s) {
    if (n <= 0) return LCODE_OK;
    zero_ints_kernel<<<1, 64, 0, s>>>(p, n);
    LCODE_HIP(hipGetLastError());
    return LCODE_OK;
}

// The tile kernel for a tile, its waves per SIMD and forms, or NULL.
using DepKernel = void (*)(DepositArgs);
template <int T, int W>
static DepKernel deposit_kernel_of(bool staged, bool grid32) {
    if (staged)
        return grid32 ? deposit_tile_kernel<T, W, true, float> : deposit_tile_kernel<T, W, true, double>;
    return grid32 ? deposit_tile_kernel<T, W, false, float> : deposit_tile_kernel<T, W, false, double>;
}
static DepKernel deposit_kernel_of(int tile, int waves, bool staged, bool grid32) {
    switch (tile * 10 + waves) {
        case 83: return deposit_kernel_of<8, 3>(staged, grid32);
        case 163: return deposit_kernel_of<16, 3>(staged, grid32);
        case 243: return deposit_kernel_of<24, 3>(staged, grid32);
        case 244: return deposit_kernel_of<24, 4>(staged, grid32);
        default: return nullptr;
    }
}

int deposit_blocks_per_cu(const DepositPlan& p) {
    int least = 0;
    for (const bool grid32 : {false, true}) {
        int n = 0;
        if (hipOccupancyMaxActiveBlocksPerMultiprocessor(
                &n, reinterpret_cast<const void*>(deposit_kernel_of(p.tile, p.waves, p.staged, grid32)),
                kDepBlock, deposit_lds_bytes(p.tile, p.fine_max, p.staged ? p.coarse_max : 0)) !=
            hipSuccess) {
            (void)hipGetLastError();   // leave no error behind for later checks
            return 0;
        }
        least = grid32 ? std::min(least, n) : n;
    }
    return least;
}

// Small grids take small tiles: 24-cell ones would leave CUs idle (36 tiles at
// 129^2) and the launch as long as the chain of one tile.  us per launch in a step,
// fineness 2, displacements to 1.2 cells, 8 / 16 / 24 cells a side:
//   coarseness 2 (24 cells: not staged)      coarseness 3
//   129^2  11.5 / 13.6 / 23.3                181^2  11.6 / 13.2 / 17.5
//   193^2  13.2 / 14.5 / 23.2                201^2  12.9 / 14.0 / 17.7
//   217^2  12.3 / 15.0 / 24.8                217^2  12.4 / 14.2 / 18.2
//   257^2  17.5 / 16.0 / 25.6                241^2  16.6 / 14.9 / 18.8
//   321^2  24.5 / 18.3 / 27.3                385^2  31.8 / 19.3 / 23.0
//   401^2  35.0 / 20.5 / 32.3                433^2  39.3 / 22.3 / 24.8
//   541^2     - / 33.2 / 40.8                481^2     - / 28.6 / 27.1
//   641^2     - / 43.7 / 46.8                641^2     - / 42.9 / 32.6
// (coarseness 3 up to 433^2: 0.5 cells.)  The sides cross where the smaller tiles take
// a second round of the block slots (8 cells beyond 216^2, 16 cells beyond 432^2 on
// 256 CUs with three blocks each); the lines at 200 and 400 lie a little below, and
// take no account of the CUs or the coarseness.
// Tiles larger than 24 cells leave too few blocks at 641^2 or too few registers
// for the waves (32 cells with 8 waves 34.8 - 52).  In launches of several
// rounds four waves per SIMD hide more of a tile's start than three (1281^2,
// fineness 3: 190 -> 178), in one round they leave the same waves and fewer
// registers (641^2: 34.7 -> 37.6).
DepositPlan deposit_plan(int N, int coarseness, int fineness, int cus) {
    DepositPlan p{};
    p.tile = N <= 200 ? 8 : N <= 400 ? 16 : 24;
    p.nt = (N + p.tile - 1) / p.tile;
    p.waves = p.tile == 24 && p.nt * p.nt > 3 * cus ? 4 : 3;
    const int ext = p.tile + 2 * kDepositHalo + 2;   // initial cells per side, at most
    // the coarse rectangle of a tile has at most ext / coarseness + 3 rows;
    // staged while three blocks share a CU's LDS (not with 24 cells at coarseness 2,
    // 54.7 KB with tables for fineness 3)
    p.fine_max = std::max(fineness, 3) * ext;
    p.coarse_max = ext / coarseness + 3;
    p.staged = deposit_lds_bytes(p.tile, p.fine_max, p.coarse_max) <= 53 * 1024;
    // The tables also take grids denser than the config says (the caller makes them):
    // 18 coarse rows and 128 fine indices, or 15 and no more of these where four
    // blocks share the LDS (more took a block of each CU: 1281^2 995 -> 1052 us a
    // step).  A denser tile is a fault.
    if (p.staged) p.coarse_max = std::max(p.coarse_max, p.waves == 4 ? 15 : 18);
    if (!p.staged || p.waves == 3) p.fine_max = std::max(p.fine_max, 128);
    return p;
}

int launch_deposit(const DepositArgs& a, hipStream_t s, Profiler* prof) {
    LCODE_REQUIRE(a.ntx == (a.N + a.tile - 1) / a.tile, "deposition: tiles per side do not match N");
    LCODE_REQUIRE(a.nsplit >= 0 && a.nsplit <= a.ntx * a.ntx &&
                      (!a.nsplit || (a.tile_order && a.split_part && a.split_count)),
                  "deposition: inconsistent split tiles");
    LCODE_REQUIRE(!a.tile_order || dep_entries_fit(a.ntx * a.ntx, a.nsplit),
                  "deposition: more tiles than the block table holds");
    const DepKernel kernel = deposit_kernel_of(a.tile, a.waves, a.staged, a.grid32);
    LCODE_REQUIRE(kernel, "deposition: no kernel for this tile");
    {
        ProfScope ps(prof, "deposit_tile", s, true);
        launch_timed(ps, kernel, dim3(a.ntx * a.ntx + a.nsplit), dim3(kDepBlock),
                     deposit_lds_bytes(a.tile, a.fine_max, a.staged ? a.coarse_max : 0), s, a);
    }
    LCODE_HIP(hipGetLastError());
    if (!a.spill_in_tiles) {
        ProfScope ps(prof, "deposit_spill", s, true);
        if (a.grid32)
            launch_timed(ps, deposit_spill_kernel<float>, dim3(kSpillBlocks), dim3(kBlock), 0, s, a);
        else
            launch_timed(ps, deposit_spill_kernel<double>, dim3(kSpillBlocks), dim3(kBlock), 0, s, a);
    }
    LCODE_HIP(hipGetLastError());
    return LCODE_OK;
}

}  // namespace lcode
