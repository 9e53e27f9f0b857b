// sdm_kernels.h -- HIP kernels of the SDM step for gfx950 (wave64).
//
// One step of every replica r of a context (LangevinIntegratorSDM::step,
// openmmapi/src/LangevinIntegratorSDM.cpp:153-183) is the launch sequence
//
//   k_bin -> k_scan -> k_scatter -> k_cellsort -> k_blockorder          spatial sort
//   k_refresh -> k_tiles   slot records, boxes; tile lists
//                          and the j-blocks near the displaced atoms at x or at x+d
//   k_forces               F0: LJ+RF of every pair at x (FP32 math, fixed-point forces)
//                          U0 on the steps that report energies (FP64 pair sums)
//                          Ub, Fb: harmonic bonds/angles at x (FP64, gathered per atom)
//                          u and F1-F0 (FP64, pairs with d_i != d_j)
//   k_deltaA_red           the sums of u and F1-F0 on displaced atoms
//   k_scalar               SoftCoreF, bias W/W', PotEnergy, noneq schedule/work, sp
//   k_mix                  F += sp (F1 - F0)
//   k_langevin             leapfrog Langevin update, Philox noise (FP64)
//   k_constrain            SHAKE on constrained clusters (FP64)
//
// U1 and F1 are never computed as a second full sweep: pairs whose displacements are
// equal (d_i == d_j) have identical minimum-image distances at x and at x+d, so
// U(x+d) - U(x) and F(x+d) - F(x) are sums over the few pairs with d_i != d_j only.
// Every grid has the replica index in its y (or z) dimension.
#pragma once
#include <type_traits>

#include "sdm_device.h"

namespace sdm {

// Box and cutoff constants of every kernel.  A non-periodic system (CutoffNonPeriodic)
// has a box of 1e30 with zero inverse: every image shift L * round(d / L) is then 0 and
// coordinates are never wrapped.
struct Geom {
    float bx, by, bz, ibx, iby, ibz;  // box and inverse (FP32 path)
    double Lx, Ly, Lz, iLx, iLy, iLz; // FP64 path
    float rc2f, krff, crff;
    double rc2, krf, crf;
    // one periodic shift s for a whole tile (two blocks with centre difference dc and
    // half-extents h_i, h_j) is exact for every pair within the list radius r_l when
    // |dc - s| + h_i + h_j <= L - r_l in each dimension: a pair that s puts k != 0 box
    // lengths off its minimum image then lies at least L - (L - r_l) = r_l away in truth,
    // and at least L/2 >= r_c as evaluated, so it is left out either way.  oix..oiz hold
    // L - r_l less a 1e-3 nm margin for FP32 rounding (1e30 if not periodic)
    float oix, oiy, oiz;
    // LJ sigma combining: 0 Lorentz-Berthelot, 1 geometric (OPLS).  The per-atom FP32 and
    // FP64-record sigma entries hold s/2 for the first, s for the second (the FP64 sigma
    // array always s); the pair kernel takes it as a template parameter
    int geo;
    // sort grid: cell c_d = floor((w_d - go_d) * gs_d), clamped to the grid, w the
    // (wrapped, if periodic) coordinate.  Periodic: go = 0, gs = cells / L; otherwise
    // the grid spans a region around the positions (atoms outside take edge cells)
    double go[3], gs[3];
};

// Tile lists kept over several steps (a Verlet skin).  The lists are built with the
// radius r_l = r_c + skin + 1e-3 nm (r2), and with oix..oiy as Geom's but for that radius
// (a shift exact for every pair within r_l).  A pair within r_c now was within
// r_c + d_i + d_j when the lists were built (d: each atom's displacement since, as a
// minimum image), so the lists hold every pair within r_c while 2 max d <= skin:
// reuse_d2 = (skin / 2)^2 (negative: build on every call).
struct TileRadius {
    float r2, oix, oiy, oiz, reuse_d2;
};
// a block displacement record that forces the next build (after a sort, or non-finite)
constexpr float DISP_STALE = 3.0e38f;
// floats between consecutive replicas' displacement records (dmax[r * DISP_STRIDE]): one
// 256-byte line each, so that the blocks' atomics of different replicas do not queue on
// one line (all on one line cost 62 us per launch at 22 x 356 blocks)
constexpr int DISP_STRIDE = 64;

// Slot-ordered FP64 record of the energy kernel: the position in the same periodic image
// as the slot's FP32 record (so one tile shift serves both), and the parameters.
struct Rec64 {
    double x, y, z, qk, sh, es;  // position; q sqrt(k_e), sigma/2, 2 sqrt(eps)
};

__device__ __forceinline__ int grid_cell(double w, double go, double gs, int n) {
    return (int)fmin(fmax(floor((w - go) * gs), 0.0), (double)(n - 1));
}

// ---------------------------------------------------------------------------
// spatial sort (deterministic): cell rank per atom, counting sort, per-cell sort by
// atom index so the slot order does not depend on atomic ordering.
// ---------------------------------------------------------------------------
__global__ void k_bin(int N, int Np, const double* __restrict__ x64, int* __restrict__ key,
                      int* __restrict__ ccount, const int* __restrict__ cellrank, Geom g,
                      int ncx, int ncy, int ncz, int NC) {
    int r = blockIdx.y;
    int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= N) return;
    const double* X = x64 + (size_t)r * 3 * Np;
    double wx = X[i], wy = X[Np + i], wz = X[2 * Np + i];
    wx -= g.Lx * floor(wx * g.iLx);
    wy -= g.Ly * floor(wy * g.iLy);
    wz -= g.Lz * floor(wz * g.iLz);
    int cx = grid_cell(wx, g.go[0], g.gs[0], ncx);
    int cy = grid_cell(wy, g.go[1], g.gs[1], ncy);
    int cz = grid_cell(wz, g.go[2], g.gs[2], ncz);
    int k = cellrank[(cx * ncy + cy) * ncz + cz];
    key[(size_t)r * Np + i] = k;
    atomicAdd(&ccount[(size_t)r * NC + k], 1);
}

// inclusive sum over the lanes up to this one
__device__ __forceinline__ int wave_scan(int v) {
    v += __builtin_amdgcn_update_dpp(0, v, 0x111, 0xf, 0xf, true);  // row_shr:1, 2, 4, 8
    v += __builtin_amdgcn_update_dpp(0, v, 0x112, 0xf, 0xf, true);
    v += __builtin_amdgcn_update_dpp(0, v, 0x114, 0xf, 0xf, true);
    v += __builtin_amdgcn_update_dpp(0, v, 0x118, 0xf, 0xf, true);
    v += __builtin_amdgcn_update_dpp(0, v, 0x142, 0xa, 0xf, true);  // row_bcast:15
    v += __builtin_amdgcn_update_dpp(0, v, 0x143, 0xc, 0xf, true);  // row_bcast:31
    return v;
}

// exclusive scan of the cell counts, one 1024-thread workgroup per replica; clears the
// counters for the next step.  8 x 1024 cells at a time, coalesced and in flight together,
// with one barrier a round: the launch is one workgroup's latency, 19.6 us for 8,000 cells with a
// run of cells per thread and a barrier per doubling, 3.8 us so.
__global__ __launch_bounds__(1024) void k_scan(int NC, int* __restrict__ ccount,
                                               int* __restrict__ cstart, int* __restrict__ cfill) {
    __shared__ int sums[2][128];  // of chunk k and wave w: [16 k + w], alternating
    const int r = blockIdx.x, t = threadIdx.x, lane = t & 63;
    const int wv = __builtin_amdgcn_readfirstlane(t >> 6);
    int* cnt = ccount + (size_t)r * NC;
    int* st = cstart + (size_t)r * (NC + 1);
    int* fl = cfill + (size_t)r * NC;
    int before = 0;  // cells of the rounds before
    for (int base = 0, row = 0; base < NC; base += 8192, row ^= 1) {
        int v[8], end[8];
#pragma unroll
        for (int k = 0; k < 8; k++) {
            const int c = base + 1024 * k + t;
            v[k] = c < NC ? cnt[c] : 0;
        }
#pragma unroll
        for (int k = 0; k < 8; k++) {
            end[k] = wave_scan(v[k]);
            if (lane == 63) sums[row][16 * k + wv] = end[k];
        }
        __syncthreads();
        // every wave finds the sums in front of its parts
        const int a = sums[row][lane], b = sums[row][64 + lane];
        const int ea = wave_scan(a), ta = __builtin_amdgcn_readlane(ea, 63);
        const int eb = wave_scan(b) + ta;
#pragma unroll
        for (int k = 0; k < 8; k++) {
            const int q = 16 * k + wv, x = k < 4 ? ea - a : eb - b;
            const int c = base + 1024 * k + t;
            if (c < NC) {
                st[c] = before + __builtin_amdgcn_readlane(x, q & 63) + end[k] - v[k];
                cnt[c] = 0;
                fl[c] = 0;
            }
        }
        before += __builtin_amdgcn_readlane(eb, 63);
    }
    if (t == 0) st[NC] = before;
}

__global__ void k_scatter(int N, int Np, int NC, const int* __restrict__ key,
                          const int* __restrict__ cstart, int* __restrict__ cfill,
                          int* __restrict__ orig_s) {
    int r = blockIdx.y;
    int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= N) return;
    int k = key[(size_t)r * Np + i];
    int s = cstart[(size_t)r * (NC + 1) + k] + atomicAdd(&cfill[(size_t)r * NC + k], 1);
    if (s >= 0 && s < N) orig_s[(size_t)r * Np + s] = i;  // always, with consistent counts
}

// per cell: order its slots by atom index
__global__ void k_cellsort(int N, int Np, int NC, const int* __restrict__ cstart,
                           int* __restrict__ orig_s) {
    int r = blockIdx.y;
    int c = blockIdx.x * blockDim.x + threadIdx.x;
    if (c >= NC) return;
    const int* st = cstart + (size_t)r * (NC + 1);
    int beg = max(st[c], 0), end = min(st[c + 1], N);
    int* o = orig_s + (size_t)r * Np;
    for (int a = beg + 1; a < end; a++) {
        int v = o[a];
        int b = a - 1;
        while (b >= beg && o[b] > v) {
            o[b + 1] = o[b];
            b--;
        }
        o[b + 1] = v;
    }
}

// Orders the 64 slots of a block so that its clusters of 8 are compact: the block is split
// at the median of its longest axis into halves of 32, these into 16 and these into 8 (one
// wave per block, bitonic sorts of the axis' coordinate, ties by atom index, so that the
// order is unique).  Writes the final orig_s and slot_of, and the atom that the periodic
// images of the block's atoms are taken about until the next sort (bfirst, the first along
// the curve).  In a disordered 22,750-atom box
// (cells of 0.305 nm) it leaves 8% fewer pairs of clusters within the list radius and 5%
// fewer with a pair within the cutoff than the order along the curve.
__global__ __launch_bounds__(64) void k_blockorder(int N, int Np, const double* __restrict__ x64,
                                                   int* __restrict__ orig_s,
                                                   int* __restrict__ slot_of,
                                                   int* __restrict__ bfirst, Geom g) {
    const int r = blockIdx.y, b = blockIdx.x, lane = threadIdx.x;
    const int sl = b * 64 + lane;
    int* O = orig_s + (size_t)r * Np;
    const double* X = x64 + (size_t)r * 3 * Np;
    const bool v = sl < N;
    int idx = v ? O[sl] : 0x7FFFFFFF;
    if (lane == 0) bfirst[(size_t)r * gridDim.x + b] = idx;  // slot b * 64 is always below N
    float p[3] = {0.f, 0.f, 0.f};
    const double* L = &g.Lx;
    const double* iL = &g.iLx;
#pragma unroll
    for (int d = 0; d < 3; d++) {  // relative to the block's first atom, in its image
        const double w = X[(size_t)d * Np + (v ? idx : O[b * 64])];
        const double dw = w - __shfl(w, 0, 64);
        p[d] = (float)(dw - L[d] * rint(dw * iL[d]));
        // The lanes of a comparison decide apart, so keys have to be in a total order, and
        // below the key of the empty slots: NaN, infinities and what is beyond FP32 (a replica
        // that has blown up) count as one far coordinate, ordered by the atoms' indices.
        if (!(fabsf(p[d]) <= 1.0e30f)) p[d] = 1.0e30f;
    }
#pragma unroll
    for (int n = 64; n >= 16; n >>= 1) {
        float ext[3];
#pragma unroll
        for (int d = 0; d < 3; d++) {
            float lo = idx != 0x7FFFFFFF ? p[d] : 3.0e38f, hi = idx != 0x7FFFFFFF ? p[d] : -3.0e38f;
            for (int o = n / 2; o > 0; o >>= 1) {
                lo = fminf(lo, __shfl_xor(lo, o, 64));
                hi = fmaxf(hi, __shfl_xor(hi, o, 64));
            }
            ext[d] = hi - lo;
        }
        const int ax = ext[0] >= ext[1] && ext[0] >= ext[2] ? 0 : ext[1] >= ext[2] ? 1 : 2;
        for (int k = 2; k <= n; k <<= 1)
            for (int j = k >> 1; j > 0; j >>= 1) {
                const float key = idx == 0x7FFFFFFF ? 3.0e38f : ax == 0 ? p[0] : ax == 1 ? p[1] : p[2];
                const float ok = __shfl_xor(key, j, 64);
                const int oi = __shfl_xor(idx, j, 64);
                const bool less = ok < key || (ok == key && oi < idx);  // the partner's is smaller
                const bool up = ((lane & (n - 1)) & k) == 0, first = (lane & j) == 0;
                // (up, first) and (!up, !first) lanes keep the smaller of the two
                const bool take = (up == first) ? less : !less;
#pragma unroll
                for (int d = 0; d < 3; d++) {
                    const float op = __shfl_xor(p[d], j, 64);
                    p[d] = take ? op : p[d];
                }
                idx = take ? oi : idx;
            }
    }
    if (v) {  // the empty slots of the last block stay last
        O[sl] = idx;
        slot_of[(size_t)r * Np + idx] = sl;
    }
}

// min / max over the 8 lanes of each group of 8 (lane ^ 7, lane ^ 2, lane ^ 1 via DPP)
__device__ __forceinline__ float min8(float v) {
    v = fminf(v, __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(v), 0x141, 0xf, 0xf, true)));
    v = fminf(v, __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(v), 0x4E, 0xf, 0xf, true)));
    return fminf(v, __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(v), 0xB1, 0xf, 0xf, true)));
}
__device__ __forceinline__ float max8(float v) {
    v = fmaxf(v, __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(v), 0x141, 0xf, 0xf, true)));
    v = fmaxf(v, __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(v), 0x4E, 0xf, 0xf, true)));
    return fmaxf(v, __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(v), 0xB1, 0xf, 0xf, true)));
}

// Boxes of one 64-slot block (one wave, lane = slot, v: the slot holds an atom at p): the
// block's corners, and per cluster of 8 slots its centre (cbox[0..7]) and half extents
// (cbox[8..15]; -1e30 for a cluster without atoms, whose gap to any box is then never in
// range).
__device__ __forceinline__ void block_boxes(float4 p, bool v, int lane, float4* __restrict__ lo,
                                            float4* __restrict__ hi, float4* __restrict__ cbox) {
    float lx = min8(v ? p.x : 3.0e38f), ly = min8(v ? p.y : 3.0e38f), lz = min8(v ? p.z : 3.0e38f);
    float hx = max8(v ? p.x : -3.0e38f), hy = max8(v ? p.y : -3.0e38f), hz = max8(v ? p.z : -3.0e38f);
    if ((lane & 7) == 0) {
        const bool any = lx <= hx;
        cbox[lane >> 3] = any ? make_float4(0.5f * (lx + hx), 0.5f * (ly + hy), 0.5f * (lz + hz), 0.f)
                              : make_float4(0.f, 0.f, 0.f, 0.f);
        cbox[8 + (lane >> 3)] = any ? make_float4(0.5f * (hx - lx), 0.5f * (hy - ly), 0.5f * (hz - lz), 0.f)
                                    : make_float4(-1.0e30f, -1.0e30f, -1.0e30f, 0.f);
    }
#pragma unroll
    for (int o = 32; o >= 8; o >>= 1) {
        lx = fminf(lx, __shfl_xor(lx, o, 64));
        ly = fminf(ly, __shfl_xor(ly, o, 64));
        lz = fminf(lz, __shfl_xor(lz, o, 64));
        hx = fmaxf(hx, __shfl_xor(hx, o, 64));
        hy = fmaxf(hy, __shfl_xor(hy, o, 64));
        hz = fmaxf(hz, __shfl_xor(hz, o, 64));
    }
    if (lane == 0) {
        *lo = make_float4(lx, ly, lz, 0.f);
        *hi = make_float4(hx, hy, hz, 0.f);
    }
}

// The slot records of one evaluation.  One wave per 64-slot block gathers its atoms'
// coordinates from the FP64 positions, wrapped into the box after a sort and then taken in
// the periodic image nearest the block's atom bfirst, so a block stays compact when one of
// its atoms crosses a face of the box; then the boxes of the block and its clusters are
// computed and the slot-ordered force accumulator cleared.  Culling and pair distances take
// minimum images of box centres or of pairs, so they hold for any image.
//   SORT = true (after a sort; the slot order is new): also the records' parameters; the
// replica's displacement record (dmax, read by k_tiles) is set to a value that makes the
// next tile-list build unconditional; and the exclusions are written in slot order:
// exs[block][k][lane], the slot of the k-th partner of the block's atom `lane` (-1: none),
// and exblocks[block], a 64-bit set that has bit b & 63 for every j-block b that holds a
// partner (mostly the block and its neighbours, now and then one far along the curve).  The
// pair and energy kernels then read them with one coalesced load instead of a chain of four
// (atom, list start, list entry, slot), and only for the tiles that need them.
//   SORT = false: the order of the last sort is kept; the displacement record of kept lists
// is updated (xb, dmax).
//   refresh_block: one wave, lane = slot of block b (v: below N), which holds atom i at
// (wx, wy, wz), the block's atom bfirst being at (rx, ry, rz).
template <bool SORT>
__device__ __forceinline__ void refresh_block(
    int r, int b, int lane, int i, bool v, double wx, double wy, double wz, double rx, double ry,
    double rz, int N, int Np, int NB, const float* __restrict__ qs,
    const float* __restrict__ sh, const float* __restrict__ se, const Geom& g,
    float4* __restrict__ arec, long long* __restrict__ F, float4* __restrict__ bb_lo,
    float4* __restrict__ bb_hi, float4* __restrict__ cbox, const double4* __restrict__ par64,
    Rec64* __restrict__ rec, const float4* __restrict__ xb, float* __restrict__ dmax,
    const int* __restrict__ slot_of, const int* __restrict__ ex_start,
    const int* __restrict__ ex_list, int max_ex, int* __restrict__ exs,
    unsigned long long* __restrict__ exblocks) {
    const int sl = b * 64 + lane;
    if (SORT) {
        wx -= g.Lx * floor(wx * g.iLx);
        wy -= g.Ly * floor(wy * g.iLy);
        wz -= g.Lz * floor(wz * g.iLz);
    } else {
        rx -= g.Lx * floor(rx * g.iLx);
        ry -= g.Ly * floor(ry * g.iLy);
        rz -= g.Lz * floor(rz * g.iLz);
        wx -= g.Lx * rint((wx - rx) * g.iLx);
        wy -= g.Ly * rint((wy - ry) * g.iLy);
        wz -= g.Lz * rint((wz - rz) * g.iLz);
    }
    const float4 p = make_float4((float)wx, (float)wy, (float)wz, qs[i]);
    size_t o = (size_t)r * Np + sl;
    const size_t bo = (size_t)r * NB + b;
    if (v) {
        arec[2 * o] = p;
        if (SORT) arec[2 * o + 1] = make_float4(sh[i], se[i], 0.f, 0.f);
        if (rec) {  // energy evaluations: the FP64 record in the same image
            double4 pr = par64[i];
            rec[o] = Rec64{wx, wy, wz, pr.x, pr.y, pr.z};
        }
        long long* Fr = F + (size_t)r * 3 * Np;
        Fr[sl] = 0;
        Fr[Np + sl] = 0;
        Fr[2 * Np + sl] = 0;
    }
    block_boxes(p, v, lane, bb_lo + bo, bb_hi + bo, cbox + 16 * bo);
    if (SORT) {
        if (lane == 0 && b == 0) dmax[(size_t)r * DISP_STRIDE] = DISP_STALE;
        unsigned long long set = 0ull;
        int nex = 0, b0 = 0;
        if (v) {
            b0 = ex_start[i];
            nex = ex_start[i + 1] - b0;
        }
        int* E = exs + bo * max_ex * 64;
        for (int k = 0; k < max_ex; k++) {
            const int es = k < nex ? slot_of[(size_t)r * Np + ex_list[b0 + k]] : -1;
            E[k * 64 + lane] = es;
            if (es >= 0) set |= 1ull << ((es >> 6) & 63);
        }
#pragma unroll
        for (int q = 32; q > 0; q >>= 1) set |= __shfl_xor(set, q, 64);
        if (lane == 0) exblocks[bo] = set;
        return;
    }
    // kept tile lists (xb: the slot coordinates when they were built): the block's
    // largest squared displacement since, as a minimum image (the block may have moved
    // to another image of the box; non-finite counts as stale), into the replica's
    // maximum by a device-scope atomic max (non-negative floats order as their bits).
    // k_scalar sets it back to 0 at the end of each evaluation; where no k_scalar runs in
    // between (pair timing, pair counts) it can only be larger, so lists are rebuilt
    // sooner, never later.  (A last-block reduction needs a device-scope fence per block,
    // which writes back the XCD's L2: +0.2 ms per step at 22 x 22,750 atoms.)  One atomic
    // per block: 356 per replica at 22,750 atoms.
    if (xb) {
        float d2 = 0.f;
        if (v) {
            const float4 q = xb[o];
            float dx = p.x - q.x, dy = p.y - q.y, dz = p.z - q.z;
            dx -= g.bx * rintf(dx * g.ibx);
            dy -= g.by * rintf(dy * g.iby);
            dz -= g.bz * rintf(dz * g.ibz);
            d2 = dx * dx + dy * dy + dz * dz;
            if (!(d2 <= 1.0e30f)) d2 = DISP_STALE;
        }
        d2 = wave_max(d2);
        if (lane == 0)
            atomicMax(reinterpret_cast<unsigned*>(dmax) + (size_t)r * DISP_STRIDE,
                      __float_as_uint(d2));
    }
}

template <bool SORT>
__global__ __launch_bounds__(64) void k_refresh(
    int N, int Np, int NB, const double* __restrict__ x64, const int* __restrict__ orig_s,
    const float* __restrict__ qs, const float* __restrict__ sh, const float* __restrict__ se,
    Geom g, float4* __restrict__ arec, long long* __restrict__ F,
    float4* __restrict__ bb_lo, float4* __restrict__ bb_hi, float4* __restrict__ cbox,
    const double4* __restrict__ par64, Rec64* __restrict__ rec, const float4* __restrict__ xb,
    float* __restrict__ dmax, const int* __restrict__ slot_of, const int* __restrict__ bfirst,
    const int* __restrict__ ex_start, const int* __restrict__ ex_list, int max_ex,
    int* __restrict__ exs, unsigned long long* __restrict__ exblocks) {
    const int r = blockIdx.y, b = blockIdx.x, lane = threadIdx.x, sl = b * 64 + lane;
    const bool v = sl < N;  // slot b * 64 (lane 0) is always below N
    const double* X = x64 + (size_t)r * 3 * Np;
    const int i = orig_s[(size_t)r * Np + (v ? sl : b * 64)];
    const int f = SORT ? i : bfirst[(size_t)r * NB + b];
    refresh_block<SORT>(r, b, lane, i, v, X[i], X[Np + i], X[2 * Np + i], X[f], X[Np + f],
                        X[2 * Np + f], N, Np, NB, qs, sh, se, g, arec, F, bb_lo, bb_hi, cbox,
                        par64, rec, xb, dmax, slot_of, ex_start, ex_list, max_ex, exs, exblocks);
}

__device__ __forceinline__ float bbox_gap2(float4 lo_i, float4 hi_i, float4 lo_j, float4 hi_j,
                                           const Geom& g) {
    float cx = 0.5f * (lo_i.x + hi_i.x) - 0.5f * (lo_j.x + hi_j.x);
    float cy = 0.5f * (lo_i.y + hi_i.y) - 0.5f * (lo_j.y + hi_j.y);
    float cz = 0.5f * (lo_i.z + hi_i.z) - 0.5f * (lo_j.z + hi_j.z);
    cx -= g.bx * rintf(cx * g.ibx);
    cy -= g.by * rintf(cy * g.iby);
    cz -= g.bz * rintf(cz * g.ibz);
    float gx = fmaxf(fabsf(cx) - 0.5f * (hi_i.x - lo_i.x) - 0.5f * (hi_j.x - lo_j.x), 0.f);
    float gy = fmaxf(fabsf(cy) - 0.5f * (hi_i.y - lo_i.y) - 0.5f * (hi_j.y - lo_j.y), 0.f);
    float gz = fmaxf(fabsf(cz) - 0.5f * (hi_i.z - lo_i.z) - 0.5f * (hi_j.z - lo_j.z), 0.f);
    return gx * gx + gy * gy + gz * gz;
}

__device__ __forceinline__ int lane_rank(unsigned long long m) {
    return __builtin_amdgcn_mbcnt_hi((unsigned)(m >> 32), __builtin_amdgcn_mbcnt_lo((unsigned)m, 0u));
}

// Which of two blocks lists their tile.  Taking j >= i would give the first blocks of the
// slot order all of their neighbours and the last ones none; by the parity of i + j every
// block lists about half of its neighbours, so that i-blocks (and with them the XCDs, which
// work on consecutive blocks) have equal work.
__device__ __forceinline__ bool lists_tile(int ib, int jb) {
    return jb == ib || (jb > ib) == (((ib ^ jb) & 1) != 0);
}

// candidate j-blocks: within rc of a displaced class's box at x or at x+d_k.  One
// workgroup of NW waves per replica (they share the class boxes' reductions and the scan
// over the blocks, so the replica's serial chain is short); candidates are written in
// ascending block order.
template <int NW>
__device__ __forceinline__ void lig_candidates(
    int r, int Np, int NB, int L, int ncls, const int* __restrict__ lig, const int* __restrict__ cls,
    const double* __restrict__ cdispl, const double* __restrict__ x64,
    const float4* __restrict__ bb_lo, const float4* __restrict__ bb_hi, int maxc,
    int* __restrict__ cand, int* __restrict__ ncand, float list_r2, const Geom& g,
    int* __restrict__ flags, int* __restrict__ cmap) {
    __shared__ float4 blo[2 * SDM_MAX_CLASSES], bhi[2 * SDM_MAX_CLASSES];
    __shared__ double red[6][NW];
    __shared__ int wcount[NW];
    const int t = threadIdx.x, lane = t & 63, wv = t >> 6;
    const double* X = x64 + (size_t)r * 3 * Np;
    for (int k = 1; k <= ncls; k++) {
        double v[6] = {1e300, 1e300, 1e300, -1e300, -1e300, -1e300};
        for (int li = t; li < L; li += 64 * NW) {
            int a = lig[li];
            if (cls[a] != k) continue;
            for (int d = 0; d < 3; d++) {
                double x = X[d * Np + a];
                v[d] = fmin(v[d], x);
                v[3 + d] = fmax(v[3 + d], x);
            }
        }
        for (int d = 0; d < 3; d++) {
            v[d] = wave_min_d(v[d]);
            v[3 + d] = wave_max_d(v[3 + d]);
        }
        if (lane == 0)
            for (int q = 0; q < 6; q++) red[q][wv] = v[q];
        __syncthreads();
        if (t == 0) {
            for (int w = 1; w < NW; w++)
                for (int d = 0; d < 3; d++) {
                    v[d] = fmin(v[d], red[d][w]);
                    v[3 + d] = fmax(v[3 + d], red[3 + d][w]);
                }
            const double* dk = cdispl + 3 * k;
            blo[2 * (k - 1)] = make_float4((float)v[0], (float)v[1], (float)v[2], 0.f);
            bhi[2 * (k - 1)] = make_float4((float)v[3], (float)v[4], (float)v[5], 0.f);
            blo[2 * (k - 1) + 1] = make_float4((float)(v[0] + dk[0]), (float)(v[1] + dk[1]),
                                               (float)(v[2] + dk[2]), 0.f);
            bhi[2 * (k - 1) + 1] = make_float4((float)(v[3] + dk[0]), (float)(v[4] + dk[1]),
                                               (float)(v[5] + dk[2]), 0.f);
        }
        __syncthreads();  // red is reused by the next class
    }
    const float4* lo = bb_lo + (size_t)r * NB;
    const float4* hi = bb_hi + (size_t)r * NB;
    int* out = cand + (size_t)r * maxc;
    int count = 0;  // candidates before this round (uniform)
    for (int base = 0; base < NB; base += 64 * NW) {
        int jb = base + t;
        bool ok = false;
        if (jb < NB) {
            float4 lj = lo[jb], hj = hi[jb];
            for (int k = 0; k < 2 * ncls; k++) ok = ok || (bbox_gap2(blo[k], bhi[k], lj, hj, g) < list_r2);
        }
        unsigned long long m = __ballot(ok);
        if (lane == 0) wcount[wv] = __popcll(m);
        __syncthreads();
        int before = count;
        for (int w = 0; w < wv; w++) before += wcount[w];
        int pos = before + lane_rank(m);
        if (ok && pos < maxc) out[pos] = jb;
        // block -> candidate index (-1: none), for the Langevin kernel's gather of the
        // displaced-state forces
        if (cmap && jb < NB) cmap[(size_t)r * NB + jb] = (ok && pos < maxc) ? pos : -1;
        for (int w = 0; w < NW; w++) count += wcount[w];
        __syncthreads();  // wcount is rewritten next round
    }
    if (t == 0) {
        ncand[r] = min(count, maxc);
        if (count > maxc) atomicOr(&flags[r], 4);
    }
}

// How the tiles of an i-block are shared out: in parts of the steps (bits of the masks) of
// its tile list, in list order, a tile counting TILE_UNITS steps more for its records, shift
// and j forces.  A tile may be cut between two parts, but not within an eighth of a part (at
// most 16 steps) of its ends.  The tile kernel finds the bounds, once for all waves of the
// block: bounds[p] = (tile, steps of it that belong to the parts before p).
// Parts are equal where one replica's waves are all resident at once (its longest wave is
// what the launch waits for), and become smaller, to a tenth of the mean, from
// TILE_SLOPE_BLOCKS blocks on, where waves start as others end: equal waves run in
// generations, in step, and the last one leaves the GPU partly idle.
// Tiles hold 1 to 64 steps: dealt out whole, every 8th tile to one of 8 waves, the longest
// wave of 22,750 atoms took 50 us and the median one 25.  Measured, the pair kernel alone
// (us): 186 atoms 9.9 -> 8.6, 2,976 atoms 28 -> 20 and 20 replicas of them 70 -> 60, 8 x
// 99,920 atoms 855 -> 790 (877 with equal parts), 22 x 22,750 atoms 403 -> 392.
constexpr int TILE_UNITS = 6, TILE_SLOPE_BLOCKS = 512;
constexpr int MAX_TILE_PARTS = 64, TILE_BOUNDS = MAX_TILE_PARTS + 1;

// one wave: the bounds of `parts` (at most 64) parts of a list of nt tiles with masks tmk,
// whose numbers of steps are in nstep for the first SHARE_LDS ones.  Lanes are tiles for the
// sums in front of them and then parts, which look for their tile.
constexpr int SHARE_LDS = 256;
__device__ __forceinline__ void share_tiles(const unsigned char* nstep,
                                            const unsigned long long* tmk, int nt, int lane,
                                            int parts, bool slope,
                                            int2* __restrict__ bounds) {
    auto steps = [&](int t) {
        return t >= nt ? 0 : t < SHARE_LDS ? (int)nstep[t] : __popcll(tmk[t]);
    };
    auto units = [](int n) { return n ? n + TILE_UNITS : 0; };
    int n = steps(lane), end = wave_scan(units(n));
    int total = __builtin_amdgcn_readlane(end, 63);
    for (int t = 64; t < nt; t += 64)
        total += __builtin_amdgcn_readlane(wave_scan(units(steps(t + lane))), 63);
    const int snap = min(16, total / parts / 8);
    const double f = (double)lane / parts;
    const int at = (int)(total * (slope ? f * (1.9 - 0.9 * f) : f));
    int2 bound = make_int2(0, 0);
    for (int t = 0, before = 0; t < nt; t += 64) {
        if (t > 0) {
            n = steps(t + lane);
            end = before + wave_scan(units(n));
        }
        int q = 0;  // tiles of these that end at or before `at`
#pragma unroll
        for (int h = 32; h > 0; h >>= 1) q += __shfl(end, q + h - 1, 64) <= at ? h : 0;
        const int qn = __shfl(n, q, 64), qe = __shfl(end, q, 64);
        if (at >= before && q < 64 && at < qe) {
            int a = max(at - (qe - qn), 0);
            if (min(a, qn - a) <= snap) a = a <= qn - a ? 0 : qn;
            bound = a < qn ? make_int2(t + q, a) : make_int2(t + q + 1, 0);
        }
        before = __builtin_amdgcn_readlane(end, 63);
    }
    if (lane < parts) bounds[lane] = bound;
    if (lane == 0) bounds[parts] = make_int2(nt, 0);
}

// the periodic shift of a whole tile (boxes of the two blocks): (kx, ky, kz) box lengths;
// returns whether it is exact for every pair within the list radius (Geom::oix)
__device__ __forceinline__ bool tile_shift(float4 bli, float4 bhi, float4 blj, float4 bhj,
                                           const Geom& g, float& kx, float& ky, float& kz) {
    float dcx = 0.5f * (bli.x + bhi.x - blj.x - bhj.x);
    float dcy = 0.5f * (bli.y + bhi.y - blj.y - bhj.y);
    float dcz = 0.5f * (bli.z + bhi.z - blj.z - bhj.z);
    kx = rintf(dcx * g.ibx);
    ky = rintf(dcy * g.iby);
    kz = rintf(dcz * g.ibz);
    return fabsf(dcx - g.bx * kx) + 0.5f * (bhi.x - bli.x + bhj.x - blj.x) < g.oix &&
           fabsf(dcy - g.by * ky) + 0.5f * (bhi.y - bli.y + bhj.y - blj.y) < g.oiy &&
           fabsf(dcz - g.bz * kz) + 0.5f * (bhi.z - bli.z + bhj.z - blj.z) < g.oiz;
}

// An entry of a tile list: the j-block and, where the lists are built for this evaluation
// (not kept from an earlier one, after which blocks may have moved to another image), the
// shift of tile_shift: box lengths by dimension, or that each pair takes its own image.
constexpr int TILE_BLOCK = (1 << 21) - 1, TILE_MI = 1 << 30;
__device__ __forceinline__ int pack_tile(int jb, bool one, float kx, float ky, float kz) {
    return jb | (one ? ((int)kx + 4) << 21 | ((int)ky + 4) << 24 | ((int)kz + 4) << 27 : TILE_MI);
}
__device__ __forceinline__ float tile_images(int entry, int d) {
    return entry & TILE_MI ? 0.f : (float)(((entry >> (21 + 3 * d)) & 7) - 4);
}

// tile list of one i-block: every j-block it lists (lists_tile) whose box is within the
// list radius r_l (r_c + skin + slack, TileRadius) of the i-block's box, ascending, each
// with a 64-bit mask of the pairs of 8-slot clusters whose boxes lie within r_l: bit
// 8 jc + ic for cluster jc of the j-block and ic of the i-block.  In the diagonal tile
// only jc >= ic.  A wave tests the 64 cluster pairs of a candidate at once (lane = bit),
// about 30 VALU instructions per candidate; the ballot is the mask.
// NW waves per i-block: in each round wave w takes 64 j-blocks (their box tests on its
// lanes, then the masks of those in range) and the waves' lists are put one after the other.
// Results do not depend on NW.
// Kept lists (tr.reuse_d2 >= 0): the workgroup returns at once while no atom of the
// replica has moved more than half the skin since the build (dmax); a build stores the
// block's slot coordinates in xb.  Last, the list is shared out among the waves of the pairs
// (waves, bounds) and, if they are not as many, of the pair energies (ewaves, ebounds).
// The first workgroup of a replica with displaced atoms finds the candidate blocks
// (LigCand::groups is 1) instead: both need the boxes only, and a launch of its own would
// take as long as this one.
struct LigCand {
    int groups, L, ncls, maxc;
    float r2;
    const int *lig, *cls;
    const double *cdispl, *x64;
    int *cand, *ncand, *cmap;
};
template <int NW>  // waves per i-block workgroup
__global__ __launch_bounds__(64 * NW) __attribute__((amdgpu_num_vgpr(64))) void k_tiles(int N, int Np, int NB, int maxj,
                                               const float4* __restrict__ arec,
                                               const float4* __restrict__ bb_lo,
                                               const float4* __restrict__ bb_hi,
                                               const float4* __restrict__ cbox,
                                               int* __restrict__ tiles,
                                               unsigned long long* __restrict__ tmask,
                                               const float* __restrict__ dmax,
                                               float4* __restrict__ xb, TileRadius tr, Geom g,
                                               int* __restrict__ flags, LigCand lc,
                                               int packed, int waves, int ewaves,
                                               int2* __restrict__ bounds,
                                               int2* __restrict__ ebounds) {
    __shared__ int nkept[2][NW];
    __shared__ unsigned char nstep[SHARE_LDS];
    const int r = blockIdx.y, ib = (int)blockIdx.x - lc.groups;
    if (ib < 0) {
        lig_candidates<NW>(r, Np, NB, lc.L, lc.ncls, lc.lig, lc.cls, lc.cdispl, lc.x64, bb_lo,
                           bb_hi, lc.maxc, lc.cand, lc.ncand, lc.r2, g, flags, lc.cmap);
        return;
    }
    const int lane = threadIdx.x & 63;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const float list_r2 = tr.r2;
    // kept lists: every workgroup of the replica reads the same record (written by the
    // slot refresh or the sort before this launch), so all of them keep or all rebuild
    if (tr.reuse_d2 >= 0.f && dmax[(size_t)r * DISP_STRIDE] <= tr.reuse_d2) return;
    const float4* lo = bb_lo + (size_t)r * NB;
    const float4* hi = bb_hi + (size_t)r * NB;
    const float4* CB = cbox + (size_t)r * NB * 16;
    const float4 li = lo[ib], hi_i = hi[ib];
    if (wave == 0 && tr.reuse_d2 >= 0.f) {  // the build coordinates
        int is = ib * 64 + lane;
        if (is < N) xb[(size_t)r * Np + is] = arec[2 * ((size_t)r * Np + is)];
    }
    // this lane's pair of clusters: ic of the i-block, jc of the candidate
    const int ic = lane & 7, jc = lane >> 3;
    const float4 ci = CB[16 * ib + ic], hc = CB[16 * ib + 8 + ic];
    auto mask_of = [&](int jb, float4 cj, float4 hj) {
        // the smallest gap over all images is the one at the centres' minimum image
        float dx = ci.x - cj.x, dy = ci.y - cj.y, dz = ci.z - cj.z;
        dx -= g.bx * rintf(dx * g.ibx);
        dy -= g.by * rintf(dy * g.iby);
        dz -= g.bz * rintf(dz * g.ibz);
        // a cluster without atoms has half extents of -1e30: its gap is never in range
        const float gx = fmaxf(fabsf(dx) - (hc.x + hj.x), 0.f),
                    gy = fmaxf(fabsf(dy) - (hc.y + hj.y), 0.f),
                    gz = fmaxf(fabsf(dz) - (hc.z + hj.z), 0.f);
        return __ballot(gx * gx + gy * gy + gz * gz < list_r2 && (jb != ib || jc >= ic));
    };
    int* out = tiles + ((size_t)r * NB + ib) * maxj;
    unsigned long long* mout = tmask + ((size_t)r * NB + ib) * maxj;
    int count = 0;  // tiles of the rounds before (uniform)
    for (int base = 0, round = 0; base < NB; base += 64 * NW, round ^= 1) {
        const int jl = base + 64 * wave + lane;  // this lane's j-block
        bool ok = false;
        if (jl < NB && lists_tile(ib, jl)) ok = bbox_gap2(li, hi_i, lo[jl], hi[jl], g) < list_r2;
        unsigned long long near = __ballot(ok), am = 0ull;
        // the masks of the candidates, each kept by its lane; four at a time, so that their
        // box loads are in flight together
        while (near) {
            int q[4];
            float4 cj[4], hj[4];
#pragma unroll
            for (int k = 0; k < 4; k++) {
                q[k] = near ? __builtin_ctzll(near) : (k ? q[k - 1] : 0);
                near &= near - 1ull;
                const float4* C = CB + 16 * (base + 64 * wave + q[k]) + jc;
                cj[k] = C[0];
                hj[k] = C[8];
            }
#pragma unroll
            for (int k = 0; k < 4; k++) {
                const unsigned long long b = mask_of(base + 64 * wave + q[k], cj[k], hj[k]);
                if (lane == q[k]) am = b;
            }
        }
        const unsigned long long keep = __ballot(am != 0ull);
        if (lane == 0) nkept[round][wave] = __popcll(keep);
        __syncthreads();  // one barrier a round: the counts alternate between two rows
        int pos = count + lane_rank(keep);
#pragma unroll
        for (int w = 0; w < NW; w++) {
            const int n = nkept[round][w];
            if (w < wave) pos += n;
            count += n;
        }
        if (am != 0ull && pos < maxj) {
            int entry = jl;
            if (packed) {
                const int lower = min(ib, jl), upper = max(ib, jl);
                float kx, ky, kz;
                const bool one = tile_shift(lo[lower], hi[lower], lo[upper], hi[upper], g, kx, ky, kz);
                entry = pack_tile(jl, one, kx, ky, kz);
            }
            out[pos] = entry;
            mout[pos] = am;
            if (pos < SHARE_LDS) nstep[pos] = (unsigned char)__popcll(am);
        }
    }
    if (threadIdx.x == 0 && count > maxj) atomicOr(&flags[r], 4);
    __syncthreads();  // the list is complete
    const size_t rb = (size_t)r * NB + ib;
    if (wave == 0) share_tiles(nstep, mout, min(count, maxj), lane, waves, NB >= TILE_SLOPE_BLOCKS, bounds + rb * TILE_BOUNDS);
    if (wave == NW - 1 && ewaves != waves)
        share_tiles(nstep, mout, min(count, maxj), lane, ewaves, NB >= TILE_SLOPE_BLOCKS, ebounds + rb * TILE_BOUNDS);
}

// ---------------------------------------------------------------------------
// The pair kernel: F0 over all pairs at x, each pair once (Newton-3 over the tile lists).
// Each i-block has one wave or several (TilePart).  A wave holds the 64 i atoms as eight
// clusters of 8: lane 8 jl + il keeps atom il of every cluster in registers, and takes one
// cluster of 8 j atoms at a time, lane 8 jl + il holding j atom jl.  One step is a pair of
// clusters, 64 pairs on 64 lanes, taken for the bits of the tile's mask (uniform branches).
// A step none of whose pairs is within the cutoff ends after the distance test.
//   i forces: FP32 in the lane (24 registers), added up over the eight lanes that share an
//     i atom and over to the int64 accumulator, rounded to nearest, at the end of each part
//     and by PAIRS_PER_FLUSH and TILES_PER_FLUSH.
//   j forces: FP32 over the cluster's steps, added up over the eight lanes that share a j
//     atom, kept in registers over the tile and added to the slot-ordered int64 accumulator
//     once per tile with coalesced atomics.
// The periodic image is one shift per tile when that is exact for every pair within the
// list radius (Geom::oix), otherwise the minimum image of each pair.  The shift is taken off
// the lower block's atoms, the i atoms (read from LDS again when it changes) or the j atoms,
// because a separation in FP32 (2e-7 nm) decides what is within the cutoff, where the
// reaction-field force ends with a step: coordinates relative to the block, with the shift in
// the j atoms' offset, took 5% less time but rounded otherwise than the box's coordinates.
// Fixed-point atomics commute, so results are bit-reproducible.
//
// What bounds it: VALU issue (93% of the cycles of 22 x 22,750 atoms, 4 waves per SIMD at
// 123 registers).  A step takes 7 instructions to the distance test and 21 after it.  One
// lane per i atom against one j atom at a time, the form before, took 37 instructions per 64
// pairs with 22% of them within the cutoff; pairs of clusters have 30% (40% after the
// distance test's early end) and no sum over the wave for each j atom.  Measured alone, 22
// x 22,750 atoms: 532 -> 405 us (297M -> 201M VALU instructions); 8 x 99,920 atoms:
// 1,054 -> 850 us; one replica of 22,750 atoms: 55 -> 44 us (before the tiles were shared out
// in parts, share_tiles; 22 x 22,750 atoms now 351 us, 195M
// instructions).  Where the i atoms' charges and
// LJ parameters came from LDS instead (122 registers), or the j forces of four clusters were
// summed together (as many instructions in all, 30% more code), it was 4% and 14% slower.
// ---------------------------------------------------------------------------

// a + b taken from the DPP partner lane.  bound_ctrl lets the mov fold into the add as
// its DPP operand; contraction is off so the add is not fused with the product that
// made a (gfx9 has no DPP form of v_fma).
template <int CTRL>
__device__ __forceinline__ float dpp_add(float a, float b) {
#pragma clang fp contract(off)
    return a + __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(b), CTRL, 0xf, 0xf, true));
}

// sum over the 8 lanes of each aligned group of 8, on every lane of the group
__device__ __forceinline__ float sum8(float y) {
    y = dpp_add<0xB1>(y, y);     // quad_perm [1,0,3,2] = lane ^ 1
    y = dpp_add<0x4E>(y, y);     // quad_perm [2,3,0,1] = lane ^ 2
    return dpp_add<0x141>(y, y); // row_half_mirror: lane i <- 7 - i within 8
}

template <int CTRL>
__device__ __forceinline__ double dpp_d(double v) {
    const long long b = __double_as_longlong(v);
    const unsigned lo = __builtin_amdgcn_update_dpp(0, (int)b, CTRL, 0xf, 0xf, true);
    const unsigned hi = __builtin_amdgcn_update_dpp(0, (int)(b >> 32), CTRL, 0xf, 0xf, true);
    return __longlong_as_double((long long)((unsigned long long)hi << 32 | lo));
}
__device__ __forceinline__ double sum8(double y) {
    y += dpp_d<0xB1>(y);
    y += dpp_d<0x4E>(y);
    return y + dpp_d<0x141>(y);
}

// Which part of which (replica, i-block) of n a wave takes: workgroup ids go to the 8 XCDs
// round-robin and each XCD has its own L2, so an XCD gets an eighth of consecutive blocks,
// first part 0 of all of them, then part 1, ..: parts become smaller (share_tiles), so the
// launch ends with short waves.
struct BlockWave {
    int rb, part;
    __device__ __forceinline__ BlockWave(int group, int waves_per_group, int wv, int n) {
        const int per = (n + 7) >> 3, q = (group >> 3) * waves_per_group + wv;
        part = q / per;
        rb = (group & 7) * per + q - part * per;
    }
};

// s_waitcnt vmcnt(0) alone (expcnt and lgkmcnt at their no-wait maxima).  The
// scheduling barrier keeps the arithmetic before it from being moved past the wait.
__device__ __forceinline__ void wait_vmem() {
    __builtin_amdgcn_sched_barrier(0);
    __builtin_amdgcn_s_waitcnt(0x0F70);
    __builtin_amdgcn_sched_barrier(0);
}

// Sums v[24] (8 i clusters x 3 components, index 3k+c) over the eight lanes with equal
// lane & 7 so that lane 8k + il ends up holding the components of cluster k, atom il.
// Three halving stages split the values between lane halves (bit 5: v_permlane32_swap,
// bit 4: v_permlane16_swap, bit 3: DPP row_ror:8).  The swaps exchange the upper half of
// their first operand with the lower half of their second, so r0 + r1 is the pairwise
// sum of the value each half keeps, with no selects.
__device__ __forceinline__ void scatter_clusters24(const float (&v)[24], int lane, float (&out)[3]) {
    float w[12], x[6];
#pragma unroll
    for (int t = 0; t < 12; t++) {
        auto r = __builtin_amdgcn_permlane32_swap(__float_as_uint(v[t]), __float_as_uint(v[t + 12]),
                                                   false, false);
        w[t] = __uint_as_float(r[0]) + __uint_as_float(r[1]);
    }
#pragma unroll
    for (int t = 0; t < 6; t++) {
        auto r = __builtin_amdgcn_permlane16_swap(__float_as_uint(w[t]), __float_as_uint(w[t + 6]),
                                                   false, false);
        x[t] = __uint_as_float(r[0]) + __uint_as_float(r[1]);
    }
    const bool b3 = (lane & 8) != 0;
#pragma unroll
    for (int t = 0; t < 3; t++) {
        float keep = b3 ? x[t + 3] : x[t];
        float send = b3 ? x[t] : x[t + 3];
        out[t] = dpp_add<0x128>(keep, send);  // row_ror:8 = lane ^ 8 within 16
    }
}

// Pairs of a block (within the cutoff), and tiles with any, after which the FP32 sums of its i
// forces go to the 64-bit accumulator, at the next tile.  A lane adds at most 8 terms to an i
// atom's sum in a tile, so 7 tiles leave 56 additions in a row and three over the lanes,
// whatever the geometry: no more than a tile's 64 terms in one lane.  The pairs bound the mean (16 to 20
// terms an atom).  The error of the forces against 64 bits, 32 frames of 22,750, 21,005 and 9,005
// atoms, as a ratio to FP32 sums of one tile added up in FP64: 0.989, 0.997, 0.994 (0.990, 0.997,
// 0.994 with one part per block); with 4,096 pairs and any number of tiles (20 frames) 0.991, 1.001,
// 0.996 (0.995, 1.008, 1.002), and 5.5e-8 where one atom has all pairs, so 1.4e-8.  Pair kernel of
// 22 x 22,750 and 8 x 99,920 atoms: 391 and 797 us, with 4,096 pairs 386 and 778, with 512 397 and 807,
// with tiles alone 387 and 781 (but 1.000, 1.004, 1.009 with one part per block).
constexpr int PAIRS_PER_FLUSH = 1024, TILES_PER_FLUSH = 7;

// m without its r lowest bits
__device__ __forceinline__ unsigned long long drop_bits(unsigned long long m, int r) {
    int p = 0, left = r;
#pragma unroll
    for (int h = 32; h > 0; h >>= 1) {
        const int c = __popcll((m >> p) & ((1ull << h) - 1ull));
        p += left >= c ? h : 0;
        left -= left >= c ? c : 0;
    }
    return left > 0 ? 0ull : m & (~0ull << p);
}

// One part of an i-block's tile list: tiles first..last (none: last < first), of the first
// one without its `skip` lowest steps, of the last one only the `upto` lowest
struct TilePart {
    int first, last, skip, upto;
    __device__ __forceinline__ TilePart(const int2* __restrict__ bounds, int rb, int part) {
        const int2 a = bounds[(size_t)rb * TILE_BOUNDS + part],
                   b = bounds[(size_t)rb * TILE_BOUNDS + part + 1];
        first = a.x;
        skip = a.y;
        last = b.y > 0 ? b.x : b.x - 1;
        upto = b.y > 0 ? b.y : 64;
        if (first == last && upto <= skip) last = -1;
    }
    __device__ __forceinline__ bool empty() const { return last < first; }
    // the part's bits of tile t's mask m
    __device__ __forceinline__ unsigned long long take(int t, unsigned long long m) const {
        unsigned long long k = m;
        if (t == last && upto < 64) k &= ~drop_bits(m, upto);
        if (t == first && skip > 0) k &= drop_bits(m, skip);
        return k;
    }
};

// The parts of a block that wave j of `waves` takes, from part_of(j) to part_of(j + 1): one
// each, or (waves < parts) first more and then fewer.  Where the waves are many, an i-block's
// atoms are then loaded for several parts at a time and the launch still ends with short waves
// (22 x 22,750 atoms, parts taken one by one 429 us, so 402, with 12 parts).
__device__ __forceinline__ int part_of(int j, int waves, int parts) {
    return waves == parts ? j : parts * j * (2 * waves - j) / (waves * waves);
}

// j atoms of block jb that i atom `lane` must not be paired with in this tile: exclusion
// partners, in the diagonal tile the atoms up to itself, slots past N; everything for a
// lane without an atom
__device__ __forceinline__ unsigned long long tile_exclusions(unsigned long long set,
                                                              int max_ex,
                                                              const int* __restrict__ exs,
                                                              int lane, bool vi, int ib, int jb,
                                                              int N) {
    unsigned long long em = 0;
    if ((set >> (jb & 63)) & 1ull) {
        for (int k = 0; k < max_ex; k++) {
            int sl = exs[k * 64 + lane];
            if ((sl >> 6) == jb) em |= 1ull << (sl & 63);  // -1 (none) is in no block
        }
    }
    if (jb == ib) em |= (2ull << lane) - 1ull;
    if (jb * 64 + 64 > N) em |= ~0ull << (N - jb * 64);  // uniform; N > jb * 64
    return vi ? em : ~0ull;
}

//   LDS per wave: two 2 KB tile buffers, 512 B of exclusion masks, 768 B of i coordinates.
//   vmcnt discipline: the only vector memory operations inside the tile loop are the
//   next tile's copy (global -> LDS by DMA), the exclusion loads of the few tiles that have
//   any, and the three flush atomics that end each tile.  Loads and stores/atomics share
//   vmcnt but need not retire in issue order, so the copy is waited for with vmcnt(0) before
//   the atomics, not with vmcnt(3) after them.
//   GEO: the geometric LJ sigma rule, the records holding sigma itself (Geom::geo).
//   rb: replica and i-block, of whose tile list the wave takes the parts from `part` up to
//   part_end; tile_s, em_s, xi_s: its LDS.
template <bool COUNT, bool GEO>
__device__ __forceinline__ void pair_wave(
    int rb, int part, int part_end, int lane, float4* tile_s, unsigned long long* em_s, float* xi_s, int R, int N, int Np,
    int NB, int maxj, int packed, const float4* __restrict__ arec,
    const int* __restrict__ tiles, const unsigned long long* __restrict__ tmask,
    const int2* __restrict__ bounds, const float4* __restrict__ bb_lo,
    const float4* __restrict__ bb_hi, const int* __restrict__ exs,
    const unsigned long long* __restrict__ exblocks, int max_ex, long long* __restrict__ F,
    int* __restrict__ flags, unsigned long long* __restrict__ pair_count, const Geom& g) {
    int r = rb / NB;
    int ib = rb - r * NB;
    const float4* A = arec + (size_t)r * Np * 2;
    unsigned long long* Fr = (unsigned long long*)(F + (size_t)r * 3 * Np);
    const int islot = ib * 64 + lane;
    const bool vi = islot < N;
    const int il = lane & 7, jl = lane >> 3;
    const float4* lo = bb_lo + (size_t)r * NB;
    const float4* hi = bb_hi + (size_t)r * NB;

    // copies the 64 slot records (32 B) of j-block jb into tile buffer b: lane L moves
    // half L&1 of record L>>1 (first instruction) and of record 32 + (L>>1) (second)
    auto stage = [&](int jb, int b) {
        float4* dst = tile_s + 128 * b;
        const char* src = (const char*)(A + 2 * jb * 64) + lane * 16;
        __builtin_amdgcn_wave_barrier();
        __builtin_amdgcn_global_load_lds((const void*)src,
                                         (__attribute__((address_space(3))) void*)dst, 16, 0, 0);
        __builtin_amdgcn_global_load_lds((const void*)(src + 1024),
                                         (__attribute__((address_space(3))) void*)(dst + 64), 16, 0, 0);
        __builtin_amdgcn_wave_barrier();
    };
    // 64 tiles of the list at a time, one per lane, so that no tile waits for its descriptor:
    // j-block (TILE_MI set where every pair needs its own minimum image), this wave's bits
    // of the mask, and the shift (hx, hy, hz) of the periodic image that the tile's pairs
    // take, which is taken off the atoms of the lower block whichever of the two lists the
    // tile, so that the rounding of a separation (and what is within the cutoff) does not
    // depend on that
    int tj = 0;
    float hx = 0.f, hy = 0.f, hz = 0.f;
    unsigned long long tm = 0ull;
    auto load_tiles = [&](int t) {
        if (t < maxj) {
            tj = tiles[(size_t)rb * maxj + t];
            tm = tmask[(size_t)rb * maxj + t];
        }
    };
    load_tiles(lane);  // mostly the whole list, in flight with the bounds
    if (part == part_end) return;  // more waves than the falling sizes need
    TilePart at(bounds, rb, part);
    while (at.empty()) {
        if (++part == part_end) return;
        at = TilePart(bounds, rb, part);
    }
    float xi[8], yi[8], zi[8], qi[8], si[8], ei[8], fi[24];
#pragma unroll
    for (int k = 0; k < 8; k++) {
        const float4 a = A[2 * (ib * 64 + 8 * k + il)];
        const float2 b = *(const float2*)&A[2 * (ib * 64 + 8 * k + il) + 1];
        xi[k] = a.x;
        yi[k] = a.y;
        zi[k] = a.z;
        qi[k] = a.w;
        si[k] = b.x;
        ei[k] = b.y;
        fi[3 * k] = fi[3 * k + 1] = fi[3 * k + 2] = 0.f;
    }
    if (vi) {  // i coordinates as stored, for tiles that shift them
        const float4 a = A[2 * islot];
        xi_s[lane] = a.x;
        xi_s[64 + lane] = a.y;
        xi_s[128 + lane] = a.z;
    }
    int ox = 0, oy = 0, oz = 0;  // what xi, yi, zi are shifted by now (bits of the floats)
    const int* E = exs + (size_t)rb * max_ex * 64;
    const unsigned long long eset = exblocks[rb];
    auto load_shifts = [&]() {
        if (packed) {
            hx = g.bx * tile_images(tj, 0);
            hy = g.by * tile_images(tj, 1);
            hz = g.bz * tile_images(tj, 2);
            return;
        }
        // the i-block's box is read here each time (opaque index): kept in registers
        // over the tile loop it made it spill
        int ibo = ib;
        asm volatile("" : "+s"(ibo));
        tj = min(tj & TILE_BLOCK, NB - 1);  // past the list's end: anything
        const int lower = min(ibo, tj), upper = max(ibo, tj);
        const bool one = tile_shift(lo[lower], hi[lower], lo[upper], hi[upper], g, hx, hy, hz);
        hx = one ? g.bx * hx : 0.f;
        hy = one ? g.by * hy : 0.f;
        hz = one ? g.bz * hz : 0.f;
        if (!one) tj |= TILE_MI;
    };
    int t = at.first;
    if (t >= 64) load_tiles((t & ~63) + lane);
    stage(__builtin_amdgcn_readlane(tj, t & 63) & TILE_BLOCK, 0);
    load_shifts();
    int bad = 0;
    // adds the i forces of the pairs so far to the accumulator: lane = i atom (atomic: other
    // waves and the side kernels add to the same accumulator)
    auto flush_i = [&]() {
        float f[3];
        scatter_clusters24(fi, lane, f);
        if (vi) {
            atomicAdd(&Fr[islot], to_fixed(f[0], &bad));
            atomicAdd(&Fr[Np + islot], to_fixed(f[1], &bad));
            atomicAdd(&Fr[2 * Np + islot], to_fixed(f[2], &bad));
        }
#pragma unroll
        for (int k = 0; k < 24; k++) fi[k] = 0.f;
    };
    int npair = 0, used = 0, buf = 0;  // pairs, and tiles with any, in the sums
    // lane that holds the sum of j atom `lane` of a tile (cluster lane >> 3 in lanes with
    // il = that cluster), as a byte address for ds_bpermute
    const int transpose = 4 * ((lane >> 3) + 8 * (lane & 7));
    const unsigned rec_lds = (unsigned)(size_t)&tile_s[2 * jl];
    wait_vmem();  // the first tile and the i atoms have arrived
    while (true) {
        const int ql = t & 63;
        const int jt = __builtin_amdgcn_readlane(tj, ql), jb = jt & TILE_BLOCK;
        const unsigned long long m = at.take(
            t, (unsigned long long)(unsigned)__builtin_amdgcn_readlane((int)(unsigned)tm, ql) |
                   (unsigned long long)(unsigned)__builtin_amdgcn_readlane((int)(unsigned)(tm >> 32), ql) << 32);
        // the shift (bits of the floats) of the i atoms, or else of each j atom as it is read
        const bool up = jb > ib;
        const int sx = __builtin_amdgcn_readlane(__float_as_int(hx), ql),
                  sy = __builtin_amdgcn_readlane(__float_as_int(hy), ql),
                  sz = __builtin_amdgcn_readlane(__float_as_int(hz), ql);
        const float ux = __int_as_float(up ? 0 : sx), uy = __int_as_float(up ? 0 : sy),
                    uz = __int_as_float(up ? 0 : sz);
        if ((up ? sx : 0) != ox || (up ? sy : 0) != oy || (up ? sz : 0) != oz) {
            ox = up ? sx : 0;
            oy = up ? sy : 0;
            oz = up ? sz : 0;
#pragma unroll
            for (int k = 0; k < 8; k++) {
                xi[k] = xi_s[8 * k + il] - __int_as_float(ox);
                yi[k] = xi_s[64 + 8 * k + il] - __int_as_float(oy);
                zi[k] = xi_s[128 + 8 * k + il] - __int_as_float(oz);
            }
        }
        // the next tile, of this part or of the wave's next one (which may begin with the rest
        // of this tile)
        const bool part_ends = t == at.last;
        int next = t + 1;
        if (part_ends) {
            next = -1;
            while (++part < part_end) {
                at = TilePart(bounds, rb, part);
                if (at.empty()) continue;
                next = at.first;
                break;
            }
        }
        if (next > t) {
            if (next >> 6 != t >> 6) {
                load_tiles((next & ~63) + lane);
                load_shifts();
            }
            stage(__builtin_amdgcn_readlane(tj, next & 63) & TILE_BLOCK, buf ^ 1);
        }
        if (!COUNT && (npair >= PAIRS_PER_FLUSH || used == TILES_PER_FLUSH)) {
            flush_i();
            npair = used = 0;
        }
        const int in_tile = npair;
        // pairs of the tile that need more than the shift (uniform): their own minimum
        // image, or a look at the exclusions and empty slots
        const bool mi = (jt & TILE_MI) != 0;
        bool ex = jb == ib || ((eset >> (jb & 63)) & 1ull) || ib * 64 + 64 > N || jb * 64 + 64 > N;
        if (ex) {
            const unsigned long long em = tile_exclusions(eset, max_ex, E, lane, vi, ib, jb, N);
            ex = __ballot(em != 0ull) != 0ull;
            em_s[lane] = em;
        }
        const int general = __builtin_amdgcn_readfirstlane(mi || ex ? 1 : 0);
        float fjx = 0.f, fjy = 0.f, fjz = 0.f;  // sum of cluster il, atom jl
        unsigned long long rest = m, done = 0ull;
        do {
            // the last cluster first: the order of the FP32 sums.  Errors as at PAIRS_PER_FLUSH (with
            // 384 pairs) 0.989, 0.996, 0.993, with the first one first 0.991, 0.997, 0.995
            const int jc8 = (63 - __builtin_clzll(rest)) & 56;  // 8 jc
            const unsigned ics = (unsigned)(m >> jc8) & 0xffu;
            rest &= ~(0xffull << jc8);
            // the cluster's records.  Written out because the compiler would otherwise put an
            // s_waitcnt vmcnt(0) (a wait for the next tile's copy, which goes to the other
            // half of the same array) in front of the reads.
            float4 pj;
            float2 pq;
            {
                const unsigned addr = rec_lds + (unsigned)(buf * 2048 + jc8 * 32);
                asm volatile(
                    "ds_read_b128 %0, %2\n\t"
                    "ds_read_b64 %1, %2 offset:16\n\t"
                    "s_waitcnt lgkmcnt(0)"
                    : "=&v"(pj), "=&v"(pq)
                    : "v"(addr)
                    : "memory");
            }
            const float xj = pj.x - ux, yj = pj.y - uy, zj = pj.z - uz;
            float fx = 0.f, fy = 0.f, fz = 0.f;
            // opaque to the compiler, which would otherwise carry the zeros through the
            // branches below as constants and copy the registers at the joins
            asm volatile("" : "+v"(fx), "+v"(fy), "+v"(fz));
            const int before = npair;
#pragma unroll
            for (int k = 0; k < 8; k++) {
                if (!(ics & (1u << k))) continue;  // uniform
                float dx = xi[k] - xj, dy = yi[k] - yj, dz = zi[k] - zj;
                float r2 = dx * dx + dy * dy + dz * dz;
                unsigned long long in = __ballot(r2 < g.rc2f);
                if (general != 0) {
                    if (mi) {
                        dx -= g.bx * rintf(dx * g.ibx);
                        dy -= g.by * rintf(dy * g.iby);
                        dz -= g.bz * rintf(dz * g.ibz);
                        r2 = dx * dx + dy * dy + dz * dz;
                        in = __ballot(r2 < g.rc2f);
                    }
                    if (ex) {  // the shift by uniform jc8 and lane jl in two steps
                        const unsigned long long em = em_s[8 * k + il];
                        const unsigned eb = (unsigned)(jc8 & 32 ? em >> 32 : em) >> (jc8 & 31);
                        in &= __ballot(!((eb >> jl) & 1u));
                    }
                }
                npair += __popcll(in);
                if (COUNT) continue;
                // lanes outside the cutoff are off; a step without any ends here
                if (__builtin_amdgcn_inverse_ballot_w64(in)) {
                    const float ir = __frsqrt_rn(r2);
                    const float ir2 = ir * ir;
                    float s2;
                    if constexpr (GEO) {
                        s2 = (si[k] * pq.x) * ir2;
                    } else {
                        const float sig = si[k] + pq.x;
                        s2 = sig * sig * ir2;
                    }
                    const float s6 = s2 * s2 * s2;
                    const float es6 = (ei[k] * pq.y) * s6;
                    const float qq = qi[k] * pj.w;
                    const float fr =
                        es6 * (12.0f * s6 - 6.0f) * ir2 + qq * (ir * ir2 - 2.0f * g.krff);
                    fi[3 * k] += fr * dx;
                    fi[3 * k + 1] += fr * dy;
                    fi[3 * k + 2] += fr * dz;
                    fx -= fr * dx;
                    fy -= fr * dy;
                    fz -= fr * dz;
                }
            }
            if (COUNT || npair == before) continue;  // uniform: no pair of the cluster
            // each j atom of the tile is in exactly one cluster: lanes with il = jc keep it
            const unsigned long long mine = 0x0101010101010101ull << (jc8 >> 3);
            done |= 0xffull << jc8;
            fx = sum8(fx);
            fy = sum8(fy);
            fz = sum8(fz);
            const bool keep = __builtin_amdgcn_inverse_ballot_w64(mine);
            fjx = keep ? fx : fjx;
            fjy = keep ? fy : fjy;
            fjz = keep ? fz : fjz;
        } while (rest);
        // flush the tile's j forces: lane = j atom, coalesced fixed-point atomics
        fjx = __int_as_float(__builtin_amdgcn_ds_bpermute(transpose, __float_as_int(fjx)));
        fjy = __int_as_float(__builtin_amdgcn_ds_bpermute(transpose, __float_as_int(fjy)));
        fjz = __int_as_float(__builtin_amdgcn_ds_bpermute(transpose, __float_as_int(fjz)));
        // the next tile's records have landed (and the previous tile's atomics, issued a
        // tile earlier, are done): waited for before this tile's atomics, because a load
        // and later atomics share vmcnt but may retire out of order
        wait_vmem();
        if (!COUNT && __builtin_amdgcn_inverse_ballot_w64(done)) {
            int s = jb * 64 + lane;
            atomicAdd(&Fr[s], fixed_from_float(fjx, &bad));
            atomicAdd(&Fr[Np + s], fixed_from_float(fjy, &bad));
            atomicAdd(&Fr[2 * Np + s], fixed_from_float(fjz, &bad));
        }
        // the i forces of each part are added up by themselves, so that results do not depend
        // on how many parts a wave takes
        if (!COUNT && part_ends) {
            flush_i();
            npair = used = 0;
        } else {
            used += npair > in_tile ? 1 : 0;
        }
        if (next < 0) break;
        buf ^= next > t ? 1 : 0;
        t = next;
    }
    if (COUNT) {
        if (lane == 0) atomicAdd(&pair_count[r], (unsigned long long)npair);
        return;
    }
    if (__ballot(bad) != 0ull && lane == 0) atomicOr(&flags[r], 2);
}

// ---------------------------------------------------------------------------
// Pair energies in FP64 (the energy evaluations: U0 and with it U1 = U0 + u and the
// potential energy).  The force kernel computes in FP32 from FP32 coordinates, whose
// rounding (an ulp is ~5e-7 nm at 4-8 nm) and arithmetic leave ~2^-24 of the summed pair
// magnitudes in U0; where U0 is a small net of large terms that exceeds 1e-5 of U0.  This
// kernel takes the FP64 positions and parameters of every pair with r < rc once, in
// Newton-3 order over the half tile lists, so U0 is exact to FP64 rounding.
//
// Waves per (replica, i-block) and their shares of the tiles as in the pair kernel
// (TilePart), pair of clusters by pair of clusters as the pair kernel does (lane 8 jl + il:
// j atom jl, i atom il), all in FP64: vector FP64 issues at the rate of unpacked FP32.  The i records
// stay in LDS (eight clusters of FP64 records would take 96 registers), the next tile's j
// records are loaded into registers while the current tile is evaluated.
// ---------------------------------------------------------------------------
// Orders the LDS accesses of a one-wave workgroup around this point.  A wave's LDS
// instructions are carried out in issue order, so a compiler barrier is enough: unlike
// __syncthreads() it does not wait for the wave's global loads in flight.
__device__ __forceinline__ void lds_order() { asm volatile("" ::: "memory"); }

//   irec, jrec, em_s: the wave's LDS
__device__ __forceinline__ void energy64_wave(
    int rb, int part, int lane, Rec64* irec, Rec64* jrec, unsigned long long* em_s, int R, int N, int Np,
    int NB, int maxj, int waves, int packed, const Rec64* __restrict__ rec,
    const int* __restrict__ tiles, const unsigned long long* __restrict__ tmask,
    const int2* __restrict__ bounds, const float4* __restrict__ bb_lo,
    const float4* __restrict__ bb_hi, const int* __restrict__ exs,
    const unsigned long long* __restrict__ exblocks, int max_ex, double* __restrict__ e_out,
    const Geom& g) {
    const int r = rb / NB, ib = rb - r * NB;
    const Rec64* RC = rec + (size_t)r * Np;
    const int islot = ib * 64 + lane;
    const bool vi = islot < N;
    const int il = lane & 7, jl = lane >> 3;
    irec[lane] = RC[vi ? islot : ib * 64];
    const int* E = exs + (size_t)(r * NB + ib) * max_ex * 64;
    const unsigned long long eset = exblocks[(size_t)r * NB + ib];
    const float4 bli = bb_lo[(size_t)r * NB + ib], bhi = bb_hi[(size_t)r * NB + ib];
    const int* tl = tiles + ((size_t)r * NB + ib) * maxj;
    const unsigned long long* tmk = tmask + ((size_t)r * NB + ib) * maxj;
    double e = 0.0;
    // the j records of the wave's next tile (a record is 3 x 16 bytes)
    double2 na = make_double2(0.0, 0.0), nb = na, nc = na;
    auto prefetch = [&](int jb) {
        const int js = jb * 64 + lane;
        if (js < N) {
            const double2* src = (const double2*)(RC + js);
            na = src[0];
            nb = src[1];
            nc = src[2];
        }
    };
    const TilePart steps(bounds, rb, part);
    if (steps.first <= steps.last) prefetch(tl[steps.first] & TILE_BLOCK);
    for (int t = steps.first; t <= steps.last; t++) {
        const int entry = tl[t], jb = entry & TILE_BLOCK;
        const unsigned long long m = steps.take(t, tmk[t]);
        lds_order();  // the previous tile's records are no longer read
        jrec[lane] = Rec64{na.x, na.y, nb.x, nb.y, nc.x, nc.y};
        if (t < steps.last) prefetch(tl[t + 1] & TILE_BLOCK);
        const unsigned long long em = tile_exclusions(eset, max_ex, E, lane, vi, ib, jb, N);
        const bool ex = __ballot(em != 0ull) != 0ull;
        if (ex) em_s[lane] = em;
        float kx, ky, kz;
        bool one_image;
        if (packed) {  // of the lower block's atoms
            const float up = jb > ib ? 1.f : -1.f;
            kx = up * tile_images(entry, 0);
            ky = up * tile_images(entry, 1);
            kz = up * tile_images(entry, 2);
            one_image = !(entry & TILE_MI);
        } else {
            one_image = tile_shift(bli, bhi, bb_lo[(size_t)r * NB + jb], bb_hi[(size_t)r * NB + jb],
                                   g, kx, ky, kz);
        }
        const double sx = g.Lx * (double)kx, sy = g.Ly * (double)ky, sz = g.Lz * (double)kz;
        lds_order();  // this tile's records are stored
        auto clusters = [&](auto mic, auto exc) {
            constexpr bool MI = decltype(mic)::value, EX = decltype(exc)::value;
            unsigned long long rest = m;
            while (rest) {
                const int jc = __builtin_ctzll(rest) >> 3;
                unsigned ics = (unsigned)(m >> (8 * jc)) & 0xffu;
                rest &= ~(0xffull << (8 * jc));
                Rec64 J = jrec[8 * jc + jl];
                if (!MI) {
                    J.x += sx;
                    J.y += sy;
                    J.z += sz;
                }
                do {
                    const int k = __builtin_ctz(ics);
                    ics &= ics - 1u;
                    const Rec64 I = irec[8 * k + il];
                    double dx = I.x - J.x, dy = I.y - J.y, dz = I.z - J.z;
                    if (MI) {
                        dx = min_image(dx, g.Lx, g.iLx);
                        dy = min_image(dy, g.Ly, g.iLy);
                        dz = min_image(dz, g.Lz, g.iLz);
                    }
                    const double r2 = dx * dx + dy * dy + dz * dz;
                    bool ok = r2 < g.rc2;
                    if (EX) ok = ok && !((em_s[8 * k + il] >> (8 * jc + jl)) & 1ull);
                    if (__ballot(ok) == 0ull) continue;  // uniform
                    const double ir = rsqrt(r2);
                    const double ir2 = ir * ir;
                    double s2;
                    if (g.geo) {  // Geom::geo: the records hold sigma itself
                        s2 = I.sh * J.sh * ir2;
                    } else {
                        const double sig = I.sh + J.sh;
                        s2 = sig * sig * ir2;
                    }
                    const double s6 = s2 * s2 * s2;
                    const double qq = I.qk * J.qk;
                    const double ee = (I.es * J.es) * s6 * (s6 - 1.0) +
                                      qq * (ir + g.krf * r2 - g.crf);
                    e += ok ? ee : 0.0;  // also clears inf or NaN of excluded or empty slots
                } while (ics);
            }
        };
        using T = std::true_type;
        using Fa = std::false_type;
        if (one_image) {
            if (ex) clusters(Fa(), T());
            else clusters(Fa(), Fa());
        } else {
            if (ex) clusters(T(), T());
            else clusters(T(), Fa());
        }
    }
    e = wave_sum(e);
    if (lane == 0) e_out[rb * waves + part] = e;
}

// ---------------------------------------------------------------------------
// group 1: harmonic bonds and angles at x (FP64), gathered per atom.  One thread per
// (atom, replica) evaluates every term its atom belongs to (a bond by both of its atoms,
// an angle by all three) and keeps only its own atom's share, so the forces need no
// atomics and are summed in a fixed order; a term's energy is counted by its first
// atom.  bcode holds (bond << 1) | role and acode (angle << 2) | role, role being the
// atom's position in the term; the lists of atom i are [bstart[i], bstart[i+1]) and
// [astart[i], astart[i+1]).  The forces go to Fb (FP64, atom order, [R][3][Np]), which
// the integrator adds to the fixed-point accumulator.
// ---------------------------------------------------------------------------
//   One wave takes 64 atoms of one replica (w: replica, then block of 64 atoms).
__device__ __forceinline__ void bonded_wave(
    int w, int lane, int R, int N, int Np, int nbw, const int* __restrict__ bstart,
    const int* __restrict__ bcode, const int* __restrict__ astart,
    const int* __restrict__ acode, const int* __restrict__ bond_atoms,
    const double* __restrict__ bond_r0, const double* __restrict__ bond_k,
    const int* __restrict__ ang_atoms, const double* __restrict__ ang_t0,
    const double* __restrict__ ang_k, const double* __restrict__ x64, double* __restrict__ Fb,
    double* __restrict__ e_bond, int* __restrict__ flags) {
    if (w >= R * nbw) return;
    const int r = w / nbw, i = (w - r * nbw) * 64 + lane;
    const double* X = x64 + (size_t)r * 3 * Np;
    double e = 0.0;
    if (i < N) {
        double f[3] = {0.0, 0.0, 0.0};
        double xi[3] = {X[i], X[Np + i], X[2 * Np + i]};
        for (int q = bstart[i], qe = bstart[i + 1]; q < qe; q++) {
            int code = bcode[q], t = code >> 1, role = code & 1;
            int j = bond_atoms[2 * t + (role ^ 1)];
            double d[3];
            for (int a = 0; a < 3; a++) d[a] = X[a * Np + j] - xi[a];
            const double rsq = d[0] * d[0] + d[1] * d[1] + d[2] * d[2];
            const double irr = rsq > 0.0 ? rsqrt(rsq) : 0.0;
            double dr = rsq * irr - bond_r0[t];
            double gg = bond_k[t] * dr * irr;
            for (int a = 0; a < 3; a++) f[a] += gg * d[a];  // pulls i toward j when stretched
            if (role == 0) e += 0.5 * bond_k[t] * dr * dr;
        }
        for (int q = astart[i], qe = astart[i + 1]; q < qe; q++) {
            int code = acode[q], k = code >> 2, role = code & 3;
            int ia = ang_atoms[3 * k], im = ang_atoms[3 * k + 1], ic = ang_atoms[3 * k + 2];
            double v1[3], v2[3];
            for (int a = 0; a < 3; a++) {
                double xm = X[a * Np + im];
                v1[a] = X[a * Np + ia] - xm;
                v2[a] = X[a * Np + ic] - xm;
            }
            // theta = atan2(|v1 x v2|, v1 . v2): one call gives the angle and, with the
            // reciprocal lengths, its sine (acos plus sin took twice the instructions and
            // is worse conditioned near 0 and pi)
            const double i1 = rsqrt(v1[0] * v1[0] + v1[1] * v1[1] + v1[2] * v1[2]);
            const double i2 = rsqrt(v2[0] * v2[0] + v2[1] * v2[1] + v2[2] * v2[2]);
            const double dot = v1[0] * v2[0] + v1[1] * v2[1] + v1[2] * v2[2];
            const double cx = v1[1] * v2[2] - v1[2] * v2[1], cy = v1[2] * v2[0] - v1[0] * v2[2],
                         cz = v1[0] * v2[1] - v1[1] * v2[0];
            const double cr = sqrt(cx * cx + cy * cy + cz * cz);
            double th = atan2(cr, dot);
            const double cs = dot * i1 * i2, sn = cr * i1 * i2;
            double dth = th - ang_t0[k];
            double gg = ang_k[k] * dth / fmax(sn, 1e-12);
            if (role == 0) e += 0.5 * ang_k[k] * dth * dth;
            const double p12 = gg * i1 * i2, p11 = gg * cs * i1 * i1, p22 = gg * cs * i2 * i2;
            for (int a = 0; a < 3; a++) {
                double fa = p12 * v2[a] - p11 * v1[a];
                double fc = p12 * v1[a] - p22 * v2[a];
                f[a] += role == 0 ? fa : (role == 2 ? fc : -(fa + fc));
            }
        }
        bool bad = false;
        double* Fr = Fb + (size_t)r * 3 * Np;
        for (int a = 0; a < 3; a++) {
            bad |= !(fabs(f[a]) < SDM_FIX_LIMIT);
            Fr[a * Np + i] = f[a];
        }
        if (bad) atomicOr(&flags[r], 2);
    }
    e = wave_sum(e);
    if (lane == 0) e_bond[w] = e;
}

// ---------------------------------------------------------------------------
// group 1: the SDMUtils restraints at x (FP64), fixed-point atomics; one wave per
// (restraint, replica).  Restates SDMUtils.py:32-257 (the energy expressions of the
// CustomCentroidBondForce and the three CustomCompoundBondForces); no periodic images.
// ---------------------------------------------------------------------------
struct DevCentroid {
    int g1, n1, g2, n2;  // ranges of the restraint atom / weight arrays (weights sum to 1)
    int do_angles, pad;
    int ref[6];          // g3, g4, g5 (receptor), g6, g7, g8 (ligand)
    double kfcm, tol, off[3], control;
    double kf[3], lo[3], hi[3];
};

struct DevAlign {
    int a[3], b[3];
    double kfd, kth, kps, off[3];
};

__device__ __forceinline__ double wrap_period(double x, double P) {
    return x - P * floor(x / P + 0.5);
}

__device__ __forceinline__ double dot3(const double* a, const double* b) {
    return a[0] * b[0] + a[1] * b[1] + a[2] * b[2];
}

__device__ __forceinline__ void cross3(const double* a, const double* b, double* c) {
    c[0] = a[1] * b[2] - a[2] * b[1];
    c[1] = a[2] * b[0] - a[0] * b[2];
    c[2] = a[0] * b[1] - a[1] * b[0];
}

// (kf/2)(step(dm) max(0,db)^2 + step(-dm) max(0,-da)^2) with db, da, dm = t - hi, t - lo,
// t - (lo+hi)/2 wrapped to the period P (step(0) = 1); *dEdt = its derivative in t
__device__ double flat_bottom(double t, double kf, double lo, double hi, double P,
                              double* dEdt) {
    double db = wrap_period(t - hi, P), da = wrap_period(t - lo, P);
    double dm = wrap_period(t - 0.5 * (lo + hi), P);
    double e = 0.0, g = 0.0;
    if (dm >= 0.0) {
        double m = fmax(0.0, db);
        e += m * m;
        g += m;
    }
    if (-dm >= 0.0) {
        double m = fmax(0.0, -da);
        e += m * m;
        g -= m;
    }
    *dEdt = kf * g;
    return 0.5 * kf * e;
}

// angle at p2 in [0, pi] and its gradient (zero when the three points are collinear)
__device__ double angle_grad(const double* p1, const double* p2, const double* p3, double* g1,
                             double* g2, double* g3) {
    double u[3], v[3], n[3], nu[3], nv[3];
    for (int d = 0; d < 3; d++) {
        u[d] = p1[d] - p2[d];
        v[d] = p3[d] - p2[d];
    }
    cross3(u, v, n);
    double nn = sqrt(dot3(n, n));
    double t = atan2(nn, dot3(u, v));
    cross3(n, u, nu);
    cross3(n, v, nv);
    double su = nn > 0.0 ? 1.0 / (nn * dot3(u, u)) : 0.0;
    double sv = nn > 0.0 ? 1.0 / (nn * dot3(v, v)) : 0.0;
    for (int d = 0; d < 3; d++) {
        g1[d] = -nu[d] * su;
        g3[d] = nv[d] * sv;
        g2[d] = -(g1[d] + g3[d]);
    }
    return t;
}

// dihedral (IUPAC sign) in (-pi, pi] and its gradient (zero when degenerate)
__device__ double dihedral_grad(const double* p1, const double* p2, const double* p3,
                                const double* p4, double* g1, double* g2, double* g3,
                                double* g4) {
    double b1[3], b2[3], b3[3], n1[3], n2[3];
    for (int d = 0; d < 3; d++) {
        b1[d] = p2[d] - p1[d];
        b2[d] = p3[d] - p2[d];
        b3[d] = p4[d] - p3[d];
    }
    cross3(b1, b2, n1);
    cross3(b2, b3, n2);
    double l2 = sqrt(dot3(b2, b2));
    double t = atan2(l2 * dot3(b1, n2), dot3(n1, n2));
    double q1 = dot3(n1, n1), q2 = dot3(n2, n2);
    bool ok = q1 > 0.0 && q2 > 0.0 && l2 > 0.0;
    double s1 = ok ? dot3(b1, b2) / (l2 * l2) : 0.0, s3 = ok ? dot3(b3, b2) / (l2 * l2) : 0.0;
    for (int d = 0; d < 3; d++) {
        g1[d] = ok ? -l2 * n1[d] / q1 : 0.0;
        g4[d] = ok ? l2 * n2[d] / q2 : 0.0;
        g2[d] = (-s1 - 1.0) * g1[d] + s3 * g4[d];
        g3[d] = s1 * g1[d] - (s3 + 1.0) * g4[d];
    }
    return t;
}

// k (1 - cos p) for cos p between the components of x3-x1 and x5-x4 perpendicular to
// x2-x1; adds the forces to f[0..4]
__device__ double psi_term(const double* x1, const double* x2, const double* x3,
                           const double* x4, const double* x5, double k, double (*f)[3]) {
    double d1[3], d0[3], d3[3], n1[3], v[3], w[3];
    for (int d = 0; d < 3; d++) {
        d1[d] = x2[d] - x1[d];
        d0[d] = x3[d] - x1[d];
        d3[d] = x5[d] - x4[d];
    }
    double l1 = sqrt(dot3(d1, d1));
    for (int d = 0; d < 3; d++) n1[d] = d1[d] / l1;
    double p0 = dot3(d0, n1), p3 = dot3(d3, n1);
    for (int d = 0; d < 3; d++) {
        v[d] = d0[d] - p0 * n1[d];
        w[d] = d3[d] - p3 * n1[d];
    }
    double lv = sqrt(dot3(v, v)), lw = sqrt(dot3(w, w));
    double c = dot3(v, w) / (lv * lw);
    for (int d = 0; d < 3; d++) {
        double gv = (w[d] / lw - c * v[d] / lv) / lv;
        double gw = (v[d] / lv - c * w[d] / lw) / lw;
        double gd1 = (-p0 * gv - p3 * gw) / l1;
        // F = -dE/dx = k d(cos p)/dx
        f[0][d] -= k * (gd1 + gv);
        f[1][d] += k * gd1;
        f[2][d] += k * gv;
        f[3][d] -= k * gw;
        f[4][d] += k * gw;
    }
    return k * (1.0 - c);
}

__global__ __launch_bounds__(64) void k_restraints(
    int Np, int ncen, int nrest, const DevCentroid* __restrict__ cen,
    const DevAlign* __restrict__ ali, const int* __restrict__ ratom,
    const double* __restrict__ rw, const double* __restrict__ x64,
    const int* __restrict__ slot_of, long long* __restrict__ F, double* __restrict__ e_rest,
    int* __restrict__ flags) {
    const double kPi = 3.14159265358979323846;
    int k = blockIdx.x, r = blockIdx.y, lane = threadIdx.x;
    const double* X = x64 + (size_t)r * 3 * Np;
    unsigned long long* Fr = (unsigned long long*)(F + (size_t)r * 3 * Np);
    const int* S = slot_of ? slot_of + (size_t)r * Np : nullptr;
    int bad = 0;
    auto addf = [&](int a, const double* f) {
        int s = S ? S[a] : a;
        atomicAdd(&Fr[s], (unsigned long long)to_fixed(f[0], &bad));
        atomicAdd(&Fr[Np + s], (unsigned long long)to_fixed(f[1], &bad));
        atomicAdd(&Fr[2 * Np + s], (unsigned long long)to_fixed(f[2], &bad));
    };
    auto pos = [&](int a, double* p) {
        p[0] = X[a];
        p[1] = X[Np + a];
        p[2] = X[2 * Np + a];
    };
    double e = 0.0;
    if (k < ncen) {
        const DevCentroid& R = cen[k];
        // weighted centres of the two groups (wave butterflies: every lane gets the sums)
        double c[6] = {0.0, 0.0, 0.0, 0.0, 0.0, 0.0};
        for (int i = lane; i < R.n1; i += 64) {
            int a = ratom[R.g1 + i];
            double w = rw[R.g1 + i];
            c[0] += w * X[a];
            c[1] += w * X[Np + a];
            c[2] += w * X[2 * Np + a];
        }
        for (int i = lane; i < R.n2; i += 64) {
            int a = ratom[R.g2 + i];
            double w = rw[R.g2 + i];
            c[3] += w * X[a];
            c[4] += w * X[Np + a];
            c[5] += w * X[2 * Np + a];
        }
        for (int d = 0; d < 6; d++) c[d] = wave_sum(c[d]);
        double dv[3] = {c[0] - R.off[0] - c[3], c[1] - R.off[1] - c[4],
                        c[2] - R.off[2] - c[5]};
        double d12 = sqrt(dot3(dv, dv));
        double gd = 0.0;
        if (d12 >= R.tol && d12 > 0.0) {
            double x = d12 - R.tol;
            e += 0.5 * R.control * R.kfcm * x * x;
            gd = R.control * R.kfcm * x / d12;  // |dE/dc1| / d12
        }
        if (gd != 0.0) {  // the same on every lane
            for (int i = lane; i < R.n1; i += 64) {
                double w = rw[R.g1 + i];
                double f[3] = {-w * gd * dv[0], -w * gd * dv[1], -w * gd * dv[2]};
                addf(ratom[R.g1 + i], f);
            }
            for (int i = lane; i < R.n2; i += 64) {
                double w = rw[R.g2 + i];
                double f[3] = {w * gd * dv[0], w * gd * dv[1], w * gd * dv[2]};
                addf(ratom[R.g2 + i], f);
            }
        }
        if (R.do_angles && lane == 0) {
            double p[6][3], f[6][3] = {}, g[4][3], dE;
            for (int j = 0; j < 6; j++) pos(R.ref[j], p[j]);
            // theta = angle(g3, g6, g7)
            double t = angle_grad(p[0], p[3], p[4], g[0], g[1], g[2]);
            e += R.control * flat_bottom(t, R.kf[0], R.lo[0], R.hi[0], kPi, &dE);
            dE *= R.control;
            const int ta[3] = {0, 3, 4};
            for (int j = 0; j < 3; j++)
                for (int d = 0; d < 3; d++) f[ta[j]][d] -= dE * g[j][d];
            // phi1 = dihedral(g4, g3, g6, g7), phi2 = dihedral(g3, g6, g7, g8)
            const int da[2][4] = {{1, 0, 3, 4}, {0, 3, 4, 5}};
            for (int q = 0; q < 2; q++) {
                const int* ix = da[q];
                t = dihedral_grad(p[ix[0]], p[ix[1]], p[ix[2]], p[ix[3]], g[0], g[1], g[2],
                                  g[3]);
                e += R.control *
                     flat_bottom(t, R.kf[1 + q], R.lo[1 + q], R.hi[1 + q], 2.0 * kPi, &dE);
                dE *= R.control;
                for (int j = 0; j < 4; j++)
                    for (int d = 0; d < 3; d++) f[ix[j]][d] -= dE * g[j][d];
            }
            for (int j = 0; j < 6; j++) addf(R.ref[j], f[j]);
        }
    } else if (lane == 0) {
        const DevAlign& A = ali[k - ncen];
        double a[3][3], b[3][3], fa[3][3] = {}, fb[3][3] = {};
        for (int j = 0; j < 3; j++) {
            pos(A.a[j], a[j]);
            pos(A.b[j], b[j]);
        }
        // displacement: (kfdispl/2)|b0 - offset - a0|^2
        double dd[3];
        for (int d = 0; d < 3; d++) dd[d] = b[0][d] - A.off[d] - a[0][d];
        e += 0.5 * A.kfd * dot3(dd, dd);
        for (int d = 0; d < 3; d++) {
            fb[0][d] -= A.kfd * dd[d];
            fa[0][d] += A.kfd * dd[d];
        }
        // theta: (ktheta/2)(1 - cos t), cos t = unit(b1 - b0).unit(a1 - a0)
        double d1[3], d2[3];
        for (int d = 0; d < 3; d++) {
            d1[d] = b[1][d] - b[0][d];
            d2[d] = a[1][d] - a[0][d];
        }
        double l1 = sqrt(dot3(d1, d1)), l2 = sqrt(dot3(d2, d2));
        double cs = dot3(d1, d2) / (l1 * l2);
        e += 0.5 * A.kth * (1.0 - cs);
        for (int d = 0; d < 3; d++) {
            double f2 = 0.5 * A.kth * (d2[d] / l2 - cs * d1[d] / l1) / l1;
            double f4 = 0.5 * A.kth * (d1[d] / l1 - cs * d2[d] / l2) / l2;
            fb[1][d] += f2;
            fb[0][d] -= f2;
            fa[1][d] += f4;
            fa[0][d] -= f4;
        }
        // psi, symmetrized: (kpsi/4)(1 - cos p) for (b0,b1,b2,a0,a2) and (a0,a1,a2,b0,b2)
        double f5[5][3] = {};
        e += psi_term(b[0], b[1], b[2], a[0], a[2], 0.25 * A.kps, f5);
        for (int d = 0; d < 3; d++) {
            fb[0][d] += f5[0][d];
            fb[1][d] += f5[1][d];
            fb[2][d] += f5[2][d];
            fa[0][d] += f5[3][d];
            fa[2][d] += f5[4][d];
        }
        double h5[5][3] = {};
        e += psi_term(a[0], a[1], a[2], b[0], b[2], 0.25 * A.kps, h5);
        for (int d = 0; d < 3; d++) {
            fa[0][d] += h5[0][d];
            fa[1][d] += h5[1][d];
            fa[2][d] += h5[2][d];
            fb[0][d] += h5[3][d];
            fb[2][d] += h5[4][d];
        }
        for (int j = 0; j < 3; j++) {
            addf(A.a[j], fa[j]);
            addf(A.b[j], fb[j]);
        }
    }
    if (bad) atomicOr(&flags[r], 2);
    if (lane == 0) e_rest[(size_t)r * nrest + k] = e;
}

// ---------------------------------------------------------------------------
// further force-field terms (FP64, one thread per term): periodic torsions, harmonic
// impropers and positional restraints (group 1), the 1-4 exceptions of the nonbonded
// force (group 2: plain LJ + Coulomb, no cutoff, no periodic image).
// ---------------------------------------------------------------------------
struct DevTerms {
    int nt, ni, nfb, nph, nex;  // term index ranges, in this order
    const int* t_atoms;
    const int* t_n;
    const double *t_phase, *t_k;
    const int* i_atoms;
    const double *i_phi0, *i_k;
    const int* fb_atom;
    const double *fb_x0, *fb_k, *fb_tol;
    const int* ph_atom;
    const double *ph_x0, *ph_k;
    const int* ex_atoms;
    const double *ex_qq, *ex_sig, *ex_eps;  // qq includes k_e
};

// group-1 forces go to Fb (slot map Sb, or atom order if null), group-2 forces to F
// (slot map S); energies per workgroup into e1 (group 1) and e2 (group 2)
__global__ __launch_bounds__(256) void k_terms(int Np, DevTerms T, const double* __restrict__ x64,
                                               const int* __restrict__ Sb_all,
                                               long long* __restrict__ Fb,
                                               const int* __restrict__ S_all,
                                               long long* __restrict__ F, double* __restrict__ e1,
                                               double* __restrict__ e2, int nblk, Geom g,
                                               int* __restrict__ flags) {
    __shared__ double red[2][256];
    int r = blockIdx.y, t = blockIdx.x * 256 + threadIdx.x;
    const double* X = x64 + (size_t)r * 3 * Np;
    const int* Sb = Sb_all ? Sb_all + (size_t)r * Np : nullptr;
    const int* S = S_all + (size_t)r * Np;
    unsigned long long* Fbr = (unsigned long long*)(Fb + (size_t)r * 3 * Np);
    unsigned long long* Fr = (unsigned long long*)(F + (size_t)r * 3 * Np);
    int bad = 0;
    double eg1 = 0.0, eg2 = 0.0;
    auto pos = [&](int a, double* p) {
        p[0] = X[a];
        p[1] = X[Np + a];
        p[2] = X[2 * Np + a];
    };
    auto addf = [&](unsigned long long* Fx, const int* map, int a, const double* f) {
        int s = map ? map[a] : a;
        atomicAdd(&Fx[s], (unsigned long long)to_fixed(f[0], &bad));
        atomicAdd(&Fx[Np + s], (unsigned long long)to_fixed(f[1], &bad));
        atomicAdd(&Fx[2 * Np + s], (unsigned long long)to_fixed(f[2], &bad));
    };
    const int e_imp = T.nt + T.ni, e_fb = e_imp + T.nfb, e_ph = e_fb + T.nph, e_ex = e_ph + T.nex;
    if (t < e_imp) {  // torsion or improper: a function of the dihedral
        bool tors = t < T.nt;
        int k = tors ? t : t - T.nt;
        const int* a = tors ? T.t_atoms + 4 * k : T.i_atoms + 4 * k;
        double p[4][3], gr[4][3];
        for (int j = 0; j < 4; j++) pos(a[j], p[j]);
        double phi = dihedral_grad(p[0], p[1], p[2], p[3], gr[0], gr[1], gr[2], gr[3]);
        double dE;
        if (tors) {
            double n = (double)T.t_n[k], arg = n * phi - T.t_phase[k];
            eg1 = T.t_k[k] * (1.0 + cos(arg));
            dE = -T.t_k[k] * n * sin(arg);
        } else {
            double d = phi - T.i_phi0[k];
            eg1 = T.i_k[k] * d * d;
            dE = 2.0 * T.i_k[k] * d;
        }
        for (int j = 0; j < 4; j++) {
            double f[3] = {-dE * gr[j][0], -dE * gr[j][1], -dE * gr[j][2]};
            addf(Fbr, Sb, a[j], f);
        }
    } else if (t < e_fb) {  // flat-bottom positional restraint, minimum image
        int k = t - e_imp, a = T.fb_atom[k];
        double p[3];
        pos(a, p);
        double d[3] = {min_image(p[0] - T.fb_x0[3 * k], g.Lx, g.iLx),
                       min_image(p[1] - T.fb_x0[3 * k + 1], g.Ly, g.iLy),
                       min_image(p[2] - T.fb_x0[3 * k + 2], g.Lz, g.iLz)};
        double dist = sqrt(dot3(d, d)), x = dist - T.fb_tol[k];
        if (x >= 0.0 && dist > 0.0) {
            eg1 = T.fb_k[k] * x * x;
            double c = -2.0 * T.fb_k[k] * x / dist;
            double f[3] = {c * d[0], c * d[1], c * d[2]};
            addf(Fbr, Sb, a, f);
        }
    } else if (t < e_ph) {  // harmonic positional restraint per axis
        int k = t - e_fb, a = T.ph_atom[k];
        double p[3], f[3];
        pos(a, p);
        for (int d = 0; d < 3; d++) {
            double dx = p[d] - T.ph_x0[3 * k + d];
            eg1 += T.ph_k[3 * k + d] * dx * dx;
            f[d] = -2.0 * T.ph_k[3 * k + d] * dx;
        }
        addf(Fbr, Sb, a, f);
    } else if (t < e_ex) {  // 1-4 exception (group 2)
        int k = t - e_ph, i = T.ex_atoms[2 * k], j = T.ex_atoms[2 * k + 1];
        double pi[3], pj[3], d[3];
        pos(i, pi);
        pos(j, pj);
        for (int q = 0; q < 3; q++) d[q] = pi[q] - pj[q];
        double r2 = dot3(d, d), ir2 = 1.0 / r2, ir = sqrt(ir2);
        double s2 = T.ex_sig[k] * T.ex_sig[k] * ir2, s6 = s2 * s2 * s2;
        double e4 = 4.0 * T.ex_eps[k];
        eg2 = e4 * s6 * (s6 - 1.0) + T.ex_qq[k] * ir;
        double fr = (e4 * s6 * (12.0 * s6 - 6.0) + T.ex_qq[k] * ir) * ir2;  // -dE/dr / r
        double fi[3] = {fr * d[0], fr * d[1], fr * d[2]};
        double fj[3] = {-fi[0], -fi[1], -fi[2]};
        addf(Fr, S, i, fi);
        addf(Fr, S, j, fj);
    }
    if (bad) atomicOr(&flags[r], 2);
    red[0][threadIdx.x] = eg1;
    red[1][threadIdx.x] = eg2;
    __syncthreads();
    for (int o = 128; o > 0; o >>= 1) {
        if (threadIdx.x < o) {
            red[0][threadIdx.x] += red[0][threadIdx.x + o];
            red[1][threadIdx.x] += red[1][threadIdx.x + o];
        }
        __syncthreads();
    }
    if (threadIdx.x == 0) {
        e1[(size_t)r * nblk + blockIdx.x] = red[0][0];
        e2[(size_t)r * nblk + blockIdx.x] = red[1][0];
    }
}

// ---------------------------------------------------------------------------
// displaced-state passes (FP64)
// ---------------------------------------------------------------------------

__device__ __forceinline__ bool excluded(const int* __restrict__ ex_start,
                                         const int* __restrict__ ex_list, int a, int b) {
    for (int k = ex_start[a]; k < ex_start[a + 1]; k++)
        if (ex_list[k] == b) return true;
    return false;
}

struct Atom64 {
    double x, y, z;      // position at x
    double dx, dy, dz;   // displacement
    double qk, sig, se;  // q*sqrt(k_e), sigma, sqrt(epsilon)
    int idx, cls;
};

__device__ __forceinline__ Atom64 load_atom64(const double* __restrict__ X, int Np, int a,
                                              const int* __restrict__ cls,
                                              const double* __restrict__ cdispl,
                                              const double* __restrict__ q,
                                              const double* __restrict__ sig,
                                              const double* __restrict__ eps) {
    Atom64 A;
    A.x = X[a];
    A.y = X[Np + a];
    A.z = X[2 * Np + a];
    A.cls = cls[a];
    A.dx = cdispl[3 * A.cls];
    A.dy = cdispl[3 * A.cls + 1];
    A.dz = cdispl[3 * A.cls + 2];
    A.qk = q[a];
    A.sig = sig[a];
    A.se = sqrt(eps[a]);
    A.idx = a;
    return A;
}

// the two geometries of one pair (i displaced by d_i, j by d_j): returns
// e(x+d) - e(x) and adds F1-F0 on i to (fx,fy,fz).
__device__ __forceinline__ double delta_pair(const Atom64& I, const Atom64& J, const Geom& g,
                                             double& fx, double& fy, double& fz, int* inside_y) {
    double qq = I.qk * J.qk;
    double sig = g.geo ? sqrt(I.sig * J.sig) : 0.5 * (I.sig + J.sig);
    double eps4 = 4.0 * I.se * J.se;
    double ex, fr_x, ey, fr_y;
    double dx = min_image(I.x - J.x, g.Lx, g.iLx);
    double dy = min_image(I.y - J.y, g.Ly, g.iLy);
    double dz = min_image(I.z - J.z, g.Lz, g.iLz);
    pair64(dx, dy, dz, qq, sig, eps4, g.rc2, g.krf, g.crf, &ex, &fr_x);
    double ex_ = min_image((I.x + I.dx) - (J.x + J.dx), g.Lx, g.iLx);
    double ey_ = min_image((I.y + I.dy) - (J.y + J.dy), g.Ly, g.iLy);
    double ez_ = min_image((I.z + I.dz) - (J.z + J.dz), g.Lz, g.iLz);
    *inside_y = pair64(ex_, ey_, ez_, qq, sig, eps4, g.rc2, g.krf, g.crf, &ey, &fr_y);
    fx += fr_y * ex_ - fr_x * dx;
    fy += fr_y * ey_ - fr_x * dy;
    fz += fr_y * ez_ - fr_x * dz;
    return ey - ex;
}

// Up to 64 atoms staged in LDS by one wave (lane t copies atom t), so that the loops over
// partner atoms read LDS broadcasts instead of chains of dependent global loads.
struct AtomTile64 {
    double x[64], y[64], z[64], dx[64], dy[64], dz[64], q[64], sig[64], se[64];
    int cls[64], idx[64];
};

__device__ __forceinline__ void stage_atom(AtomTile64& T, int t, const Atom64& A) {
    T.x[t] = A.x;
    T.y[t] = A.y;
    T.z[t] = A.z;
    T.dx[t] = A.dx;
    T.dy[t] = A.dy;
    T.dz[t] = A.dz;
    T.q[t] = A.qk;
    T.sig[t] = A.sig;
    T.se[t] = A.se;
    T.cls[t] = A.cls;
    T.idx[t] = A.idx;
}

__device__ __forceinline__ Atom64 tile_atom(const AtomTile64& T, int t) {
    Atom64 A;
    A.x = T.x[t];
    A.y = T.y[t];
    A.z = T.z[t];
    A.cls = T.cls[t];
    A.dx = T.dx[t];
    A.dy = T.dy[t];
    A.dz = T.dz[t];
    A.qk = T.q[t];
    A.sig = T.sig[t];
    A.se = T.se[t];
    A.idx = T.idx[t];
    return A;
}

// The displaced-state pairs: every (displaced atom i, undisplaced atom j) within the
// cutoff at x or at x+d, evaluated once in FP64 at both geometries (delta_pair); every sum
// has one owner and a fixed order (no atomics).  A wave takes eight displaced atoms of each
// ligand block, one of DISP_WAVES groups, and the 64 slots of candidate block c, a cluster
// of 8 slots at a time (lane 8 q + k: displaced atom k, slot q of the cluster):
//   An FP32 screen (at x and at x+d, with a margin that covers FP32 rounding) finds the
//   clusters with a pair in range.
//   u and F1-F0 on the displaced atoms are summed in the lane over the clusters and then
//   over the eight lanes of an atom; one partial per candidate block (dA), added in block
//   order by k_deltaA_red.
//   F1-F0 on the slots is summed over the eight displaced atoms at each step, and lane
//   8 q + k keeps it for cluster k; one part per wave (dB, env_force).
// Excluded pairs are left out: exclusions with a displaced atom of another class (or of an
// undisplaced atom with a displaced one: a bond from the ligand to the receptor) are rare, so
// only atoms that have one (ex_cross) search their list per pair.
//
// What bounds it is the chain of loads and of up to 8 steps of FP64 pairs of one wave (a few
// blocks near the displaced atoms hold most pairs) and, with many replicas, FP64 issue.  With
// lanes = slots and lanes = displaced atoms in turn, each lane walking its list of partners,
// every pair was evaluated twice and most lanes waited for the longest list: as a part of
// k_forces it added 58 us to 22 x 22,750 atoms, so 26 us.
constexpr float DSCREEN_MARGIN = 1e-3f;  // nm; FP32 position rounding is below 1e-6 nm
constexpr int DISP_WAVES = 8;            // groups of eight displaced atoms of a ligand block
// candidate blocks of a replica that have waves of their own; further ones take turns
constexpr int DISP_BLOCKS = 64;

// the slots of one wave's candidate block
struct EnvTile {
    double x[64], y[64], z[64], q[64], sig[64], se[64];
    int idx[64];
};

// F1-F0 on slot `lane` of candidate block cb (r * maxc + c): its waves' parts in order
__device__ __forceinline__ double4 env_force(const double4* __restrict__ dB, int parts, size_t cb,
                                             int lane) {
    const double4* p = dB + cb * parts * 64 + lane;
    double4 t = p[0];
    for (int w = 1; w < parts; w++) {
        const double4 q = p[64 * w];
        t.x += q.x;
        t.y += q.y;
        t.z += q.z;
    }
    return t;
}

//   w: replica, then candidate block and group, of which a wave takes `subs` in turn; waves:
//   those of one replica; E: LDS.
//   COUNT: adds the pairs within the cutoff at x+d to pair_count instead.
template <bool COUNT>
__device__ __forceinline__ void displaced_wave(
    int w, int waves, int subs, int lane, EnvTile& E, int R, int N, int Np, int L, int LB,
    const int* __restrict__ lig, const int* __restrict__ lb_start,
    const int* __restrict__ lb_count, const int* __restrict__ cls,
    const double* __restrict__ cdispl, const double* __restrict__ q64,
    const double* __restrict__ sig64, const double* __restrict__ eps64,
    const int* __restrict__ ex_start, const int* __restrict__ ex_list, const int* __restrict__ ex_cross,
    const double* __restrict__ x64, const int* __restrict__ orig_s,
    const int* __restrict__ cand, const int* __restrict__ ncand, int maxc,
    double4* __restrict__ dA, double4* __restrict__ dB,
    unsigned long long* __restrict__ pair_count, const Geom& g) {
    const int r = w / waves;
    if (r >= R) return;
    const int nc = ncand[r], parts = DISP_WAVES / subs, sub0 = (w - r * waves) % parts * subs;
    const int kk = lane & 7, q = lane >> 3;
    const double* X = x64 + (size_t)r * 3 * Np;
    const float rs = (float)sqrt(g.rc2) + DSCREEN_MARGIN, rs2 = rs * rs;
    for (int c = (w - r * waves) / parts; c < nc; c += waves / parts) {
        const size_t cb = (size_t)r * maxc + c;
        const int s = cand[cb] * 64 + lane;
        const bool v = s < N;
        const int b = v ? orig_s[(size_t)r * Np + s] : 0;
        const bool env = v && cls[b] == 0;
        lds_order();  // the previous block's atoms have been read
        E.x[lane] = X[b];
        E.y[lane] = X[Np + b];
        E.z[lane] = X[2 * Np + b];
        E.q[lane] = q64[b];
        E.sig[lane] = sig64[b];
        E.se[lane] = sqrt(eps64[b]);
        E.idx[lane] = b;
        const unsigned long long envm = __ballot(env);
        const unsigned long long exm =
            __ballot(env && ex_cross[b] != 0);
        lds_order();
        // the groups' sums are added in order here as in env_force, so that results do not
        // depend on how many of them a wave takes
        double tx = 0.0, ty = 0.0, tz = 0.0;
        for (int sub = sub0; sub < sub0 + subs; sub++) {
            double fx = 0.0, fy = 0.0, fz = 0.0;  // on slot 8 kk + q
            for (int lb = 0; lb < LB; lb++) {
                const int base = lb_start[lb], n = lb_count[lb], k = 8 * sub + kk;
                if (8 * sub >= n) continue;  // uniform
                const Atom64 I = load_atom64(X, Np, lig[base + min(k, n - 1)], cls, cdispl, q64, sig64,
                                             eps64);
                const float ix = (float)I.x, iy = (float)I.y, iz = (float)I.z;
                const float jx = (float)(I.x + I.dx), jy = (float)(I.y + I.dy),
                            jz = (float)(I.z + I.dz);
                double gx = 0.0, gy = 0.0, gz = 0.0, du = 0.0;
                int cnt = 0;
                for (int jc = 0; jc < 8; jc++) {
                    if (((envm >> (8 * jc)) & 0xffull) == 0ull) continue;  // uniform
                    const int t = 8 * jc + q;
                    Atom64 J;
                    J.x = E.x[t];
                    J.y = E.y[t];
                    J.z = E.z[t];
                    const float x = (float)J.x, y = (float)J.y, z = (float)J.z;
                    float dx = x - ix, dy = y - iy, dz = z - iz;
                    dx -= g.bx * rintf(dx * g.ibx);
                    dy -= g.by * rintf(dy * g.iby);
                    dz -= g.bz * rintf(dz * g.ibz);
                    float ex = x - jx, ey = y - jy, ez = z - jz;
                    ex -= g.bx * rintf(ex * g.ibx);
                    ey -= g.by * rintf(ey * g.iby);
                    ez -= g.bz * rintf(ez * g.ibz);
                    bool in = k < n && ((envm >> t) & 1ull) &&
                              (dx * dx + dy * dy + dz * dz < rs2 || ex * ex + ey * ey + ez * ez < rs2);
                    if (((exm >> t) & 1ull) && in) in = !excluded(ex_start, ex_list, E.idx[t], I.idx);
                    if (__ballot(in) == 0ull) continue;  // uniform
                    double px = 0.0, py = 0.0, pz = 0.0;
                    if (in) {
                        J.dx = J.dy = J.dz = -0.0;  // x + -0.0 is x
                        J.qk = E.q[t];
                        J.sig = E.sig[t];
                        J.se = E.se[t];
                        int iny;
                        du += delta_pair(I, J, g, px, py, pz, &iny);
                        cnt += iny;
                    }
                    gx += px;
                    gy += py;
                    gz += pz;
                    if (COUNT) continue;
                    px = sum8(px);
                    py = sum8(py);
                    pz = sum8(pz);
                    const bool keep = kk == jc;
                    fx -= keep ? px : 0.0;
                    fy -= keep ? py : 0.0;
                    fz -= keep ? pz : 0.0;
                }
                if (COUNT) {
                    const double sc = wave_sum((double)cnt);
                    if (lane == 0 && sc > 0.0) atomicAdd(&pair_count[r], (unsigned long long)(sc + 0.5));
                    continue;
                }
    #pragma unroll
                for (int o = 8; o < 64; o <<= 1) {
                    gx += __shfl_xor(gx, o, 64);
                    gy += __shfl_xor(gy, o, 64);
                    gz += __shfl_xor(gz, o, 64);
                    du += __shfl_xor(du, o, 64);
                }
                if (q == 0 && k < n) dA[(cb * LB + lb) * 64 + k] = make_double4(gx, gy, gz, du);
            }
            tx = sub == sub0 ? fx : tx + fx;
            ty = sub == sub0 ? fy : ty + fy;
            tz = sub == sub0 ? fz : tz + fz;
        }
        if (!COUNT)
            dB[(cb * parts + sub0 / subs) * 64 + 8 * kk + q] = make_double4(tx, ty, tz, 0.0);
    }
}

// The forces of one evaluation in one launch: workgroups of one wave (WPW, by tuning) take
// first the displaced-state pairs (the longest chain of dependent loads), then the FP64 pair
// energies where they are asked for, the pairs, and the bonded terms (short waves that wait
// for memory, which fill the slots that the last pairs leave: 22 x 22,750 atoms, 10 steps
// 6.03 ms so, 6.12 ms with them in front).  The parts need the slot records, tile lists and
// candidates only and write to different places (or by integer atomics), so they run side by
// side without the streams and events that separate launches would take: a dependency
// between queues costs 4 to 12 us, and a step had five of them.  Each count is a multiple
// of 8 workgroups, so that every part spreads over the XCDs alike.  Measured, separate
// launches on three streams against this: 10 steps of 150 atoms without a box 0.89 -> 0.43 ms,
// 20 steps of 22,750 atoms 2.24 -> 1.95 ms; 22 replicas of them, 10 steps, 6.14 -> 6.03 ms.
//   COUNT: pairs within the cutoff (pair_count) and displaced-state pairs (pair_count + R).
struct ForceGroups {
    int displaced, energy, pairs;  // workgroups of each part; the rest are the bonded terms'
    int displaced_waves;           // waves per replica, and groups of displaced atoms per wave
    int displaced_subs;
};

template <int WPW, bool COUNT, bool GEO>
__global__ __launch_bounds__(64 * WPW) __attribute__((amdgpu_waves_per_eu(4))) void k_forces(
    ForceGroups fg, int R, int N, int Np, int NB, int maxj, int waves, int parts, int packed,
    const float4* __restrict__ arec, const int* __restrict__ tiles,
    const unsigned long long* __restrict__ tmask, const int2* __restrict__ bounds,
    const float4* __restrict__ bb_lo, const float4* __restrict__ bb_hi,
    const int* __restrict__ exs, const unsigned long long* __restrict__ exblocks, int max_ex,
    long long* __restrict__ F, int* __restrict__ flags,
    unsigned long long* __restrict__ pair_count, int ewaves, const int2* __restrict__ ebounds,
    const Rec64* __restrict__ rec, double* __restrict__ e64, int nbw,
    const int* __restrict__ bstart, const int* __restrict__ bcode,
    const int* __restrict__ astart, const int* __restrict__ acode,
    const int* __restrict__ bond_atoms, const double* __restrict__ bond_r0,
    const double* __restrict__ bond_k, const int* __restrict__ ang_atoms,
    const double* __restrict__ ang_t0, const double* __restrict__ ang_k,
    const double* __restrict__ x64, double* __restrict__ Fb, double* __restrict__ e_bond,
    int L, int LB, const int* __restrict__ lig, const int* __restrict__ lb_start,
    const int* __restrict__ lb_count, const int* __restrict__ cls,
    const double* __restrict__ cdispl, const double* __restrict__ q64,
    const double* __restrict__ sig64, const double* __restrict__ eps64,
    const int* __restrict__ ex_start, const int* __restrict__ ex_list, const int* __restrict__ ex_cross,
    const int* __restrict__ orig_s, const int* __restrict__ cand,
    const int* __restrict__ ncand, int maxc, double4* __restrict__ dA,
    double4* __restrict__ dB, Geom g) {
    // one wave's LDS: the pairs' two tiles, or the energies' records, or the displaced atoms
    constexpr int LDS16 = 2 * 64 * sizeof(Rec64) / 16;
    static_assert(LDS16 >= 256 && 16 * LDS16 >= sizeof(EnvTile), "LDS");
    __shared__ float4 wave_s[WPW][LDS16];
    __shared__ unsigned long long em_s[WPW][64];
    __shared__ float xi_s[WPW][192];
    // wave-uniform by construction; readfirstlane lets the compiler keep everything
    // derived from it (replica, block, tile, mask) in scalar registers
    const int wv = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int lane = threadIdx.x & 63;
    int b = blockIdx.x;
    if (b < fg.displaced) {
        displaced_wave<COUNT>(b * WPW + wv, fg.displaced_waves, fg.displaced_subs, lane,
                              *(EnvTile*)wave_s[wv], R, N, Np, L, LB, lig, lb_start, lb_count, cls, cdispl, q64, sig64, eps64,
                              ex_start, ex_list, ex_cross, x64, orig_s, cand, ncand, maxc, dA, dB,
                              pair_count + R, g);
        return;
    }
    b -= fg.displaced;
    if (!COUNT && b < fg.energy) {
        Rec64* irec = (Rec64*)wave_s[wv];
        const BlockWave bw(b, WPW, wv, R * NB);
        if (bw.part < ewaves && bw.rb < R * NB)
            energy64_wave(bw.rb, bw.part, lane, irec, irec + 64, em_s[wv], R, N, Np, NB, maxj,
                          ewaves, packed, rec, tiles, tmask, ebounds, bb_lo, bb_hi, exs, exblocks,
                          max_ex, e64, g);
        return;
    }
    b -= fg.energy;
    if (b < fg.pairs) {
        const BlockWave bw(b, WPW, wv, R * NB);
        if (bw.part < waves && bw.rb < R * NB)
            pair_wave<COUNT, GEO>(bw.rb, part_of(bw.part, waves, parts),
                                  part_of(bw.part + 1, waves, parts), lane, wave_s[wv],
                                  em_s[wv], xi_s[wv], R, N, Np, NB, maxj, packed, arec, tiles, tmask, bounds, bb_lo,
                                  bb_hi, exs, exblocks, max_ex, F, flags, pair_count, g);
        return;
    }
    b -= fg.pairs;
    if (!COUNT)
        bonded_wave(b * WPW + wv, lane, R, N, Np, nbw, bstart, bcode, astart, acode, bond_atoms,
                    bond_r0, bond_k, ang_atoms, ang_t0, ang_k, x64, Fb, e_bond, flags);
}

// The FP64 pair energies alone, beside the forces on another stream, for long launches: in
// k_forces they have its 4 waves per SIMD, here 6, and other waves to run with.
__global__ __launch_bounds__(64) void k_energy64(
    int R, int N, int Np, int NB, int maxj, int waves, int packed, const Rec64* __restrict__ rec,
    const int* __restrict__ tiles, const unsigned long long* __restrict__ tmask,
    const int2* __restrict__ bounds, const float4* __restrict__ bb_lo,
    const float4* __restrict__ bb_hi, const int* __restrict__ exs,
    const unsigned long long* __restrict__ exblocks, int max_ex, double* __restrict__ e_out,
    Geom g) {
    __shared__ Rec64 irec[64], jrec[64];
    __shared__ unsigned long long em_s[64];
    const BlockWave bw(blockIdx.x, 1, 0, R * NB);
    if (bw.part < waves && bw.rb < R * NB)
        energy64_wave(bw.rb, bw.part, threadIdx.x, irec, jrec, em_s, R, N, Np, NB, maxj, waves,
                      packed, rec, tiles, tmask, bounds, bb_lo, bb_hi, exs, exblocks, max_ex, e_out, g);
}

// per displaced atom of ligand block lb: the block partials of displaced_wave, plus pairs with
// displaced atoms of a different class (D x D); writes dlig and returns the ligand block's u
// (in the first wave).  A workgroup of RW waves.
template <int RW>
__device__ __forceinline__ double delta_sums(
    int lb, int r, int Np, int L, int LB, int ncls, const int* __restrict__ lig,
    const int* __restrict__ lb_start, const int* __restrict__ lb_count,
    const int* __restrict__ cls, const double* __restrict__ cdispl,
    const double* __restrict__ q64, const double* __restrict__ sig64,
    const double* __restrict__ eps64, const int* __restrict__ ex_start,
    const int* __restrict__ ex_list, const int* __restrict__ ex_cross, const double* __restrict__ x64,
    const int* __restrict__ ncand, int maxc, const double4* __restrict__ dA,
    double4* __restrict__ dlig, const Geom& g, unsigned long long* __restrict__ pair_count) {
    // RW waves: wave w adds the partials of blocks w, w + RW, .. and the D x D pairs of
    // displaced atoms w, w + RW, ..; the waves' sums are added in wave order
    const int lane = threadIdx.x & 63, wv = threadIdx.x >> 6;
    const double* X = x64 + (size_t)r * 3 * Np;
    int li = lb_start[lb] + lane;
    bool v = lane < lb_count[lb];
    Atom64 I = load_atom64(X, Np, v ? lig[li] : lig[lb_start[lb]], cls, cdispl, q64, sig64, eps64);
    double du = 0.0, fx = 0.0, fy = 0.0, fz = 0.0;
    const int nc = ncand[r];
#pragma unroll 4
    for (int c = wv; c < nc; c += RW) {
        double4 p = dA[(((size_t)r * maxc + c) * LB + lb) * 64 + lane];
        fx += p.x;
        fy += p.y;
        fz += p.z;
        du += p.w;
    }
    __shared__ AtomTile64 T;
    __shared__ double4 part[RW][64];
    int cnt = 0;
    if (ncls > 1) {  // uniform
        const bool exI = v && ex_cross[I.idx] != 0;
        for (int base = 0; base < L; base += 64) {
            int n = min(64, L - base);
            // (the list is in order of classes, and a ligand block is of one class)
            const int own = cls[lig[lb_start[lb]]];
            if (cls[lig[base]] == own && cls[lig[base + n - 1]] == own) continue;  // uniform
            __syncthreads();  // the previous chunk has been read
            if ((int)threadIdx.x < n)
                stage_atom(T, threadIdx.x, load_atom64(X, Np, lig[base + threadIdx.x], cls, cdispl, q64,
                                                       sig64, eps64));
            __syncthreads();
            for (int k = wv; k < n; k += RW) {
                Atom64 J = tile_atom(T, k);
                if (!v || J.cls == I.cls) continue;
                if (exI && excluded(ex_start, ex_list, I.idx, J.idx)) continue;
                int iny;
                du += 0.5 * delta_pair(I, J, g, fx, fy, fz, &iny);
                cnt += (iny && I.idx < J.idx) ? 1 : 0;
            }
        }
    }
    if (pair_count) {
        double s = wave_sum((double)cnt);
        if (lane == 0) atomicAdd(&pair_count[r], (unsigned long long)(s + 0.5));
        return 0.0;
    }
    part[wv][lane] = make_double4(fx, fy, fz, du);
    __syncthreads();
    if (wv != 0) return 0.0;
    double4 t = part[0][lane];
    for (int w = 1; w < RW; w++) {
        t.x += part[w][lane].x;
        t.y += part[w][lane].y;
        t.z += part[w][lane].z;
        t.w += part[w][lane].w;
    }
    if (v) dlig[(size_t)r * L + li] = t;
    return wave_sum(v ? t.w : 0.0);
}

// the sums of one ligand block (and, with pair_count, only the count of its pairs)
template <int RW>
__global__ __launch_bounds__(64 * RW) void k_deltaA_red(
    int Np, int L, int LB, int ncls, const int* __restrict__ lig, const int* __restrict__ lb_start,
    const int* __restrict__ lb_count, const int* __restrict__ cls,
    const double* __restrict__ cdispl, const double* __restrict__ q64,
    const double* __restrict__ sig64, const double* __restrict__ eps64,
    const int* __restrict__ ex_start, const int* __restrict__ ex_list, const int* __restrict__ ex_cross,
    const double* __restrict__ x64, const int* __restrict__ ncand, int maxc,
    const double4* __restrict__ dA, double4* __restrict__ dlig, double* __restrict__ u_part,
    Geom g, unsigned long long* __restrict__ pair_count) {
    const double u = delta_sums<RW>(blockIdx.x, blockIdx.y, Np, L, LB, ncls, lig, lb_start, lb_count, cls,
                                    cdispl, q64, sig64, eps64, ex_start, ex_list, ex_cross, x64, ncand,
                                    maxc, dA, dlig, g, pair_count);
    if (threadIdx.x == 0 && !pair_count) u_part[(size_t)blockIdx.y * LB + blockIdx.x] = u;
}
constexpr int DRED_WAVES = 16;
// ligand blocks whose sums k_scalar takes itself; more of them get workgroups of their own (the
// figures are at k_scalar)
constexpr int DRED_FUSED = 1;

// ---------------------------------------------------------------------------
// scalar stage (one workgroup per replica): energies, SoftCoreF, bias, sp, schedule.
// Restates ReferenceSDMKernels.cpp:202-309 and LangevinIntegratorSDM.cpp:125-149.
// ---------------------------------------------------------------------------
__device__ double softcore_dev(int method, double u, double umax, double a, double ub,
                               double* fp) {
    if (u <= ub || method == 0) {
        *fp = 1.0;
        return u;
    }
    if (method == 1) {
        double t = tanh((u - ub) / umax);
        *fp = 1.0 - t * t;
        return umax * t + ub;
    }
    double gu = (u - ub) / (a * (umax - ub));
    double zeta = 1.0 + 2.0 * gu * (gu + 1.0);
    double zetap = pow(zeta, a);
    double s = 4.0 * (2.0 * gu + 1.0) / zeta;
    *fp = s * zetap / ((1.0 + zetap) * (1.0 + zetap));
    return (umax - ub) * (zetap - 1.0) / (zetap + 1.0) + ub;
}

// ne: pair-energy slots per replica (one per part of an i-block's tiles)
// SUMS: first the sums on the displaced atoms (delta_sums), with one ligand block: a launch of
// its own for them took 7.2 us of 22,750 atoms and 10 us of 22 replicas before this one's 9.9
// and 7.5 us; together, and with the state and the Langevin parameters off the last thread's
// chain of loads and divisions, 9.3 and 12.7 us.  Two ligand blocks one after the other took
// 36 us of 8 x 99,920 atoms, in workgroups of their own 13.5 us and 8 us here.
template <bool SUMS>
__global__ __launch_bounds__(64 * DRED_WAVES) void k_scalar(
    int ne, int nbw, int LB, const double* __restrict__ e_pair,
    const double* __restrict__ e_bond, const double* __restrict__ u_part,
    DevState* __restrict__ state, DevRecord* __restrict__ rec, int* __restrict__ flags,
    int advance, int energy, int hist_every, int hist_cap, double* __restrict__ uhist,
    const double* __restrict__ e_rest, int nrest, const double* __restrict__ e_t1,
    const double* __restrict__ e_t2, int ntb, float* __restrict__ dmax, int Np, int L, int ncls,
    const int* __restrict__ lig, const int* __restrict__ lb_start,
    const int* __restrict__ lb_count, const int* __restrict__ cls,
    const double* __restrict__ cdispl, const double* __restrict__ q64,
    const double* __restrict__ sig64, const double* __restrict__ eps64,
    const int* __restrict__ ex_start, const int* __restrict__ ex_list, const int* __restrict__ ex_cross,
    const double* __restrict__ x64, const int* __restrict__ ncand, int maxc,
    const double4* __restrict__ dA, double4* __restrict__ dlig, Geom g) {
    constexpr int T = 64 * DRED_WAVES;
    __shared__ double red[2][DRED_WAVES];
    __shared__ DevState S;  // in flight with the sums
    int r = blockIdx.x, t = threadIdx.x;
    constexpr int words = sizeof(DevState) / 4;
    static_assert(sizeof(DevState) % 4 == 0 && words <= 192, "DevState");
    if (t >= 64 && t < 64 + words) ((int*)&S)[t - 64] = ((const int*)&state[r])[t - 64];
    const double old_U0 = t == 0 ? rec[r].U0 : 0.0;
    // the displacement record of kept tile lists restarts with the next slot refresh:
    // this evaluation's k_tiles has read it and kept or rebuilt the lists (after a sort,
    // rebuilt), and the next refresh measures the displacement since that build again
    if (t == 0) dmax[(size_t)r * DISP_STRIDE] = 0.f;
    double s0 = 0.0, s1 = 0.0;
    if (energy)
        for (int k = t; k < ne; k += T) s0 += e_pair[(size_t)r * ne + k];
    for (int k = t; k < nbw; k += T) s1 += e_bond[(size_t)r * nbw + k];
    s0 = wave_sum(s0);
    s1 = wave_sum(s1);
    if ((t & 63) == 0) {
        red[0][t >> 6] = s0;
        red[1][t >> 6] = s1;
    }
    double u = 0.0;
    if constexpr (SUMS) {
        for (int lb = 0; lb < LB; lb++) {
            u += delta_sums<DRED_WAVES>(lb, r, Np, L, LB, ncls, lig, lb_start, lb_count, cls, cdispl, q64,
                                        sig64, eps64, ex_start, ex_list, ex_cross, x64, ncand, maxc, dA,
                                        dlig, g, nullptr);
            __syncthreads();  // its LDS is used again
        }
    }
    __syncthreads();
    if (t == 64) {
        // Langevin parameters (OpenCLSDMKernels.cpp:331-355; equal to
        // ReferenceStochasticDynamicsSDM.cpp:144-148 for friction > 0)
        const double vscale = exp(-S.step_size * S.friction);
        rec[r].vscale = vscale;
        rec[r].fscale = (S.friction == 0.0) ? S.step_size : (1.0 - vscale) / S.friction;
        rec[r].noisescale = sqrt(SDM_BOLTZ * S.temperature * (1.0 - vscale * vscale));
        rec[r].dt = S.step_size;
    }
    if (t != 0) return;
    double U0 = 0.0, Ub = 0.0;
    for (int w = 0; w < DRED_WAVES; w++) {
        U0 += red[0][w];
        Ub += red[1][w];
    }
    // energy == 0: the pair energies were left out; U0, U1 and pot_energy keep the values of
    // the last evaluation that had them (nothing else depends on U0)
    if (!energy) U0 = old_U0;
    for (int k = 0; k < nrest; k++) Ub += e_rest[(size_t)r * nrest + k];  // restraints
    for (int k = 0; k < ntb; k++) {  // further force-field terms: groups 1 and 2
        Ub += e_t1[(size_t)r * ntb + k];
        if (energy) U0 += e_t2[(size_t)r * ntb + k];
    }
    if constexpr (!SUMS)
        for (int k = 0; k < LB; k++) u += u_part[(size_t)r * LB + k];
    DevRecord& Rr = rec[r];
    // nonequilibrium schedule (ReferenceSDMKernels.cpp:221-245)
    double stepSize = S.step_size;
    double lambdac = S.lambda, dlambdac = 0.0, gamma = 0.0, wbcoeff = lambdac, w0coeff = 0.0;
    double lambda1 = lambdac, lambda2 = lambdac, alpha = 1.0, u0 = 0.0;
    double alpha_now = S.alpha;  // alpha of this step (scheduled while switching)
    if (S.nonequilibrium == 1) {
        lambdac = S.time / S.noneq_tmax;
        S.lambda = lambdac;
        S.lambda1 = S.m_l1 * lambdac + S.b_l1;
        S.lambda2 = S.m_l2 * lambdac + S.b_l2;
        S.u0 = S.m_u0 * lambdac + S.b_u0;
        S.w0coeff = S.m_w0 * lambdac + S.b_w0;
        dlambdac = stepSize / S.noneq_tmax;
        alpha_now = S.alpha + S.m_alpha * lambdac;
    }
    int method = S.bias_method;
    if (method == 1) {
        gamma = S.gamma;
        wbcoeff = S.wbcoeff;
        w0coeff = S.w0coeff;
    } else if (method == 2) {
        lambda1 = S.lambda1;
        lambda2 = S.lambda2;
        alpha = alpha_now;
        u0 = S.u0;
        w0coeff = S.w0coeff;
    }
    double fp;
    double be = softcore_dev(S.softcore_method, u, S.umax, S.acore, S.ubcore, &fp);
    double ebias, bfp;
    if (method == 1) {
        ebias = 0.5 * gamma * be * be + wbcoeff * be + w0coeff;
        bfp = gamma * be + wbcoeff;
    } else if (method == 2) {
        double z = -alpha * (be - u0);  // ee = 1 + e^z
        ebias = (alpha > 0) ? ((lambda2 - lambda1) / alpha) * softplus(z) : 0.0;
        ebias += lambda2 * be + w0coeff;
        bfp = (lambda2 - lambda1) * inv_one_plus_exp(z) + lambda1;
    } else {
        ebias = lambdac * be;
        bfp = lambdac;
    }
    if (S.nonequilibrium == 1) {
        double z = -alpha * (be - u0);
        double lee = softplus(z);
        double dwdl1 = -lee / alpha;
        double dwdl2 = be + lee / alpha;
        double dwdu0 = (lambda2 - lambda1) * (1.0 - inv_one_plus_exp(z));
        // dW/dalpha of the ILogistic bias: -(l2-l1) ln(1+e^z)/alpha^2 - (u'-u0) dW/du0/alpha
        double dwdalpha = (alpha > 0) ? -(lambda2 - lambda1) * lee / (alpha * alpha) -
                                            (be - u0) * dwdu0 / alpha
                                      : 0.0;
        double dwdlambda = dwdl1 * S.m_l1 + dwdl2 * S.m_l2 + dwdu0 * S.m_u0 + 1.0 * S.m_w0 +
                           dwdalpha * S.m_alpha;
        S.work += dlambdac * dwdlambda;
    }
    double sp = bfp * fp;
    double pot = U0 + ebias + Ub;
    int fl = 0;
    if (!isfinite(u) || !isfinite(be) || !isfinite(sp)) fl |= 1;
    if (energy && (!isfinite(U0) || !isfinite(pot))) fl |= 1;
    if (fl) atomicOr(&flags[r], fl);
    if (energy) {
        Rr.U0 = U0;
        Rr.U1 = U0 + u;
        Rr.pot_energy = pot;
    }
    Rr.u = u;
    Rr.Ub = Ub;
    Rr.bind_e = be;
    Rr.fp = fp;
    Rr.W = ebias;
    Rr.Wp = bfp;
    Rr.sp = sp;
    Rr.lambda = lambdac;
    Rr.lambda1 = (method == 2) ? lambda1 : S.lambda1;
    Rr.lambda2 = (method == 2) ? lambda2 : S.lambda2;
    Rr.u0 = (method == 2) ? u0 : S.u0;
    Rr.w0 = S.w0coeff;
    Rr.work = S.work;
    Rr.noise_step = S.step;
    if (hist_every > 0 && advance && (S.step % hist_every) == 0) {
        uhist[(size_t)r * hist_cap + (size_t)(S.hist_n % hist_cap)] = be;
        S.hist_n += 1;
    }
    if (advance) {
        S.time += stepSize;
        S.step += 1;
    }
    Rr.time = S.time;
    Rr.step = S.step;
    Rr.flags = flags[r];
    state[r] = S;
}

// F += sp (F1 - F0): candidate-block atoms from dB, displaced atoms from dlig (the
// accumulator is in slot order).
__global__ __launch_bounds__(64) void k_mix(int N, int Np, int L, int maxc,
                                            const int* __restrict__ lig, const int* __restrict__ cls,
                                            const int* __restrict__ orig_s,
                                            const int* __restrict__ cand, const int* __restrict__ ncand,
                                            int parts, const double4* __restrict__ dB,
                                            const double4* __restrict__ dlig,
                                            const DevRecord* __restrict__ rec,
                                            const int* __restrict__ slot_of,
                                            long long* __restrict__ F, int* __restrict__ flags) {
    int r = blockIdx.y, lane = threadIdx.x;
    double sp = rec[r].sp;
    long long* Fr = F + (size_t)r * 3 * Np;
    const int* S = slot_of + (size_t)r * Np;
    int bad = 0;
    if ((int)blockIdx.x < maxc) {
        int c = blockIdx.x;
        if (c >= ncand[r]) return;
        int s = cand[(size_t)r * maxc + c] * 64 + lane;
        if (s >= N) return;
        int b = orig_s[(size_t)r * Np + s];
        if (cls[b] != 0) return;
        const double4 d = env_force(dB, parts, (size_t)r * maxc + c, lane);
        Fr[s] += to_fixed(sp * d.x, &bad);
        Fr[Np + s] += to_fixed(sp * d.y, &bad);
        Fr[2 * Np + s] += to_fixed(sp * d.z, &bad);
    } else {
        int li = (blockIdx.x - maxc) * 64 + lane;
        if (li >= L) return;
        int a = S[lig[li]];
        double4 d = dlig[(size_t)r * L + li];
        Fr[a] += to_fixed(sp * d.x, &bad);
        Fr[Np + a] += to_fixed(sp * d.y, &bad);
        Fr[2 * Np + a] += to_fixed(sp * d.z, &bad);
    }
    if (bad) atomicOr(&flags[r], 2);
}

// leapfrog Langevin (langevin.cl:7-69, double-precision branch).  The force is the
// fixed-point accumulator (slot order) plus, when there are bonded terms, their FP64
// forces Fb (atom order).  Atoms with a constraint (cflag) leave their displacement
// dt*v in dxs for k_constrain.
// MixGather: k_mix's work done here instead, per atom (one launch fewer per step): the
// displaced-state force sp * dF of atom i, from the ligand sums (lig_of: the atom's
// ligand index, -1 for environment atoms) or from its block's environment sums (cmap:
// block -> candidate index of this step, -1 for none), added to the accumulator as k_mix
// adds it, so the accumulator holds the same bits afterwards.
struct MixGather {
    const int* lig_of;
    const int* cmap;
    const double4* dB;
    const double4* dlig;
    int NB, maxc, L, parts;
};

//   langevin_atom: atom i in slot `slot`; x: its new position (unless it is constrained).
// KEEP: the accumulator keeps the forces with the displaced-state part.
template <bool KEEP>
__device__ __forceinline__ void langevin_atom(
    int r, int i, int slot, int Np, const double* __restrict__ invm, long long* __restrict__ F,
    const double* __restrict__ Fb, double* __restrict__ x64, double* __restrict__ v64,
    const DevRecord* __restrict__ rec, const DevState* __restrict__ state,
    const int* __restrict__ cflag, double* __restrict__ dxs, const MixGather& mg,
    int* __restrict__ flags, double (&x)[3]) {
    // everything that is read is asked for first, and the noise computed meanwhile: a thread's
    // time is its chain of loads and FP64 logarithms, square roots and sines (22,750 atoms 9.0 ->
    // 6.9 us)
    const DevRecord& Rr = rec[r];
    const double im = invm[i];
    const bool con = cflag && cflag[i];
    long long* Fr = F + (size_t)r * 3 * Np;
    double* X = x64 + (size_t)r * 3 * Np;
    double* V = v64 + (size_t)r * 3 * Np;
    long long fi[3];
    double fb[3], v[3];
#pragma unroll
    for (int d = 0; d < 3; d++) {
        x[d] = X[d * Np + i];
        v[d] = V[d * Np + i];
        fb[d] = Fb ? Fb[((size_t)r * 3 + d) * Np + i] : 0.0;
        fi[d] = Fr[d * Np + slot];
    }
    int li = -1, cb = -1;
    if (mg.lig_of) {
        li = mg.lig_of[i];
        const int env = mg.cmap[(size_t)r * mg.NB + (slot >> 6)];
        cb = li >= 0 ? 0 : env;
    }
    double gz[3];
    gauss3(state[r].seed, (uint32_t)r, (uint64_t)Rr.noise_step, (uint32_t)i, gz);
    if (cb >= 0) {  // the displaced-state forces, into the accumulator too
        const double4 d = li >= 0 ? mg.dlig[(size_t)r * mg.L + li]
                                  : env_force(mg.dB, mg.parts, (size_t)r * mg.maxc + cb, slot & 63);
        const double sp = Rr.sp;
        int bad = 0;
        fi[0] += to_fixed(sp * d.x, &bad);
        fi[1] += to_fixed(sp * d.y, &bad);
        fi[2] += to_fixed(sp * d.z, &bad);
        if (KEEP)
#pragma unroll
            for (int k = 0; k < 3; k++) Fr[k * Np + slot] = fi[k];
        if (bad) atomicOr(&flags[r], 2);
    }
    if (im == 0.0) return;
    double vscale = Rr.vscale, fscale = Rr.fscale, noise = Rr.noisescale, dt = Rr.dt;
    double sim = sqrt(im);
    double inv = 1.0 / dt;
#pragma unroll
    for (int d = 0; d < 3; d++) {
// (products and sums written out: both kernels that this is part of have to round alike)
#pragma clang fp contract(off)
        double f = from_fixed(fi[d]);
        if (Fb) f += fb[d];
        const double vel = fma(noise * sim, gz[d], fma(fscale * im, f, vscale * v[d]));
        const double delta = dt * vel;
        if (con) {
            dxs[(size_t)r * 3 * Np + d * Np + i] = delta;
        } else {
            x[d] += delta;
            X[d * Np + i] = x[d];
            V[d * Np + i] = inv * delta;
        }
    }
}

__global__ __launch_bounds__(256) void k_langevin(
    int N, int Np, const double* __restrict__ invm, long long* __restrict__ F,
    const double* __restrict__ Fb, double* __restrict__ x64, double* __restrict__ v64,
    const DevRecord* __restrict__ rec, const DevState* __restrict__ state,
    const int* __restrict__ slot_of, const int* __restrict__ cflag, double* __restrict__ dxs,
    MixGather mg, int* __restrict__ flags) {
    const int r = blockIdx.y, i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= N) return;
    double x[3];
    langevin_atom<true>(r, i, slot_of[(size_t)r * Np + i], Np, invm, F, Fb, x64, v64, rec, state,
                        cflag, dxs, mg, flags, x);
}

// The Langevin update and, for a next step in the same order, that step's slot records
// (k_refresh<false>): one wave per block of 64 slots moves its atoms and has their new
// positions at hand.  Two launches, one in atom order and one that gathers the positions
// again, against this: 22,750 atoms 6.8 + 5.1 -> 9.0 us, 152 atoms 6.0 + 3.3 -> 7.4 us (10
// steps 367 -> 355 us).
__global__ __launch_bounds__(64) void k_move(
    int N, int Np, int NB, const double* __restrict__ invm, long long* __restrict__ F,
    const double* __restrict__ Fb, double* __restrict__ x64, double* __restrict__ v64,
    const DevRecord* __restrict__ rec, const DevState* __restrict__ state,
    const int* __restrict__ orig_s, MixGather mg, int* __restrict__ flags,
    const float* __restrict__ qs, Geom g, float4* __restrict__ arec, float4* __restrict__ bb_lo,
    float4* __restrict__ bb_hi, float4* __restrict__ cbox, const double4* __restrict__ par64,
    Rec64* __restrict__ rec64, const float4* __restrict__ xb, float* __restrict__ dmax,
    const int* __restrict__ bfirst) {
    const int r = blockIdx.y, b = blockIdx.x, lane = threadIdx.x, sl = b * 64 + lane;
    const bool v = sl < N;
    const int i = orig_s[(size_t)r * Np + (v ? sl : b * 64)];
    const int f = bfirst[(size_t)r * NB + b];  // one of the block's atoms
    double x[3] = {0.0, 0.0, 0.0};
    if (v)
        langevin_atom<false>(r, i, sl, Np, invm, F, Fb, x64, v64, rec, state, nullptr, nullptr, mg,
                             flags, x);
    const int q = __builtin_ctzll(__ballot(v && i == f));
    const double rx = __shfl(x[0], q, 64), ry = __shfl(x[1], q, 64), rz = __shfl(x[2], q, 64);
    refresh_block<false>(r, b, lane, i, v, x[0], x[1], x[2], rx, ry, rz, N, Np, NB, qs, nullptr,
                         nullptr, g, arec, F, bb_lo, bb_hi, cbox, par64, rec64, xb, dmax, nullptr,
                         nullptr, nullptr, 0, nullptr, nullptr);
}

// Virtual sites (massless atoms placed from others; the reference's integrator places
// them after every step, ReferenceStochasticDynamicsSDM.cpp:264, from the definitions the
// DMS reader makes, desmonddmsfile75.py _addVirtualSitesToSystem).  Site k: at[k] = (site,
// p1, p2, p3), weights w[3k..3k+2]:
//   VSITE_AVERAGE2:      x = w0 x1 + w1 x2
//   VSITE_AVERAGE3:      x = w0 x1 + w1 x2 + w2 x3
//   VSITE_OUT_OF_PLANE:  x = x1 + w0 r12 + w1 r13 + w2 (r12 x r13),  r1k = xk - x1
// (coordinates as stored, without periodic images, as OpenMM 7 places them).
constexpr int VSITE_AVERAGE2 = 0, VSITE_AVERAGE3 = 1, VSITE_OUT_OF_PLANE = 2;

__device__ __forceinline__ void vsite_cross(const double a[3], const double b[3], double o[3]) {
    o[0] = a[1] * b[2] - a[2] * b[1];
    o[1] = a[2] * b[0] - a[0] * b[2];
    o[2] = a[0] * b[1] - a[1] * b[0];
}

// before the Langevin update: each site's force (fixed-point accumulator plus the FP64
// bonded forces) moves to its parents by the transpose of the site's Jacobian, through
// fixed-point atomics (parents are never sites, so no site's own entry is written by
// another thread); the site's entries are left at zero.  Out of plane: a parent k's share
// is w f plus w2 times the cross-product term's derivative (r13 x f for p2, f x r12 for p3),
// and p1 takes the rest, so the three shares sum to f.
__global__ __launch_bounds__(256) void k_vsite_forces(int nvs, int Np,
                                                      const int* __restrict__ kind,
                                                      const int4* __restrict__ at,
                                                      const double* __restrict__ w,
                                                      const double* __restrict__ x64,
                                                      const int* __restrict__ slot_of,
                                                      long long* __restrict__ F,
                                                      double* __restrict__ Fb,
                                                      int* __restrict__ flags) {
    const int k = blockIdx.x * blockDim.x + threadIdx.x, r = blockIdx.y;
    if (k >= nvs) return;
    const int4 a = at[k];
    const int K = kind[k];
    const double w0 = w[3 * k], w1 = w[3 * k + 1], w2 = w[3 * k + 2];
    long long* Fr = F + (size_t)r * 3 * Np;
    double* Fbr = Fb ? Fb + (size_t)r * 3 * Np : nullptr;
    const int* S = slot_of + (size_t)r * Np;
    const double* X = x64 + (size_t)r * 3 * Np;
    const int ss = S[a.x];
    double f[3];
#pragma unroll
    for (int d = 0; d < 3; d++) {
        f[d] = from_fixed(Fr[d * Np + ss]);
        Fr[d * Np + ss] = 0;
        if (Fbr) {
            f[d] += Fbr[d * Np + a.x];
            Fbr[d * Np + a.x] = 0.0;
        }
    }
    double g1[3], g2[3], g3[3];
    if (K == VSITE_OUT_OF_PLANE) {
        double r12[3], r13[3], c2[3], c3[3];
#pragma unroll
        for (int d = 0; d < 3; d++) {
            r12[d] = X[d * Np + a.z] - X[d * Np + a.y];
            r13[d] = X[d * Np + a.w] - X[d * Np + a.y];
        }
        vsite_cross(r13, f, c2);
        vsite_cross(f, r12, c3);
#pragma unroll
        for (int d = 0; d < 3; d++) {
            g2[d] = w0 * f[d] + w2 * c2[d];
            g3[d] = w1 * f[d] + w2 * c3[d];
            g1[d] = f[d] - g2[d] - g3[d];
        }
    } else {
#pragma unroll
        for (int d = 0; d < 3; d++) {
            g1[d] = w0 * f[d];
            g2[d] = w1 * f[d];
            g3[d] = K == VSITE_AVERAGE3 ? w2 * f[d] : 0.0;
        }
    }
    int bad = 0;
    const int s1 = S[a.y], s2 = S[a.z];
#pragma unroll
    for (int d = 0; d < 3; d++) {
        atomicAdd(reinterpret_cast<unsigned long long*>(&Fr[d * Np + s1]),
                  (unsigned long long)to_fixed(g1[d], &bad));
        atomicAdd(reinterpret_cast<unsigned long long*>(&Fr[d * Np + s2]),
                  (unsigned long long)to_fixed(g2[d], &bad));
    }
    if (K != VSITE_AVERAGE2) {
        const int s3 = S[a.w];
#pragma unroll
        for (int d = 0; d < 3; d++)
            atomicAdd(reinterpret_cast<unsigned long long*>(&Fr[d * Np + s3]),
                      (unsigned long long)to_fixed(g3[d], &bad));
    }
    if (bad) atomicOr(&flags[r], 2);
}

// after the update and the constraints: the sites' positions from their parents'
__global__ __launch_bounds__(256) void k_vsite_pos(int nvs, int Np, const int* __restrict__ kind,
                                                   const int4* __restrict__ at,
                                                   const double* __restrict__ w,
                                                   double* __restrict__ x64) {
    const int k = blockIdx.x * blockDim.x + threadIdx.x, r = blockIdx.y;
    if (k >= nvs) return;
    const int4 a = at[k];
    const int K = kind[k];
    const double w0 = w[3 * k], w1 = w[3 * k + 1], w2 = w[3 * k + 2];
    double* X = x64 + (size_t)r * 3 * Np;
    double p1[3], p2[3], p3[3] = {0.0, 0.0, 0.0}, o[3];
#pragma unroll
    for (int d = 0; d < 3; d++) {
        p1[d] = X[d * Np + a.y];
        p2[d] = X[d * Np + a.z];
        if (K != VSITE_AVERAGE2) p3[d] = X[d * Np + a.w];
    }
    if (K == VSITE_OUT_OF_PLANE) {
        double r12[3], r13[3], c[3];
#pragma unroll
        for (int d = 0; d < 3; d++) {
            r12[d] = p2[d] - p1[d];
            r13[d] = p3[d] - p1[d];
        }
        vsite_cross(r12, r13, c);
#pragma unroll
        for (int d = 0; d < 3; d++) o[d] = p1[d] + w0 * r12[d] + w1 * r13[d] + w2 * c[d];
    } else {
#pragma unroll
        for (int d = 0; d < 3; d++)
            o[d] = w0 * p1[d] + w1 * p2[d] + (K == VSITE_AVERAGE3 ? w2 * p3[d] : 0.0);
    }
#pragma unroll
    for (int d = 0; d < 3; d++) X[d * Np + a.x] = o[d];
}

// centre-of-mass motion removal (one workgroup per replica) on steps whose index (the
// step count before the step, as OpenMM's CMMotionRemover tests it in the
// updateContextState call that starts the step, LangevinIntegratorSDM.cpp:158) is a
// multiple of `every`: v -= sum(m v) / sum(m) for every atom with mass.  Launched after
// the scalar stage has advanced the count, so the step's index is state.step - 1.
__global__ __launch_bounds__(1024) void k_cm_remove(int N, int Np, int every,
                                                    const double* __restrict__ mass,
                                                    double* __restrict__ v64,
                                                    const DevState* __restrict__ state) {
    __shared__ double red[4][1024];
    int r = blockIdx.x, t = threadIdx.x;
    if ((state[r].step - 1) % every != 0) return;  // uniform over the workgroup
    double* V = v64 + (size_t)r * 3 * Np;
    double p[4] = {0.0, 0.0, 0.0, 0.0};
    for (int i = t; i < N; i += 1024) {
        double m = mass[i];
        p[0] += m * V[i];
        p[1] += m * V[Np + i];
        p[2] += m * V[2 * Np + i];
        p[3] += m;
    }
    for (int d = 0; d < 4; d++) red[d][t] = p[d];
    __syncthreads();
    for (int o = 512; o > 0; o >>= 1) {
        if (t < o)
            for (int d = 0; d < 4; d++) red[d][t] += red[d][t + o];
        __syncthreads();
    }
    double im = red[3][0] > 0.0 ? 1.0 / red[3][0] : 0.0;
    double cx = red[0][0] * im, cy = red[1][0] * im, cz = red[2][0] * im;
    for (int i = t; i < N; i += 1024) {
        if (mass[i] == 0.0) continue;
        V[i] -= cx;
        V[Np + i] -= cy;
        V[2 * Np + i] -= cz;
    }
}

// Position constraints of the Langevin step: SHAKE on one cluster of constrained atoms
// per thread (Ryckaert, Ciccotti, Berendsen, J. Comput. Phys. 23, 327 (1977)): each
// constraint in turn moves its two atoms along their bond vector before the step, in
// inverse proportion to their masses, until every |r_ij|^2 is within tol of d_ij^2.
// Then x = x', v = (x' - x)/dt.  Sets flag 8 if a cluster does not converge.
//
// What bounds it is the chain of constraints of one cluster (each needs the positions the
// one before left), a few dozen FP64 divisions long.  A rigid three-site molecule
// (constraints 0-1, 0-2, 1-2) is worked on in registers; other clusters keep their atoms in
// LDS ([atom][value][lane], no bank conflicts), since arrays indexed by the constraint
// lists would lie in scratch memory.  990 rigid waters: 67 us with the arrays in scratch and
// 256 threads per workgroup, 9 us so.
constexpr int SHAKE_MAX_ATOMS = 16, SHAKE_MAX_CONS = 32, SHAKE_MAX_ITER = 500;
constexpr int SHAKE_LDS = 7 * 64 * sizeof(double);  // bytes of LDS per atom of the largest cluster

// one constraint: moves atoms i and j along ro, their separation before the step; returns
// whether it was within the tolerance
__device__ __forceinline__ bool shake(const double (&ro)[3], double (&xi)[3], double (&xj)[3],
                                      double mi, double mj, double d2, double tol) {
    double rn[3];
#pragma unroll
    for (int d = 0; d < 3; d++) rn[d] = xi[d] - xj[d];
    const double diff = d2 - dot3(rn, rn);
    const double g = diff / (2.0 * (mi + mj) * dot3(ro, rn));
#pragma unroll
    for (int d = 0; d < 3; d++) {
        xi[d] += g * mi * ro[d];
        xj[d] -= g * mj * ro[d];
    }
    return !(fabs(diff) > tol * d2);
}

__global__ __launch_bounds__(64) void k_constrain(
    int Np, int ncl, const int* __restrict__ cl_start, const int* __restrict__ cl_atoms,
    const int* __restrict__ con_start, const int* __restrict__ con_ij,
    const double* __restrict__ con_d2, double tol, const double* __restrict__ invm,
    const double* __restrict__ dxs, double* __restrict__ x64, double* __restrict__ v64,
    const DevRecord* __restrict__ rec, int* __restrict__ flags) {
    extern __shared__ double atoms_s[];  // atom k, value f of lane: [(7 k + f) * 64 + lane]
    const int r = blockIdx.y, lane = threadIdx.x, q = blockIdx.x * 64 + lane;
    if (q >= ncl) return;
    double* X = x64 + (size_t)r * 3 * Np;
    double* V = v64 + (size_t)r * 3 * Np;
    const double* D = dxs + (size_t)r * 3 * Np;
    const int a0 = cl_start[q], na = cl_start[q + 1] - a0;
    const int c0 = con_start[q], nc = con_start[q + 1] - c0;
    const int* ij = con_ij + 2 * c0;
    const double inv = 1.0 / rec[r].dt;
    bool done = false;
    if (na == 3 && nc == 3 && ij[0] == 0 && ij[1] == 1 && ij[2] == 0 && ij[3] == 2 && ij[4] == 1 &&
        ij[5] == 2) {
        double xo[3][3], xn[3][3], im[3], ro[3][3];
        int a[3];
#pragma unroll
        for (int k = 0; k < 3; k++) {
            a[k] = cl_atoms[a0 + k];
            im[k] = invm[a[k]];
#pragma unroll
            for (int d = 0; d < 3; d++) {
                xo[k][d] = X[d * Np + a[k]];
                xn[k][d] = xo[k][d] + D[d * Np + a[k]];
            }
        }
#pragma unroll
        for (int d = 0; d < 3; d++) {
            ro[0][d] = xo[0][d] - xo[1][d];
            ro[1][d] = xo[0][d] - xo[2][d];
            ro[2][d] = xo[1][d] - xo[2][d];
        }
        const double d01 = con_d2[c0], d02 = con_d2[c0 + 1], d12 = con_d2[c0 + 2];
        for (int it = 0; it < SHAKE_MAX_ITER && !done; it++) {
            done = shake(ro[0], xn[0], xn[1], im[0], im[1], d01, tol);
            done &= shake(ro[1], xn[0], xn[2], im[0], im[2], d02, tol);
            done &= shake(ro[2], xn[1], xn[2], im[1], im[2], d12, tol);
        }
#pragma unroll
        for (int k = 0; k < 3; k++)
#pragma unroll
            for (int d = 0; d < 3; d++) {
                V[d * Np + a[k]] = inv * (xn[k][d] - xo[k][d]);
                X[d * Np + a[k]] = xn[k][d];
            }
    } else {
        // values 0-2: position before the step, 3-5: new position, 6: inverse mass
        auto at = [&](int k, int f) -> double& { return atoms_s[(7 * k + f) * 64 + lane]; };
        for (int k = 0; k < na; k++) {
            const int a = cl_atoms[a0 + k];
            for (int d = 0; d < 3; d++) {
                const double x = X[d * Np + a];
                at(k, d) = x;
                at(k, 3 + d) = x + D[d * Np + a];
            }
            at(k, 6) = invm[a];
        }
        for (int it = 0; it < SHAKE_MAX_ITER && !done; it++) {
            done = true;
            for (int k = 0; k < nc; k++) {
                const int i = ij[2 * k], j = ij[2 * k + 1];
                double ro[3], xi[3], xj[3];
#pragma unroll
                for (int d = 0; d < 3; d++) {
                    ro[d] = at(i, d) - at(j, d);
                    xi[d] = at(i, 3 + d);
                    xj[d] = at(j, 3 + d);
                }
                done &= shake(ro, xi, xj, at(i, 6), at(j, 6), con_d2[c0 + k], tol);
#pragma unroll
                for (int d = 0; d < 3; d++) {
                    at(i, 3 + d) = xi[d];
                    at(j, 3 + d) = xj[d];
                }
            }
        }
        for (int k = 0; k < na; k++) {
            const int a = cl_atoms[a0 + k];
            for (int d = 0; d < 3; d++) {
                const double x = at(k, 3 + d);
                V[d * Np + a] = inv * (x - at(k, d));
                X[d * Np + a] = x;
            }
        }
    }
    if (!done) atomicOr(&flags[r], 8);
}

// Kinetic energy 0.5 sum m v^2 of every replica (one workgroup per replica), with the
// velocities of constrained atoms first projected onto the constraints, as
// ReferenceSDMKernels.cpp:108-135 does (applyToVelocities on a copy; the stored
// velocities are not changed): per cluster, each constraint in turn removes the relative
// velocity of its two atoms along their current bond vector in inverse proportion to
// their masses (momentum is conserved), repeated until |r . dv| <= tol |r| (|v_i|+|v_j|)
// for every constraint.  The converged result is the mass-weighted projection onto
// r_c . (v_i - v_j) = 0, whatever solver reaches it.  Unconstrained atoms (cflag 0, or no
// clusters) are summed as they are.  Sets flag 8 if a cluster does not converge.
constexpr int KE_MAX_ITER = 500;
__global__ __launch_bounds__(256) void k_kinetic(
    int N, int Np, const double* __restrict__ mass, const double* __restrict__ invm,
    const double* __restrict__ x64, const double* __restrict__ v64, int ncl,
    const int* __restrict__ cl_start, const int* __restrict__ cl_atoms,
    const int* __restrict__ con_start, const int* __restrict__ con_ij,
    const int* __restrict__ cflag, double tol, int* __restrict__ flags,
    double* __restrict__ out) {
    __shared__ double red[256];
    int r = blockIdx.x, t = threadIdx.x;
    const double* V = v64 + (size_t)r * 3 * Np;
    const double* X = x64 + (size_t)r * 3 * Np;
    double e = 0.0;
    for (int i = t; i < N; i += 256) {
        double m = mass[i];
        if (m > 0 && !(ncl > 0 && cflag[i]))
            e += m * (V[i] * V[i] + V[Np + i] * V[Np + i] + V[2 * Np + i] * V[2 * Np + i]);
    }
    bool bad = false;
    for (int q = t; q < ncl; q += 256) {
        int a0 = cl_start[q], na = cl_start[q + 1] - a0;
        int c0 = con_start[q], nc = con_start[q + 1] - c0;
        double xv[SHAKE_MAX_ATOMS][3], vv[SHAKE_MAX_ATOMS][3], im[SHAKE_MAX_ATOMS];
        for (int k = 0; k < na; k++) {
            int a = cl_atoms[a0 + k];
            im[k] = invm[a];
            for (int d = 0; d < 3; d++) {
                xv[k][d] = X[d * Np + a];
                vv[k][d] = V[d * Np + a];
            }
        }
        bool done = false;
        for (int it = 0; it < KE_MAX_ITER && !done; it++) {
            done = true;
            for (int k = 0; k < nc; k++) {
                int i = con_ij[2 * (c0 + k)], j = con_ij[2 * (c0 + k) + 1];
                double rr[3], dv[3];
                for (int d = 0; d < 3; d++) {
                    rr[d] = xv[i][d] - xv[j][d];
                    dv[d] = vv[i][d] - vv[j][d];
                }
                double r2 = dot3(rr, rr), rv = dot3(rr, dv);
                double vs = sqrt(dot3(vv[i], vv[i])) + sqrt(dot3(vv[j], vv[j]));
                if (fabs(rv) > tol * sqrt(r2) * vs) done = false;
                double g = rv / (r2 * (im[i] + im[j]));
                for (int d = 0; d < 3; d++) {
                    vv[i][d] -= g * im[i] * rr[d];
                    vv[j][d] += g * im[j] * rr[d];
                }
            }
        }
        bad = bad || !done;
        for (int k = 0; k < na; k++) {
            double m = mass[cl_atoms[a0 + k]];
            e += m * dot3(vv[k], vv[k]);
        }
    }
    if (bad) atomicOr(&flags[r], 8);
    red[t] = e;
    __syncthreads();
    for (int o = 128; o > 0; o >>= 1) {
        if (t < o) red[t] += red[t + o];
        __syncthreads();
    }
    if (t == 0) out[r] = 0.5 * red[0];
}

// ---------------------------------------------------------------------------
// adjoint (parameter gradients of u over many frames).  Frames are [F][N][3] doubles in
// atom order; pair terms are recomputed from the positions, never stored.
//
// k_adj: one workgroup per (256 atoms of a frame, frame, 64 selected atoms).  Its atoms
// within reach of a displaced class (its box at x or at x+d, FP64, any image) are listed in
// LDS with their parameters, in atom order; then lanes = selected atoms and the listed
// atoms are taken one after the other (LDS broadcasts), so every selected atom's sums have
// one owner and no cross-lane reduction: the parts of the list that the workgroup's waves
// (or, for 32 selected atoms or fewer, parts of waves) take are added in order.  One partial
// per workgroup goes to the context's buffer and k_adj_u / k_adj_grad add the frame's
// partials in order: bit-reproducible, whatever number of frames fits the buffer.
//   GRAD = false: u (selected = the displaced atoms; pairs of two displaced atoms once).
//   GRAD = true: du/d(q, sigma, eps) of the selected atoms that are displaced.
// What bounds it: FP64 issue on the listed pairs.  One workgroup per frame over all (displaced
// atom, atom) pairs with an integer division each left 3/4 of the GPU idle and took 8.1 ms
// for u and 0.60 ms for the gradient (a wave per selected atom and frame over all atoms) for
// 64 frames of 22,750 atoms with 50 displaced; 481 and 80 us for 3,000 atoms with 30.
// ---------------------------------------------------------------------------
__device__ __forceinline__ void load_frame_atom(const double* __restrict__ X, int a, double& x,
                                                double& y, double& z) {
    x = X[3 * a];
    y = X[3 * a + 1];
    z = X[3 * a + 2];
}

constexpr int ADJ_ATOMS = 256;  // atoms (and threads) per workgroup
constexpr int ADJ_SEL = 64;     // selected atoms per workgroup
constexpr int ADJ_PART = 3 * ADJ_SEL;  // doubles of a workgroup's gradient partial

// what the two geometries of one pair (I displaced by I.d, J by J.d) add to the sums
struct AdjSums {
    double u, q, s, e;
};

template <bool GRAD>
__device__ __forceinline__ void adj_pair(const Atom64& I, const Atom64& J, const Geom& g, AdjSums& a) {
    double ex = min_image(I.x - J.x, g.Lx, g.iLx), ey = min_image(I.y - J.y, g.Ly, g.iLy),
           ez = min_image(I.z - J.z, g.Lz, g.iLz);
    const double r0 = ex * ex + ey * ey + ez * ez;
    ex = min_image((I.x + I.dx) - (J.x + J.dx), g.Lx, g.iLx);
    ey = min_image((I.y + I.dy) - (J.y + J.dy), g.Ly, g.iLy);
    ez = min_image((I.z + I.dz) - (J.z + J.dz), g.Lz, g.iLz);
    const double r1 = ex * ex + ey * ey + ez * ez;
    if (!(r0 < g.rc2) && !(r1 < g.rc2)) return;
    const double sig = g.geo ? sqrt(I.sig * J.sig) : 0.5 * (I.sig + J.sig);
    const double sig2 = sig * sig;
    double c = 0.0, A = 0.0, B = 0.0;  // sums over the geometries, x with sign -
#pragma unroll
    for (int t = 0; t < 2; t++) {
        const double r2 = t ? r1 : r0, sgn = t ? 1.0 : -1.0;
        if (r2 < g.rc2) {
            const double ir = rsqrt(r2);
            const double s2 = sig2 * (ir * ir);
            const double s6 = s2 * s2 * s2;
            c += sgn * (ir + g.krf * r2 - g.crf);
            B += sgn * (s6 * (s6 - 1.0));
            if (GRAD) A += sgn * (s6 * (12.0 * s6 - 6.0));
        }
    }
    if (GRAD) {
        a.q += J.qk * c;
        a.e += J.se * B;
        // d sigma_ij / d sigma_i / sigma_ij: 1 / (2 sigma_ij), or 1 / (2 sigma_i) for the
        // geometric rule (the terms vanish with sigma_ij = 0)
        if (sig > 0.0) a.s += J.se * A / (g.geo ? I.sig : sig);
    } else {
        a.u += 4.0 * I.se * J.se * B + I.qk * J.qk * c;
    }
}

template <bool GRAD>
__global__ __launch_bounds__(ADJ_ATOMS) void k_adj(
    int N, int L, int ncls, const int* __restrict__ sel, int nsel, const int* __restrict__ lig,
    const int* __restrict__ cls, const double* __restrict__ cdispl,
    const double* __restrict__ q64, const double* __restrict__ sig64,
    const double* __restrict__ eps64, const int* __restrict__ ex_start,
    const int* __restrict__ ex_list, const double* __restrict__ frames, int tile0,
    double* __restrict__ part, Geom g) {
    constexpr int NW = ADJ_ATOMS / 64;
    __shared__ double box[SDM_MAX_CLASSES][6];  // per class: centre and half extent
    __shared__ double jx[ADJ_ATOMS], jy[ADJ_ATOMS], jz[ADJ_ATOMS], jq[ADJ_ATOMS], js[ADJ_ATOMS],
        je[ADJ_ATOMS];
    __shared__ int jc[ADJ_ATOMS], ji[ADJ_ATOMS];
    __shared__ double red[GRAD ? 3 : 1][ADJ_ATOMS];
    __shared__ int wcount[NW];
    const int t = threadIdx.x, lane = t & 63, wv = t >> 6;
    const int chunk = blockIdx.x, f = blockIdx.y, tile = tile0 + blockIdx.z;
    const double* X = frames + (size_t)f * 3 * N;
    for (int k = 1 + wv; k <= ncls; k += NW) {
        double v[6] = {1e300, 1e300, 1e300, -1e300, -1e300, -1e300};
        for (int li = lane; li < L; li += 64) {
            const int a = lig[li];
            if (cls[a] != k) continue;
            for (int d = 0; d < 3; d++) {
                v[d] = fmin(v[d], X[3 * a + d]);
                v[3 + d] = fmax(v[3 + d], X[3 * a + d]);
            }
        }
        for (int d = 0; d < 3; d++) {
            const double lo = wave_min_d(v[d]), hi = wave_max_d(v[3 + d]);
            if (lane == 0) {
                box[k - 1][d] = 0.5 * (lo + hi);
                box[k - 1][3 + d] = 0.5 * (hi - lo);
            }
        }
    }
    __syncthreads();
    // the chunk's atoms that can have a partner
    const int j = chunk * ADJ_ATOMS + t;
    bool near = false;
    double xj = 0.0, yj = 0.0, zj = 0.0;
    int cj = 0;
    if (j < N) {
        load_frame_atom(X, j, xj, yj, zj);
        cj = cls[j];
        const double reach = sqrt(g.rc2) + 1e-6, reach2 = reach * reach;
        const double* dj = cdispl + 3 * cj;
        for (int k = 1; k <= ncls; k++) {
            if (k == cj) continue;
            const double* dk = cdispl + 3 * k;
            const double* b = box[k - 1];
            for (int geo = 0; geo < 2; geo++) {  // at x, at x + d
                const double dx = xj - b[0] + (geo ? dj[0] - dk[0] : 0.0),
                             dy = yj - b[1] + (geo ? dj[1] - dk[1] : 0.0),
                             dz = zj - b[2] + (geo ? dj[2] - dk[2] : 0.0);
                const double gx = fmax(fabs(min_image(dx, g.Lx, g.iLx)) - b[3], 0.0),
                             gy = fmax(fabs(min_image(dy, g.Ly, g.iLy)) - b[4], 0.0),
                             gz = fmax(fabs(min_image(dz, g.Lz, g.iLz)) - b[5], 0.0);
                near = near || !(gx * gx + gy * gy + gz * gz >= reach2);
            }
        }
    }
    const unsigned long long m = __ballot(near);
    if (lane == 0) wcount[wv] = __popcll(m);
    __syncthreads();
    int n = 0, pos = lane_rank(m);
    for (int w = 0; w < NW; w++) {
        if (w < wv) pos += wcount[w];
        n += wcount[w];
    }
    if (near) {
        jx[pos] = xj;
        jy[pos] = yj;
        jz[pos] = zj;
        jq[pos] = q64[j];
        js[pos] = sig64[j];
        je[pos] = sqrt(eps64[j]);
        jc[pos] = cj;
        ji[pos] = j;
    }
    __syncthreads();
    // lanes = selected atoms; the list in 256 / W parts
    const int ns = min(ADJ_SEL, nsel - tile * ADJ_SEL);
    const int W = ns <= 16 ? 16 : ns <= 32 ? 32 : 64;
    const int k = t & (W - 1), p = t / W, parts = ADJ_ATOMS / W;
    AdjSums a{0.0, 0.0, 0.0, 0.0};
    double ise = 0.0, ses = 0.0;
    if (k < ns && n > 0) {
        const int i = sel[tile * ADJ_SEL + k];
        const int ci = cls[i];
        if (ci != 0) {
            Atom64 I;
            load_frame_atom(X, i, I.x, I.y, I.z);
            I.dx = cdispl[3 * ci];
            I.dy = cdispl[3 * ci + 1];
            I.dz = cdispl[3 * ci + 2];
            I.qk = q64[i];
            I.sig = sig64[i];
            I.se = sqrt(eps64[i]);
            const int e0 = ex_start[i], e1 = ex_start[i + 1];
            // exclusions across classes are rare: only atoms that have one search their list
            bool exI = false;
            for (int q = e0; q < e1; q++) exI = exI || cls[ex_list[q]] != ci;
            for (int e = p; e < n; e += parts) {
                const int cq = jc[e], jj = ji[e];
                if (cq == ci || (!GRAD && cq != 0 && jj < i)) continue;
                if (exI && excluded(ex_start, ex_list, i, jj)) continue;
                Atom64 J;
                J.x = jx[e];
                J.y = jy[e];
                J.z = jz[e];
                J.dx = cdispl[3 * cq];
                J.dy = cdispl[3 * cq + 1];
                J.dz = cdispl[3 * cq + 2];
                J.qk = jq[e];
                J.sig = js[e];
                J.se = je[e];
                adj_pair<GRAD>(I, J, g, a);
            }
            ses = I.se;
            ise = I.se > 0.0 ? 1.0 / I.se : 0.0;
        }
    }
    if constexpr (GRAD) {
        red[0][t] = sqrt(SDM_ONE_4PI_EPS0) * a.q;  // q64 holds q sqrt(k_e)
        red[1][t] = 2.0 * ses * a.s;
        red[2][t] = 2.0 * ise * a.e;
        __syncthreads();
        if (p == 0) {
            double* o = part + (((size_t)f * gridDim.z + blockIdx.z) * gridDim.x + chunk) * ADJ_PART;
            for (int c = 0; c < 3; c++) {
                double v = 0.0;
                for (int q = 0; q < parts; q++) v += red[c][q * W + k];
                o[c * ADJ_SEL + k] = v;
            }
        }
    } else {
        red[0][t] = a.u;
        __syncthreads();
        for (int o = ADJ_ATOMS / 2; o > 0; o >>= 1) {
            if (t < o) red[0][t] += red[0][t + o];
            __syncthreads();
        }
        if (t == 0) part[((size_t)f * gridDim.z + blockIdx.z) * gridDim.x + chunk] = red[0][0];
    }
}

// u of frame f: its np partials in order (one wave per frame, a lane's in stride 64)
__global__ __launch_bounds__(64) void k_adj_u(int np, const double* __restrict__ part,
                                              double* __restrict__ u_out) {
    const int f = blockIdx.x;
    double v = 0.0;
    for (int k = threadIdx.x; k < np; k += 64) v += part[(size_t)f * np + k];
    v = wave_sum(v);
    if (threadIdx.x == 0) u_out[f] = v;
}

// one component of the gradient of 64 selected atoms in a frame: the chunks' partials in
// four interleaved runs, added in order; atoms that are not displaced are left to k_adj_env
__global__ __launch_bounds__(256) void k_adj_grad(int nchunk, const int* __restrict__ sel, int nsel,
                                                  const int* __restrict__ cls, int tile0,
                                                  const double* __restrict__ part,
                                                  double* __restrict__ grad) {
    __shared__ double red[4][64];
    const int c = blockIdx.x, f = blockIdx.y, k = threadIdx.x & 63, p = threadIdx.x >> 6;
    const double* P = part + ((size_t)f * gridDim.z + blockIdx.z) * nchunk * ADJ_PART + c * ADJ_SEL + k;
    const int s = (tile0 + blockIdx.z) * ADJ_SEL + k;
    const bool mine = s < nsel && cls[sel[s]] != 0;
    double v = 0.0;
    if (mine)
#pragma unroll 4
        for (int q = p; q < nchunk; q += 4) v += P[(size_t)q * ADJ_PART];
    red[p][k] = v;
    __syncthreads();
    if (p == 0 && mine)
        grad[((size_t)f * nsel + s) * 3 + c] = ((red[0][k] + red[1][k]) + red[2][k]) + red[3][k];
}

// du/d(q, sigma, eps) of a selected atom that is not displaced: its partners are the
// displaced atoms.  One wave per (selected atom, frame)
__global__ __launch_bounds__(64) void k_adj_env(
    int N, int L, const int* __restrict__ sel, int nsel, const int* __restrict__ lig,
    const int* __restrict__ cls, const double* __restrict__ cdispl,
    const double* __restrict__ q64, const double* __restrict__ sig64,
    const double* __restrict__ eps64, const int* __restrict__ ex_start,
    const int* __restrict__ ex_list, const double* __restrict__ frames,
    double* __restrict__ grad, Geom g) {
    const int k = blockIdx.x, f = blockIdx.y, lane = threadIdx.x;
    const int s = sel[k];
    if (cls[s] != 0) return;
    const double* X = frames + (size_t)f * 3 * N;
    Atom64 I;
    load_frame_atom(X, s, I.x, I.y, I.z);
    I.dx = I.dy = I.dz = 0.0;
    I.qk = q64[s];
    I.sig = sig64[s];
    I.se = sqrt(eps64[s]);
    AdjSums a{0.0, 0.0, 0.0, 0.0};
    for (int li = lane; li < L; li += 64) {
        const int j = lig[li], cj = cls[j];
        if (excluded(ex_start, ex_list, s, j)) continue;
        Atom64 J;
        load_frame_atom(X, j, J.x, J.y, J.z);
        J.dx = cdispl[3 * cj];
        J.dy = cdispl[3 * cj + 1];
        J.dz = cdispl[3 * cj + 2];
        J.qk = q64[j];
        J.sig = sig64[j];
        J.se = sqrt(eps64[j]);
        adj_pair<true>(I, J, g, a);
    }
    const double dq = wave_sum(a.q), ds = wave_sum(a.s), de = wave_sum(a.e);
    if (lane == 0) {
        double* o = grad + ((size_t)f * nsel + k) * 3;
        o[0] = sqrt(SDM_ONE_4PI_EPS0) * dq;
        o[1] = 2.0 * I.se * ds;
        o[2] = I.se > 0.0 ? 2.0 / I.se * de : 0.0;
    }
}

// ---------------------------------------------------------------------------
// diagnostics: dense component forces (FP64) for sdm_compute_components.
// ---------------------------------------------------------------------------
__global__ void k_fill_ll(long long* __restrict__ p, size_t n) {
    size_t i = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i < n) p[i] = 0;
}
__global__ void k_fill_d(double* __restrict__ p, size_t n) {
    size_t i = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i < n) p[i] = 0.0;
}
__global__ void k_fill_u64(unsigned long long* __restrict__ p, size_t n) {
    size_t i = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i < n) p[i] = 0ull;
}

// dF (dense, [R][3][Np]) from dB and dlig
__global__ __launch_bounds__(64) void k_scatter_dF(int N, int Np, int L, int maxc,
                                                   const int* __restrict__ lig,
                                                   const int* __restrict__ cls,
                                                   const int* __restrict__ orig_s,
                                                   const int* __restrict__ cand,
                                                   const int* __restrict__ ncand,
                                                   int parts, const double4* __restrict__ dB,
                                                   const double4* __restrict__ dlig,
                                                   double* __restrict__ dF) {
    int r = blockIdx.y, lane = threadIdx.x;
    double* D = dF + (size_t)r * 3 * Np;
    if ((int)blockIdx.x < maxc) {
        int c = blockIdx.x;
        if (c >= ncand[r]) return;
        int s = cand[(size_t)r * maxc + c] * 64 + lane;
        if (s >= N) return;
        int b = orig_s[(size_t)r * Np + s];
        if (cls[b] != 0) return;
        const double4 d = env_force(dB, parts, (size_t)r * maxc + c, lane);
        D[b] = d.x;
        D[Np + b] = d.y;
        D[2 * Np + b] = d.z;
    } else {
        int li = (blockIdx.x - maxc) * 64 + lane;
        if (li >= L) return;
        int a = lig[li];
        double4 d = dlig[(size_t)r * L + li];
        D[a] = d.x;
        D[Np + a] = d.y;
        D[2 * Np + a] = d.z;
    }
}

// ---------------------------------------------------------------------------
// Data between the host and the device.  These read or write pinned host memory as well as
// device memory, with consecutive threads on consecutive words of it, so that no copy
// command waits between the kernels of the stream: bounded by the host link and the
// launch.  Copies of pageable memory with a wait each, against these: 22,750 atoms
// set, evaluated and their forces read 380 -> 244 us, 20 replicas of 2,976 atoms 616 -> 427
// us, a step of 186 atoms read back 132 -> 89 us.
// ---------------------------------------------------------------------------
// [R][N][3] -> [R][3][Np] and back
__global__ void k_aos_to_soa(int N, int Np, const double* __restrict__ in, double* __restrict__ out) {
    const int r = blockIdx.y, k = blockIdx.x * blockDim.x + threadIdx.x;
    if (k >= 3 * N) return;
    out[((size_t)r * 3 + k % 3) * Np + k / 3] = in[(size_t)r * 3 * N + k];
}
__global__ void k_soa_to_aos(int N, int Np, const double* __restrict__ in, double* __restrict__ out) {
    const int r = blockIdx.y, k = blockIdx.x * blockDim.x + threadIdx.x;
    if (k >= 3 * N) return;
    out[(size_t)r * 3 * N + k] = in[((size_t)r * 3 + k % 3) * Np + k / 3];
}
// words of a and then of b
__global__ void k_words(const unsigned* __restrict__ a, size_t na, const unsigned* __restrict__ b,
                        size_t nb, unsigned* __restrict__ dst) {
    const size_t k = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (k < na) dst[k] = a[k];
    else if (k < na + nb) dst[k] = b[k - na];
}
// hybrid forces of one replica [N][3]: the fixed-point accumulator (slot order) and, where
// there are any, the bonded forces (atom order)
__global__ void k_hybrid_forces(int N, int Np, const long long* __restrict__ F,
                                const int* __restrict__ slot_of, const double* __restrict__ Fb,
                                double* __restrict__ out) {
    const int k = blockIdx.x * blockDim.x + threadIdx.x;
    if (k >= 3 * N) return;
    const int i = k / 3, d = k - 3 * i;
    out[k] = (double)F[(size_t)d * Np + slot_of[i]] / SDM_FIX_SCALE + (Fb ? Fb[(size_t)d * Np + i] : 0.0);
}
// the forms of the nonbonded parameters (charges, sigmas, epsilons: [3][N]) that the kernels read
__global__ void k_nb_params(int N, int geo, const double* __restrict__ p, float* __restrict__ qs,
                            float* __restrict__ sh, float* __restrict__ se,
                            double* __restrict__ q64, double* __restrict__ sig64,
                            double* __restrict__ eps64, double4* __restrict__ par64) {
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= N) return;
    const double q = p[i] * sqrt(SDM_ONE_4PI_EPS0), sig = p[N + i], eps = p[2 * (size_t)N + i];
    const double s = geo ? sig : 0.5 * sig, e = 2.0 * sqrt(eps);  // the entry each rule combines
    qs[i] = (float)q;
    sh[i] = (float)s;
    se[i] = (float)e;
    q64[i] = q;
    sig64[i] = sig;
    eps64[i] = eps;
    par64[i] = make_double4(q, s, e, 0.0);
}

}  // namespace sdm
