// d2bi_bin.cuh -- link-cell binning of the replica atoms: findGdotR and
// LinkCell3D add as a stable counting sort (classify, scan, scatter, scan,
// place, emit).
//
// One part of the single translation unit d2bi_gpu.hip, which includes the
// parts in order so that kernels and the device helpers they call compile
// together; each part uses the definitions of the parts before it.
#pragma once

namespace d2bi {

// ------------------------------------------------------------------ (a) binning

static constexpr int BIN_BLOCK = 256;
static constexpr int MAX_REPL = 32;

// Workgroups of the counting passes, an atom per thread: with four atoms per
// thread in turn (a quarter of the counts to scan) a 16,000-atom set had 16
// workgroups and k_bin_scatter took 43 us of latency against 14; 8.0e6 atoms
// bin in 0.65 ms either way.
static int bin_blocks(int64_t n) { return (int)std::max<int64_t>(1, (n + BIN_BLOCK - 1) / BIN_BLOCK); }

// FP64 offset of a point in its link cell, in cell units
struct Frac3 {
    double x, y, z;
};

struct BinParams {
    double RU[9];               // column-major
    double delta[3];
    double lc_delta[3];
    double ia[9];               // link-cell inverse (column-major)
    double gg[3];
    double Ruvw[3 * MAX_REPL];
    int nuvw;
    int Ex, Ey, Ez;
    int64_t n;                  // atoms
    int generic;                // 1: LinkCell3D add1 (no transform, no filter)
    int fast;                   // FAST imaging: phases in FP32 beside the positions, else FP64
    int keep_src;               // also keep each slot's atom and replica (aperture phases)
    int keep_ids;               // link-cell API: point numbers (and g.r if not generic), no phases
    double cell_a[3];           // diagonal of the link-cell matrix (FP32 positions)
    // replica pre-classification: c ~= M x + off[nn] approximates the
    // link-cell coordinates of replica nn (products folded, so a few
    // roundings away from the reference's order); a replica is decided
    // from it unless a coordinate lies within eps of a box face
    int prefilter;
    double M[9];                // ia . RU (column-major)
    double off[3 * MAX_REPL];   // ia . (RU . Ruvw[nn] + delta - lc_delta)
    double mabs, oabs;          // magnitude bounds: per unit |x|, and the rest
};

// Link-cell index of a reduced coordinate: mod(floor(y) + 16*N, N)
// (whichCell, Lib_SimpleSupercells.f90:371-373).  For points further than
// 16 boxes away the reference's expression goes negative; here the floor is
// clamped and the modulo kept non-negative, which changes nothing for
// points within range and keeps every index inside the cell array.
__device__ inline int cell_of(double fl, int n)
{
    const double c = fmin(fmax(fl, -1.0e9), 1.0e9);
    const int r = ((int)c + 16 * n) % n;
    return r < 0 ? r + n : r;
}

// Transform atom j for replica nn: yy (rotated lab position), zz (link-cell
// frame), and whether it lies in the link-cell box.  Operation order of
// findGdotR (Lib_DynamicalTwoBeamImaging.f90:1225-1240) and pointInSupercell0
// (Lib_SimpleSupercells.f90:1077-1084).
__device__ inline bool bin_point(const BinParams& P, const double* x3, int nn, double yy[3],
                                 double cyy[3])
{
    if (P.generic) {
        yy[0] = x3[0]; yy[1] = x3[1]; yy[2] = x3[2];
        for (int i = 0; i < 3; i++)
            cyy[i] = (P.ia[i] * yy[0] + P.ia[3 + i] * yy[1]) + P.ia[6 + i] * yy[2];
        return true;
    }
    double y0[3], zz[3];
    for (int i = 0; i < 3; i++) y0[i] = x3[i] + P.Ruvw[3 * nn + i];
    for (int i = 0; i < 3; i++) yy[i] = (P.RU[i] * y0[0] + P.RU[3 + i] * y0[1]) + P.RU[6 + i] * y0[2];
    for (int i = 0; i < 3; i++) {
        yy[i] = yy[i] + P.delta[i];
        zz[i] = yy[i] - P.lc_delta[i];
    }
    for (int i = 0; i < 3; i++)
        cyy[i] = (P.ia[i] * zz[0] + P.ia[3 + i] * zz[1]) + P.ia[6 + i] * zz[2];
    // |floor| beyond 2^30 cannot be inside the box; clamping keeps int conversion defined
    int ix = (int)fmin(fmax(floor(cyy[0]), -1.0e9), 1.0e9);
    int iy = (int)fmin(fmax(floor(cyy[1]), -1.0e9), 1.0e9);
    int iz = (int)fmin(fmax(floor(cyy[2]), -1.0e9), 1.0e9);
    bool is = (ix == (ix + 256 * P.Ex) % P.Ex);
    is = is && (iy == (iy + 256 * P.Ey) % P.Ey);
    is = is && (iz == (iz + 256 * P.Ez) % P.Ez);
    return is;
}

// Replica bits set in any lane of the wave (wave-uniform).
__device__ __forceinline__ uint32_t wave_or(uint32_t m)
{
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) m |= (uint32_t)__shfl_xor((int)m, o, 64);
    return __builtin_amdgcn_readfirstlane(m);
}

// Pass 1: replica predicate bits per atom and per-(replica, block) counts.  It
// also clears what the later passes count into (Z): a launch less.
__global__ __launch_bounds__(BIN_BLOCK) void k_bin_classify(const double* __restrict__ x, BinParams P,
                                                            uint32_t* __restrict__ mask,
                                                            int* __restrict__ blk_cnt, int nblk, ZeroRanges Z)
{
    __shared__ int cnt[MAX_REPL];
    zero_share(Z);
    if (threadIdx.x < MAX_REPL) cnt[threadIdx.x] = 0;
    __syncthreads();
    const int lane = threadIdx.x & 63;
    const int64_t j = (int64_t)blockIdx.x * BIN_BLOCK + threadIdx.x;
    uint32_t m = 0;
    if (j < P.n) {
        double x3[3] = {x[3 * j], x[3 * j + 1], x[3 * j + 2]};
        if (P.prefilter) {
            double cb[3];
            for (int i = 0; i < 3; i++) cb[i] = P.M[i] * x3[0] + P.M[3 + i] * x3[1] + P.M[6 + i] * x3[2];
            // |approximate - exact| is a few units of roundoff (1e-16) of
            // the magnitudes involved; eps is 1e-10 of their bound
            const double eps = 1.0e-10 * (1.0 + P.mabs * (fabs(x3[0]) + fabs(x3[1]) + fabs(x3[2])) + P.oabs);
            // c in [0, E) per axis is |c - E/2| < E/2: certainly outside
            // when |c - E/2| >= E/2 + eps, certainly inside when <= E/2 - eps
            const double h[3] = {0.5 * P.Ex, 0.5 * P.Ey, 0.5 * P.Ez};
            double ch[3], hout[3], hin[3];
            for (int i = 0; i < 3; i++) {
                ch[i] = cb[i] - h[i];
                hout[i] = h[i] + eps;
                hin[i] = h[i] - eps;
            }
            for (int nn = 0; nn < P.nuvw; nn++) {
                bool out = false, sure = true;
                for (int i = 0; i < 3; i++) {
                    const double u = fabs(ch[i] + P.off[3 * nn + i]);
                    out = out || u >= hout[i];
                    sure = sure && u <= hin[i];
                }
                if (out) continue;                       // outside on some axis for certain
                if (sure) { m |= 1u << nn; continue; }   // inside on every axis for certain
                double yy[3], cyy[3];
                if (bin_point(P, x3, nn, yy, cyy)) m |= 1u << nn;
            }
        } else {
            for (int nn = 0; nn < P.nuvw; nn++) {
                double yy[3], cyy[3];
                if (bin_point(P, x3, nn, yy, cyy)) m |= 1u << nn;
            }
        }
        mask[j] = m;
    }
    // only the replicas some lane of the wave lies in
    for (uint32_t wm = wave_or(m); wm; wm &= wm - 1) {
        const int nn = __builtin_ctz(wm);
        const unsigned long long b = __ballot((m >> nn) & 1u);
        if (lane == 0) atomicAdd(&cnt[nn], (int)__popcll(b));
    }
    __syncthreads();
    if (threadIdx.x < P.nuvw) blk_cnt[(int64_t)threadIdx.x * nblk + blockIdx.x] = cnt[threadIdx.x];
}

// Pass 2: point number ii in (replica, atom) order, link cell, atom number and
// a per-cell arrival slot from an atomic counter.
__global__ __launch_bounds__(BIN_BLOCK) void k_bin_scatter(const double* __restrict__ x, BinParams P,
                                                           const uint32_t* __restrict__ mask,
                                                           const int* __restrict__ blk_off, int nblk,
                                                           int* __restrict__ pt_cell,
                                                           int* __restrict__ pt_slot,
                                                           int* __restrict__ pt_j,
                                                           int* __restrict__ cell_cnt, PointCount N)
{
    __shared__ int first[MAX_REPL];
    __shared__ int wcnt[BIN_BLOCK / 64][MAX_REPL];
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    if (threadIdx.x < P.nuvw) first[threadIdx.x] = blk_off[(int64_t)threadIdx.x * nblk + blockIdx.x];
    const unsigned long long lt = (lane == 0) ? 0ull : (~0ull >> (64 - lane));
    const int64_t j = (int64_t)blockIdx.x * BIN_BLOCK + threadIdx.x;
    const uint32_t m = (j < P.n) ? mask[j] : 0u;
    if (N.over()) return;
    // the wave's count per replica: zero, then the replicas some lane lies in
    const uint32_t wm0 = wave_or(m);
    if (lane < P.nuvw) wcnt[wave][lane] = 0;
    for (uint32_t wm = wm0; wm; wm &= wm - 1) {
        const int nn = __builtin_ctz(wm);
        const unsigned long long b = __ballot((m >> nn) & 1u);
        if (lane == 0) wcnt[wave][nn] = (int)__popcll(b);
    }
    __syncthreads();
    if (!m) return;
    const double x3[3] = {x[3 * j], x[3 * j + 1], x[3 * j + 2]};
    for (uint32_t wm = wm0; wm; wm &= wm - 1) {
        const int nn = __builtin_ctz(wm);
        const unsigned long long b = __ballot((m >> nn) & 1u);   // uniform among lanes with m != 0
        if (!((m >> nn) & 1u)) continue;
        int off = first[nn];
        for (int w = 0; w < wave; w++) off += wcnt[w][nn];
        const int ii = off + (int)__popcll(b & lt);
        double yy[3], cyy[3];
        bin_point(P, x3, nn, yy, cyy);
        const double fl[3] = {floor(cyy[0]), floor(cyy[1]), floor(cyy[2])};
        // a replica point passed pointInSupercell, so 0 <= floor < E
        // and mod(floor + 16E, E) is the floor itself
        const int cx = P.generic ? cell_of(fl[0], P.Ex) : (int)fl[0];
        const int cy = P.generic ? cell_of(fl[1], P.Ey) : (int)fl[1];
        const int cz = P.generic ? cell_of(fl[2], P.Ez) : (int)fl[2];
        const int cell = cx + P.Ex * (cy + P.Ey * cz);
        pt_cell[ii] = cell;
        pt_j[ii] = (int)j;
        // arrival slot: lanes of this wave landing in one cell share
        // one atomic (the lowest such lane adds the group's size);
        // the grouping is ALU-only, so each lane waits for one atomic
        // return.  Order inside a cell is restored by ii later.
        unsigned long long rem = __ballot(1), grp = 0;
        int leader = lane;
        while (rem) {
            const int l = __ffsll((long long)rem) - 1;
            const int lc = __builtin_amdgcn_readlane(cell, l);
            const unsigned long long gm = __ballot(cell == lc);
            if (cell == lc) { leader = l; grp = gm; }
            rem &= ~gm;
        }
        int base = 0;
        if (lane == leader) base = atomicAdd(&cell_cnt[cell], (int)__popcll(grp));
        base = __shfl(base, leader, 64);
        pt_slot[ii] = base + (int)__popcll(grp & lt);
    }
}

// f(t) for the items t of a thread among n, workgroups of 256 in a grid of
// xcd_grid(n) or more, or (LOOP) fewer, where a thread goes on at the grid's
// stride: a contiguous range of items per XCD (workgroups go round-robin to the
// eight), so that neighbours in cell or atom order, which share lines of the
// arrays they gather from and scatter into, share one L2.  Against
// workgroups in order: k_bin_emit 39.5 -> 26.7 us and k_bin_place 9.6 -> 6.8 at
// 1.2e6 atoms, 222 -> 212 and 54 -> 46 at 8e6 (k_bin_scatter, whose atomics
// meet in memory either way, lost 7 % there and keeps its order).
template <bool LOOP, class F>
__device__ __forceinline__ void xcd_items(int64_t n, F f)
{
    const int64_t per = (n + 2047) / 2048;
    int64_t b = blockIdx.x >> 3;
    do {
        const int64_t t = ((blockIdx.x & 7) * per + b) * 256 + threadIdx.x;
        if (b < per && t < n) f(t);
        b += gridDim.x >> 3;
    } while (LOOP && b < per);
}
static unsigned xcd_grid(int64_t n) { return (unsigned)(8 * ((n + 2047) / 2048)); }

// Pass 3: place each point at its cell's start + arrival slot.
template <bool LOOP>
__global__ void k_bin_place(PointCount N, const int* __restrict__ pt_cell, const int* __restrict__ pt_slot,
                            const int* __restrict__ cell_start, int* __restrict__ cell_ids)
{
    xcd_items<LOOP>(N.stored(), [&](int64_t ii) { cell_ids[cell_start[pt_cell[ii]] + pt_slot[ii]] = (int)ii; });
}

// What pass 4 writes per slot (null: not wanted).
struct EmitOut {
    float4* p32;                // offset from the cell origin in A (cuboidal cells); FAST: cos g.r
    float* sn32;                // FAST: sin g.r
    double2* cs64;              // FP64: (cos, sin) of g.r
    Frac3* frac;                // FP64 offset in cell
    int2* src;                  // atom, replica
    int* id;                    // 1-based point number
    double* gdotr;              // g.r, by point number
};

// Pass 4, one thread per placed point: its slot is its cell's start plus the
// number of points of the cell with a smaller number, which restores the
// reference's insertion order (a cell's handful of numbers is read from cache
// by neighbouring threads; sorting each cell first, a thread per cell, took a
// launch of its own and up to 19 us where a cell holds more than 16).  The
// point is evaluated again from its atom and replica (the transform of
// k_bin_scatter, so the same cell offsets to the bit).  The replica of point
// ii is the last one whose first point number is <= ii (numbers run in
// (replica, atom) order; rep_first is padded to 32 entries with INT_MAX).
// Bound: HBM and, in imaging, FP64 sincos with full argument reduction.
template <bool FAST, bool LOOP>
__global__ __launch_bounds__(256) void k_bin_emit(PointCount N, const int* __restrict__ cell_ids,
                                                  const int* __restrict__ pt_cell, const int* __restrict__ pt_j,
                                                  const int* __restrict__ cell_start, const double* __restrict__ x,
                                                  BinParams P, const int* __restrict__ blk_off, int nblk, EmitOut O)
{
    __shared__ int rep_first[MAX_REPL];
    if (threadIdx.x < MAX_REPL)
        rep_first[threadIdx.x] = threadIdx.x < P.nuvw ? blk_off[(int64_t)threadIdx.x * nblk] : 0x7fffffff;
    __syncthreads();
    xcd_items<LOOP>(N.stored(), [&](int64_t t) {
        const int ii = cell_ids[t];
        const int64_t j = pt_j[ii];
        const int c = pt_cell[ii];
        const int s0 = cell_start[c], s1 = cell_start[c + 1];
        int nn = 0;                                       // rep_first[0] = 0 <= ii
#pragma unroll
        for (int step = MAX_REPL / 2; step > 0; step >>= 1)
            if (rep_first[nn + step] <= ii) nn += step;
        const double x3[3] = {x[3 * j], x[3 * j + 1], x[3 * j + 2]};
        int64_t s = s0;
        for (int k = s0; k < s1; k++) s += cell_ids[k] < ii ? 1 : 0;
        double yy[3], cyy[3];
        bin_point(P, x3, nn, yy, cyy);
        const Frac3 f{cyy[0] - floor(cyy[0]), cyy[1] - floor(cyy[1]), cyy[2] - floor(cyy[2])};
        const double gd = (P.gg[0] * yy[0] + P.gg[1] * yy[1]) + P.gg[2] * yy[2];
        O.frac[s] = f;
        float4 p = make_float4((float)(P.cell_a[0] * f.x), (float)(P.cell_a[1] * f.y), (float)(P.cell_a[2] * f.z), 0.0f);
        if (FAST) {
            double sn, cs;
            sincos(gd, &sn, &cs);
            p.w = (float)cs;
            O.sn32[s] = (float)sn;
        } else if (O.cs64) {
            double sn, cs;
            sincos(gd, &sn, &cs);
            O.cs64[s] = make_double2(cs, sn);
        }
        O.p32[s] = p;
        if (O.src) O.src[s] = make_int2((int)j, nn);
        if (O.id) O.id[s] = ii + 1;
        if (O.gdotr) O.gdotr[ii] = gd;
    });
}

// g-vectors of up to four aperture points (findGdotR_aperture,
// Lib_DynamicalTwoBeamImaging.f90:1269-1396: the points of a condition differ
// only in g, so they share its binned points and take their own g.r)
struct AppG {
    double g[4][3];
};

// cos and sin of g_a.r for every slot and the NA aperture points of G, the
// slot's point evaluated again from its atom and replica as k_bin_emit does,
// so the phases are those a binning at g_a would give.  F64: double2 (cos,
// sin) at out64[a stride + slot].  FAST: NA = 1 rewrites the FP32 phase of the
// slot's record in place (slot_p32.w, slot_sn32); NA > 1 writes float2 (cos,
// sin) at out32[a stride + slot].
template <bool F64, int NA>
__global__ __launch_bounds__(256) void k_app_phase(int64_t nr, const int2* __restrict__ slot_src,
                                                   const double* __restrict__ x, BinParams P, AppG G, int64_t stride,
                                                   double2* __restrict__ out64, float2* __restrict__ out32,
                                                   float4* __restrict__ slot_p32, float* __restrict__ slot_sn32)
{
    xcd_items<false>(nr, [&](int64_t s) {
        const int2 src = slot_src[s];
        const int64_t j = src.x;
        const double x3[3] = {x[3 * j], x[3 * j + 1], x[3 * j + 2]};
        double yy[3], cyy[3];
        bin_point(P, x3, src.y, yy, cyy);
#pragma unroll
        for (int a = 0; a < NA; a++) {
            const double gd = (G.g[a][0] * yy[0] + G.g[a][1] * yy[1]) + G.g[a][2] * yy[2];
            double sn, cs;
            sincos(gd, &sn, &cs);
            if (F64) {
                out64[a * stride + s] = make_double2(cs, sn);
            } else if (NA == 1) {
                reinterpret_cast<float*>(slot_p32 + s)[3] = (float)cs;
                slot_sn32[s] = (float)sn;
            } else {
                out32[a * stride + s] = make_float2((float)cs, (float)sn);
            }
        }
    });
}

struct Binned {
    int64_t nr = -1;            // points; -1: not known on the host yet
    PointCount N{};             // on the device, and what the point arrays hold
    int ncell = 0;
};

// Passes 2 to 4 on workspace w, once the points are counted on the device (*N.n
// of them, about `expect`): d_x, mask, blk_off and nblk are the condition's atoms,
// replica predicates and per-(replica, block) point offsets; w.cell_cnt is zero.
// The largest cell count goes to *mpc.
static int launch_bin_points(const double* d_x, const BinParams& P, const uint32_t* mask, const int* blk_off, int nblk,
                             int ncell, PointCount N, int64_t expect, int* scan_tmp, int* mpc, hipStream_t s, Workspace& w)
{
    if (P.n > 0 && N.cap > 0) {
        hipLaunchKernelGGL(k_bin_scatter, dim3(nblk), dim3(BIN_BLOCK), 0, s, d_x, P, mask, blk_off, nblk,
                           w.pt_cell.as<int>(), w.pt_slot.as<int>(), w.pt_j.as<int>(), w.cell_cnt.as<int>(), N);
        HIPCHK(hipGetLastError());
    }
    CHK(scan_exclusive_tmp(w.cell_cnt.as<int>(), w.cell_start.as<int>(), ncell, scan_tmp, s,
                           ScanEnds{nullptr, mpc, N}));
    if (P.n > 0 && N.cap > 0) {
        // a thread per point that the arrays hold, or, where an earlier condition
        // left them far larger, per point expected (k_bin_emit's loop costs it a
        // wave per SIMD: 213 -> 220 us at 8e6 points)
        const bool loop = N.cap > 2 * expect;
        const dim3 grid(xcd_grid(loop ? expect : N.cap));
        auto place = [&](auto kern) {
            hipLaunchKernelGGL(kern, grid, dim3(256), 0, s, N, w.pt_cell.as<int>(), w.pt_slot.as<int>(),
                               w.cell_start.as<int>(), w.cell_ids.as<int>());
        };
        if (loop) place(k_bin_place<true>);
        else place(k_bin_place<false>);
        EmitOut O{w.slot_p32.as<float4>(), w.slot_sn32.as<float>(), nullptr, w.slot_frac.as<Frac3>(),
                  P.keep_src ? w.slot_src.as<int2>() : nullptr, nullptr, nullptr};
        if (!P.fast) {
            O.sn32 = nullptr;
            if (P.keep_ids) {
                O.id = w.slot_id.as<int>();
                O.gdotr = P.generic ? nullptr : w.pt_gdotr.as<double>();
            } else {
                O.cs64 = w.slot_cs64.as<double2>();
            }
        }
        auto go = [&](auto kern) {
            hipLaunchKernelGGL(kern, grid, dim3(256), 0, s, N, w.cell_ids.as<int>(), w.pt_cell.as<int>(),
                               w.pt_j.as<int>(), w.cell_start.as<int>(), d_x, P, blk_off, nblk, O);
        };
        if (loop && P.fast) go(k_bin_emit<true, true>);
        else if (loop) go(k_bin_emit<false, true>);
        else if (P.fast) go(k_bin_emit<true, false>);
        else go(k_bin_emit<false, false>);
    }
    HIPCHK(hipGetLastError());
    return D2BI_OK;
}

// The per-point and per-slot buffers of a condition and their bytes per point.
template <class F>
static void point_buffers(Workspace& w, bool fast, bool keep_ids, bool generic, bool keep_src, F f)
{
    f(w.pt_cell, sizeof(int));
    f(w.pt_slot, sizeof(int));
    f(w.pt_j, sizeof(int));
    f(w.cell_ids, sizeof(int));
    f(w.slot_p32, sizeof(float4));
    f(w.slot_frac, sizeof(Frac3));
    if (fast) f(w.slot_sn32, sizeof(float));
    else if (!keep_ids) f(w.slot_cs64, sizeof(double2));
    if (keep_ids) f(w.slot_id, sizeof(int));
    if (keep_ids && !generic) f(w.pt_gdotr, sizeof(double));
    if (keep_src) f(w.slot_src, sizeof(int2));
}

// Points a condition is expected to have, with a margin: its atoms' density
// in the supercell times the link-cell box (at most all its replicas).
static int64_t expected_points(const d2bi_record* r, const d2bi_plan* p, int64_t n)
{
    double A[9];
    for (int j = 0; j < 3; j++)
        for (int i = 0; i < 3; i++) A[3 * j + i] = r->super_a[3 * j + i] * r->super_n[j];
    const double box = p->a_col[0] * p->Ex * (p->a_col[4] * p->Ey) * (p->a_col[8] * p->Ez), super = std::fabs(det3(A));
    const double most = (double)r->nuvw * (double)n;
    const double e = super > 0.0 ? 1.1 * (box / super) * (double)n + 4096.0 : most;
    return (int64_t)std::min(std::min(e, most), 2147483647.0);
}

// Run binning for either a condition (generic = 0) or plain points, on
// workspace w.  expect > 0: the point arrays are sized for that many points
// (or what they hold) and nothing waits for the count, which stays in the
// workspace's counters; the caller compares it with out->N.cap at its own end
// and bins again with expect = 0 if they did not fit (the kernels after the
// count have then done nothing).  expect = 0: the host waits for the count and
// sizes the arrays by it.
static int run_binning(const double* d_x, int64_t n, BinParams& P, Binned* out, hipStream_t s, Workspace& w,
                       int64_t expect = 0)
{
    const int64_t ncell64 = (int64_t)P.Ex * P.Ey * P.Ez;
    if (ncell64 > (int64_t)INT32_MAX / 2) return seterr(D2BI_ERR_CAPACITY, "too many link cells");
    const int ncell = (int)ncell64;
    const int nblk = bin_blocks(n);
    if (n > (int64_t)INT32_MAX) return seterr(D2BI_ERR_CAPACITY, "more than 2^31 - 1 atoms");
    P.n = n;
    const int64_t nbc = (int64_t)P.nuvw * nblk;
    CHK(w.mask.ensure(sizeof(uint32_t) * std::max<int64_t>(n, 1)));
    CHK(w.blk_cnt.ensure(sizeof(int) * (nbc + 1)));
    CHK(w.blk_off.ensure(sizeof(int) * (nbc + 1)));
    CHK(w.cell_cnt.ensure(sizeof(int) * (ncell + 1)));
    CHK(w.cell_start.ensure(sizeof(int) * (ncell + 1)));
    CHK(w.counters.ensure(sizeof(Counters)));
    CHK(w.scan_tmp.ensure(sizeof(int) * std::max(scan_tmp_ints(nbc), scan_tmp_ints(ncell))));
    Counters* ct = w.counters.as<Counters>();
    const ZeroRanges Z{{w.cell_cnt.as<int>(), (int*)ct}, {ncell + 1, sizeof(Counters) / sizeof(int)}};
    if (n > 0)
        hipLaunchKernelGGL(k_bin_classify, dim3(nblk), dim3(BIN_BLOCK), 0, s, d_x, P, w.mask.as<uint32_t>(),
                           w.blk_cnt.as<int>(), nblk, Z);
    else
        zero_i32(s, Z.p[0], Z.n[0], Z.p[1], Z.n[1], w.blk_cnt.as<int>(), nbc);
    HIPCHK(hipGetLastError());
    CHK(scan_exclusive_tmp(w.blk_cnt.as<int>(), w.blk_off.as<int>(), nbc, w.scan_tmp.as<int>(), s,
                           ScanEnds{&ct->n_points, nullptr, {}}));
    int64_t cap = expect;
    if (expect <= 0) {
        int nr_host = 0;
        HIPCHK(hipMemcpyAsync(&nr_host, &ct->n_points, sizeof(int), hipMemcpyDeviceToHost, s));
        HIPCHK(hipStreamSynchronize(s));
        if (nr_host < 0) return seterr(D2BI_ERR_CAPACITY, "point count overflow");
        out->nr = cap = nr_host;
    }
    int rc = D2BI_OK;
    int64_t held = INT64_MAX;
    point_buffers(w, P.fast, P.keep_ids, P.generic, P.keep_src, [&](Buf& b, size_t bytes) {
        if (rc == D2BI_OK) rc = b.ensure(bytes * std::max<int64_t>(cap, 1));
        held = std::min(held, (int64_t)(b.cap / bytes));
    });
    CHK(rc);
    out->N = PointCount{&ct->n_points, expect > 0 ? held : cap};
    CHK(launch_bin_points(d_x, P, w.mask.as<uint32_t>(), w.blk_off.as<int>(), nblk, ncell, out->N, cap,
                          w.scan_tmp.as<int>(), &ct->max_per_cell, s, w));
    out->ncell = ncell;
    return D2BI_OK;
}

// Fill the binning parameters of a condition from the plan.
static int bin_params(const d2bi_record* r, const d2bi_plan* p, BinParams* P)
{
    std::memset(P, 0, sizeof *P);
    if (r->nuvw < 1 || r->nuvw > MAX_REPL)
        return seterr(D2BI_ERR_ARG, "nuvw = %d not supported (1..%d)", r->nuvw, MAX_REPL);
    std::memcpy(P->RU, p->RU, sizeof P->RU);
    std::memcpy(P->delta, r->delta, sizeof P->delta);
    std::memcpy(P->lc_delta, p->lc_delta, sizeof P->lc_delta);
    std::memcpy(P->ia, p->ia_col, sizeof P->ia);
    std::memcpy(P->gg, p->gg, sizeof P->gg);
    for (int nn = 0; nn < r->nuvw; nn++) {
        const int* u = &r->uvw[3 * nn];
        for (int i = 0; i < 3; i++) {       // getSuperVector (Lib_SimpleSupercells.f90:904-918)
            double s1 = r->super_a[i] * r->super_n[0];
            double s2 = r->super_a[3 + i] * r->super_n[1];
            double s3 = r->super_a[6 + i] * r->super_n[2];
            P->Ruvw[3 * nn + i] = (u[0] * s1 + u[1] * s2) + u[2] * s3;
        }
    }
    P->nuvw = r->nuvw;
    P->Ex = p->Ex; P->Ey = p->Ey; P->Ez = p->Ez;
    P->generic = 0;
    P->cell_a[0] = p->a_col[0]; P->cell_a[1] = p->a_col[4]; P->cell_a[2] = p->a_col[8];
    // folded transform of the pre-classification (any rounding order: it
    // only decides replicas that are further than eps from a box face)
    double ia_max = 0.0, ru_max = 0.0, t_max = 0.0;
    for (int i = 0; i < 9; i++) {
        ia_max = std::max(ia_max, std::fabs(P->ia[i]));
        ru_max = std::max(ru_max, std::fabs(P->RU[i]));
    }
    for (int i = 0; i < 3; i++)
        for (int j = 0; j < 3; j++) {
            double v = 0.0;
            for (int k = 0; k < 3; k++) v += P->ia[3 * k + i] * P->RU[3 * j + k];
            P->M[3 * j + i] = v;
        }
    for (int nn = 0; nn < P->nuvw; nn++) {
        double z[3];
        for (int k = 0; k < 3; k++) {
            double v = P->delta[k] - P->lc_delta[k];
            double t = std::fabs(P->delta[k]) + std::fabs(P->lc_delta[k]);
            for (int j = 0; j < 3; j++) {
                v += P->RU[3 * j + k] * P->Ruvw[3 * nn + j];
                t += std::fabs(P->RU[3 * j + k] * P->Ruvw[3 * nn + j]) + std::fabs(P->Ruvw[3 * nn + j]);
            }
            z[k] = v;
            t_max = std::max(t_max, t);
        }
        for (int i = 0; i < 3; i++) {
            double v = 0.0;
            for (int k = 0; k < 3; k++) v += P->ia[3 * k + i] * z[k];
            P->off[3 * nn + i] = v;
        }
    }
    // bounds on the magnitude of every intermediate of both evaluations:
    // |x| terms scale with 3 max|ia| max(1, max|RU|), the rest with
    // 3 max|ia| (|RU Ruvw| + |Ruvw| + |delta| + |lc_delta|)
    P->mabs = 3.0 * ia_max * std::max(1.0, ru_max) * std::max(1.0, 3.0 * ru_max);
    P->oabs = 3.0 * ia_max * t_max;
    // box faces at 0 and E <= 2^20, so that E + eps and the exact path's
    // integer test are exact
    P->prefilter = (P->Ex <= (1 << 20) && P->Ey <= (1 << 20) && P->Ez <= (1 << 20)) ? 1 : 0;
    return D2BI_OK;
}

}  // namespace d2bi
