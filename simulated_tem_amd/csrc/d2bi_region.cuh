// d2bi_region.cuh -- candidate staging of the region voxel kernels: the points
// near an 8 x 8 x 8 block of voxels, listed once for the whole workgroup.
//
// One part of the single translation unit d2bi_gpu.hip, which includes the
// parts in order so that kernels and the device helpers they call compile
// together; each part uses the definitions of the parts before it.
#pragma once

namespace d2bi {

// ------------------------------------------------------------------ region staging

// A workgroup of NW waves owns a region of 8 x 8 x 8 voxels, cut into eight
// subtiles of 4 x 4 x 4.  The points that can matter to
// it (those of the link cells of the unwrapped range [cell(first voxel) - 1,
// cell(last voxel) + 1] that lie within 3 sigma of the region's box) are found
// once by all waves; each subtile then keeps those within 3 sigma of its own
// box.  For bcc at four voxels per lattice parameter an 8 x 8 x 8 region has
// ~169 candidates, a subtile ~71 (a 4 x 4 x 8 tile has ~95), against 28 inside
// 3 sigma of a voxel: smaller boxes test fewer pairs, and the region shares
// the listing, loading and culling that a tile of its own would repeat for
// every 64 voxels.
//
// An unwrapped cell u stands for cell mod(u, E) displaced by u - mod(u, E)
// cells, the periodic image neighbourList1b sees through its mod()
// (Lib_LinkCell3D.f90:1567-1575).
static constexpr int REG = 8;                        // voxels along each side of a region
static constexpr int REG_MAXC = 256;                 // link cells in a region's unwrapped range

struct RegionParams {
    VoxParams v;
    int nrx, nry, nrz;          // regions per axis
    int nreg, per_xcd;          // regions; workgroups per XCD (the grid is 8 per_xcd)
    float rc_cull2;             // (3 sigma)^2 widened for the FP32 box culls
    float cellf[3];             // link-cell sides in FP32
};

// Region of a workgroup: rows of regions along x dealt to the XCDs in turn
// (consecutive workgroups go round-robin to them), so that neighbours along a
// row, which read the same link cells, share one L2 and every XCD holds rows
// at every depth.  A region's sums do not depend on the order.
__device__ __forceinline__ int region_of(const RegionParams& R, int bid)
{
    const int idx = bid >> 3, row = (idx / R.nrx) * 8 + (bid & 7);
    return row * R.nrx + (idx - (idx / R.nrx) * R.nrx);
}

// set bits of a wave mask below this lane (v_mbcnt)
__device__ __forceinline__ int bits_below(unsigned long long m)
{
    return (int)__builtin_amdgcn_mbcnt_hi((unsigned)(m >> 32), __builtin_amdgcn_mbcnt_lo((unsigned)m, 0u));
}

// LDS writes of this wave visible to its own later reads (LDS operations of
// one wave execute in order; this keeps the compiler from moving them)
__device__ __forceinline__ void wave_sync()
{
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
}

// The region's link cells, needed while its candidates are staged.
template <int NW>
struct RegionCells {
    static_assert(64 * NW >= REG_MAXC, "a thread per link cell");
    float4 crec[REG_MAXC];      // kept cells: origin in the region frame, slot - candidate index
    int cupk[REG_MAXC];         // kept cells: dx | dy << 8 | dz << 16 from the first cell of the range
    int cstart[REG_MAXC];       // kept cells' first candidate
    int flag[NW][64];           // cells starting at a lane's candidate
};

template <int NW>
struct RegionStage {
    static constexpr int CAP = 64 * NW;     // one round of candidates always fits
    int wk[NW], wt[NW];         // kept cells and their points, per wave
    int wcnt[2][NW];            // candidates kept, per wave and parity of the round
    float4 pos[CAP];            // staged candidates: position in the region frame, slot
    int upk[CAP];               // staged candidates: their cell (as cupk)
    float q[3][REG];            // voxel positions in the region frame (clamped at the grid's edge)
    int lc[3][REG];             // voxel cells from the region's first
    double zi[3][REG];          // FP64 voxel offsets in their cells
};

// The region's frame: origin voxel, last voxel, cells from the first voxel's,
// box.  All values are the same in every thread.
struct RegionBox {
    int o[3], l[3];             // first and last voxel
    int u0[3], nc[3];           // unwrapped cell range: first cell, cells
    float cc[3], hf[3];         // centre relative to the first voxel's cell, half sides
};

// Axis tables of the region into LDS, and its box (a barrier follows in
// region_cells).  A voxel's FP32 position is rounded once from FP64, relative
// to the link cell of the region's first voxel, then centred.
template <int NW>
__device__ __forceinline__ void region_box(const RegionParams& R, int region, RegionStage<NW>& S, RegionBox& B)
{
    const VoxParams& P = R.v;
    const int r[3] = {region % R.nrx, (region / R.nrx) % R.nry, region / (R.nrx * R.nry)};
    const int M[3] = {P.Mx, P.My, P.Mz};
#pragma unroll
    for (int a = 0; a < 3; a++) {
        B.o[a] = r[a] * REG;
        B.l[a] = min(M[a], B.o[a] + REG) - 1;
        const int c0 = P.ax.cell[a][B.o[a]], c1 = P.ax.cell[a][B.l[a]];
        const float q0 = (float)(P.a[a] * P.ax.zi[a][B.o[a]]);
        const float q1 = (float)(P.a[a] * (P.ax.zi[a][B.l[a]] + (c1 - c0)));
        B.u0[a] = c0 - 1;
        B.nc[a] = c1 - c0 + 3;
        B.cc[a] = 0.5f * (q0 + q1);
        B.hf[a] = q1 - B.cc[a];
        if (threadIdx.x < REG) {
            const int i = min(B.o[a] + (int)threadIdx.x, B.l[a]);
            const int lc = P.ax.cell[a][i] - c0;
            const double zi = P.ax.zi[a][i];
            S.q[a][threadIdx.x] = (float)(P.a[a] * (zi + lc)) - B.cc[a];
            S.lc[a][threadIdx.x] = lc;
            S.zi[a][threadIdx.x] = zi;
        }
    }
}

// Kept cells of the region: within 3 sigma of its box and not empty, in cell
// order.  K cells, T points in them.
template <int NW>
__device__ __forceinline__ void region_cells(const RegionParams& R, const RegionBox& B, RegionStage<NW>& S,
                                             RegionCells<NW>& C, const int* __restrict__ cell_start, int& K, int& T)
{
    const VoxParams& P = R.v;
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    const int ncx = B.nc[0], ncy = B.nc[1], ncell = ncx * ncy * B.nc[2];   // <= REG_MAXC (checked on the host)
    const int c = threadIdx.x;
    int cnt = 0, b = 0, upk = 0;
    float l[3] = {0.0f, 0.0f, 0.0f};
    if (c < ncell) {
        // (c + 0.5) / n lies at least 1/(2n) >= 1/512 from an integer, far
        // beyond the error of v_rcp_f32, so the truncations are exact
        const int dz = (int)(((float)c + 0.5f) * __builtin_amdgcn_rcpf((float)(ncx * ncy)));
        const int rem = c - dz * (ncx * ncy);
        const int dy = (int)(((float)rem + 0.5f) * __builtin_amdgcn_rcpf((float)ncx));
        const int d[3] = {rem - dy * ncx, dy, dz};
        float g2 = 0.0f;
#pragma unroll
        for (int a = 0; a < 3; a++) {
            l[a] = R.cellf[a] * (float)(d[a] - 1) - B.cc[a];
            const float g = fmaxf(0.0f, fmaxf(l[a] - B.hf[a], -B.hf[a] - (l[a] + R.cellf[a])));
            g2 = fmaf(g, g, g2);
        }
        if (g2 <= R.rc_cull2) {
            const int E[3] = {P.Ex, P.Ey, P.Ez};
            int w[3];
#pragma unroll
            for (int a = 0; a < 3; a++) {
                w[a] = B.u0[a] + d[a];                      // in [-1, E]: cells are monotonic
                w[a] = w[a] < 0 ? w[a] + E[a] : (w[a] >= E[a] ? w[a] - E[a] : w[a]);
            }
            const int rc = w[0] + P.Ex * (w[1] + P.Ey * w[2]);
            b = cell_start[rc];
            cnt = cell_start[rc + 1] - b;
            upk = d[0] | (d[1] << 8) | (d[2] << 16);
        }
    }
    const int incl = wave_incl_scan(cnt);
    const unsigned long long m = __ballot(cnt > 0);
    if (lane == 63) {
        S.wk[wave] = (int)__popcll(m);
        S.wt[wave] = incl;
    }
    __syncthreads();
    int k0 = 0, t0 = 0;
    K = 0;
    T = 0;
#pragma unroll
    for (int w = 0; w < NW; w++) {
        k0 += w < wave ? S.wk[w] : 0;
        t0 += w < wave ? S.wt[w] : 0;
        K += S.wk[w];
        T += S.wt[w];
    }
    if (cnt > 0) {
        const int k = k0 + bits_below(m), st = t0 + incl - cnt;
        C.crec[k] = make_float4(l[0], l[1], l[2], __int_as_float(b - st));
        C.cupk[k] = upk;
        C.cstart[k] = st;
    }
    __syncthreads();
    K = __builtin_amdgcn_readfirstlane(K);
    T = __builtin_amdgcn_readfirstlane(T);
}

// One pass of staging: candidates from t_next on, 64 per wave and round, those
// within 3 sigma of the region's box compacted into S.pos and S.upk in
// candidate order, until they are all seen or a round's do not fit.  Returns
// the number staged; t_next (the same in every thread) moves on.  A barrier
// precedes and follows each use of the staged arrays.
template <int NW>
__device__ __forceinline__ int region_stage(const RegionParams& R, const RegionBox& B, RegionStage<NW>& S,
                                            RegionCells<NW>& C, const float4* __restrict__ p32, int K, int T,
                                            int& t_next)
{
    const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    int base = 0;
    for (int r = 0; t_next < T; r ^= 1) {
        const int t0 = t_next + 64 * wave, t = t0 + lane;
        bool keep = false;
        int k = 0;
        float4 p = make_float4(0.0f, 0.0f, 0.0f, 0.0f);
        if (t0 < T) {
            // cell of candidate t: the kept cells that start at or before it,
            // less one, from the cells before this wave's 64 candidates and a
            // mask of those that start inside them
            int kb = 0;
            C.flag[wave][lane] = 0;
            wave_sync();
            for (int q = 0; q < K; q += 64) {
                const int s = q + lane < K ? C.cstart[q + lane] : 0x7fffffff;
                kb += (int)__popcll(__ballot(s < t0));
                if (s >= t0 && s < t0 + 64) C.flag[wave][s - t0] = 1;
            }
            wave_sync();
            const unsigned long long sm = __ballot(C.flag[wave][lane] != 0);
            k = kb + bits_below(sm) + ((sm >> lane) & 1ull ? 1 : 0) - 1;
            if (t < T) {
                const float4 cr = C.crec[k];
                const int slot = t + __float_as_int(cr.w);
                const float4 pc = p32[slot];
                p = make_float4(pc.x + cr.x, pc.y + cr.y, pc.z + cr.z, __int_as_float(slot));
                const float ex = fmaxf(0.0f, fabsf(p.x) - B.hf[0]);
                const float ey = fmaxf(0.0f, fabsf(p.y) - B.hf[1]);
                const float ez = fmaxf(0.0f, fabsf(p.z) - B.hf[2]);
                keep = fmaf(ex, ex, fmaf(ey, ey, ez * ez)) <= R.rc_cull2;
            }
        }
        const unsigned long long m = __ballot(keep);
        if (lane == 0) S.wcnt[r][wave] = (int)__popcll(m);
        __syncthreads();
        int off = base, end = base;
#pragma unroll
        for (int w = 0; w < NW; w++) {
            const int n = S.wcnt[r][w];
            off += w < wave ? n : 0;
            end += n;
        }
        if (end > S.CAP) break;                             // this round starts the next pass
        if (keep) {
            const int i = off + bits_below(m);
            S.pos[i] = p;
            S.upk[i] = C.cupk[k];
        }
        base = end;
        t_next += 64 * NW;
    }
    return __builtin_amdgcn_readfirstlane(base);
}

// Box of the subtile of 4 x 4 x 4 voxels at s of the region: centre, half sides.
template <int NW>
__device__ __forceinline__ void subtile_box(const RegionStage<NW>& S, const int s[3], float c[3], float h[3])
{
#pragma unroll
    for (int a = 0; a < 3; a++) {
        const float q0 = S.q[a][s[a]], q1 = S.q[a][s[a] + TILE - 1];
        c[a] = 0.5f * (q0 + q1);
        h[a] = q1 - c[a];
    }
}

// Candidates c0 .. c0 + nc - 1 within 3 sigma of a subtile's box, as byte
// offsets (of their numbers from c0) into records of `size` bytes, padded to a
// multiple of four entries with record `pad`.  One wave; returns their number.
template <int NW>
__device__ __forceinline__ int subtile_list(const RegionStage<NW>& S, float rc_cull2, int c0, int nc, const float c[3],
                                            const float h[3], int size, int pad, unsigned short* list)
{
    const int lane = threadIdx.x & 63;
    int nl = 0;
    wave_sync();                                            // the previous list is read
    for (int b = 0; b < nc; b += 64) {
        const float4 p = S.pos[min(c0 + b + lane, S.CAP - 1)];
        const float ex = fmaxf(0.0f, fabsf(p.x - c[0]) - h[0]);
        const float ey = fmaxf(0.0f, fabsf(p.y - c[1]) - h[1]);
        const float ez = fmaxf(0.0f, fabsf(p.z - c[2]) - h[2]);
        const bool keep = b + lane < nc && fmaf(ex, ex, fmaf(ey, ey, ez * ez)) <= rc_cull2;
        const unsigned long long m = __ballot(keep);
        if (keep) list[nl + bits_below(m)] = (unsigned short)(size * (b + lane));
        nl += (int)__popcll(m);
    }
    if (lane < 4) list[nl + lane] = (unsigned short)(size * pad);
    wave_sync();
    return __builtin_amdgcn_readfirstlane(nl);
}

// Sum over the four candidate parts (16 lanes each) of per-part values of a
// lane's four voxels v[0..3]; part p ends with voxel p's total, added as
// (p0 + p2) + (p1 + p3).  A permlane swap exchanges two registers' halves, so
// each step halves the values a lane holds.
__device__ __forceinline__ float swap_add32(float a, float b)
{
    const auto s = __builtin_amdgcn_permlane32_swap(__float_as_uint(a), __float_as_uint(b), false, false);
    return __uint_as_float(s[0]) + __uint_as_float(s[1]);
}
__device__ __forceinline__ float swap_add16(float a, float b)
{
    const auto s = __builtin_amdgcn_permlane16_swap(__float_as_uint(a), __float_as_uint(b), false, false);
    return __uint_as_float(s[0]) + __uint_as_float(s[1]);
}
template <bool HALF>
__device__ __forceinline__ void swap64(double& a, double& b)
{
    unsigned al = (unsigned)__double2loint(a), ah = (unsigned)__double2hiint(a);
    unsigned bl = (unsigned)__double2loint(b), bh = (unsigned)__double2hiint(b);
    const auto l = HALF ? __builtin_amdgcn_permlane32_swap(al, bl, false, false)
                        : __builtin_amdgcn_permlane16_swap(al, bl, false, false);
    const auto h = HALF ? __builtin_amdgcn_permlane32_swap(ah, bh, false, false)
                        : __builtin_amdgcn_permlane16_swap(ah, bh, false, false);
    a = __hiloint2double((int)h[0], (int)l[0]);
    b = __hiloint2double((int)h[1], (int)l[1]);
}
__device__ __forceinline__ double part_sum(double v0, double v1, double v2, double v3)
{
    swap64<true>(v0, v2);
    swap64<true>(v1, v3);
    double a = v0 + v2, b = v1 + v3;
    swap64<false>(a, b);
    return a + b;
}
__device__ __forceinline__ double part_min(double v0, double v1, double v2, double v3)
{
    swap64<true>(v0, v2);
    swap64<true>(v1, v3);
    double a = fmin(v0, v2), b = fmin(v1, v3);
    swap64<false>(a, b);
    return fmin(a, b);
}
__device__ __forceinline__ float part_sum(float v0, float v1, float v2, float v3)
{
    return swap_add16(swap_add32(v0, v2), swap_add32(v1, v3));
}

}  // namespace d2bi
