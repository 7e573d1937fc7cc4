// d2bi_fp64.cuh -- FP64 voxelisation: by regions, and the per-voxel walk over
// the 27 neighbour cells.
//
// One part of the single translation unit d2bi_gpu.hip, which includes the
// parts in order so that kernels and the device helpers they call compile
// together; each part uses the definitions of the parts before it.
#pragma once

namespace d2bi {

// ------------------------------------------------------------------ (b) voxelise, FP64

// One thread per voxel; the 27 neighbour cells in (kz,ky,kx) order and the
// points of each cell in insertion order, exactly the neighbour list order
// of neighbourList1b, summed as the reference sums it (:1877-1892).  NA > 1:
// the aperture branch's shared neighbour loop (:1905-1922), one weight per
// member and one sum per aperture point a, whose phases are cs64[a cs_stride
// + slot] and whose fields go to out_re/out_im[a out_stride + voxel]; each
// point's sum takes the same terms in the same order as an NA = 1 pass over
// that point's phases.
template <int NA>
__global__ __launch_bounds__(256) void k_voxel_fp64(VoxParams P, const int* __restrict__ cell_start,
                                                    const Frac3* __restrict__ frac,
                                                    const double2* __restrict__ cs64, int64_t cs_stride,
                                                    double* __restrict__ out_re,
                                                    double* __restrict__ out_im, int64_t out_stride,
                                                    double* __restrict__ out_rho,
                                                    int* __restrict__ out_cnt,
                                                    double* __restrict__ out_r2m)
{
    const int ix = blockIdx.x * 8 + (threadIdx.x & 7);
    const int iy = blockIdx.y * 8 + ((threadIdx.x >> 3) & 7);
    const int iz = blockIdx.z * 4 + (threadIdx.x >> 6);
    if (ix >= P.Mx || iy >= P.My || iz >= P.Mz) return;
    const int cx = P.ax.cell[0][ix], cy = P.ax.cell[1][iy], cz = P.ax.cell[2][iz];
    const double zx = P.ax.zi[0][ix], zy = P.ax.zi[1][iy], zz = P.ax.zi[2][iz];
    double sre[NA], sim[NA];
#pragma unroll
    for (int a = 0; a < NA; a++) { sre[a] = 0.0; sim[a] = 0.0; }
    double r2min = 3.4028234663852886e38;
    int n = 0;
    for (int kz = -1; kz <= 1; kz++) {
        const int jz = (cz + P.Ez + kz) % P.Ez;
        const double dzi3 = kz - zz;
        for (int ky = -1; ky <= 1; ky++) {
            const int jy = (cy + P.Ey + ky) % P.Ey;
            const double dzi2 = ky - zy;
            for (int kx = -1; kx <= 1; kx++) {
                const int jx = (cx + P.Ex + kx) % P.Ex;
                const double dzi1 = kx - zx;
                const int c = jx + P.Ex * (jy + P.Ey * jz);
                const int s1 = cell_start[c + 1];
                for (int s = cell_start[c]; s < s1; s++) {
                    const Frac3 f = frac[s];
                    const double d1 = P.a[0] * (f.x + dzi1);
                    const double d2 = P.a[1] * (f.y + dzi2);
                    const double d3 = P.a[2] * (f.z + dzi3);
                    const double dd = (d1 * d1 + d2 * d2) + d3 * d3;
                    if (dd <= P.rc2) {
                        n++;
                        r2min = r2min < dd ? r2min : dd;
                        const double e = exp(-dd * P.i2s2);
#pragma unroll
                        for (int a = 0; a < NA; a++) {
                            const double2 cs = cs64[a * cs_stride + s];
                            sre[a] = sre[a] + e * cs.x;
                            sim[a] = sim[a] + e * cs.y;
                        }
                    }
                }
            }
        }
    }
    const int64_t o = (int64_t)ix + (int64_t)P.Mx * (iy + (int64_t)P.My * iz);
#pragma unroll
    for (int a = 0; a < NA; a++) {
        double ww = hypot(sre[a], sim[a]);
        ww = 1 / (1.0e-16 > ww ? 1.0e-16 : ww);
        out_re[a * out_stride + o] = sre[a] * ww;
        out_im[a * out_stride + o] = sim[a] * ww;
    }
    out_rho[o] = P.use_density ? rho_of(r2min, P.sigma) : 1.0;
    if (out_cnt) out_cnt[o] = n;
    if (out_r2m) out_r2m[o] = r2min;
}

// Region form (default).  A workgroup of four waves per 8 x 8 x 8 region, a
// wave per column of two 4 x 4 x 4 subtiles (staging: d2bi_region.cuh).  Per axis, the
// squared offset of a candidate from a voxel depends on the voxel's index
// along that axis only, so neighbourList1b's range
//     dd = (d1^2 + d2^2) + d3^2,   d = a (frac + (k - zi))
// (Lib_LinkCell3D.f90:1565-1596) is an add of squares that are evaluated once
// per candidate and axis position, with the reference's expression: every
// range is the reference's to the bit, and so are the members and the nearest
// range.  A voxel whose cell is not next to the candidate's along an axis
// gets an infinite square there (the 27-cell rule).  The weight factorises the
// same way, into exp(-d^2 / 2s^2) of the three axes, each an exponential of its
// own: of a member none is below exp(-4.5), whatever the voxels' sides, and the
// product is nearer the exact weight than one exponential of the rounded range
// (relative rms 1.8e-16 against 2.7e-16).  A recurrence along each axis,
// exp(-d0^2 / 2s^2) exp(d0 h / s^2)^i from the region's first voxel, would take
// two exponentials for eight, but carries exponents of the whole region: weights
// off by up to 1e-14 at four voxels per lattice parameter, and under- and
// overflow where voxels are taller than about 5 sigma.  Lane (xy, part) walks
// every fourth candidate of the subtile's list for the four voxels along z at
// its x and y: an add, a compare, a select, a multiply and two FMAs per pair, in
// FP64.
//
// Bound: FP64 VALU issue (an add, multiply or compare ~4.7 cycles per wave,
// measured) in the pair loop; the per-voxel 27-cell walk above evaluates 180
// pairs per voxel with an exponential per member and gathers every point from
// memory.  MFMA does not help: v_mfma_f64_4x4x4 takes 16 cycles for the two
// FMAs' 10 and does not overlap the vector pipe.

static constexpr int F64R_NW = 4;                    // waves per workgroup
// Candidates whose records are held at once.  A workgroup's phases (cells,
// points, records, pairs) are parted by barriers and start with loads, so it
// is the number of workgroups per CU that hides their latencies: 64 records
// (30 KB of LDS) ran 1.58 ms on a 400 x 360 x 200 field, 88 1.75, 128 (three
// workgroups instead of four) 2.31, regions of 8 x 8 x 16 with eight waves
// 2.18, of 8 x 8 x 4 1.89, and the per-voxel walk 10.4 ms.  (With an axis per
// wave in the records, no quieting before the minimum and a square root for
// the modulus 1.31 without, 1.45 with the density; with an exponential per
// weight, 32 KB, 3 % more on the same box: 1.40 -> 1.44 with the density.)
static constexpr int F64R_REC = 64;

template <int NA>
struct F64Record {
    double2 x[REG], y[REG], z[REG];                  // (square, weight) per voxel position
    double2 cs[NA];                                  // cos and sin of g.r
};

template <int NA, bool MIN, bool DIAG>
__global__ __launch_bounds__(64 * F64R_NW, NA == 4 ? 2 : 4) void k_voxel_fp64_region(
    RegionParams R, const int* __restrict__ cell_start, const Frac3* __restrict__ frac,
    const float4* __restrict__ p32, const double2* __restrict__ cs64, int64_t cs_stride, double* __restrict__ out_re,
    double* __restrict__ out_im, int64_t out_stride, double* __restrict__ out_rho, int* __restrict__ out_cnt,
    double* __restrict__ out_r2m)
{
    constexpr int NW = F64R_NW, NS = REG / TILE;
    typedef F64Record<NA> Rec;
    __shared__ RegionStage<NW> S;
    // the link cells are done with once a pass is staged, the records after it
    __shared__ union {
        RegionCells<NW> cells;
        Rec rec[F64R_REC + 1];                       // the last one pads lists
    } U;
    __shared__ unsigned short lists[NW][F64R_REC + 4];           // byte offsets of records
    static_assert(sizeof U.rec < 65536, "16-bit record offsets");
    const int region = region_of(R, blockIdx.x);
    if (region >= R.nreg) return;
    const VoxParams& P = R.v;
    const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    RegionBox B;
    region_box(R, region, S, B);

    // the wave's subtiles (two along z) and the lane's voxels: x, y, and four
    // along z in each
    const int s0 = (wave & 1) * TILE, s1 = (wave >> 1) * TILE;
    const int part = lane >> 4, lx = s0 + (lane & 3), ly = s1 + ((lane >> 2) & 3);
    const bool active = B.o[0] + s0 <= B.l[0] && B.o[1] + s1 <= B.l[1];
    double sre[NS][NA][TILE], sim[NS][NA][TILE], dmin[NS][TILE];
    int cnt[NS][TILE];
#pragma unroll
    for (int z = 0; z < NS; z++)
#pragma unroll
        for (int i = 0; i < TILE; i++) {
#pragma unroll
            for (int a = 0; a < NA; a++) { sre[z][a][i] = 0.0; sim[z][a][i] = 0.0; }
            dmin[z][i] = 3.4028234663852886e38;
            cnt[z][i] = 0;
        }

    // records of a chunk, a candidate per lane: three waves an axis each, the
    // fourth the phases.  The parts go round the waves from chunk to chunk and
    // region to region, so that no SIMD has the phases' share every time.  A
    // lane's inputs are loaded before the previous chunk's pairs.
    static_assert(NW == 4 && F64R_REC == 64, "a wave per part, a lane per candidate");
    double in[2 * NA];
    int turn = region;
    auto load = [&](int c0, int nc) {
        const int part = (wave + turn + 1) & 3;
        if (lane >= nc) return;
        const int slot = __float_as_int(S.pos[c0 + lane].w);
        if (part < 3) {
            in[0] = reinterpret_cast<const double*>(frac + slot)[part];
        } else {
#pragma unroll
            for (int a = 0; a < NA; a++) {
                const double2 c = cs64[a * cs_stride + slot];
                in[2 * a] = c.x;
                in[2 * a + 1] = c.y;
            }
        }
    };
    auto record = [&](int c0, int nc) {
        turn++;
        const int ax = (wave + turn) & 3;
        Rec& q = U.rec[lane];
        if (lane >= nc) {
        } else if (ax == 3) {
#pragma unroll
            for (int a = 0; a < NA; a++) q.cs[a] = make_double2(in[2 * a], in[2 * a + 1]);
        } else {
            const int u = ((S.upk[c0 + lane] >> (8 * ax)) & 255) - 1;
            const double side = ax == 0 ? P.a[0] : ax == 1 ? P.a[1] : P.a[2];
            double2* const out = ax == 0 ? q.x : ax == 1 ? q.y : q.z;
#pragma unroll
            for (int v = 0; v < REG; v++) {
                const int k = u - S.lc[ax][v];
                const double d = side * (in[0] + (k - S.zi[ax][v]));
                const double d2 = d * d;
                out[v] = make_double2((unsigned)(k + 1) <= 2u ? d2 : HUGE_VAL, exp(-d2 * P.i2s2));
            }
        }
        // the padding record: no voxel is in range of it
        static_assert(sizeof(Rec) == sizeof(double2) * (3 * REG + NA), "x, y and z, then the phases");
        if (threadIdx.x < 3 * REG + NA)
            reinterpret_cast<double2*>(&U.rec[F64R_REC])[threadIdx.x] =
                make_double2(threadIdx.x < 3 * REG ? HUGE_VAL : 0.0, 0.0);
    };

    for (int t_next = 0, T = 1; t_next < T;) {
        int K;
        region_cells(R, B, S, U.cells, cell_start, K, T);
        const int n = region_stage(R, B, S, U.cells, p32, K, T, t_next);
        // equal chunks of at most F64R_REC candidates
        const int nch = (n + F64R_REC - 1) / F64R_REC, per = nch > 0 ? (n + nch - 1) / nch : 0;
        __syncthreads();                             // staged points written, cells read
        load(0, min(per, n));
        for (int c0 = 0; c0 < n; c0 += per) {
            const int nc = min(per, n - c0);
            if (c0 > 0) __syncthreads();             // earlier records read
            record(c0, nc);
            __syncthreads();
            if (c0 + per < n) load(c0 + per, min(per, n - c0 - per));
            if (!active) continue;
#pragma unroll
            for (int z = 0; z < NS; z++) {
                const int s[3] = {s0, s1, z * TILE};
                if (B.o[2] + s[2] > B.l[2]) continue;
                float tc[3], th[3];
                subtile_box(S, s, tc, th);
                const int nl = subtile_list(S, R.rc_cull2, c0, nc, tc, th, (int)sizeof(Rec), F64R_REC, lists[wave]);
                const char* rec = reinterpret_cast<const char*>(U.rec);
#pragma unroll 1
                for (int k = 0; k < nl; k += 4) {
                    const Rec& q = *reinterpret_cast<const Rec*>(rec + lists[wave][k + part]);
                    const double2 qx = q.x[lx], qy = q.y[ly];
                    const double s12 = qx.x + qy.x, wxy = qx.y * qy.y;
                    double2 cs[NA];
#pragma unroll
                    for (int a = 0; a < NA; a++) cs[a] = q.cs[a];
#pragma unroll
                    for (int v = 0; v < TILE; v++) {
                        const double2 qz = q.z[z * TILE + v];
                        const double dd = s12 + qz.x, p = wxy * qz.y;
                        const bool in = dd <= P.rc2;
                        // a pair out of range keeps the low word of its
                        // weight: < 1e-313, dropped from the sums at the end
                        const double w = __hiloint2double(in ? __double2hiint(p) : 0, __double2loint(p));
#pragma unroll
                        for (int a = 0; a < NA; a++) {
                            sre[z][a][v] = fma(w, cs[a].x, sre[z][a][v]);
                            sim[z][a][v] = fma(w, cs[a].y, sim[z][a][v]);
                        }
                        // fmin() would first quiet its operands, one more
                        // operation per pair
                        if (MIN) asm("v_min_f64 %0, %0, %1" : "+v"(dmin[z][v]) : "v"(dd));
                        if (DIAG) cnt[z][v] += in ? 1 : 0;
                    }
                }
            }
        }
        __syncthreads();                             // staged points and records read
    }
    if (!active) return;

    // lane (xy, part) finishes the voxel `part` along z of each subtile
    auto drop = [](double v) { return fabs(v) < 1.0e-280 ? 0.0 : v; };
#pragma unroll
    for (int z = 0; z < NS; z++) {
        const int vx = B.o[0] + lx, vy = B.o[1] + ly, vz = B.o[2] + z * TILE + part;
        const bool out = vx < P.Mx && vy < P.My && vz < P.Mz;
        const int64_t o = (int64_t)vx + (int64_t)P.Mx * (vy + (int64_t)P.My * vz);
#pragma unroll
        for (int a = 0; a < NA; a++) {
            const double re = drop(part_sum(sre[z][a][0], sre[z][a][1], sre[z][a][2], sre[z][a][3]));
            const double im = drop(part_sum(sim[z][a][0], sim[z][a][1], sim[z][a][2], sim[z][a][3]));
            // (|S| counts from 1e-16 on, so its square is in range)
            double ww = sqrt(fma(re, re, im * im));
            ww = 1 / (1.0e-16 > ww ? 1.0e-16 : ww);
            if (out) {
                out_re[a * out_stride + o] = re * ww;
                out_im[a * out_stride + o] = im * ww;
            }
        }
        double r2 = 3.4028234663852886e38;
        if (MIN) {
            // over every candidate: the nearest is a member if there is one
            const double v = part_min(dmin[z][0], dmin[z][1], dmin[z][2], dmin[z][3]);
            if (v <= P.rc2) r2 = v;
        }
        // without the density field rho = 1, which the integrators do not read
        if (MIN && out) out_rho[o] = P.use_density ? rho_of(r2, P.sigma) : 1.0;
        if (DIAG) {
            const float c = part_sum((float)cnt[z][0], (float)cnt[z][1], (float)cnt[z][2], (float)cnt[z][3]);
            if (out && out_cnt) out_cnt[o] = (int)c;
            if (out && out_r2m) out_r2m[o] = r2;
        }
    }
}

}  // namespace d2bi
