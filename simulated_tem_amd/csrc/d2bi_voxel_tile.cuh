// d2bi_voxel_tile.cuh -- the FAST voxel kernel k_voxel_tile: LDS-staged voxel
// tiles, the row variants and the FP64 guard re-test.
//
// One part of the single translation unit d2bi_gpu.hip, which includes the
// parts in order so that kernels and the device helpers they call compile
// together; each part uses the definitions of the parts before it.
#pragma once

namespace d2bi {

// ------------------------------------------------------------------ (b) voxelise, FAST

static constexpr int TILE_MAXC = 128;                // cells in a tile's unwrapped range (<= 5^3)
static constexpr int ROW_BLOCK = 32;                 // row kernel: steps per guard test and Kahan merge
static constexpr int TILE_WIN = 1024;                // candidates whose cell starts are flagged at once

struct FastParams {
    VoxParams v;
    int ntx, nty, ntz;          // tiles per axis
    int ntiles, per_xcd;        // tiles; workgroups per XCD (the grid is 8 per_xcd)
    float e_rc, e_band;         // k2 (3 sigma)^2 and the guard half-width around it
    float rc_cull2;             // (3 sigma)^2 widened for the tile-box cull
    float k2;                   // -log2(e)/(2 sigma^2)
    float w_scale;              // 2^e_rc
    float m2_min;               // (1e-16)^2 / w_scale^2
    float inv_k2;               // 1 / k2
    float cellf[3];             // link-cell sides in FP32
    int thin_z;                 // link cells thinner than 3 sigma along z
    int order;                  // tiles over workgroups: 0 contiguous ranges per XCD, 1 linear, 2 rows dealt to XCDs
    // aperture points sharing one pass (kernels with NA > 1): point a's
    // (cos, sin) of g.r at app_cs[a app_stride + slot], its field at
    // field[a field_stride + voxel]
    const float2* app_cs;
    int64_t app_stride, field_stride;
};

// One wave per voxel tile: 4x4x4 voxels, 4x4x8 or 4x8x8 for the row kernel
// (x, y, z; x fastest).  The tile's candidates are the points of
// every link cell in the unwrapped range [cell(first voxel)-1,
// cell(last voxel)+1] on each axis; an unwrapped cell u stands for cell
// mod(u, E) displaced by u - mod(u, E) cells, which is exactly the periodic
// image neighbourList1b sees through its mod() (Lib_LinkCell3D.f90:1567-1575).
// Cells, then points, farther than 3 sigma from the tile's voxel box are
// dropped; the rest are compacted into LDS (ballot + popcount).
//
// What bounds it: FP32 vector instructions, not memory or LDS (counters on
// 800 x 800 x 400 voxels: the vector units issue all the time).  The tile
// lists about 400 points, keeps about 127 of them, and a voxel has 28 members,
// so the kernel is arranged to spend few instructions on a listed point, few
// on a kept one, and to leave out most of the pairs beyond 3 sigma:
//   - a listed point is only moved to the tile frame, culled and compacted
//     (the Gaussian factors were once evaluated here, for a quarter of the
//     lanes); the records are made for 64 kept candidates at a time;
//   - the rows of voxels form groups (2 along y by TZ / 2 along z), each with
//     its own list of the candidates within 3 sigma of its box: 59 instead of
//     127 of a 4 x 8 x 8 tile, 59 instead of 95 of a 4 x 4 x 8;
//   - the larger tile stages fewer points per voxel.
// 800 x 800 x 400 voxels, ms (before all three, 4 x 4 x 8 tiles: 5.5): 5.0,
// 4.65, 4.2 (4.06 with the guard band watched by steps and voxels); 2020 vector
// instructions per 128 voxels became 1280.
//
// Staging.  The kept non-empty cells are listed once per tile with their
// origin in the tile frame and the offset from candidate index to point
// slot.  Candidates are then taken 64 at a time; the cell of candidate t is
// the number of kept cells, after the first, that start at or before t: a
// 64-bit mask of starts, from flags set for TILE_WIN candidates at a time.
//
// Arithmetic.  Positions are taken relative to the tile centre c (FP32,
// rounded once from FP64 values).  For a candidate p and voxel q the Gaussian
// exponent e = k2*|p - q|^2 (k2 = -log2(e)/(2 sigma^2), so the weight is 2^e)
// is evaluated as
//     e = (-2 k2 p).q + (k2 |p|^2 + k2 |q|^2)
// from a per-candidate record (-2 k2 p, k2 |p|^2): three FMAs and an add.
// Membership is e >= k2 (3 sigma)^2; where |e - k2 (3 sigma)^2| is within
// the guard band the pair is re-tested in FP64 with the expression of
// neighbourList1b (and the neighbour offset must be -1, 0 or +1, as in its
// 27-cell loop), so the set of summed atoms is exactly the FP64 set.
// cos/sin of g.r were evaluated in FP64.
//
// ROW = false: lane = voxel; S = sum w (cos, sin) is accumulated in blocks of
// 32 candidates whose sums are merged with Kahan compensation.
//
// ROW = true: the wave is the tile's voxel rows along x (one per (y, z): 16,
// 32 or 64) times NQ candidate parts (4, 2 or 1); lane (row, s)
// walks entries s, s+NQ, s+2NQ, ... of its group's list for the four voxels of
// its row.  The Gaussian factorises along x:
//     2^(e_i - e_rc) = X_i * 2^t,   X_i = 2^(k2 ((p_x - q_x,i)^2 + p_y^2 + p_z^2)),
//     t = -2 k2 (p_y q_y + p_z q_z) + k2 (q_y^2 + q_z^2) - e_rc   (e_rc = k2 (3 sigma)^2),
// and the four x positions q_x,i are the tile's, common to every row, so
// X_0..X_3 (which carry the candidate's own y-z term) are evaluated once
// per candidate when it is staged and a lane spends two FMAs and one
// v_exp_f32 per candidate on four voxels.  Membership e_i >= e_rc
// is u_i = X_i 2^t - 1 >= 0; the steps and voxels of a block (even or
// odd, 0-1 or 2-3) in which some |u_i| lies within the guard band are walked
// again and the pairs of the band re-tested in FP64, correcting the sums where
// the FP64 test disagrees.  The parts' sums are
// added in a fixed order through LDS at the end, after which lane (row, s)
// holds voxels s NV .. s NV + NV - 1 of its row (NV = 4 / NQ).
//
// Thin cells.  Link cells are at least 3 sigma wide along x and y (Ex <=
// Dx/deltaM + 2 with deltaM >= 3 sigma / min(a_x, a_y)), so along those axes
// every point within 3 sigma of a voxel lies in a neighbouring cell and the
// range test alone decides membership (the guard band covers rounding of the
// cell sides).  Along z the cell height Mz a_z / Ez can be smaller (a_z <
// min(a_x, a_y) with deltaM dividing Mz, or Ez = 3 for thin foils); then a
// point two cells away can lie within 3 sigma, and neighbourList1b does not
// see it.  ROW = 2 applies that rule: a candidate whose cell is not within one
// cell of the row's along z gets weight 0 for the row.  The diagnostic kernel
// tests the z offset of every pair when F.thin_z is set.
//
// Aperture points (NA = 2 or 4, row kernels of 4 x 4 x TZ tiles): the NA
// points of a condition's aperture sum share its binned points, weights and
// membership and differ only in g.r (Lib_DynamicalTwoBeamImaging.f90:
// 1905-1922 sums them in one neighbour loop).  Each staged candidate carries
// NA (cos, sin) pairs, every step adds the pair's weight into NA sums, and a
// guard correction is applied to each.  Point a's sums take the same terms in
// the same order as an NA = 1 pass with that point's phases, so its field is
// that pass's to the bit.
template <bool DENSITY, bool DIAG, int ROW, int TZ, int TY = 4, int NA = 1>
__global__ __launch_bounds__(64) void k_voxel_tile(FastParams F, const int* __restrict__ cell_start,
                                                   const Frac3* __restrict__ slot_frac,
                                                   const float4* __restrict__ p32,
                                                   const float* __restrict__ sn32,
                                                   float4* __restrict__ field,
                                                   int* __restrict__ out_cnt,
                                                   float* __restrict__ out_r2m,
                                                   unsigned long long* __restrict__ guard_count)
{
    static_assert(!(DIAG && ROW), "the diagnostic kernel tests every pair itself");
    static_assert(TZ == 4 || (ROW && TZ == 8), "tiles of 4 x 4 x 4, or deeper ones of the row kernel");
    static_assert(TY == 4 || (ROW && TY == 8 && TZ == 8), "tiles of 4 x 8 x 8: a lane per row");
    static_assert(NA == 1 || ((NA == 2 || NA == 4) && ROW && TY == 4), "aperture points: 2 or 4, tiles 4 voxels wide");
    constexpr int TX = 4;
    // ROW: candidate parts per row, voxels a lane finishes
    constexpr int NQ = ROW ? 256 / (TY * TZ * TX) : 1;
    constexpr int NV = ROW ? TX / NQ : 1;
    // ROW: groups of rows, 2 along y and TZ / 2 along z, with a list each
    constexpr int GLANES = NQ * TZ, GROWS = TZ;
    constexpr int NG = ROW ? 64 / GLANES : 1;
    constexpr int GY = TY / 2;
    // candidates staged at once: one pass for most tiles at four voxels per
    // lattice parameter (about 95 candidates, 127 for 4 x 8 x 8)
    constexpr int CAP = TY == 8 ? 144 : 112;
    // XCD-aware order: consecutive workgroups go round-robin to the 8 XCDs;
    // order 0 gives each XCD a contiguous range of tiles so neighbouring
    // tiles, which read the same link cells, share one L2 (the ranges are
    // slabs along z); order 1 is linear; order 2 deals rows of tiles along x
    // to the XCDs in turn (row r to XCD r mod 8), so that every XCD holds
    // rows at every depth and a row's tiles share one L2.  A tile's sums do
    // not depend on the order.
    const int bid = blockIdx.x;
    int L;
    if (F.order == 0) L = (bid & 7) * F.per_xcd + (bid >> 3);
    else if (F.order == 1) L = bid;
    else {
        const int idx = bid >> 3, row = (idx / F.ntx) * 8 + (bid & 7);
        L = row * F.ntx + (idx - (idx / F.ntx) * F.ntx);
    }
    if (L >= F.ntiles) return;
    const VoxParams& P = F.v;
    const int tx = L % F.ntx, ty = (L / F.ntx) % F.nty, tz = L / (F.ntx * F.nty);
    const int lane = threadIdx.x;
    const int x0 = tx * TX, y0 = ty * TY, z0 = tz * TZ;
    const int x1 = min(P.Mx, x0 + TX) - 1, y1 = min(P.My, y0 + TY) - 1, z1 = min(P.Mz, z0 + TZ) - 1;
    // the lane's row of voxels along x (y fastest) and, lane per voxel, its x
    const int rrow = ROW ? lane / NQ : (lane >> 2);
    const int grp = lane / GLANES, rg = rrow & (GROWS - 1);    // ROW: the lane's group and its row there
    const int ix = x0 + (lane & 3);
    const int iy = y0 + (ROW ? 2 * (grp % GY) + (rg & 1) : rrow & 3);
    const int iz = z0 + (ROW ? (TZ / 2) * (grp / GY) + (rg >> 1) : rrow >> 2);
    const bool row_act = iy <= y1 && iz <= z1;
    const bool act = ix <= x1 && row_act;
    const int jx = min(ix, x1), jy = min(iy, y1), jz = min(iz, z1);
    const QL* const qlz_tab = TZ == 8 ? P.ax.ql[3] : P.ax.ql[2];   // z relative to the tile's first cell
    const QL* const qly_tab = TY == 8 ? P.ax.ql[4] : P.ax.ql[1];   // y relative to the tile's first cell

    // origin cell of the tile; the voxel's FP32 position relative to it and
    // its cell offset (host tables)
    const int c0x = P.ax.cell[0][x0], c0y = P.ax.cell[1][y0], c0z = P.ax.cell[2][z0];
    const QL qlx = P.ax.ql[0][jx], qly = qly_tab[jy], qlz = qlz_tab[jz];
    const int lcx = qlx.lc, lcy = qly.lc, lcz = qlz.lc;
    const float qx = qlx.q, qy = qly.q, qz = qlz.q;
    // the tile's voxel box: positions do not decrease with the voxel index
    // (link cells are monotonic along each axis), so its corners are the
    // first and last voxels
    const QL ex0 = P.ax.ql[0][x0], ex1 = P.ax.ql[0][x1];
    const QL ey0 = qly_tab[y0], ey1 = qly_tab[y1];
    const QL ez0 = qlz_tab[z0], ez1 = qlz_tab[z1];
    const float bx0 = ex0.q, bx1 = ex1.q, by0 = ey0.q, by1 = ey1.q, bz0 = ez0.q, bz1 = ez1.q;
    // tile-centred frame
    const float ccx = 0.5f * (bx0 + bx1), ccy = 0.5f * (by0 + by1), ccz = 0.5f * (bz0 + bz1);
    const float hx = bx1 - ccx, hy = by1 - ccy, hz = bz1 - ccz;
    const float qcx = qx - ccx, qcy = qy - ccy, qcz = qz - ccz;
    const float k2 = F.k2;
    const float kq2 = k2 * fmaf(qcx, qcx, fmaf(qcy, qcy, qcz * qcz));
    const int squart = lane & (NQ - 1);
    const float kyz = fmaf(k2, fmaf(qcy, qcy, qcz * qcz), -F.e_rc);

    // unwrapped cell range (cells are monotonic, so ux0 + dx lies in [-1, E])
    const int ux0 = c0x - 1, uy0 = c0y - 1, uz0 = c0z - 1;
    const int ncx = ex1.lc + 3, ncy = ey1.lc + 3, ncz = ez1.lc + 3;
    const int ncell = ncx * ncy * ncz;                 // <= TILE_MAXC (checked on the host)

    // records of the staged candidates, part c of candidate j at
    // sM[c (CAP + 1) + j]: ROW = false, (-2 k2 p, k2 |p|^2) tile-centred,
    // then (cos, sin) of g.r; ROW = true, (X_0..X_3), then (-2 k2 p_y,
    // -2 k2 p_z, sin, cos), NA > 1 then (cos, sin) of the aperture points two
    // to a part.  Until its record is made part 0 holds a candidate's position
    // in the tile frame and its cosine.  ROW = true: candidate CAP is the
    // zero record that fills the groups' lists.
    constexpr int NPH = NA > 1 ? NA / 2 : 0;
    constexpr int REC = ROW ? 2 + NPH : 2;
    constexpr int RST = CAP + 1;
    __shared__ float4 sM[RST * REC];
    __shared__ float4 crec[TILE_MAXC];         // kept cells: origin in the tile frame, slot - index
    __shared__ unsigned short cupk[TILE_MAXC]; // kept cells: dx | dy << 4 | dz << 8 (each below 16)
    __shared__ unsigned sflag[TILE_WIN / 32];  // bit s - 1 of the window: a cell starts at candidate s
    __shared__ int sslot[CAP];            // staged candidates' slots ...
    __shared__ unsigned char scell[CAP + 1];     // ... and kept cells
    __shared__ __align__(16) unsigned short slist[ROW ? NG * CAP : 8];   // groups' candidates: 16 j
    int* const cstart = reinterpret_cast<int*>(sM);
    // ROW: the tile's x positions and the boxes of its GY parts along y and two
    // along z (centre and half-width of each), tile-centred; clamped at the
    // grid's edge.  Kept in LDS: as registers, live over the whole tile, they
    // cost a wave per SIMD.
    __shared__ __align__(16) float sbox[ROW ? TX + 2 * GY + 4 : 4];
    if (ROW && lane < TX) sbox[lane] = P.ax.ql[0][min(x0 + lane, x1)].q - ccx;
    if (ROW && lane < GY + 2) {
        const bool z = lane >= GY;
        const int v0 = z ? z0 + TZ / 2 * (lane - GY) : y0 + 2 * lane, v1 = z ? v0 + TZ / 2 - 1 : v0 + 1;
        const float lo = z ? qlz_tab[min(v0, z1)].q : qly_tab[min(v0, y1)].q;
        const float hi = z ? qlz_tab[min(v1, z1)].q : qly_tab[min(v1, y1)].q;
        const float c = 0.5f * (lo + hi);
        sbox[TX + 2 * lane] = c - (z ? ccz : ccy);
        sbox[TX + 2 * lane + 1] = hi - c;
    }
    static_assert(TILE_MAXC / (3 * 3) < 16, "cell offsets in four bits");
    static_assert(sizeof(int) * TILE_MAXC <= sizeof(sM), "cstart overlay");
    static_assert(NQ == 1 || 3 * 64 * TX * sizeof(float) <= sizeof(sM), "row sums overlay");
    static_assert(16 * CAP < 65536 && CAP % 8 == 0, "list entries, 16-byte stores");

    // base plus the set bits of a wave mask below this lane (v_mbcnt)
    auto below = [](unsigned long long m, int base) -> int {
        return (int)__builtin_amdgcn_mbcnt_hi((unsigned)(m >> 32), __builtin_amdgcn_mbcnt_lo((unsigned)m, (unsigned)base));
    };

    // kept cells: in range of the tile box and not empty, in cell order with x
    // the slowest: where the candidates take several passes, each then has its
    // share of every group's (the groups split y and z), and the longest list,
    // which all walk, is shorter (three voxels per lattice parameter, 300 x
    // 300 x 180: 432 us with z the slowest, 392 so; at four 3990 either way)
    int K = 0, T = 0;
    {
        // (c + 0.5) / n lies at least 1/(2n) >= 1/256 from an integer, far
        // beyond the error of v_rcp_f32, so the truncations below are exact
        const float inz = __builtin_amdgcn_rcpf((float)ncz), inyz = __builtin_amdgcn_rcpf((float)(ncy * ncz));
        for (int cb = 0; cb < ncell; cb += 64) {
            const int c = cb + lane;
            int cnt = 0, b = 0, upk = 0;
            float lx = 0.0f, ly = 0.0f, lz = 0.0f;
            if (c < ncell) {
                // c = dz + ncz (dy + ncy dx); c < 128 so the float quotients are exact
                const int dx = (int)(((float)c + 0.5f) * inyz);
                const int r = c - dx * (ncy * ncz);
                const int dy = (int)(((float)r + 0.5f) * inz);
                const int dz = r - dy * ncz;
                lx = F.cellf[0] * (float)(dx - 1) - ccx;
                ly = F.cellf[1] * (float)(dy - 1) - ccy;
                lz = F.cellf[2] * (float)(dz - 1) - ccz;
                const float gx = fmaxf(0.0f, fmaxf(lx - hx, -hx - (lx + F.cellf[0])));
                const float gy = fmaxf(0.0f, fmaxf(ly - hy, -hy - (ly + F.cellf[1])));
                const float gz = fmaxf(0.0f, fmaxf(lz - hz, -hz - (lz + F.cellf[2])));
                if (fmaf(gx, gx, fmaf(gy, gy, gz * gz)) <= F.rc_cull2) {
                    int rx = ux0 + dx, ry = uy0 + dy, rz = uz0 + dz;
                    rx = rx < 0 ? rx + P.Ex : (rx >= P.Ex ? rx - P.Ex : rx);
                    ry = ry < 0 ? ry + P.Ey : (ry >= P.Ey ? ry - P.Ey : ry);
                    rz = rz < 0 ? rz + P.Ez : (rz >= P.Ez ? rz - P.Ez : rz);
                    const int rc = rx + P.Ex * (ry + P.Ey * rz);
                    b = cell_start[rc];
                    cnt = cell_start[rc + 1] - b;
                    upk = dx | (dy << 4) | (dz << 8);
                }
            }
            const int incl = wave_incl_scan(cnt);
            const unsigned long long m = __ballot(cnt > 0);
            if (cnt > 0) {
                const int k = below(m, K);
                const int st = T + incl - cnt;
                cstart[k] = st;
                crec[k] = make_float4(lx, ly, lz, __int_as_float(b - st));
                cupk[k] = (unsigned short)upk;
            }
            K += (int)__popcll(m);
            T += __shfl(incl, 63, 64);
        }
    }
    __syncthreads();
    T = __builtin_amdgcn_readfirstlane(T);
    K = __builtin_amdgcn_readfirstlane(K);
    // starts of kept cells lane and lane + 64 (K <= 128)
    const int s_lo = lane < K ? cstart[lane] : 0x7fffffff;
    const int s_hi = lane + 64 < K ? cstart[lane + 64] : 0x7fffffff;
    __syncthreads();

    // exact FP64 test of neighbourList1b (Lib_LinkCell3D.f90:1565-1596) for
    // staged candidate j and the voxel of x index vx (cell offset lx) in the lane's row
    auto exact_at = [&](int lx, int vx, int j) -> bool {
        const int slot = sslot[j], u = cupk[scell[j]];
        const int kx = (u & 15) - 1 - lx, ky = ((u >> 4) & 15) - 1 - lcy, kz = (u >> 8) - 1 - lcz;
        if (kx < -1 || kx > 1 || ky < -1 || ky > 1 || kz < -1 || kz > 1) return false;
        const Frac3 f = slot_frac[slot];                              // FP64 offset in cell
        const double zix = P.ax.zi[0][vx], ziy = P.ax.zi[1][jy], ziz = P.ax.zi[2][jz];
        const double d1 = P.a[0] * (f.x + (kx - zix));
        const double d2 = P.a[1] * (f.y + (ky - ziy));
        const double d3 = P.a[2] * (f.z + (kz - ziz));
        return ((d1 * d1 + d2 * d2) + d3 * d3) <= P.rc2;
    };
    auto kahan_add = [](float& s, float& c, float v) {
        const float y = v - c;
        const float t = s + y;
        c = (t - s) - y;
        s = t;
    };
    float sre = 0.0f, sim = 0.0f, cre = 0.0f, cim = 0.0f;
    float emax = -3.4028234663852886e38f;
    int cnt = 0;
    unsigned nguard = 0;
    // ROW: sums per aperture point (with their Kahan compensations) and
    // largest u of the row's voxels over this lane's part of the candidates
    float rre[NA][TX], rim[NA][TX], kre[NA][TX], kim[NA][TX], umax[TX];
#pragma unroll
    for (int i = 0; i < TX; i++) {
#pragma unroll
        for (int a = 0; a < NA; a++) {
            rre[a][i] = 0.0f; rim[a][i] = 0.0f; kre[a][i] = 0.0f; kim[a][i] = 0.0f;
        }
        umax[i] = -1.0f;
    }

    int t_next = 0, kbase = 0;
    while (t_next < T) {
        // compact the candidates within 3 sigma of the tile box
        int n = 0;
        while (t_next < T) {
            if ((t_next & (TILE_WIN - 1)) == 0) {
                __syncthreads();
                if (lane < TILE_WIN / 32) sflag[lane] = 0;
                __syncthreads();
                const int a = s_lo - 1 - t_next, b = s_hi - 1 - t_next;
                if ((unsigned)a < (unsigned)TILE_WIN) atomicOr(&sflag[a >> 5], 1u << (a & 31));
                if ((unsigned)b < (unsigned)TILE_WIN) atomicOr(&sflag[b >> 5], 1u << (b & 31));
                __syncthreads();
            }
            // cell of candidate t: the starts after the first at or before t
            const int wd = (t_next & (TILE_WIN - 1)) >> 5;
            const unsigned mlo = __builtin_amdgcn_readfirstlane(sflag[wd]);
            const unsigned mhi = __builtin_amdgcn_readfirstlane(sflag[wd + 1]);
            const int k = below((unsigned long long)mhi << 32 | mlo, kbase);
            const int t = min(t_next + lane, T - 1);
            const float4 cr = crec[k];
            const int slot = t + __float_as_int(cr.w);
            float4 pc = p32[slot];
            pc.x += cr.x; pc.y += cr.y; pc.z += cr.z;
            const float ex = fmaxf(0.0f, fabsf(pc.x) - hx);
            const float ey = fmaxf(0.0f, fabsf(pc.y) - hy);
            const float ez = fmaxf(0.0f, fabsf(pc.z) - hz);
            const bool keep = fmaf(ex, ex, fmaf(ey, ey, ez * ez)) <= F.rc_cull2 && t_next + lane < T;
            const unsigned long long m = __ballot(keep);
            const int nk = (int)__popcll(m);
            if (n + nk > CAP) break;                  // these 64 open the next pass
            if (keep) {
                const int p = below(m, n);
                sM[p] = pc;
                sslot[p] = slot;
                scell[p] = (unsigned char)k;
            }
            n += nk;
            kbase += __popc(mlo) + __popc(mhi);
            t_next += 64;
        }
        __syncthreads();
        // records, one candidate per lane, and the groups' lists of the
        // candidates within 3 sigma of their voxels, filled up with the zero
        // record (X = 0: never a member and never in the guard band, u = -1)
        int gn[NG] = {0};
        if (ROW) {
            const unsigned z2 = 16u * CAP * 0x10001u;
            for (int k = lane; k < NG * CAP / 8; k += 64) reinterpret_cast<uint4*>(slist)[k] = make_uint4(z2, z2, z2, z2);
            if (lane < REC) sM[lane * RST + CAP] = make_float4(0.0f, 0.0f, 0.0f, 0.0f);
            if (ROW == 2 && lane == 0) scell[CAP] = 0;
            __syncthreads();
        }
        for (int jb = 0; jb < n; jb += 64) {
            const bool live = jb + lane < n;
            const int j = live ? jb + lane : n - 1;
            const float4 pc = sM[j];
            const int slot = sslot[j];
            const float m2k = -2.0f * k2;
            const float sn = NA == 1 ? sn32[slot] : 0.0f;
            if (ROW) {
                float ey2[GY], ez2[2];
                const float ex = fmaxf(0.0f, fabsf(pc.x) - hx), ex2 = live ? ex * ex : 3.4028234663852886e38f;
#pragma unroll
                for (int h = 0; h < GY; h++) {
                    const float ey = fmaxf(0.0f, fabsf(pc.y - sbox[TX + 2 * h]) - sbox[TX + 2 * h + 1]);
                    ey2[h] = fmaf(ey, ey, ex2);
                }
#pragma unroll
                for (int h = GY; h < GY + 2; h++) {
                    const float ez = fmaxf(0.0f, fabsf(pc.z - sbox[TX + 2 * h]) - sbox[TX + 2 * h + 1]);
                    ez2[h - GY] = ez * ez;
                }
#pragma unroll
                for (int g = 0; g < NG; g++) {
                    const bool in = ey2[g % GY] + ez2[g / GY] <= F.rc_cull2;
                    const unsigned long long m = __ballot(in);
                    if (in) slist[g * CAP + below(m, gn[g])] = (unsigned short)(16 * j);
                    gn[g] += (int)__popcll(m);
                }
            }
            if (live) {
                if (ROW) {
                    const float kyzp = k2 * fmaf(pc.y, pc.y, pc.z * pc.z);
                    float xv[TX];
#pragma unroll
                    for (int i = 0; i < TX; i++) {
                        const float d = pc.x - sbox[i];
                        xv[i] = __builtin_amdgcn_exp2f(fmaf(k2, d * d, kyzp));
                    }
                    sM[j] = make_float4(xv[0], xv[1], xv[2], xv[3]);
                    sM[RST + j] = make_float4(m2k * pc.y, m2k * pc.z, sn, pc.w);
#pragma unroll
                    for (int h = 0; h < NPH; h++) {
                        const float2 c0 = F.app_cs[(2 * h) * F.app_stride + slot];
                        const float2 c1 = F.app_cs[(2 * h + 1) * F.app_stride + slot];
                        sM[(2 + h) * RST + j] = make_float4(c0.x, c0.y, c1.x, c1.y);
                    }
                } else {
                    sM[j] = make_float4(m2k * pc.x, m2k * pc.y, m2k * pc.z,
                                        k2 * fmaf(pc.x, pc.x, fmaf(pc.y, pc.y, pc.z * pc.z)));
                    sM[RST + j] = make_float4(pc.w, sn, 0.0f, 0.0f);
                }
            }
        }
        __syncthreads();
        if (DIAG) {
            // every voxel against every staged candidate, per-pair exact
            // membership with the counts and nearest ranges of the diagnostics
            for (int jb = 0; jb < n; jb += 16) {
                const int je = min(jb + 16, n);
                float pr = 0.0f, pi = 0.0f;
                for (int j = jb; j < je; j++) {
                    const float4 A = sM[j];
                    const float4 C = sM[RST + j];
                    const float e = fmaf(A.x, qcx, fmaf(A.y, qcy, fmaf(A.z, qcz, A.w + kq2)));
                    bool in = act && e >= F.e_rc;
                    if (act && fabsf(e - F.e_rc) <= F.e_band) {
                        nguard++;
                        in = exact_at(lcx, jx, j);
                    }
                    if (F.thin_z) in = in && (unsigned)((cupk[scell[j]] >> 8) - lcz) <= 2u;
                    const float w = in ? __builtin_amdgcn_exp2f(e) : 0.0f;
                    pr = fmaf(w, C.x, pr);
                    pi = fmaf(w, C.y, pi);
                    emax = in ? fmaxf(emax, e) : emax;
                    cnt += in ? 1 : 0;
                }
                kahan_add(sre, cre, pr);
                kahan_add(sim, cim, pi);
            }
        } else if (!ROW) {
            // Branch-free pass over blocks of 32 candidates in the frame
            // t = e - k2 (3 sigma)^2 (member iff t >= 0, weight 2^t scaled by
            // 2^-e_rc), tracking the smallest |t|.  A block in which some
            // lane came within the guard band is summed again with the exact
            // FP64 test for those pairs (uniform branch, rare).
            const float kq2r = kq2 - F.e_rc;
            for (int jb = 0; jb < n; jb += 32) {
                const int je = min(jb + 32, n);
                float pr = 0.0f, pi = 0.0f, dmin = 3.4028234663852886e38f;
#pragma unroll 4
                for (int j = jb; j < je; j++) {
                    const float4 A = sM[j];
                    const float4 C = sM[RST + j];
                    const float t = fmaf(A.x, qcx, fmaf(A.y, qcy, fmaf(A.z, qcz, A.w + kq2r)));
                    const float w = t >= 0.0f ? __builtin_amdgcn_exp2f(t) : 0.0f;
                    pr = fmaf(w, C.x, pr);
                    pi = fmaf(w, C.y, pi);
                    dmin = fminf(dmin, fabsf(t));
                    if (DENSITY) emax = fmaxf(emax, t);
                }
                if (__ballot(dmin <= F.e_band)) {
                    pr = 0.0f; pi = 0.0f;
                    for (int j = jb; j < je; j++) {
                        const float4 A = sM[j];
                        const float4 C = sM[RST + j];
                        const float t = fmaf(A.x, qcx, fmaf(A.y, qcy, fmaf(A.z, qcz, A.w + kq2r)));
                        bool in = t >= 0.0f;
                        if (fabsf(t) <= F.e_band) {
                            nguard++;
                            in = exact_at(lcx, jx, j);
                        }
                        const float w = in ? __builtin_amdgcn_exp2f(t) : 0.0f;
                        pr = fmaf(w, C.x, pr);
                        pi = fmaf(w, C.y, pi);
                    }
                }
                kahan_add(sre, cre, pr);
                kahan_add(sim, cim, pi);
            }
        } else {
            // ROW: steps of NQ candidates (one per part), blocks of ROW_BLOCK
            // steps; the guard band in u is the exponent's band (|u| ~ ln2 |t|
            // near the threshold, so it is 1.44 times as wide).  The member
            // weight is X E = u + 1, taken as w = s (u + 1) with the step
            // s = clamp(2^40 u) in [0, 1]: 1 for u >= 2^-40, 0 for u <= 0, and
            // fractional only inside the guard band, whose pairs the block's
            // re-walk settles.  Each block's sums are added to the running
            // sums with Kahan compensation, and so are the re-walk's
            // corrections (the block sums are not live across the re-walk,
            // which sets the register peak).
            int gmax = gn[0];
#pragma unroll
            for (int g = 1; g < NG; g++) gmax = max(gmax, gn[g]);
            const int nst = (gmax + NQ - 1) / NQ;
            const unsigned short* const list = slist + grp * CAP + squart;
            auto step = [](float u) { return __builtin_amdgcn_fmed3f(u * 1099511627776.0f, 0.0f, 1.0f); };
            // part c of the candidate with list entry e
            auto part = [&](int e, int c) -> float4 {
                return *reinterpret_cast<const float4*>(reinterpret_cast<const char*>(sM) + e + 16 * RST * c);
            };
            auto load_x = [&](int e, float* xv) {
                const float4 X = part(e, 0);
                xv[0] = X.x; xv[1] = X.y; xv[2] = X.z; xv[3] = X.w;
            };
            // its (cos, sin) pairs (B = its part 1)
            auto load_ph = [&](int e, const float4& B, float* pc, float* ps) {
                if (NA == 1) {
                    pc[0] = B.w;
                    ps[0] = B.z;
                } else {
#pragma unroll
                    for (int h = 0; h < NPH; h++) {
                        const float4 Ph = part(e, 2 + h);
                        pc[2 * h] = Ph.x; ps[2 * h] = Ph.y; pc[2 * h + 1] = Ph.z; ps[2 * h + 1] = Ph.w;
                    }
                }
            };
            // z offset of its cell
            auto zoff = [&](int e) -> int { return cupk[scell[e >> 4]] >> 8; };
            for (int kb = 0; kb < nst; kb += ROW_BLOCK) {
                const int ke = min(kb + ROW_BLOCK, nst);
                // smallest |u| of the block's even and odd steps, voxels 0-1 and 2-3
                constexpr float far = 3.4028234663852886e38f;
                float dmin[2][2] = {{far, far}, {far, far}};
                float bre[NA][TX], bim[NA][TX];
#pragma unroll
                for (int i = 0; i < TX; i++)
#pragma unroll
                    for (int a = 0; a < NA; a++) { bre[a][i] = 0.0f; bim[a][i] = 0.0f; }
                auto pairs = [&](int kk, float* near) {
                    const int e = list[NQ * kk];
                    float xv[TX];
                    load_x(e, xv);
                    const float4 B = part(e, 1);
                    float E = __builtin_amdgcn_exp2f(fmaf(B.x, qcy, fmaf(B.y, qcz, kyz)));
                    if (ROW == 2) {
                        E = (unsigned)(zoff(e) - lcz) <= 2u ? E : 0.0f;
                    }
                    float pc[NA], ps[NA];
                    load_ph(e, B, pc, ps);
#pragma unroll
                    for (int i = 0; i < TX; i++) {
                        const float u = fmaf(xv[i], E, -1.0f);
                        const float s = step(u);
                        const float w = fmaf(s, u, s);
#pragma unroll
                        for (int a = 0; a < NA; a++) {
                            bre[a][i] = fmaf(w, pc[a], bre[a][i]);
                            bim[a][i] = fmaf(w, ps[a], bim[a][i]);
                        }
                        near[i >> 1] = fminf(near[i >> 1], fabsf(u));
                        if (DENSITY) umax[i] = fmaxf(umax[i], u);
                    }
                };
                int kk = kb;
                for (; kk + 1 < ke; kk += 2) {
                    pairs(kk, dmin[0]);
                    pairs(kk + 1, dmin[1]);
                }
                if (kk < ke) pairs(kk, dmin[0]);
#pragma unroll
                for (int i = 0; i < TX; i++)
#pragma unroll
                    for (int a = 0; a < NA; a++) {
                        kahan_add(rre[a][i], kre[a][i], bre[a][i]);
                        kahan_add(rim[a][i], kim[a][i], bim[a][i]);
                    }
#pragma unroll
                for (int hh = 0; hh < 4; hh++) {
                    const int h = hh & 1, v0 = hh & 2;
                    if (!__ballot(dmin[h][v0 >> 1] <= F.e_band)) continue;
                    for (int kk = kb + h; kk < ke; kk += 2) {
                        const int e = list[NQ * kk];
                        float xv[TX];
                        load_x(e, xv);
                        const float4 B = part(e, 1);
                        float E = __builtin_amdgcn_exp2f(fmaf(B.x, qcy, fmaf(B.y, qcz, kyz)));
                        if (ROW == 2) E = (unsigned)(zoff(e) - lcz) <= 2u ? E : 0.0f;
#pragma unroll
                        for (int i = v0; i < v0 + 2; i++) {
                            const float u = fmaf(xv[i], E, -1.0f);
                            if (fabsf(u) <= F.e_band) {
                                const int vx = min(x0 + i, x1);
                                // one re-test per aperture point it settles
                                if (row_act && x0 + i <= x1) nguard += NA;
                                const bool in = exact_at(P.ax.ql[0][vx].lc, vx, e >> 4);
                                // replace the pass's s (u + 1) by the exact test's weight
                                const float s = step(u);
                                const float d = (in ? u + 1.0f : 0.0f) - fmaf(s, u, s);
                                float pc[NA], ps[NA];
                                load_ph(e, B, pc, ps);
#pragma unroll
                                for (int a = 0; a < NA; a++) {
                                    kahan_add(rre[a][i], kre[a][i], d * pc[a]);
                                    kahan_add(rim[a][i], kim[a][i], d * ps[a]);
                                }
                            }
                        }
                    }
                }
            }
        }
        __syncthreads();
    }

    // the lane's voxels: ROW, voxels s NV .. s NV + NV - 1 of its row, from
    // the parts' sums added in part order through LDS; otherwise its own
    float vre[NA][NV], vim[NA][NV], vem[NV];
    if (ROW && NQ > 1) {
        float2* red = reinterpret_cast<float2*>(sM);                  // [64 lanes][TX voxels]
        float* redm = reinterpret_cast<float*>(sM) + 2 * 64 * TX;     // [64 lanes][TX voxels]
        const int rb = lane & ~(NQ - 1);
#pragma unroll
        for (int ap = 0; ap < NA; ap++) {
            if (ap > 0) __syncthreads();                              // the previous point's reads
#pragma unroll
            for (int i = 0; i < TX; i++) {
                red[TX * lane + i] = make_float2(rre[ap][i], rim[ap][i]);
                if (DENSITY && ap == 0) redm[TX * lane + i] = umax[i];
            }
            __syncthreads();
#pragma unroll
            for (int t = 0; t < NV; t++) {
                const int i = squart * NV + t;
                float a = 0.0f, b = 0.0f, um = -1.0f;
#pragma unroll
                for (int q = 0; q < NQ; q++) {
                    const float2 v = red[TX * (rb + q) + i];
                    a += v.x;
                    b += v.y;
                    if (DENSITY && ap == 0) um = fmaxf(um, redm[TX * (rb + q) + i]);
                }
                vre[ap][t] = a;
                vim[ap][t] = b;
                // largest exponent in the t frame: 2^t = u + 1 (u = -1: no candidate)
                if (ap == 0)
                    vem[t] = (DENSITY && um > -1.0f) ? __builtin_amdgcn_logf(um + 1.0f) : -3.4028234663852886e38f;
            }
        }
    } else if (ROW) {
#pragma unroll
        for (int t = 0; t < NV; t++) {
#pragma unroll
            for (int ap = 0; ap < NA; ap++) {
                vre[ap][t] = rre[ap][t];
                vim[ap][t] = rim[ap][t];
            }
            vem[t] = (DENSITY && umax[t] > -1.0f) ? __builtin_amdgcn_logf(umax[t] + 1.0f) : -3.4028234663852886e38f;
        }
    } else {
        vre[0][0] = sre;
        vim[0][0] = sim;
        vem[0] = emax;
    }

#pragma unroll
    for (int t = 0; t < NV; t++) {
        const int vx = ROW ? x0 + squart * NV + t : ix;
        if (!(ROW ? vx <= x1 && row_act : act)) continue;
        const int64_t o = (int64_t)vx + (int64_t)P.Mx * (iy + (int64_t)P.My * iz);
        const float emax_ = vem[t];
        // nearest squared range from the largest exponent (huge(1.0) if none).
        // Without DIAG the largest exponent is over every candidate, members
        // or not: it differs from the members' only when no candidate is
        // nearer than about 3 sigma, where the density is 0 either way.
        float r2m;
        if (DIAG) r2m = emax_ > -3.4028234663852886e38f ? emax_ / k2 : 3.4028234663852886e38f;
        else r2m = emax_ > -3.4028234663852886e38f ? (emax_ + F.e_rc) * F.inv_k2 : 3.4028234663852886e38f;
        float rh = 1.0f;
        if (DENSITY && P.use_density) {
            // convertScaledRangeToRho (Lib_DynamicalTwoBeamImaging.f90:1973-1994) in FP32
            const float sg = (float)P.sigma;
            if (r2m < sg * sg) rh = 1.0f;
            else if (r2m > 4 * sg * sg) rh = 0.0f;
            else {
                const float xx = sqrtf(r2m) / sg - 1.0f;
                rh = 1.0f - xx * xx * xx * fmaf(6.0f * xx, xx, fmaf(-15.0f, xx, 10.0f));
            }
        }
#pragma unroll
        for (int ap = 0; ap < NA; ap++) {
            const float sre_ = vre[ap][t], sim_ = vim[ap][t];
            // x = S / max(|S|, 1e-16).  Without DIAG the sums carry the factor
            // 2^-e_rc of the t frame (weights 2^t = 2^(e - e_rc)); it cancels in
            // S/|S| and moves the threshold.
            const float m2 = fmaf(sre_, sre_, sim_ * sim_);
            const float ww = m2 > (DIAG ? 1.0e-32f : F.m2_min) ? __builtin_amdgcn_rsqf(m2)
                                                              : (DIAG ? 1.0e16f : 1.0e16f * F.w_scale);
            const int64_t oa = o + ap * F.field_stride;
            if (DENSITY) field[oa] = make_float4(sre_ * ww, sim_ * ww, rh, 0.0f);
            else reinterpret_cast<float2*>(field)[oa] = make_float2(sre_ * ww, sim_ * ww);
        }
        if (DIAG) {
            out_cnt[o] = cnt;
            out_r2m[o] = r2m;
        }
    }
    // spread over GUARD_SLOTS lines: many waves adding into one address
    // serialise.  ROW lanes counted only their active voxels.
    if ((ROW || act) && nguard)
        atomicAdd(guard_count + GUARD_STRIDE * (blockIdx.x & (GUARD_SLOTS - 1)), (unsigned long long)nguard);
}

}  // namespace d2bi
