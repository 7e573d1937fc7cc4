// d2bi_axis.cuh -- per-axis voxel tables (link cell, offset in the cell, FP32
// position of each voxel coordinate), uploaded once per condition.
//
// One part of the single translation unit d2bi_gpu.hip, which includes the
// parts in order so that kernels and the device helpers they call compile
// together; each part uses the definitions of the parts before it.
#pragma once

namespace d2bi {

// ------------------------------------------------------------------ voxel axis tables

// The voxel and link cells are cuboidal (findTransformedSupercell gives a
// diagonal D, Lib_DiffractionConditions.f90:1074-1077), so a voxel's link
// cell and in-cell offset factorise per axis: for axis x,
//   xx = a_vox(1,1)*ix - lc_delta(1),  zi = ia(1,1)*xx,
//   cell = mod(floor(zi) + 16*Ex, Ex), zi = zi - cell
// (neighbourList1b, Lib_LinkCell3D.f90:1549-1565).  The zero off-diagonal
// terms of the reference's 3x3 products add +-0 and change no bit.
static constexpr int TILE = 4;                       // FAST voxel tiles: 4 voxels along x (y and z: 4 or 8)

// FP32 voxel position along one axis relative to the link cell of its
// FAST tile's first voxel, and that cell offset
struct QL {
    float q;
    int lc;
};

// Voxel positions relative to the first link cell of their tile: table k
// holds axis QL_AXIS[k] for tiles of QL_TILE[k] voxels along it.
static constexpr int NQL = 5;
static constexpr int QL_AXIS[NQL] = {0, 1, 2, 2, 1};
static constexpr int QL_TILE[NQL] = {4, 4, 4, 8, 8};

struct AxisTables {
    std::vector<int> cell[3];
    std::vector<double> zi[3];
    std::vector<QL> ql[NQL];       // x, y, z for 4-voxel tiles; z, y for 8-voxel tiles
    std::vector<char> packed;      // the tables as uploaded without pinned memory
};

static bool diagonal(const double* m)
{
    return m[1] == 0.0 && m[2] == 0.0 && m[3] == 0.0 && m[5] == 0.0 && m[6] == 0.0 && m[7] == 0.0;
}

static int axis_tables(const d2bi_record* r, const d2bi_plan* p, AxisTables* t)
{
    if (!diagonal(r->gk_a) || !diagonal(p->a_col) || !diagonal(p->ia_col))
        return seterr(D2BI_ERR_ARG, "voxel/link cells must be cuboidal (diagonal cell matrices)");
    const int M[3] = {p->Mx, p->My, p->Mz};
    const int E[3] = {p->Ex, p->Ey, p->Ez};
    for (int a = 0; a < 3; a++) {
        t->cell[a].resize(M[a]);
        t->zi[a].resize(M[a]);
        const double av = r->gk_a[4 * a], ia = p->ia_col[4 * a];
        for (int i = 0; i < M[a]; i++) {
            double xx = av * i - p->lc_delta[a];
            double zi = ia * xx;
            int c = ((int)floor(zi) + 16 * E[a]) % E[a];
            t->cell[a][i] = c;
            t->zi[a][i] = zi - c;
        }
        for (int i = 1; i < M[a]; i++)
            if (t->cell[a][i] < t->cell[a][i - 1])
                return seterr(D2BI_ERR_ARG, "voxel column wraps the link-cell box (axis %d)", a);
        const double side = p->a_col[4 * a];
        for (int k = 0; k < NQL; k++) {
            if (QL_AXIS[k] != a) continue;
            const int ts = QL_TILE[k];
            t->ql[k].resize(M[a]);
            for (int i = 0; i < M[a]; i++) {
                const int lc = t->cell[a][i] - t->cell[a][(i / ts) * ts];
                t->ql[k][i] = QL{(float)(side * (t->zi[a][i] + lc)), lc};
            }
        }
    }
    return D2BI_OK;
}

struct AxisDev {
    const int* cell[3];
    const double* zi[3];
    const QL* ql[NQL];
};

// The axis tables of one condition as one block: doubles zi, then QL, then
// ints cell.
static size_t axis_bytes(const AxisTables& t)
{
    size_t n = 0;
    for (int k = 0; k < NQL; k++) n += sizeof(QL) * t.ql[k].size();
    for (int a = 0; a < 3; a++) n += (sizeof(double) + sizeof(int)) * t.cell[a].size();
    return (n + 15) & ~(size_t)15;
}

// Write the block into host memory h, and d's pointers for a block at dev.
static void axis_pack(const AxisTables& t, char* h, const char* dev, AxisDev* d)
{
    size_t o = 0;
    auto put = [&](const auto& v, auto* ptr) {
        const size_t bytes = sizeof(v[0]) * v.size();
        std::memcpy(h + o, v.data(), bytes);
        *ptr = reinterpret_cast<std::remove_reference_t<decltype(*ptr)>>(dev + o);
        o += bytes;
    };
    for (int a = 0; a < 3; a++) put(t.zi[a], &d->zi[a]);
    for (int k = 0; k < NQL; k++) put(t.ql[k], &d->ql[k]);
    for (int a = 0; a < 3; a++) put(t.cell[a], &d->cell[a]);
}

// Copy the axis tables into workspace w.  t must stay alive until the
// stream has executed the copy.
static int upload_axis(AxisTables& t, AxisDev* d, hipStream_t s, Workspace& w)
{
    const size_t bytes = axis_bytes(t);
    CHK(w.ax_tab.ensure(bytes));
    void* h;
    if (w.ax_tab.arena) {
        // a workspace that must not allocate: copy from pageable memory, not
        // through the (growable) pinned staging buffer
        t.packed.resize(bytes);
        h = t.packed.data();
    } else {
        CHK(pinned(bytes, &h));
    }
    axis_pack(t, (char*)h, w.ax_tab.as<char>(), d);
    HIPCHK(hipMemcpyAsync(w.ax_tab.p, h, bytes, hipMemcpyHostToDevice, s));
    if (!w.ax_tab.arena) {
        // the pinned buffer is reused by later calls: they wait for this event
        HIPCHK(hipEventRecord(g.ev[9], s));
        g.pinned_busy = true;
    }
    return D2BI_OK;
}

struct VoxParams {
    int Mx, My, Mz;
    int Ex, Ey, Ez;
    double a[3];                // link-cell sides (diagonal of a_col)
    double rc2, i2s2, sigma;
    int use_density;
    AxisDev ax;
};

// convertScaledRangeToRho (Lib_DynamicalTwoBeamImaging.f90:1973-1994)
__device__ inline double rho_of(double r2_min, double sig)
{
    if (r2_min < sig * sig) return 1.0;
    if (r2_min > 4 * sig * sig) return 0.0;
    double xx = sqrt(r2_min) / sig - 1.0;
    return 1 - ((xx * xx) * xx) * ((10 - 15 * xx) + (6 * xx) * xx);
}

}  // namespace d2bi
