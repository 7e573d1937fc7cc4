// d2bi_run.cuh -- one imaging condition: planning, binning, voxelisation (with the
// FAST variant choice), integration, the aperture sum and the field API.
//
// One part of the single translation unit d2bi_gpu.hip, which includes the
// parts in order so that kernels and the device helpers they call compile
// together; each part uses the definitions of the parts before it.
#pragma once

namespace d2bi {

// ------------------------------------------------------------------ orchestration

struct Timer {
    hipEvent_t* ev;
    hipStream_t s;
    int record(int i)
    {
        HIPCHK(hipEventRecord(ev[i], s));
        return D2BI_OK;
    }
    double ms(int a, int b)
    {
        float t = 0.0f;
        (void)hipEventElapsedTime(&t, ev[a], ev[b]);
        return t;
    }
};

static void fill_vox_params(const d2bi_record* r, const d2bi_plan* p, const AxisDev& ax, VoxParams* V)
{
    V->Mx = p->Mx; V->My = p->My; V->Mz = p->Mz;
    V->Ex = p->Ex; V->Ey = p->Ey; V->Ez = p->Ez;
    V->a[0] = p->a_col[0]; V->a[1] = p->a_col[4]; V->a[2] = p->a_col[8];
    V->rc2 = p->rc2; V->i2s2 = p->i2s2; V->sigma = p->sigma;
    V->use_density = r->use_density ? 1 : 0;
    V->ax = ax;
}

// Tile of a FAST kernel variant, 4 voxels along x: variants 0 (a lane per
// voxel) and 1 (rows) use 4 x 4 x 4, 2 4 x 4 x 8 and 3 4 x 8 x 8.
static int variant_tz(int variant) { return variant >= 2 ? 8 : 4; }
static int variant_ty(int variant) { return variant == 3 ? 8 : 4; }

// The order of the FAST voxel kernel's tiles over its workgroups and the
// grid it needs (8 per_xcd workgroups): orders 0 and 1 launch one workgroup
// per tile (rounded up to a multiple of 8); order 2 deals whole rows of ntx
// tiles, so each XCD gets ceil(rows / 8) rows.
static void set_tile_order(FastParams* F, int order)
{
    F->order = order;
    if (order == 2) {
        const int rows = (F->ntiles + F->ntx - 1) / F->ntx;
        F->per_xcd = ((rows + 7) / 8) * F->ntx;
    } else {
        F->per_xcd = (F->ntiles + 7) / 8;
    }
}

// Link cells in the largest unwrapped cell range of a 4 x ty x tz tile.
static int tile_cells(const d2bi_plan* p, const AxisTables& tab, int tz, int ty = TILE)
{
    int worst = 1;
    for (int a = 0; a < 3; a++) {
        const int M = a == 0 ? p->Mx : a == 1 ? p->My : p->Mz;
        const int ts = a == 2 ? tz : a == 1 ? ty : TILE;
        int mx = 0;
        for (int t0 = 0; t0 < M; t0 += ts)
            mx = std::max(mx, tab.cell[a][std::min(M, t0 + ts) - 1] - tab.cell[a][t0] + 3);
        worst *= mx;
    }
    return worst;
}

// Binary exponents that the factors of a member's weight take in a tile of 4 x
// ty x tz voxels: those of the range from the tile's centre (x: along x too;
// the row kernels' factors take that from each voxel).
static double tile_bits(const d2bi_plan* p, int tz, int ty, bool x)
{
    const double hx = x ? 0.5 * (std::min(TILE, p->Mx) - 1) * p->xmax[0] / p->Mx : 0.0;
    const double hy = 0.5 * (std::min(ty, p->My) - 1) * p->xmax[1] / p->My;
    const double hz = 0.5 * (std::min(tz, p->Mz) - 1) * p->xmax[2] / p->Mz;
    const double q = std::sqrt(hx * hx + hy * hy + hz * hz) + 3.0 * p->sigma;
    return q * q * p->i2s2 * 1.4426950408889634;
}

// What the FAST kernels allow them.  A member's X is at least 2^-bits and its
// 2^t at most 2^(bits + 6.5), FP32's range ends at 2^-126, and eight roundings of
// 85 leave u within half the guard band.  A 4 x 8 x 8 tile has 22 at four cubic
// voxels per lattice parameter and 46 at two; 4 x 4 x 8 has 81 at one; voxels of
// 1.4 x 1.4 x 2.7 sigma have 134 in a 4 x 8 x 8 tile (NaN) and 41 in 4 x 4 x 4.
// The kernel of a lane per voxel has no such factors, but its exponent is a
// difference of the range from the tile's centre in x too: 130 keep its
// roundings within the guard band.
static constexpr double TILE_BITS = 85.0, VOXEL_BITS = 130.0;

static bool fast_fits(const d2bi_plan* p)
{
    return tile_bits(p, TILE, TILE, false) <= TILE_BITS && tile_bits(p, TILE, TILE, true) <= VOXEL_BITS;
}

// Launch parameters of the FAST voxel kernel for a plan, tiles of 4 x ty x tz.
static int fast_params(const d2bi_plan* p, const AxisTables& tab, const VoxParams& V, FastParams* Fo, int tz,
                       int ty = TILE)
{
    FastParams& F = *Fo;
    F.v = V;
    F.ntx = (p->Mx + TILE - 1) / TILE;
    F.nty = (p->My + ty - 1) / ty;
    F.ntz = (p->Mz + tz - 1) / tz;
    F.ntiles = F.ntx * F.nty * F.ntz;
    set_tile_order(&F, 2);
    F.app_cs = nullptr;
    F.app_stride = 0;
    F.field_stride = 0;
    // guard band: the FP32 exponent carries <= ~2e-6 relative error (inputs
    // rounded once from FP64, three FMAs); +-1e-5 relative covers it 5x
    const double k2 = -p->i2s2 * 1.4426950408889634;
    F.k2 = (float)k2;
    F.e_rc = (float)(k2 * p->rc2);
    F.e_band = (float)(std::fabs(k2 * p->rc2) * 1.0e-5);
    F.w_scale = (float)std::exp2((double)F.e_rc);
    F.m2_min = (float)(1.0e-32 / ((double)F.w_scale * (double)F.w_scale));
    F.inv_k2 = (float)(1.0 / k2);
    F.rc_cull2 = (float)(p->rc2 * (1.0 + 1.0e-4));
    F.cellf[0] = (float)p->a_col[0]; F.cellf[1] = (float)p->a_col[4]; F.cellf[2] = (float)p->a_col[8];
    // cells thinner than 3 sigma by more than rounding (the guard band, ~2e-5
    // A, covers less): only z can be, x and y are wide by construction
    const double rc = std::sqrt(p->rc2), thin = rc * (1.0 - 1.0e-7);
    if (p->a_col[0] < thin || p->a_col[4] < thin)
        return seterr(D2BI_ERR_ARG, "link cells %.6f x %.6f narrower than 3 sigma = %.6f", p->a_col[0],
                      p->a_col[4], rc);
    F.thin_z = p->a_col[8] < thin ? 1 : 0;
    // the unwrapped cell range of a tile must fit the per-tile cell table
    const int worst = tile_cells(p, tab, tz, ty);
    if (worst > TILE_MAXC) return seterr(D2BI_ERR_CAPACITY, "voxel tile spans %d link cells (max %d)", worst, TILE_MAXC);
    return D2BI_OK;
}

// The arithmetic that images a condition in *mode: FP64 where a voxel is so
// tall (about 5 sigma) that even the smallest FAST tile has too many bits.  What
// the FAST kernels refuse is refused there too.
static int condition_mode(const d2bi_plan* p, const AxisTables& tab, int* mode)
{
    if (*mode != D2BI_MODE_FAST || fast_fits(p)) return D2BI_OK;
    FastParams F;
    CHK(fast_params(p, tab, VoxParams{}, &F, TILE));
    *mode = D2BI_MODE_FP64;
    return D2BI_OK;
}

// Launch parameters of the region kernels for a plan; false where they do not
// apply: a region spanning more link cells than its table holds (voxels
// coarser than about a third of the lattice parameter), or so long that the
// culls' FP32 positions might lose a member.  A position takes at most ten
// roundings of 2^-24 of the range's length L, 1e-6 L over three axes, and the
// culls allow half of 1e-4 of 3 sigma: 150 sigma, of which 100 are used (15 at
// four voxels per lattice parameter, 28 at one).
static bool region_params(const d2bi_plan* p, const AxisTables& tab, const VoxParams& V, RegionParams* R)
{
    R->v = V;
    const int M[3] = {p->Mx, p->My, p->Mz};
    int n[3];
    int64_t worst = 1;
    for (int a = 0; a < 3; a++) {
        int mx = 0;
        for (int t0 = 0; t0 < M[a]; t0 += REG)
            mx = std::max(mx, tab.cell[a][std::min(M[a], t0 + REG) - 1] - tab.cell[a][t0] + 3);
        worst *= mx;
        if (!(mx * p->a_col[4 * a] <= 100.0 * p->sigma)) return false;
        n[a] = (M[a] + REG - 1) / REG;
        R->cellf[a] = (float)p->a_col[4 * a];
    }
    if (worst > REG_MAXC) return false;
    R->nrx = n[0];
    R->nry = n[1];
    R->nrz = n[2];
    R->nreg = n[0] * n[1] * n[2];
    R->per_xcd = ((n[1] * n[2] + 7) / 8) * n[0];
    R->rc_cull2 = (float)(p->rc2 * (1.0 + 1.0e-4));
    return true;
}

// FP64 voxelisation of na aperture points (1, 2 or 4; phases cs at a stride
// of cs_stride slots, fields at a stride of out_stride voxels) from workspace
// w's binned points; cnt and r2m: optional diagnostics.  The per-voxel walk
// takes over where a region spans too many link cells.
static int launch_voxel_fp64(const d2bi_plan* p, const AxisTables& tab, const VoxParams& V, int na, Workspace& w,
                             const double2* cs, int64_t cs_stride, int64_t out_stride, int* cnt, double* r2m,
                             hipStream_t s)
{
    RegionParams R;
    if (region_params(p, tab, V, &R)) {
        auto go = [&](auto kern) {
            hipLaunchKernelGGL(kern, dim3(8 * R.per_xcd), dim3(64 * F64R_NW), 0, s, R, w.cell_start.as<int>(),
                               w.slot_frac.as<Frac3>(), w.slot_p32.as<float4>(), cs, cs_stride, w.f64_re.as<double>(),
                               w.f64_im.as<double>(), out_stride, w.f64_rho.as<double>(), cnt, r2m);
        };
        const bool dens = V.use_density != 0;
        if (cnt || r2m) go(k_voxel_fp64_region<1, true, true>);
        else if (dens && na == 4) go(k_voxel_fp64_region<4, true, false>);
        else if (dens && na == 2) go(k_voxel_fp64_region<2, true, false>);
        else if (dens) go(k_voxel_fp64_region<1, true, false>);
        else if (na == 4) go(k_voxel_fp64_region<4, false, false>);
        else if (na == 2) go(k_voxel_fp64_region<2, false, false>);
        else go(k_voxel_fp64_region<1, false, false>);
    } else {
        const dim3 grid((p->Mx + 7) / 8, (p->My + 7) / 8, (p->Mz + 3) / 4);
        auto go = [&](auto kern) {
            hipLaunchKernelGGL(kern, grid, dim3(256), 0, s, V, w.cell_start.as<int>(), w.slot_frac.as<Frac3>(), cs,
                               cs_stride, w.f64_re.as<double>(), w.f64_im.as<double>(), out_stride,
                               w.f64_rho.as<double>(), cnt, r2m);
        };
        if (na == 4) go(k_voxel_fp64<4>);
        else if (na == 2) go(k_voxel_fp64<2>);
        else go(k_voxel_fp64<1>);
    }
    HIPCHK(hipGetLastError());
    return D2BI_OK;
}

// A variant whose tiles span more link cells than the per-tile table holds, or
// whose factors span more than TILE_BITS, gives way to the next smaller tile (3
// to 2, 2 to 1).
static int effective_variant(const d2bi_plan* p, const AxisTables& tab, int variant)
{
    if (variant == 3 && (tile_cells(p, tab, 8, 8) > TILE_MAXC || tile_bits(p, 8, 8, false) > TILE_BITS)) variant = 2;
    if (variant == 2 && (tile_cells(p, tab, 8) > TILE_MAXC || tile_bits(p, 8, 4, false) > TILE_BITS)) variant = 1;
    return variant;
}

static int variant_params(const d2bi_plan* p, const AxisTables& tab, const VoxParams& V, int* variant,
                          FastParams* F)
{
    *variant = effective_variant(p, tab, *variant);
    return fast_params(p, tab, V, F, variant_tz(*variant), variant_ty(*variant));
}

// Kernel instance for (diagnostics, density, variant); link cells thinner
// than 3 sigma along z take a row kernel (variant 1, 2 or 3) with the
// z-offset test.
template <bool DENS, int ROW, class Go>
static void pick_row(int tz, int ty, Go go)
{
    if (ty == 8) go(k_voxel_tile<DENS, false, ROW, 8, 8>);
    else if (tz == 8) go(k_voxel_tile<DENS, false, ROW, 8>);
    else go(k_voxel_tile<DENS, false, ROW, 4>);
}

template <class Go>
static void pick_tile(bool diag, bool dens, int variant, bool thin_z, Go go)
{
    if (diag) { go(k_voxel_tile<true, true, 0, 4>); return; }
    const int tz = variant_tz(variant), ty = variant_ty(variant);
    if (!thin_z && variant == 0) {
        if (dens) go(k_voxel_tile<true, false, 0, 4>);
        else go(k_voxel_tile<false, false, 0, 4>);
    } else if (thin_z) {
        if (dens) pick_row<true, 2>(tz, ty, go);
        else pick_row<false, 2>(tz, ty, go);
    } else {
        if (dens) pick_row<true, 1>(tz, ty, go);
        else pick_row<false, 1>(tz, ty, go);
    }
}

template <bool DIAG>
static void launch_tile(const FastParams& F, int variant, bool dens, const int* cell_start,
                        const Frac3* slot_frac, const float4* p32, const float* sn32, float4* field, int* cnt,
                        float* r2m, unsigned long long* gc, hipStream_t s)
{
    pick_tile(DIAG, dens, variant, F.thin_z != 0, [&](auto kern) {
        hipLaunchKernelGGL(kern, dim3(8 * F.per_xcd), dim3(64), 0, s, F, cell_start, slot_frac, p32, sn32,
                           field, cnt, r2m, gc);
    });
}

// Choice of the FAST voxel kernel variant (0: a lane per voxel; rows of four
// voxels: 1: a lane per row and quarter of the candidates of a 4 x 4 x 4 tile,
// 2: per row and half of the candidates of a 4 x 4 x 8 tile, 3: per row of a
// 4 x 8 x 8 tile).  The variants sum the same atoms in different orders, so
// their fields agree to FP32 rounding, not bit for bit; the choice is
// therefore fixed by the grid's size, so that a condition images the same in
// every process (variant_params falls back to a smaller tile where a cell
// range does not fit).  A larger tile stages fewer candidates per voxel, but
// needs enough tiles to fill the chip: 16 waves of variant 3 fit a CU, 20 of
// 1 and 2, and below a few rounds of 4096 the waves' own latency counts.
// Measured (voxel kernel, us, variants 1/2/3 at four voxels per lattice
// parameter; tiles of variant 3): 14^3 cells 16/20/28 (686), 20^3 25/25/31
// (2000), 28^3 48/44/47 (5488), 36^3 82/69/70 (11664), 40^3 109/89/88 (16000),
// 50^3 204/163/153 (31250), 150 x 150 x 100 3463/2528/2292 (562500).
// D2BI_FAST_VARIANT=0|1|2|3 forces a variant; D2BI_FAST_TUNE=1 instead times
// all on the first condition of each voxel-grid shape and keeps the fastest
// (results then depend on the timing).
static int default_variant(const d2bi_plan* p, int most = 3)
{
    const int64_t t2 = (int64_t)((p->Mx + 3) / 4) * ((p->My + 3) / 4) * ((p->Mz + 7) / 8);
    const int64_t t3 = (int64_t)((p->Mx + 3) / 4) * ((p->My + 7) / 8) * ((p->Mz + 7) / 8);
    return std::min(most, t3 >= 16000 ? 3 : t2 >= 5000 ? 2 : 1);
}

// The aperture sum's variant, the same for a shared pass and for a pass per
// point: tiles of 4 x 8 x 8 with four points' sums leave room for two or
// three waves per SIMD and are no faster (60 x 60 x 40 cells, eight points,
// whole call: 1377 us, variant 2 1338, variant 1 1537).
static constexpr int APERTURE_VARIANT = 2;

static std::map<std::array<int, 7>, int> g_variant_cache;

static bool tune_variants()
{
    const char* e = std::getenv("D2BI_FAST_TUNE");
    return e && e[0] == '1' && e[1] == 0;
}

static int forced_variant()
{
    const char* env = std::getenv("D2BI_FAST_VARIANT");
    if (env && env[0] >= '0' && env[0] <= '3' && env[1] == 0) return env[0] - '0';
    return -1;
}

// the variant for a shape: forced, fixed, or tuned (-1 if not tuned yet)
static int known_variant(const d2bi_plan* p, bool dens)
{
    const int f = forced_variant();
    if (f >= 0) return f;
    if (!tune_variants()) return default_variant(p);
    const std::array<int, 7> key{p->Mx, p->My, p->Mz, p->Ex, p->Ey, p->Ez, dens ? 1 : 0};
    auto it = g_variant_cache.find(key);
    return it == g_variant_cache.end() ? -1 : it->second;
}

template <class TimeFn>
static int fast_variant(const d2bi_plan* p, bool dens, bool diag, bool thin_z, int most, TimeFn time_variant)
{
    auto& cache = g_variant_cache;
    const int f = forced_variant();
    if (f >= 0) return f;
    if (diag) return 0;
    if (!tune_variants()) return default_variant(p, most);
    const std::array<int, 7> key{p->Mx, p->My, p->Mz, p->Ex, p->Ey, p->Ez, dens ? 1 : 0};
    auto it = cache.find(key);
    if (it != cache.end()) return it->second;
    // each variant twice, the second (warm-cache) timing counts; thin z
    // cells have only the row kernels
    const int v0 = thin_z ? 1 : 0;
    float t[4] = {0.0f, 0.0f, 0.0f, 0.0f};
    for (int rep = 0; rep < 2; rep++)
        for (int v = v0; v < 4; v++) {
            t[v] = time_variant(v);
            if (t[v] < 0) return seterr(D2BI_ERR_HIP, "variant timing failed");
        }
    int best = v0;
    for (int v = v0 + 1; v < 4; v++)
        if (t[v] < t[best]) best = v;
    cache[key] = best;
    return best;
}

// Tile orders the tuner may choose; 2 (rows dealt to the XCDs) is the
// default, the fastest of the three on c1, c2 and c3 (up to 12 % over per-XCD
// ranges, whose z slabs leave the XCDs given vacuum above and below a padded
// foil idle early).
static const int TILE_ORDERS[3] = {0, 1, 2};

// Tuner key of the FAST voxel kernel's tile order: the shape and the variant
// that runs (after the fallback of variant_params).
static TuneKey tile_order_key(const d2bi_plan* p, const AxisTables& tab, bool dens, int variant)
{
    const int v = effective_variant(p, tab, variant);
    return TuneKey{TUNE_TILE_ORDER, p->Mx, p->My, p->Mz, p->Ex, p->Ey, p->Ez, dens ? 1 : 0, v};
}

// Voxelise into the mode's field buffers of workspace w; optional count /
// r2min outputs.  fresh: the workspace's guard counters are zero (they were
// cleared for this condition's binning).  most: the largest variant the
// default choice may take.
static int run_voxel(const d2bi_record* r, const d2bi_plan* p, const AxisTables& tab, const AxisDev& ax,
                     int mode, bool want_diag, bool fresh, hipStream_t s, Workspace& w, int most = 3)
{
    const int64_t nvox = (int64_t)p->Mx * p->My * p->Mz;
    VoxParams V;
    fill_vox_params(r, p, ax, &V);
    int* dcnt = nullptr;
    void* dr2 = nullptr;
    if (want_diag) {
        CHK(w.cnt.ensure(sizeof(int) * nvox));
        CHK(w.r2m.ensure(sizeof(double) * nvox));
        dcnt = w.cnt.as<int>();
        dr2 = w.r2m.p;
    }
    if (mode == D2BI_MODE_FP64) {
        CHK(w.f64_re.ensure(sizeof(double) * nvox));
        CHK(w.f64_im.ensure(sizeof(double) * nvox));
        CHK(w.f64_rho.ensure(sizeof(double) * nvox));
        return launch_voxel_fp64(p, tab, V, 1, w, w.slot_cs64.as<double2>(), 0, 0, dcnt, (double*)dr2, s);
    }
    CHK(w.f32_field.ensure(sizeof(float4) * nvox));
    FastParams F;
    CHK(fast_params(p, tab, V, &F, 4));
    unsigned long long* gp = w.counters.as<Counters>()->guard;
    const bool dens = r->use_density != 0;
    // launch parameters follow the variant's tile depth; order: the tiles'
    // order over the workgroups (0 per XCD, 1 linear)
    auto run_variant = [&](int v, int order = 2) -> int {
        FastParams Fv;
        fresh = false;
        CHK(variant_params(p, tab, V, &v, &Fv));
        set_tile_order(&Fv, order);
        pick_tile(want_diag, dens, v, Fv.thin_z != 0, [&](auto kern) {
            hipLaunchKernelGGL(kern, dim3(8 * Fv.per_xcd), dim3(64), 0, s, Fv, w.cell_start.as<int>(),
                               w.slot_frac.as<Frac3>(), w.slot_p32.as<float4>(),
                               w.slot_sn32.as<float>(), w.f32_field.as<float4>(), dcnt, (float*)dr2, gp);
        });
        return D2BI_OK;
    };
    const int variant = fast_variant(p, dens, want_diag, F.thin_z != 0, most, [&](int v) -> float {
        // a variant whose tiles span too many link cells is not timed
        if (tile_cells(p, tab, variant_tz(v), variant_ty(v)) > TILE_MAXC) return 3.4e38f;
        HIPCHK(hipEventRecord(g.ev[7], s));
        CHK(run_variant(v));
        HIPCHK(hipEventRecord(g.ev[8], s));
        HIPCHK(hipEventSynchronize(g.ev[8]));
        float ms = 0.0f;
        (void)hipEventElapsedTime(&ms, g.ev[7], g.ev[8]);
        return ms;
    });
    if (variant < 0) return variant;
    // the tile order: timed the first time a shape is seen (each launch
    // overwrites the whole field, so the timing runs leave no trace)
    int order = 2;
    if (!want_diag) {
        order = tune_choose(tile_order_key(p, tab, dens, variant), "D2BI_TILE_ORDER", TILE_ORDERS, 3, 2, true, s,
                            [&](int o) { (void)run_variant(variant, o); });
    }
    // tuning launches counted too
    if (!fresh) zero_i32(s, (int*)gp, (int64_t)(sizeof(Counters::guard) / (sizeof(int))));
    CHK(run_variant(variant, order));
    HIPCHK(hipGetLastError());
    return D2BI_OK;
}

// FAST integration of 8 or more precession points per launch through the
// shared step matrix, also where a column's points are split over waves that
// fewer would march faster stage by stage (its images are nearer the FP64
// ones: relative rms 4.3e-7 against 5.3e-7, 180^3 voxels, 8 points);
// D2BI_FAST_INTEGRATOR=stage marches every point stage by stage.
static bool fast_integrator_poly()
{
    const char* e = std::getenv("D2BI_FAST_INTEGRATOR");
    return !(e && std::strcmp(e, "stage") == 0);
}

// Points of the next FAST integration launch when `left` remain.
static int pass_points(int left) { return std::min(left, INT_POINTS); }

// Tuner key of the FAST integrators' workgroup size for a pass of np points.
static TuneKey int_block_key(const d2bi_plan* p, int np, bool dens)
{
    return TuneKey{TUNE_INT_BLOCK, p->Mx, p->My, p->Mz, np, dens ? 1 : 0, fast_integrator_poly() ? 1 : 0, 0, 0};
}

// Whether every tuned launch choice of a FAST condition is forced, already
// timed, or not tuned at all.
static bool condition_tuned(const d2bi_plan* p, const AxisTables& tab, bool dens, int variant)
{
    if (!tuning_on()) return true;
    if (forced_int("D2BI_TILE_ORDER", 0, 2) < 0 && tune_get(tile_order_key(p, tab, dens, variant)) < 0) return false;
    if (forced_int("D2BI_INT_BLOCK", 64, 256) >= 0) return true;
    for (int p0 = 0; p0 < p->nPrec;) {
        const int np = pass_points(p->nPrec - p0);
        if (tune_get(int_block_key(p, np, dens)) < 0) return false;
        p0 += np;
    }
    return true;
}

// How a FAST integration of np points over `plane` columns is split: points
// per wave, waves per column, column groups per workgroup.
struct IntSplit {
    int n, ns, cg;
};

// The cheapest split by a model of k_integrate_fast: vector operations per
// wave and double step (85 per point stage by stage, 40 per point after 230
// through the step matrix, 60 for the density) times the cycles one takes on
// the fullest SIMD (4.8 for a wave alone, 3.1 per wave together), workgroups
// dealt to 256 CUs and a workgroup's waves to their four SIMDs; `waves` is
// what an instance's registers let a SIMD hold.  More waves per column have to
// win 7 %.  Measured, us by points per wave: 400 x 400 columns of 120 samples,
// 5 points 1/2/4: 107/106/126, 32 points 8/16/32: 377/321/370; 80 x 80 of 80,
// 5 points 1/2/4: 17/21/31; 800 x 800 of 120, 5 points 1/4/5: 353/447/285, 32
// points 8/16/32: 1471/1215/1128; 236 x 268, 8 points of 4 per wave, 65 with
// workgroups of two column groups, 95 of one.  Powers of two in passes, one
// wave per column, took 110, 380, 40, 338, 1185 and 70.
struct IntInst {
    int n, waves, most;         // points per wave, waves a SIMD holds, waves per workgroup
    double ops;                 // vector operations per double step
};

// together: cycles per operation and wave where a SIMD holds several; gain:
// what more waves per column have to come down to
template <size_t N>
static IntSplit cheapest_split(const IntInst (&inst)[N], int64_t plane, int np, double together, double gain)
{
    const int64_t groups = (plane + 63) / 64;
    IntSplit best{0, 1, 4};
    double cost = 1.0e300;
    for (const IntInst& I : inst) {
        const int ns = (np + I.n - 1) / I.n;
        for (int cg = ns > 1 ? 1 : 4; cg <= (ns > 1 ? I.most / ns : 4); cg++) {
            const int64_t load = ((groups + cg - 1) / cg + 255) / 256 * ((ns * cg + 3) / 4);
            auto cyc = [&](int w) { return w > 0 ? std::max(4.8, together * w) : 0.0; };
            const double c = I.ops * ((double)(load / I.waves) * cyc(I.waves) + cyc((int)(load % I.waves)));
            if (c < (ns > best.ns ? gain : 1.0) * cost) {
                cost = c;
                best = IntSplit{I.n, ns, cg};
            }
        }
    }
    return best;
}

static IntSplit int_split(int64_t plane, int np, bool dens)
{
    const double d = dens ? 60 : 0;
    auto st = [&](int n, int waves) { return IntInst{n, waves, int_threads(n) / 64, 15 + 85.0 * n + d}; };
    auto mx = [&](int n, int waves) { return IntInst{n, waves, int_threads(n) / 64, 230 + 40.0 * n + d}; };
    const IntInst stage[] = {st(7, 7), st(6, 8), st(5, 8), st(4, 5), st(3, 6), st(2, 7), st(1, 7)};
    const IntInst matrix[] = {mx(32, 2), mx(16, 3), mx(8, 4), mx(4, 5), mx(2, 5)};
    if (np >= 8 && fast_integrator_poly()) return cheapest_split(matrix, plane, np, 3.1, 0.93);
    return cheapest_split(stage, plane, np, 3.1, 0.93);
}

// The same for FP64, whose operations do not overlap (a SIMD's waves take 4.8
// cycles each) and whose columns are 24 bytes a sample: splitting them has to
// win 20 % (400 x 360 columns of 200 samples with density, 2 points: 135 us in
// one wave, 196 in two).  136 x 136 of 136, one wave per column -> split: 2
// points 32 -> 26, 4 51 -> 35, 8 81 -> 56; 400 x 360, 32 points 1213 -> 1050
// (two launches before).
static IntSplit int_split64(int64_t plane, int np)
{
    auto st = [&](int n, int waves) { return IntInst{n, waves, int_threads64(n) / 64, 15 + 80.0 * n}; };
    auto mx = [&](int n, int waves) { return IntInst{n, waves, int_threads64(n) / 64, 230 + 40.0 * n}; };
    const IntInst inst[] = {mx(16, 1), mx(12, 1), mx(8, 2), mx(6, 2), st(4, 3), st(3, 4), st(2, 4), st(1, 4)};
    return cheapest_split(inst, plane, np, 4.8, 0.8);
}

// Whether one launch integrates nf fields of np points each: their
// deviations fit its parameters and a column's waves one workgroup.
static bool fields_fit(int64_t plane, int np, int nf, bool dens)
{
    const IntSplit sp = int_split(plane, np, dens);
    return nf * np <= INT_POINTS && 64 * nf * sp.ns <= int_threads(sp.n);
}

// One FAST integration launch, workgroups of about `block` threads (any size
// gives the same image).
static void launch_int_pass(FastIntParams P, const IntSplit& sp, int nf, bool dens, const void* f, double* img,
                            int acc, double inv, int block, hipStream_t s)
{
    const int64_t plane = (int64_t)P.Mx * P.My;
    const bool poly = P.np >= 8 && fast_integrator_poly();
    P.split = sp.ns;
    P.nsplit = nf * sp.ns;
    // `block` sizes the workgroups of unsplit columns
    const int cg = P.nsplit == 1 ? std::max(1, block / 64) : std::max(1, sp.cg / nf);
    const dim3 grid((unsigned)((plane + 64 * cg - 1) / (64 * cg))), thr(64 * cg * P.nsplit);
    auto go = [&](auto np_c, auto poly_c) {
        constexpr int N = decltype(np_c)::value;
        constexpr bool M = decltype(poly_c)::value;
        auto run = [&](auto kern) { hipLaunchKernelGGL(kern, grid, thr, 0, s, P, f, img, acc, inv); };
        if (P.nsplit > 1 && dens) run(k_integrate_fast<N, true, M, true>);
        else if (P.nsplit > 1) run(k_integrate_fast<N, false, M, true>);
        else if (dens) run(k_integrate_fast<N, true, M, false>);
        else run(k_integrate_fast<N, false, M, false>);
    };
    const std::true_type t{};
    const std::false_type f_{};
    switch (poly ? -sp.n : sp.n) {
        case 1: go(std::integral_constant<int, 1>{}, f_); break;
        case 2: go(std::integral_constant<int, 2>{}, f_); break;
        case 3: go(std::integral_constant<int, 3>{}, f_); break;
        case 4: go(std::integral_constant<int, 4>{}, f_); break;
        case 5: go(std::integral_constant<int, 5>{}, f_); break;
        case 6: go(std::integral_constant<int, 6>{}, f_); break;
        case 7: go(std::integral_constant<int, 7>{}, f_); break;
        case -2: go(std::integral_constant<int, 2>{}, t); break;
        case -4: go(std::integral_constant<int, 4>{}, t); break;
        case -8: go(std::integral_constant<int, 8>{}, t); break;
        case -16: go(std::integral_constant<int, 16>{}, t); break;
        default: go(std::integral_constant<int, 32>{}, t); break;
    }
}

// FAST integration of all precession points, INT_POINTS a launch.
// dens: the field holds float4 {x, rho} (density field on), else float2 x.
// acc_in: add to d_img from the first pass on; inv: weight of one
// integration (0: 1/nPrec).  tune_ws: a workspace whose tune_img buffer may
// grow, for timing the workgroup sizes of a pass that adds to d_img (null:
// such a pass is not timed).  nf > 1: fields at a stride of `stride` records
// with nPrec deviations each in aa (fields_fit), one launch for all.
static int launch_integrate_fast(const d2bi_plan* p, bool dens, const void* f, double* d_img, hipStream_t s,
                                 bool acc_in = false, double inv = 0.0, Workspace* tune_ws = nullptr, int nf = 1,
                                 int64_t stride = 0, const double* aa = nullptr, PointCount N = {})
{
    if (!aa) aa = p->aa;
    if (inv == 0.0) inv = 1.0 / p->nPrec;
    for (int p0 = 0, first = acc_in ? 0 : 1; p0 < p->nPrec; first = 0) {
        const int np = pass_points(p->nPrec - p0);
        FastIntParams P;
        P.Mx = p->Mx; P.My = p->My; P.Mz = p->Mz; P.np = np;
        P.b0 = (float)p->b0; P.bg = (float)p->bg; P.dz = (float)p->dz;
        P.stride = stride;
        P.N = N;
        for (int i = 0; i < INT_SLOTS; i++) {
            P.aa[i] = i < nf * np ? (float)aa[p0 + i] : 0.0f;
            P.al[i] = i < nf * np ? (float)(2.0 * p->dz * aa[p0 + i]) : 0.0f;
        }
        // workgroup size: timed on a launch that writes (not adds to) an
        // image, the output itself for the first pass, else a tuning buffer
        // (split columns size their own: nothing to time, and 256 stands for it
        // in the key, which several fields share with one of their shape)
        const TuneKey key = int_block_key(p, np, dens);
        const IntSplit sp = int_split((int64_t)P.Mx * P.My, np, dens);
        const bool split = nf > 1 || sp.ns > 1;
        if (split && nf == 1 && tuning_on() && forced_int("D2BI_INT_BLOCK", 64, 256) < 0 && tune_get(key) < 0)
            tune_put(key, 256);
        double* timg = first && !split ? d_img : nullptr;
        if (!timg && !split && tune_ws && !tune_ws->tune_img.arena && !g_capturing && tuning_on() && tune_get(key) < 0) {
            CHK(tune_ws->tune_img.ensure(sizeof(double) * (int64_t)P.Mx * P.My));
            timg = tune_ws->tune_img.as<double>();
        }
        static const int cand[3] = {64, 128, 256};
        const int block = split ? 256 : tune_choose(key, "D2BI_INT_BLOCK", cand, 3, 256, timg != nullptr, s, [&](int b) {
            launch_int_pass(P, sp, nf, dens, f, timg, 0, inv, b, s);
        });
        launch_int_pass(P, sp, nf, dens, f, d_img, !first, inv, block, s);
        HIPCHK(hipGetLastError());
        p0 += np;
    }
    return D2BI_OK;
}

// Double steps after which the FP64 march rescales its points, 0 for never.
// With x a bound of |2 dz H|, a double step I + D has |D| <= x + x^2/2 + x^3/6 +
// x^4/24 =: d, so it lengthens phi to at most 1 + d and shortens it to at least
// 1 - d; while the column's steps together stay within 2^+-400, so do the
// squares in FP64's range.  Four voxels per lattice parameter and s_g = 0.01
// (x = 0.17) reach that after 1300 double steps.  Larger steps have no such
// lower bound: every fourth is rescaled, which leaves them 2^100 each.
static int rescale_every(const d2bi_plan* p)
{
    double a = 0.0;
    for (int i = 0; i < p->nPrec; i++) a = std::max(a, std::fabs(p->aa[i]));
    const double x = 2.0 * p->dz * (std::fabs(p->b0) + std::fabs(p->bg) + a);
    const double d = x * (1.0 + x * (1.0 / 2 + x * (1.0 / 6 + x / 24)));
    const double bits = d < 1.0 ? std::max(std::log2(1.0 + d), -std::log2(1.0 - d)) : 1.0e300;
    if (bits * (p->Mz / 2) <= 400.0) return 0;
    return d < 1.0 ? std::max(1, (int)(400.0 / bits)) : d < 1.0e30 ? 4 : 1;
}

// FP64 integration of all precession points, INT_POINTS a launch.
// accumulate: add each column's sum over precession points to d_img; otherwise
// write sum / nPrec (div = 0) or sum / div.  The field is read from workspace
// w, field_off voxels on.
static int launch_integrate_fp64(const d2bi_plan* p, bool dens, double* d_img, hipStream_t s, Workspace& w,
                                 int accumulate = 0, double div = 0.0, int64_t field_off = 0, PointCount N = {})
{
    const int64_t plane = (int64_t)p->Mx * p->My;
    const int every = rescale_every(p);
    for (int p0 = 0; p0 < p->nPrec;) {
        const int np = pass_points(p->nPrec - p0);
        const IntSplit sp = int_split64(plane, np);
        IntParams P;
        P.Mx = p->Mx; P.My = p->My; P.Mz = p->Mz; P.np = np;
        P.nsplit = sp.ns;
        P.every = every;
        P.N = N;
        P.b0 = p->b0; P.bg = p->bg; P.dz = p->dz;
        for (int i = 0; i < INT_SLOTS; i++) {
            P.aa[i] = i < np ? p->aa[p0 + i] : 0.0;
            P.al[i] = 2.0 * p->dz * P.aa[i];
        }
        P.accumulate = accumulate || p0 > 0;
        P.div = accumulate || p0 + np < p->nPrec ? 0.0 : div == 0.0 ? (double)p->nPrec : div;
        // unsplit: small workgroups spread a small image over the CUs
        const int cg = sp.ns > 1 ? sp.cg : plane < 256 * 1024 ? 1 : 4;
        auto go = [&](auto kern) {
            hipLaunchKernelGGL(kern, dim3((unsigned)((plane + 64 * cg - 1) / (64 * cg))), dim3(64 * cg * sp.ns), 0, s, P,
                               w.f64_re.as<double>() + field_off, w.f64_im.as<double>() + field_off,
                               w.f64_rho.as<double>(), d_img);
        };
        auto pick = [&](auto np_c) {
            constexpr int N = decltype(np_c)::value;
            auto inst = [&](auto rs_c) {
                constexpr bool RS = decltype(rs_c)::value;
                if (sp.ns > 1 && dens) go(k_integrate_fp64<N, true, true, RS>);
                else if (sp.ns > 1) go(k_integrate_fp64<N, false, true, RS>);
                else if (dens) go(k_integrate_fp64<N, true, false, RS>);
                else go(k_integrate_fp64<N, false, false, RS>);
            };
            if (every > 0) inst(std::true_type{});
            else inst(std::false_type{});
        };
        switch (sp.n) {
            case 1: pick(std::integral_constant<int, 1>{}); break;
            case 2: pick(std::integral_constant<int, 2>{}); break;
            case 3: pick(std::integral_constant<int, 3>{}); break;
            case 4: pick(std::integral_constant<int, 4>{}); break;
            case 6: pick(std::integral_constant<int, 6>{}); break;
            case 8: pick(std::integral_constant<int, 8>{}); break;
            case 12: pick(std::integral_constant<int, 12>{}); break;
            default: pick(std::integral_constant<int, 16>{}); break;
        }
        HIPCHK(hipGetLastError());
        p0 += np;
    }
    return D2BI_OK;
}

// Integrate the field of workspace w into d_img (Mx*My doubles).
static int run_integrate(const d2bi_plan* p, bool dens, int mode, PointCount N, hipStream_t s, Workspace& w,
                         double* d_img)
{
    if (mode == D2BI_MODE_FP64) return launch_integrate_fp64(p, dens, d_img, s, w, 0, 0.0, 0, N);
    return launch_integrate_fast(p, dens, w.f32_field.p, d_img, s, false, 0.0, &w, 1, 0, nullptr, N);
}

// Whole condition: bin -> voxelise -> integrate on workspace w, the image
// written to d_img (device memory of Mx*My doubles) or, when d_img is null,
// left in w.img (copied to h_img when that is given).  The host waits once, at
// the end: the point arrays are sized by an estimate, and a condition that
// has more points is imaged again with the exact count (the wait for the
// count between the counting and the scatter left the GPU idle for 45-50 us).
// The exact count comes first where the arrays are carved from a fixed block,
// where the launch tuner has yet to time this shape (it should time real
// work), or where the estimate does not fit in device memory.
static int image_condition(const d2bi_record* r, const double* d_x, int64_t n, double precAngle, int nPrec,
                           int mode, d2bi_stats* st, d2bi_plan* plan_out, Workspace& w, double* d_img = nullptr,
                           double* h_img = nullptr)
{
    if (mode != D2BI_MODE_FP64 && mode != D2BI_MODE_FAST) return seterr(D2BI_ERR_ARG, "unknown mode %d", mode);
    d2bi_plan plan;
    CHK(plan_image(r, n, precAngle, nPrec, &plan));
    AxisTables tab;
    CHK(axis_tables(r, &plan, &tab));
    CHK(condition_mode(&plan, tab, &mode));
    BinParams BP;
    CHK(bin_params(r, &plan, &BP));
    const bool dens = r->use_density != 0;
    BP.fast = mode == D2BI_MODE_FAST ? 1 : 0;
    const int64_t plane = (int64_t)plan.Mx * plan.My;
    // results come back through pinned memory, small images too: those are
    // integrated right behind the counters, so that one copy brings both
    const bool small = h_img && plane <= 64 * 1024, joint = small && !d_img && !w.counters.arena;
    if (joint) {
        CHK(w.counters.ensure(sizeof(Counters) + sizeof(double) * plane));
        d_img = reinterpret_cast<double*>(w.counters.as<char>() + sizeof(Counters));
    } else if (!d_img) {
        CHK(w.img.ensure(sizeof(double) * plane));
        d_img = w.img.as<double>();
    }
    hipStream_t s = g.stream;
    Timer T{g.ev, s};
    Counters* ct;
    void* hp;
    if (w.counters.arena) {
        CHK(pinned_result(sizeof(Counters), &hp));       // held from initialisation on
    } else {
        CHK(pinned_result(sizeof(Counters) + (small ? sizeof(double) * plane : 0), &hp));
    }
    ct = (Counters*)hp;
    double* hi = (double*)((char*)hp + sizeof(Counters));
    Binned b;
    auto enqueue = [&](int64_t expect) -> int {
        CHK(T.record(0));
        AxisDev ax;
        CHK(upload_axis(tab, &ax, s, w));
        b = Binned();
        CHK(run_binning(d_x, n, BP, &b, s, w, expect));
        CHK(T.record(1));
        CHK(run_voxel(r, &plan, tab, ax, mode, false, true, s, w));
        CHK(T.record(2));
        CHK(run_integrate(&plan, dens, mode, b.N, s, w, d_img));
        CHK(T.record(3));
        HIPCHK(hipMemcpyAsync(ct, w.counters.p, sizeof(Counters) + (joint ? sizeof(double) * plane : 0),
                              hipMemcpyDeviceToHost, s));
        if (small && !joint) HIPCHK(hipMemcpyAsync(hi, d_img, sizeof(double) * plane, hipMemcpyDeviceToHost, s));
        HIPCHK(hipStreamSynchronize(s));
        return D2BI_OK;
    };
    const int v = known_variant(&plan, dens);
    double lost = 0.0;                                  // device time of a pass that did not fit
    bool exact = w.counters.arena || n == 0;
    if (mode == D2BI_MODE_FAST && (v < 0 || !condition_tuned(&plan, tab, dens, v))) exact = true;
    if (!exact) {
        const int rc = enqueue(expected_points(r, &plan, n));
        if (rc != D2BI_OK) {
            // memory for the estimate, or a failure the exact pass reports again;
            // arrays of the estimate would take the exact pass's room
            (void)hipGetLastError();
            HIPCHK(hipStreamSynchronize(s));
            if (rc == D2BI_ERR_HIP) {
                g_alloc_gen++;
                point_buffers(w, BP.fast, false, false, false, [](Buf& q, size_t) { q.release(); });
            }
            exact = true;
        } else if (ct->n_points < 0 || ct->n_points > b.N.cap) {
            exact = true;
            lost = T.ms(0, 3);
        }
    }
    if (exact) CHK(enqueue(0));
    if (small) std::memcpy(h_img, hi, sizeof(double) * plane);
    else if (h_img) HIPCHK(hipMemcpy(h_img, d_img, sizeof(double) * plane, hipMemcpyDeviceToHost));
    if (st) {
        st->n_points += ct->n_points;
        st->n_guard += mode == D2BI_MODE_FAST ? ct->n_guard() : 0;
        st->max_per_cell = std::max(st->max_per_cell, ct->max_per_cell);
        st->n_cells = b.ncell;
        st->ms_bin += T.ms(0, 1);
        st->ms_voxel += T.ms(1, 2);
        st->ms_integrate += T.ms(2, 3);
        st->ms_total += lost + T.ms(0, 3);
    }
    if (plan_out) *plan_out = plan;
    return D2BI_OK;
}

__global__ void k_div_f64(double* __restrict__ p, int64_t n, double d)
{
    const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i < n) p[i] = p[i] / d;
}

// Aperture points per shared voxel pass: D2BI_APERTURE_SHARED=0 bins and
// voxelises every point on its own instead (the same image to the bit).
static bool aperture_shared()
{
    const char* e = std::getenv("D2BI_APERTURE_SHARED");
    return !(e && e[0] == '0' && e[1] == 0);
}

// One shared voxel pass over na = 2 or 4 aperture points whose phases are in
// w.app_cs (a stride of nr slots): FP64 fields to f64_re/f64_im at a stride of
// nvox, FAST to f32_field at a stride of nvox records; variant is the FAST
// row kernel (1 or 2).
static int run_voxel_apps(const d2bi_record* r, const d2bi_plan* p, const AxisTables& tab, const AxisDev& ax,
                          int mode, int na, int variant, int64_t nr, hipStream_t s, Workspace& w)
{
    const int64_t nvox = (int64_t)p->Mx * p->My * p->Mz;
    VoxParams V;
    fill_vox_params(r, p, ax, &V);
    if (mode == D2BI_MODE_FP64) {
        CHK(w.f64_re.ensure(sizeof(double) * nvox * na));
        CHK(w.f64_im.ensure(sizeof(double) * nvox * na));
        CHK(w.f64_rho.ensure(sizeof(double) * nvox));
        return launch_voxel_fp64(p, tab, V, na, w, w.app_cs.as<double2>(), nr, nvox, nullptr, nullptr, s);
    }
    const bool dens = r->use_density != 0;
    CHK(w.f32_field.ensure((dens ? sizeof(float4) : sizeof(float2)) * nvox * na));
    FastParams F;
    CHK(variant_params(p, tab, V, &variant, &F));
    if (variant != 1 && variant != 2) return seterr(D2BI_ERR_ARG, "shared aperture pass: variant %d", variant);
    F.app_cs = w.app_cs.as<float2>();
    F.app_stride = nr;
    F.field_stride = nvox;
    const int fo = forced_int("D2BI_TILE_ORDER", 0, 2);
    set_tile_order(&F, fo >= 0 ? fo : 2);
    unsigned long long* gp = w.counters.as<Counters>()->guard;
    zero_i32(s, (int*)gp, (int64_t)(sizeof(Counters::guard) / (sizeof(int))));
    auto go = [&](auto kern) {
        hipLaunchKernelGGL(kern, dim3(8 * F.per_xcd), dim3(64), 0, s, F, w.cell_start.as<int>(),
                           w.slot_frac.as<Frac3>(), w.slot_p32.as<float4>(), w.slot_sn32.as<float>(),
                           w.f32_field.as<float4>(), (int*)nullptr, (float*)nullptr, gp);
    };
    auto pick = [&](auto dens_c, auto row_c, auto na_c) {
        constexpr bool D = decltype(dens_c)::value;
        constexpr int R = decltype(row_c)::value, N = decltype(na_c)::value;
        if (variant == 2) go(k_voxel_tile<D, false, R, 8, 4, N>);
        else go(k_voxel_tile<D, false, R, 4, 4, N>);
    };
    auto pick_na = [&](auto dens_c, auto row_c) {
        if (na == 4) pick(dens_c, row_c, std::integral_constant<int, 4>{});
        else pick(dens_c, row_c, std::integral_constant<int, 2>{});
    };
    auto pick_row_c = [&](auto dens_c) {
        if (F.thin_z) pick_na(dens_c, std::integral_constant<int, 2>{});
        else pick_na(dens_c, std::integral_constant<int, 1>{});
    };
    if (dens) pick_row_c(std::true_type{});
    else pick_row_c(std::false_type{});
    HIPCHK(hipGetLastError());
    return D2BI_OK;
}

// computeD2BI_img with apertureAngle and nAperturePoints > 1
// (Lib_DynamicalTwoBeamImaging.f90:1775-1786, 1853-1866, 1905-1951).  Every
// aperture point has its own g-vector for g.r (findGdotR_aperture :1269-1396)
// and so its own phase field; the link cells, ranges and densities are those
// of the unshifted condition.  The atoms are binned once; each pass then
// evaluates the phases of up to four points per slot (k_app_phase) and
// voxelises them together, one neighbour walk for all of them as the
// reference's loop over the neighbour list does (:1905-1922), and each
// point's field is integrated at its nPrec deviation parameters aa(app, :).
// The column sums are added up point by point and the image is divided by
// nApp * nPrec at the end (the reference adds over (prec, app) in the other
// nesting; FP64 sums agree to rounding).  Result left in ws.img.
static int image_aperture(const d2bi_record* r, const double* d_x, int64_t n, double precAngle, int nPrec,
                          double apAngle, int nApp, int mode, d2bi_stats* st, d2bi_plan* plan_out)
{
    if (mode != D2BI_MODE_FP64 && mode != D2BI_MODE_FAST) return seterr(D2BI_ERR_ARG, "unknown mode %d", mode);
    d2bi_plan plan;
    CHK(plan_image(r, n, precAngle, nPrec, &plan));
    std::vector<double> gshift(3 * (size_t)nApp), aa((size_t)nApp * nPrec);
    CHK(aperture_setup(r, precAngle, nPrec, apAngle, nApp, gshift.data(), aa.data()));
    AxisTables tab;
    CHK(axis_tables(r, &plan, &tab));
    CHK(condition_mode(&plan, tab, &mode));
    hipStream_t s = g.stream;
    Workspace& w = g.ws;
    AxisDev ax;
    CHK(upload_axis(tab, &ax, s, w));
    const int64_t plane = (int64_t)plan.Mx * plan.My;
    const int64_t nvox = plane * plan.Mz;
    CHK(w.img.ensure(sizeof(double) * plane));
    double* d_img = w.img.as<double>();
    const bool dens = r->use_density != 0;
    const double total = (double)nApp * nPrec;
    const bool f64 = mode == D2BI_MODE_FP64;
    // the plan of aperture point app: its g and deviation parameters
    auto point_plan = [&](int app) {
        d2bi_plan pk = plan;
        for (int i = 0; i < 3; i++) pk.gg[i] = gshift[3 * app + i];
        for (int q = 0; q < nPrec; q++) pk.aa[q] = aa[app + (size_t)nApp * q];
        return pk;
    };
    // aperture point app's field (FP64: offset into f64_re/f64_im; FAST: the
    // field record array) integrated into d_img
    auto integrate_point = [&](int app, int64_t f64_off, const void* f32) -> int {
        const d2bi_plan pk = point_plan(app);
        if (f64) {
            // point 0 writes its sum (div 1), the others add theirs
            CHK(launch_integrate_fp64(&pk, dens, d_img, s, w, app > 0 ? 1 : 0, 1.0, f64_off));
        } else {
            CHK(launch_integrate_fast(&pk, dens, f32, d_img, s, app > 0, 1.0 / total, &w));
        }
        return D2BI_OK;
    };
    auto add_stats = [&](const Binned& b, int points) -> int {
        void* hp;
        CHK(pinned_result(sizeof(Counters), &hp));
        const Counters* ct = (const Counters*)hp;
        if (st) HIPCHK(hipMemcpyAsync(hp, w.counters.p, sizeof(Counters), hipMemcpyDeviceToHost, s));
        HIPCHK(hipStreamSynchronize(s));
        if (st) {
            st->n_points += b.nr * points;
            st->n_guard += f64 ? 0 : ct->n_guard();
            st->max_per_cell = std::max(st->max_per_cell, ct->max_per_cell);
            st->n_cells = b.ncell;
        }
        return D2BI_OK;
    };

    const int most = nApp > 1 ? APERTURE_VARIANT : 3;      // a single point is the plain image
    if (!aperture_shared()) {
        // every point binned and voxelised on its own
        for (int app = 0; app < nApp; app++) {
            d2bi_plan pk = point_plan(app);
            BinParams BP;
            CHK(bin_params(r, &pk, &BP));
            BP.fast = f64 ? 0 : 1;
            Binned b;
            CHK(run_binning(d_x, n, BP, &b, s, w));
            CHK(run_voxel(r, &pk, tab, ax, mode, false, true, s, w, most));
            CHK(integrate_point(app, 0, w.f32_field.p));
            CHK(add_stats(b, 1));
        }
    } else {
        // one binning, at point 0's g (its phases are the binning's own)
        d2bi_plan p0 = point_plan(0);
        BinParams BP;
        CHK(bin_params(r, &p0, &BP));
        BP.fast = f64 ? 0 : 1;
        BP.keep_src = 1;
        Binned b;
        CHK(run_binning(d_x, n, BP, &b, s, w));
        const int64_t nr = b.nr;
        // shared passes of four or two points: FP64, or the FAST row kernels
        // of rows (variants 1 and 2; a forced 0 or 3 walks once per point)
        int variant = forced_variant();
        if (variant < 0) variant = default_variant(&plan, most);
        variant = effective_variant(&plan, tab, variant);
        const int na_max = (f64 || variant == 1 || variant == 2) ? 4 : 1;
        if (na_max > 1) CHK(w.app_cs.ensure((f64 ? sizeof(double2) : sizeof(float2)) * std::max<int64_t>(nr, 1) * na_max));
        for (int app = 0; app < nApp;) {
            const int left = nApp - app;
            const int na = na_max >= 4 && left >= 4 ? 4 : (na_max >= 2 && left >= 2 ? 2 : 1);
            if (nr > 0 && (app > 0 || na > 1)) {
                AppG G;
                std::memset(&G, 0, sizeof G);
                for (int a = 0; a < na; a++)
                    for (int i = 0; i < 3; i++) G.g[a][i] = gshift[3 * (app + a) + i];
                const dim3 grid(xcd_grid(nr));
                auto go = [&](auto kern) {
                    hipLaunchKernelGGL(kern, grid, dim3(256), 0, s, nr, w.slot_src.as<int2>(), d_x, BP, G, nr,
                                       na > 1 ? w.app_cs.as<double2>() : w.slot_cs64.as<double2>(),
                                       w.app_cs.as<float2>(), w.slot_p32.as<float4>(), w.slot_sn32.as<float>());
                };
                if (f64) {
                    if (na == 4) go(k_app_phase<true, 4>);
                    else if (na == 2) go(k_app_phase<true, 2>);
                    else go(k_app_phase<true, 1>);
                } else {
                    if (na == 4) go(k_app_phase<false, 4>);
                    else if (na == 2) go(k_app_phase<false, 2>);
                    else go(k_app_phase<false, 1>);
                }
                HIPCHK(hipGetLastError());
            }
            if (na == 1) {
                const d2bi_plan pk = point_plan(app);
                CHK(run_voxel(r, &pk, tab, ax, mode, false, false, s, w, most));
                CHK(integrate_point(app, 0, w.f32_field.p));
            } else {
                CHK(run_voxel_apps(r, &plan, tab, ax, mode, na, variant, nr, s, w));
                const size_t rec = dens ? sizeof(float4) : sizeof(float2);
                if (!f64 && fields_fit(plane, nPrec, na, dens)) {
                    std::vector<double> da((size_t)na * nPrec);
                    for (int a = 0; a < na; a++)
                        for (int q = 0; q < nPrec; q++) da[(size_t)nPrec * a + q] = aa[app + a + (size_t)nApp * q];
                    CHK(launch_integrate_fast(&plan, dens, w.f32_field.p, d_img, s, app > 0, 1.0 / total, nullptr, na,
                                              nvox, da.data()));
                } else {
                    for (int a = 0; a < na; a++)
                        CHK(integrate_point(app + a, nvox * a, w.f32_field.as<char>() + rec * nvox * a));
                }
            }
            CHK(add_stats(b, na));
            app += na;
        }
    }
    if (f64) {
        hipLaunchKernelGGL(k_div_f64, dim3((unsigned)((plane + 255) / 256)), dim3(256), 0, s, d_img, plane, total);
        HIPCHK(hipGetLastError());
        HIPCHK(hipStreamSynchronize(s));
    }
    if (plan_out) *plan_out = plan;
    return D2BI_OK;
}

static int upload_atoms_tmp(const double* x, int64_t ld, int64_t n, double** d_x)
{
    if (n < 0 || (n > 0 && (!x || ld < 3))) return seterr(D2BI_ERR_ARG, "bad atom array");
    CHK(g.ws.x.ensure(sizeof(double) * 3 * std::max<int64_t>(n, 1)));
    void* hp;
    CHK(pinned(sizeof(double) * 3 * std::max<int64_t>(n, 1), &hp));
    double* h = (double*)hp;
    for (int64_t j = 0; j < n; j++) {
        h[3 * j] = x[ld * j]; h[3 * j + 1] = x[ld * j + 1]; h[3 * j + 2] = x[ld * j + 2];
    }
    if (n > 0) HIPCHK(hipMemcpyAsync(g.ws.x.p, h, sizeof(double) * 3 * n, hipMemcpyHostToDevice, g.stream));
    HIPCHK(hipStreamSynchronize(g.stream));
    *d_x = g.ws.x.as<double>();
    return D2BI_OK;
}


}  // namespace d2bi
