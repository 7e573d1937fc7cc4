// d2bi_batch.cuh -- batched conditions on concurrent branches: launched as they
// are the first time, captured into one HIP graph when the batch comes again.
//
// One part of the single translation unit d2bi_gpu.hip, which includes the
// parts in order so that kernels and the device helpers they call compile
// together; each part uses the definitions of the parts before it.
#pragma once

namespace d2bi {

// ------------------------------------------------------------------ batched conditions

// One condition of a batch: its plan, tables and slices of the batch buffers.
struct Cond {
    d2bi_plan plan;
    AxisTables tab;
    BinParams BP;
    const double* d_x = nullptr;
    int64_t n = 0;
    int nblk = 0, ncell = 0, variant = 0, mode = 0;
    bool dens = false;
    int64_t nr = 0, nbc = 0, nvox = 0, plane = 0;
    int64_t o_mask = 0, o_blk = 0, o_scan = 0, o_img = 0;
    size_t o_ax = 0;
    AxisDev ax;
};

// Conditions of a batch run on up to MAX_BRANCH concurrent branches, each a
// chain of conditions on its own stream and workspace (branch 0
// on the library's stream and workspace), so that small conditions fill the
// GPU together.  A condition's arithmetic does not depend on its branch.
static constexpr int MAX_BRANCH = 4;

struct Batch {
    Buf mask, blkcnt, blkoff, scan, ax, img, counters, tot;
    std::vector<unsigned char> key;
    uint64_t gen = 0;
    std::vector<Cond> conds;                    // the planned conditions of key
    hipGraphExec_t exec = nullptr;              // their graph, from the second call on
    int64_t total_plane = 0;
    int nbr = 1;                                // branches the conditions run on
    int64_t branch_bytes = 0;                   // device bytes of one branch's workspace
    Workspace ws[MAX_BRANCH - 1];               // branches 1..MAX_BRANCH-1
    hipStream_t stream[MAX_BRANCH - 1] = {};
    hipEvent_t fork = nullptr, join[MAX_BRANCH - 1] = {};
    void reset()
    {
        if (exec) (void)hipGraphExecDestroy(exec);
        exec = nullptr;
        key.clear();
        conds.clear();
    }
    void release()
    {
        reset();
        Buf* all[] = {&mask, &blkcnt, &blkoff, &scan, &ax, &img, &counters, &tot};
        for (Buf* b : all) b->release();
        for (int k = 0; k < MAX_BRANCH - 1; k++) {
            ws[k].release_all();
            if (stream[k]) (void)hipStreamDestroy(stream[k]);
            if (join[k]) (void)hipEventDestroy(join[k]);
            stream[k] = nullptr;
            join[k] = nullptr;
        }
        if (fork) (void)hipEventDestroy(fork);
        fork = nullptr;
    }
    Workspace& branch_ws(int k) { return k == 0 ? g.ws : ws[k - 1]; }
};

// Branches a batch uses (D2BI_BATCH_BRANCHES=1..4, default 4: an uneven batch
// of 163 conditions from 64 configurations took 0.115 s with one branch, 0.099
// with two, 0.092 with four; a 42-condition tilt series of 800 x 800 x 400
// voxels is within 1 % of its best, two).
static int batch_branches()
{
    const char* e = std::getenv("D2BI_BATCH_BRANCHES");
    if (e && e[0] >= '1' && e[0] <= '0' + MAX_BRANCH && e[1] == 0) return e[0] - '0';
    return MAX_BRANCH;
}

static Batch g_batch;

static void key_append(std::vector<unsigned char>& k, const void* p, size_t n)
{
    const unsigned char* c = (const unsigned char*)p;
    k.insert(k.end(), c, c + n);
}

// counting pass of one condition: replica predicate, per-block offsets, and
// the number of points in the batch's totals
static int enqueue_count(const Cond& c, int idx, Batch& B, hipStream_t s)
{
    uint32_t* mask = B.mask.as<uint32_t>() + c.o_mask;
    int* cnt = B.blkcnt.as<int>() + c.o_blk;
    int* off = B.blkoff.as<int>() + c.o_blk;
    if (c.n > 0)
        hipLaunchKernelGGL(k_bin_classify, dim3(c.nblk), dim3(BIN_BLOCK), 0, s, c.d_x, c.BP, mask, cnt, c.nblk,
                           ZeroRanges{});
    else
        zero_i32(s, cnt, c.nbc);
    HIPCHK(hipGetLastError());
    return scan_exclusive_tmp(cnt, off, c.nbc, B.scan.as<int>() + c.o_scan, s,
                              ScanEnds{B.tot.as<int>() + idx, nullptr, {}});
}

// the rest of one condition: bin, voxelise, integrate into its image slice,
// on workspace w
static int enqueue_rest(const Cond& c, int idx, Batch& B, Workspace& w, hipStream_t s)
{
    const d2bi_plan* p = &c.plan;
    Counters* ct = B.counters.as<Counters>() + idx;
    zero_i32(s, w.cell_cnt.as<int>(), c.ncell + 1, (int*)ct, sizeof(Counters) / sizeof(int));
    CHK(launch_bin_points(c.d_x, c.BP, B.mask.as<uint32_t>() + c.o_mask, B.blkoff.as<int>() + c.o_blk, c.nblk, c.ncell,
                          PointCount{B.tot.as<int>() + idx, c.nr}, c.nr, w.scan_tmp.as<int>(), &ct->max_per_cell, s, w));
    VoxParams V;
    d2bi_record dummy;
    dummy.use_density = c.dens ? 1 : 0;
    fill_vox_params(&dummy, p, c.ax, &V);
    double* d_img = B.img.as<double>() + c.o_img;
    if (c.mode == D2BI_MODE_FP64) {
        CHK(launch_voxel_fp64(p, c.tab, V, 1, w, w.slot_cs64.as<double2>(), 0, 0, nullptr, nullptr, s));
        return launch_integrate_fp64(p, c.dens, d_img, s, w);
    }
    FastParams F;
    int variant = c.variant;
    CHK(variant_params(p, c.tab, V, &variant, &F));
    // the tile order timed eagerly before capture (nothing is timed here)
    set_tile_order(&F, tune_choose(tile_order_key(p, c.tab, c.dens, c.variant), "D2BI_TILE_ORDER", TILE_ORDERS, 3,
                                   2, false, s, [](int) {}));
    launch_tile<false>(F, variant, c.dens, w.cell_start.as<int>(), w.slot_frac.as<Frac3>(),
                       w.slot_p32.as<float4>(), w.slot_sn32.as<float>(), w.f32_field.as<float4>(), nullptr, nullptr,
                       ct->guard, s);
    HIPCHK(hipGetLastError());
    return launch_integrate_fast(p, c.dens, w.f32_field.p, d_img, s);
}

// Sizes of one branch's workspace: the largest condition of the batch.
struct BranchSizes {
    bool fast, f64;             // what its conditions run in
    int64_t max_nr, max_cell, max_vox, max_scan;
};

// The buffers of a branch workspace that a batch uses, with their sizes.
template <class F>
static void branch_buffers(Workspace& w, const BranchSizes& z, F f)
{
    for (int fast = 0; fast < 2; fast++)
        if (fast ? z.fast : z.f64)
            point_buffers(w, fast, false, false, false, [&](Buf& b, size_t bytes) {
                if (!fast || !z.f64 || &b == &w.slot_sn32) f(b, bytes * z.max_nr);      // (each once)
            });
    f(w.cell_cnt, sizeof(int) * z.max_cell);
    f(w.cell_start, sizeof(int) * z.max_cell);
    if (z.f64) {
        f(w.f64_re, sizeof(double) * z.max_vox);
        f(w.f64_im, sizeof(double) * z.max_vox);
        f(w.f64_rho, sizeof(double) * z.max_vox);
    }
    if (z.fast) f(w.f32_field, sizeof(float4) * z.max_vox);
    f(w.scan_tmp, sizeof(int) * z.max_scan);
}

// Device bytes that sizing w for the batch would add.
static double branch_growth(Workspace& w, const BranchSizes& z)
{
    double d = 0.0;
    branch_buffers(w, z, [&](Buf& b, size_t bytes) { d += b.growth(bytes); });
    return d;
}

// Device bytes of one branch workspace sized for the batch.
static int64_t branch_bytes(const BranchSizes& z)
{
    Workspace tmp;
    int64_t n = 0;
    branch_buffers(tmp, z, [&](Buf&, size_t bytes) { n += (int64_t)Buf::alloc_size(bytes); });
    return n;
}

// The batch of B.conds on nb branches, launched on the library's stream and
// the branch streams (or captured from them): conditions to branches largest
// first, each to the least loaded branch (a fixed rule: the same inputs give
// the same assignment).  count: the counting passes too.
static int enqueue_batch(Batch& B, int nb, bool count)
{
    const std::vector<Cond>& C = B.conds;
    const int nRec = (int)C.size();
    hipStream_t s = g.stream;
    std::vector<int> order(nRec), branch(nRec, 0);
    for (int i = 0; i < nRec; i++) order[i] = i;
    auto work = [&](int i) { return (double)C[i].nvox * (1.0 + C[i].plan.nPrec / 8.0) + 8.0 * C[i].n; };
    std::stable_sort(order.begin(), order.end(), [&](int a, int b) { return work(a) > work(b); });
    std::vector<double> load(nb, 0.0);
    for (int i : order) {
        int k = 0;
        for (int j = 1; j < nb; j++)
            if (load[j] < load[k]) k = j;
        branch[i] = k;
        load[k] += work(i);
    }
    int rc = D2BI_OK;
    auto bstream = [&](int k) { return k == 0 ? s : B.stream[k - 1]; };
    if (nb > 1) {
        if (hipEventRecord(B.fork, s) != hipSuccess) rc = seterr(D2BI_ERR_HIP, "batch fork failed");
        for (int k = 1; k < nb && rc == D2BI_OK; k++)
            if (hipStreamWaitEvent(bstream(k), B.fork, 0) != hipSuccess)
                rc = seterr(D2BI_ERR_HIP, "batch fork failed");
    }
    for (int i = 0; i < nRec && rc == D2BI_OK; i++) {
        if (count) rc = enqueue_count(C[i], i, B, bstream(branch[i]));
        if (rc == D2BI_OK) rc = enqueue_rest(C[i], i, B, B.branch_ws(branch[i]), bstream(branch[i]));
    }
    // join every branch back, also after an error, so that a capture can end
    for (int k = 1; k < nb; k++)
        if (hipEventRecord(B.join[k - 1], bstream(k)) != hipSuccess ||
            hipStreamWaitEvent(s, B.join[k - 1], 0) != hipSuccess)
            if (rc == D2BI_OK) rc = seterr(D2BI_ERR_HIP, "batch join failed");
    return rc;
}

// Capture the batch (counting passes included) into B.exec.
static int capture_batch(Batch& B)
{
    hipStream_t s = g.stream;
    hipGraph_t graph;
    g_capturing = true;
    if (hipStreamBeginCapture(s, hipStreamCaptureModeThreadLocal) != hipSuccess) {
        g_capturing = false;
        return seterr(D2BI_ERR_HIP, "graph capture failed to begin");
    }
    const int rc = enqueue_batch(B, B.nbr, true);
    hipError_t e = hipStreamEndCapture(s, &graph);
    g_capturing = false;
    if (rc != D2BI_OK) {
        if (e == hipSuccess) (void)hipGraphDestroy(graph);
        return rc;
    }
    if (e != hipSuccess) return seterr(D2BI_ERR_HIP, "graph capture failed: %s", hipGetErrorString(e));
    e = hipGraphInstantiate(&B.exec, graph, nullptr, nullptr, 0);
    (void)hipGraphDestroy(graph);
    if (e != hipSuccess) {
        B.exec = nullptr;
        return seterr(D2BI_ERR_HIP, "graph instantiation failed: %s", hipGetErrorString(e));
    }
    return D2BI_OK;
}

// Plan a batch's conditions, count their points (one host synchronisation for
// the sizes), size the workspaces and image every condition, leaving the
// images in B.img.  Launch choices not yet timed for a shape are timed here.
static int first_run(Batch& B, const d2bi_record* recs, const d2bi_atoms* atoms, int nRec, const double* precAngle,
                     const int32_t* nPrec, int mode)
{
    hipStream_t s = g.stream;
    std::vector<Cond>& C = B.conds;
    C.assign(nRec, Cond());
    int64_t o_mask = 0, o_blk = 0, o_scan = 0, o_img = 0;
    size_t o_ax = 0;
    int64_t max_scan = 1;
    for (int i = 0; i < nRec; i++) {
        Cond& c = C[i];
        CHK(plan_image(&recs[i], atoms[i]->n, precAngle[i], nPrec[i], &c.plan));
        CHK(axis_tables(&recs[i], &c.plan, &c.tab));
        CHK(bin_params(&recs[i], &c.plan, &c.BP));
        c.mode = mode;
        CHK(condition_mode(&c.plan, c.tab, &c.mode));
        c.BP.fast = c.mode == D2BI_MODE_FAST ? 1 : 0;
        c.d_x = atoms[i]->x;
        c.n = atoms[i]->n;
        c.BP.n = c.n;
        c.nblk = bin_blocks(c.n);
        c.nbc = (int64_t)c.BP.nuvw * c.nblk;
        c.ncell = c.plan.Ex * c.plan.Ey * c.plan.Ez;
        c.dens = recs[i].use_density != 0;
        c.plane = (int64_t)c.plan.Mx * c.plan.My;
        c.nvox = c.plane * c.plan.Mz;
        c.o_mask = o_mask; o_mask += std::max<int64_t>(c.n, 1);
        c.o_blk = o_blk; o_blk += c.nbc + 1;
        c.o_scan = o_scan; o_scan += scan_tmp_ints(c.nbc);
        c.o_ax = o_ax; o_ax += axis_bytes(c.tab);
        c.o_img = o_img; o_img += c.plane;
        max_scan = std::max(max_scan, scan_tmp_ints(c.ncell));
    }
    CHK(B.mask.ensure(sizeof(uint32_t) * o_mask));
    CHK(B.blkcnt.ensure(sizeof(int) * o_blk));
    CHK(B.blkoff.ensure(sizeof(int) * o_blk));
    CHK(B.scan.ensure(sizeof(int) * o_scan));
    CHK(B.ax.ensure(o_ax));
    CHK(B.img.ensure(sizeof(double) * o_img));
    CHK(B.counters.ensure(sizeof(Counters) * nRec));
    CHK(B.tot.ensure(sizeof(int) * nRec));
    B.total_plane = o_img;
    // branch streams and the events that fork and join them (default priority)
    const int want = std::min(batch_branches(), nRec);
    int nbr = want;
    if (!B.fork) HIPCHK(hipEventCreateWithFlags(&B.fork, hipEventDisableTiming));
    for (int k = 1; k < nbr; k++) {
        if (!B.stream[k - 1]) HIPCHK(hipStreamCreateWithFlags(&B.stream[k - 1], hipStreamNonBlocking));
        if (!B.join[k - 1]) HIPCHK(hipEventCreateWithFlags(&B.join[k - 1], hipEventDisableTiming));
    }
    // counting passes, dealt to the branch streams; the tables go up meanwhile
    HIPCHK(hipEventRecord(B.fork, s));
    for (int k = 1; k < nbr; k++) HIPCHK(hipStreamWaitEvent(B.stream[k - 1], B.fork, 0));
    int rc = D2BI_OK;
    for (int i = 0; i < nRec && rc == D2BI_OK; i++)
        rc = enqueue_count(C[i], i, B, i % nbr == 0 ? s : B.stream[i % nbr - 1]);
    for (int k = 1; k < nbr; k++) {
        HIPCHK(hipEventRecord(B.join[k - 1], B.stream[k - 1]));
        HIPCHK(hipStreamWaitEvent(s, B.join[k - 1], 0));
    }
    CHK(rc);
    void* hp;
    CHK(pinned(o_ax, &hp));
    for (int i = 0; i < nRec; i++) axis_pack(C[i].tab, (char*)hp + C[i].o_ax, B.ax.as<char>() + C[i].o_ax, &C[i].ax);
    HIPCHK(hipMemcpyAsync(B.ax.p, hp, o_ax, hipMemcpyHostToDevice, s));
    void* hr;
    CHK(pinned_result(sizeof(int) * nRec, &hr));
    const int* tot = (const int*)hr;
    HIPCHK(hipMemcpyAsync(hr, B.tot.p, sizeof(int) * nRec, hipMemcpyDeviceToHost, s));
    HIPCHK(hipStreamSynchronize(s));
    int64_t max_nr = 1, max_cell = 1, max_vox = 1;
    bool fast = false, f64 = false;
    for (int i = 0; i < nRec; i++) {
        (C[i].mode == D2BI_MODE_FAST ? fast : f64) = true;
        if (tot[i] < 0) return seterr(D2BI_ERR_CAPACITY, "point count overflow");
        C[i].nr = tot[i];
        max_nr = std::max(max_nr, C[i].nr);
        max_cell = std::max<int64_t>(max_cell, C[i].ncell + 1);
        max_vox = std::max(max_vox, C[i].nvox);
    }
    const BranchSizes bz{fast, f64, max_nr, max_cell, max_vox, max_scan};
    // every branch gets a workspace sized for the largest condition; the
    // branches beyond the first run only where what their workspaces
    // would add (branch 0's growth included) fits in 85 % of the free
    // device memory, so that a batch one workspace can hold does not
    // fail for want of four
    if (nbr > 1) {
        size_t freeb = 0, totalb = 0;
        const char* e = std::getenv("D2BI_BATCH_MEM");         // free bytes to assume (tests)
        if (e && *e) freeb = (size_t)std::strtoull(e, nullptr, 10);
        else if (hipMemGetInfo(&freeb, &totalb) != hipSuccess) {
            (void)hipGetLastError();
            freeb = 0;
        }
        auto fitting = [&] {
            double used = branch_growth(B.branch_ws(0), bz);
            int fit = 1;
            for (int k = 1; k < want; k++) {
                used += branch_growth(B.branch_ws(k), bz);
                if (used > 0.85 * (double)freeb) break;
                fit = k + 1;
            }
            return fit;
        };
        nbr = fitting();
        if (nbr < want) {
            // what earlier batches left in the branches that do not fit
            for (int k = nbr; k < MAX_BRANCH; k++) {
                freeb += B.branch_ws(k).bytes();
                B.branch_ws(k).release_all();
            }
            nbr = fitting();
        }
    }
    // branch count: forced, cached, or tuned below by timing a run on each
    // count (images are the same on any count); the count that fits is kept
    // unless another is 3 % faster.  A cached count sizes its own branches
    // only: a workspace for the others, given back after the run, cost a
    // batch of eight conditions of 1e4 to 4e5 atoms on three of four branches
    // 1.89 ms a call against 1.37, in some processes 8.4
    const bool pick = nbr > 1 && !std::getenv("D2BI_BATCH_BRANCHES") && tuning_on();
    TuneKey bkey{};
    int chosen = nbr;
    bool tune = false;
    if (pick) {
        int64_t sum_vox = 0, max_vox_c = 0, sum_n = 0, sum_p = 0;
        for (int i = 0; i < nRec; i++) {
            sum_vox += C[i].nvox;
            max_vox_c = std::max(max_vox_c, C[i].nvox);
            sum_n += C[i].n;
            sum_p += C[i].plan.nPrec;
        }
        bkey = TuneKey{TUNE_BRANCHES, nRec, mode, sum_vox, max_vox_c, sum_n, sum_p, nbr, 0};
        const int c = tune_get(bkey);
        tune = c < 1 || c > nbr;
        if (!tune) chosen = c;
    }
    for (int k = 0; k < chosen; k++) {
        int rc_ = D2BI_OK;
        branch_buffers(B.branch_ws(k), bz, [&](Buf& b, size_t bytes) {
            if (rc_ == D2BI_OK) rc_ = b.ensure(bytes);
        });
        CHK(rc_);
    }
    B.branch_bytes = branch_bytes(bz);
    // FAST kernel variants (fixed, forced, or with D2BI_FAST_TUNE=1 tuned
    // for unseen shapes), and the launch choices of shapes the tuner has not
    // timed yet: one condition of each such shape, on its own, times them
    for (int i = 0; i < nRec; i++) {
        if (C[i].mode != D2BI_MODE_FAST) continue;
        int v = known_variant(&C[i].plan, C[i].dens);
        if (v < 0 || !condition_tuned(&C[i].plan, C[i].tab, C[i].dens, v)) {
            d2bi_plan tmp;
            CHK(image_condition(&recs[i], C[i].d_x, C[i].n, precAngle[i], nPrec[i], mode, nullptr, &tmp, g.ws));
            v = known_variant(&C[i].plan, C[i].dens);
            if (v < 0) v = 0;
        }
        C[i].variant = v;
    }
    HIPCHK(hipEventRecord(g.ev[0], s));
    if (tune) {
        float tbest = 3.4e38f;
        for (int q = 0; q < nbr; q++) {
            const int nb = q == 0 ? nbr : q;                // the default first
            int rq = D2BI_OK;
            const float t = time_launch([&] { rq = enqueue_batch(B, nb, false); }, s, 1);
            CHK(rq);
            if (q == 0) tbest = t >= 0.0f ? 0.97f * t : 3.4e38f;
            else if (t >= 0.0f && t < tbest) {
                tbest = t;
                chosen = nb;
            }
        }
        tune_put(bkey, chosen);
    } else {                                                // (each timed run imaged every condition)
        CHK(enqueue_batch(B, chosen, false));
    }
    HIPCHK(hipStreamSynchronize(s));
    // workspaces of branches that timing has just left unused, or that are
    // unused where device memory is short, go back to the device (the others
    // already have)
    if (tune || nbr < want)
        for (int k = std::max(1, chosen); k < nbr; k++) B.branch_ws(k).release_all();
    B.nbr = chosen;
    return D2BI_OK;
}

// Batched conditions.  New inputs (records, atom uploads, precession) are
// planned, counted and imaged with plain launches on the branches; when the
// next call brings the same inputs and the workspaces are unchanged, the whole
// batch (counting, binning, voxelisation, integration of every condition) is
// captured into one HIP graph, which that call and later ones replay: every
// replay recomputes everything from the atoms.  A batch that comes once, as
// the frames of a series do, does not pay for a graph (capture and
// instantiation took 0.6 ms of 2.4 for eight conditions of 1e4 to 4e5 atoms).
// img_out: host memory, or device memory when dev_out.
static int run_batch(const d2bi_record* recs, const d2bi_atoms* atoms, int nRec, const double* precAngle,
                     const int32_t* nPrec, int mode, double* img_out, bool dev_out, d2bi_stats* st)
{
    if (mode != D2BI_MODE_FP64 && mode != D2BI_MODE_FAST) return seterr(D2BI_ERR_ARG, "unknown mode %d", mode);
    Batch& B = g_batch;
    hipStream_t s = g.stream;
    std::vector<unsigned char> key;
    key_append(key, &mode, sizeof mode);
    key_append(key, &nRec, sizeof nRec);
    // settings that a graph holds as they were when it was captured
    const int set[] = {forced_variant(), tune_variants() ? 1 : 0, batch_branches(), fast_integrator_poly() ? 1 : 0,
                       tuning_on() ? 1 : 0, forced_int("D2BI_TILE_ORDER", 0, 2), forced_int("D2BI_INT_BLOCK", 64, 256)};
    key_append(key, set, sizeof set);
    for (int i = 0; i < nRec; i++) {
        key_append(key, &recs[i], sizeof(d2bi_record));
        // the plan holds each set's point counts: key on the upload, not on
        // addresses that a later upload may reuse
        key_append(key, &atoms[i]->serial, sizeof(uint64_t));
        key_append(key, &atoms[i]->n, sizeof(int64_t));
        key_append(key, &precAngle[i], sizeof(double));
        key_append(key, &nPrec[i], sizeof(int32_t));
    }
    if (B.conds.empty() || key != B.key || B.gen != g_alloc_gen) {
        B.reset();
        const int rc = first_run(B, recs, atoms, nRec, precAngle, nPrec, mode);
        if (rc != D2BI_OK) {
            // nothing of the batch may run on: its inputs belong to the caller
            (void)hipStreamSynchronize(s);
            for (auto& bs : B.stream)
                if (bs) (void)hipStreamSynchronize(bs);
            B.reset();
            return rc;
        }
        B.key = key;
        B.gen = g_alloc_gen;
    } else {
        if (!B.exec) CHK(capture_batch(B));
        HIPCHK(hipEventRecord(g.ev[0], s));
        HIPCHK(hipGraphLaunch(B.exec, s));
    }
    HIPCHK(hipEventRecord(g.ev[1], s));
    HIPCHK(hipMemcpyAsync(img_out, B.img.p, sizeof(double) * B.total_plane,
                          dev_out ? hipMemcpyDeviceToDevice : hipMemcpyDeviceToHost, s));
    void* hr = nullptr;
    if (st) {
        CHK(pinned_result(sizeof(Counters) * nRec, &hr));
        HIPCHK(hipMemcpyAsync(hr, B.counters.p, sizeof(Counters) * nRec, hipMemcpyDeviceToHost, s));
    }
    HIPCHK(hipStreamSynchronize(s));
    if (st) {
        const Counters* ct = (const Counters*)hr;
        for (int i = 0; i < nRec; i++) {
            st->n_points += B.conds[i].nr;
            st->n_guard += B.conds[i].mode == D2BI_MODE_FAST ? ct[i].n_guard() : 0;
            st->max_per_cell = std::max(st->max_per_cell, ct[i].max_per_cell);
        }
        float ms = 0.0f;
        (void)hipEventElapsedTime(&ms, g.ev[0], g.ev[1]);
        st->ms_total += ms;
        st->n_branches = B.nbr;
        st->branch_bytes = B.branch_bytes;
    }
    return D2BI_OK;
}

}  // namespace d2bi
