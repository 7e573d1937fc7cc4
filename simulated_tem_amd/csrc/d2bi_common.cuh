// d2bi_common.cuh -- error state, device buffers and the library state, device
// atom sets, and the generic exclusive scan.
//
// One part of the single translation unit d2bi_gpu.hip, which includes the
// parts in order so that kernels and the device helpers they call compile
// together; each part uses the definitions of the parts before it.
#pragma once

namespace d2bi {

// ------------------------------------------------------------------ errors

static char g_err[1024] = "";

int seterr(int code, const char* fmt, ...)
{
    va_list ap;
    va_start(ap, fmt);
    vsnprintf(g_err, sizeof g_err, fmt, ap);
    va_end(ap);
    return code;
}

#define HIPCHK(call)                                                                     \
    do {                                                                                 \
        hipError_t e_ = (call);                                                          \
        if (e_ != hipSuccess)                                                            \
            return seterr(D2BI_ERR_HIP, "%s failed: %s (%s:%d)", #call, hipGetErrorString(e_), \
                          __FILE__, __LINE__);                                           \
    } while (0)

#define CHK(call)                        \
    do {                                 \
        int r_ = (call);                 \
        if (r_ != D2BI_OK) return r_;    \
    } while (0)

// ------------------------------------------------------------------ device buffers

static uint64_t g_alloc_gen = 0;         // bumped on every device reallocation
static size_t g_alloc_bytes = 0;         // device bytes in buffers

// hipMalloc of a buffer, within D2BI_MEM_LIMIT bytes for all of them (tests).
static hipError_t alloc_device(void** p, size_t bytes)
{
    const char* e = std::getenv("D2BI_MEM_LIMIT");
    if (e && *e && g_alloc_bytes + bytes > (size_t)std::strtoull(e, nullptr, 10)) return hipErrorOutOfMemory;
    return hipMalloc(p, bytes);
}

// A fixed block of device memory handed out front to back (256-byte
// aligned pieces); buffers bound to an arena never call the allocator.
struct Arena {
    char* base = nullptr;
    size_t size = 0, off = 0;
};

struct Buf {
    void* p = nullptr;
    size_t cap = 0;
    Arena* arena = nullptr;                  // set: pieces of the arena instead of hipMalloc
    int ensure(size_t bytes)
    {
        if (bytes <= cap && p) return D2BI_OK;
        if (arena) {
            const size_t off = (arena->off + 255) & ~(size_t)255;
            if (off > arena->size || bytes > arena->size - off)
                return seterr(D2BI_ERR_CAPACITY,
                              "the no-allocation scratch (%zu bytes) cannot hold this condition: "
                              "%zu bytes in use, %zu more requested",
                              arena->size, arena->off, bytes);
            p = arena->base + off;
            cap = bytes;
            arena->off = off + bytes;
            return D2BI_OK;
        }
        g_alloc_gen++;
        release();
        const size_t want = alloc_size(bytes);       // headroom for slightly larger conditions
        hipError_t e = alloc_device(&p, want);
        if (e != hipSuccess) {
            p = nullptr;
            return seterr(D2BI_ERR_HIP, "hipMalloc(%zu) failed: %s (%zu bytes held)", want, hipGetErrorString(e),
                          g_alloc_bytes);
        }
        cap = want;
        g_alloc_bytes += cap;
        return D2BI_OK;
    }
    void release()
    {
        if (p && !arena) {
            (void)hipFree(p);
            g_alloc_bytes -= cap;
        }
        p = nullptr;
        cap = 0;
    }
    // bytes ensure(bytes) allocates: the request with its headroom
    static size_t alloc_size(size_t bytes)
    {
        const size_t want = std::max<size_t>(bytes, 256);
        return want + want / 8;
    }
    // net device bytes ensure(bytes) would add (it frees the old block first)
    double growth(size_t bytes) const
    {
        if (bytes <= cap && p) return 0.0;
        return (double)alloc_size(bytes) - (double)cap;
    }
    template <class T> T* as() const { return static_cast<T*>(p); }
};

struct Workspace {
    // binning
    Buf x;                      // atoms (temporary upload)
    Buf mask, blk_cnt, blk_off;
    Buf pt_cell, pt_slot, pt_j;             // link cell, arrival in it and atom number of each point
    Buf pt_gdotr;                           // g.r of each point (link-cell API)
    Buf cell_cnt, cell_start, cell_ids;     // cell_ids: points by cell, unordered inside each
    Buf slot_id, slot_frac, slot_cs64, slot_p32, slot_sn32;
    Buf slot_src;                           // atom and replica of each slot (aperture sums)
    Buf app_cs;                 // per-slot phases of the aperture points of one shared pass
    Buf scan_tmp;
    Buf counters;               // device counters of a condition (struct Counters)
    Buf ax_tab;                 // voxel axis tables
    // fields and image
    Buf f64_re, f64_im, f64_rho, f32_field;
    Buf cnt, r2m;
    Buf img;
    Buf tune_img;               // image written by timing launches of the tuner
    Buf blur_in, blur_tmp, blur_out, blur_w, blur_wy, blur_k;
    // pinned host staging
    void* pinned = nullptr;
    size_t pinned_cap = 0;
    template <class F> void each(F f)
    {
        Buf* all[] = {&x, &mask, &blk_cnt, &blk_off, &pt_cell, &pt_slot, &pt_j, &pt_gdotr,
                      &cell_cnt, &cell_start, &cell_ids, &slot_id, &slot_frac, &slot_cs64,
                      &slot_p32, &slot_sn32, &slot_src, &app_cs, &scan_tmp, &counters, &ax_tab, &f64_re,
                      &f64_im, &f64_rho, &f32_field, &cnt, &r2m, &img, &tune_img, &blur_in, &blur_tmp,
                      &blur_out, &blur_w, &blur_wy, &blur_k};
        for (Buf* b : all) f(*b);
    }
    // every buffer a piece of arena a (no device allocation from then on)
    void bind(Arena* a)
    {
        each([&](Buf& b) { b.arena = a; });
    }
    // device bytes held
    size_t bytes()
    {
        size_t n = 0;
        each([&](Buf& b) { n += b.cap; });
        return n;
    }
    void release_all()
    {
        each([](Buf& b) { b.release(); });
        if (pinned) (void)hipHostFree(pinned);
        pinned = nullptr;
        pinned_cap = 0;
    }
};

struct State {
    int device = -1;
    bool init = false;
    hipStream_t stream = nullptr;
    hipEvent_t ev[10] = {};
    bool pinned_busy = false;       // ev[9] marks the last copy out of the pinned staging buffer
    void* res = nullptr;            // pinned memory that results are copied into
    size_t res_cap = 0;
    Workspace ws;
};

static State g;

static int need_init()
{
    if (!g.init) return seterr(D2BI_ERR_NOINIT, "d2bi_gpu_init has not been called");
    return D2BI_OK;
}

// The pinned staging buffer: a caller that leaves an asynchronous copy from
// it in flight records ev[9] and sets pinned_busy; the next user waits for
// that copy before writing into (or replacing) the buffer.
static int pinned(size_t bytes, void** out)
{
    if (g.pinned_busy) {
        HIPCHK(hipEventSynchronize(g.ev[9]));
        g.pinned_busy = false;
    }
    if (bytes > g.ws.pinned_cap) {
        if (g.ws.pinned) (void)hipHostFree(g.ws.pinned);
        g.ws.pinned = nullptr;
        g.ws.pinned_cap = 0;
        HIPCHK(hipHostMalloc(&g.ws.pinned, bytes, hipHostMallocDefault));
        g.ws.pinned_cap = bytes;
    }
    *out = g.ws.pinned;
    return D2BI_OK;
}

// Pinned memory for results on their way to the caller (a call that copies
// into it waits for its stream before it returns).
static int pinned_result(size_t bytes, void** out)
{
    if (bytes > g.res_cap) {
        if (g.res) (void)hipHostFree(g.res);
        g.res = nullptr;
        g.res_cap = 0;
        HIPCHK(hipHostMalloc(&g.res, bytes, hipHostMallocDefault));
        g.res_cap = bytes;
    }
    *out = g.res;
    return D2BI_OK;
}

// Counters of one condition, cleared before it is binned.  The FAST guard
// re-tests are spread over GUARD_SLOTS lines (many waves adding into one
// address serialise) and added up on the host.
static constexpr int GUARD_SLOTS = 16;               // power of two ...
static constexpr int GUARD_STRIDE = 8;               // ... 64 bytes apart

struct Counters {
    int max_per_cell;           // largest link-cell population
    int n_points;               // points in the link cells
    int pad[14];
    unsigned long long guard[GUARD_SLOTS * GUARD_STRIDE];
    int64_t n_guard() const
    {
        unsigned long long v = 0;
        for (int i = 0; i < GUARD_SLOTS; i++) v += guard[i * GUARD_STRIDE];
        return (int64_t)v;
    }
};

// ------------------------------------------------------------------ device atoms

}  // namespace d2bi

struct d2bi_atoms_s {
    double* x = nullptr;        // 3*n doubles, AoS
    int64_t n = 0;
    // unique per upload: a freed set's device address (and this struct's)
    // can come back for the next upload, with other positions
    uint64_t serial = 0;
};

namespace d2bi {

// ------------------------------------------------------------------ fills

// Kernels clear counters and flags (rather than hipMemsetAsync, which must not
// be recorded into a captured graph): up to four arrays in one launch.
struct ZeroRanges {
    int* p[4];
    int64_t n[4];
};

__global__ void k_zero(ZeroRanges Z)
{
    int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
#pragma unroll
    for (int r = 0; r < 4; r++) {
        if (i >= 0 && i < Z.n[r]) Z.p[r][i] = 0;
        i -= Z.n[r];
    }
}

// The first two arrays, by a kernel that has other work too.
__device__ __forceinline__ void zero_share(const ZeroRanges& Z)
{
    const int64_t step = (int64_t)gridDim.x * blockDim.x, first = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
#pragma unroll
    for (int r = 0; r < 2; r++)
        for (int64_t i = first; i < Z.n[r]; i += step) Z.p[r][i] = 0;
}

static void zero_i32(hipStream_t s, int* p0, int64_t n0, int* p1 = nullptr, int64_t n1 = 0, int* p2 = nullptr,
                     int64_t n2 = 0, int* p3 = nullptr, int64_t n3 = 0)
{
    const ZeroRanges Z{{p0, p1, p2, p3}, {n0, n1, n2, n3}};
    const int64_t n = n0 + n1 + n2 + n3;
    if (n > 0) hipLaunchKernelGGL(k_zero, dim3((unsigned)((n + 255) / 256)), dim3(256), 0, s, Z);
}

// ------------------------------------------------------------------ generic scan

// Inclusive prefix sum over the 64 lanes of a wave in six DPP steps: within
// each row of 16 lanes (row_shr 1, 2, 4, 8 with zero fill), then row 0's
// total into row 1 and row 2's into row 3 (row_bcast:15), then rows 0-1's
// into rows 2-3 (row_bcast:31).  All lanes must be active.
__device__ __forceinline__ int wave_incl_scan(int v)
{
    v += __builtin_amdgcn_update_dpp(0, v, 0x111, 0xf, 0xf, true);
    v += __builtin_amdgcn_update_dpp(0, v, 0x112, 0xf, 0xf, true);
    v += __builtin_amdgcn_update_dpp(0, v, 0x114, 0xf, 0xf, true);
    v += __builtin_amdgcn_update_dpp(0, v, 0x118, 0xf, 0xf, true);
    v += __builtin_amdgcn_update_dpp(0, v, 0x142, 0xa, 0xf, false);
    v += __builtin_amdgcn_update_dpp(0, v, 0x143, 0xc, 0xf, false);
    return v;
}

static constexpr int SCAN_BLOCK = 256;
static constexpr int SCAN_ITEMS = 4;
static constexpr int SCAN_TILE = SCAN_BLOCK * SCAN_ITEMS;

// Block-wide exclusive scan of one int per thread (wave64 prefix sums + LDS);
// lds holds a word per wave and one more.
__device__ inline int block_exclusive_scan(int v, int* total, int* lds)
{
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    const int incl = wave_incl_scan(v);
    if (lane == 63) lds[wave] = incl;
    __syncthreads();
    if (threadIdx.x == 0) {
        int s = 0;
        for (int w = 0; w < (int)(blockDim.x >> 6); w++) { int t = lds[w]; lds[w] = s; s += t; }
        lds[blockDim.x >> 6] = s;
    }
    __syncthreads();
    int r = incl - v + lds[wave];
    *total = lds[blockDim.x >> 6];
    __syncthreads();
    return r;
}

// Largest value of the block, in every thread.
__device__ inline int block_max(int v, int* lds)
{
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) v = max(v, __shfl_xor(v, o, 64));
    if ((threadIdx.x & 63) == 0) lds[threadIdx.x >> 6] = v;
    __syncthreads();
    for (int w = 0; w < (int)(blockDim.x >> 6); w++) v = max(v, lds[w]);
    __syncthreads();
    return v;
}

// The number of points, which only the device knows when the passes after the
// count are launched, and what the point arrays hold.  A condition with more
// points than that is imaged again: the kernels after the count return at once,
// and the link cells come out empty, so that nothing reads past the arrays.
struct PointCount {
    const int* n = nullptr;     // null: no such limit
    int64_t cap = 0;
    // (a count that overflowed is negative)
    __device__ bool over() const { return n && (int64_t)(unsigned)*n > cap; }
    __device__ int64_t stored() const { return over() ? 0 : *n; }
};

// What a scan hands on besides the array: its total and largest value (null:
// not wanted); N: the scan of the cell counts is that of empty cells if over.
struct ScanEnds {
    int* total_out;
    int* max_out;
    PointCount N;
};

// Short arrays (a small condition's block counts or link cells) in one
// workgroup and one launch: on an 80^3 condition the launch gaps of a
// three-phase scan cost more than its work (3 x ~5 us against 5).
static constexpr int SCAN_ONE_BLOCK = 1024;
static constexpr int SCAN_ONE_ITEMS = 16;
static constexpr int SCAN_ONE = SCAN_ONE_BLOCK * SCAN_ONE_ITEMS;

__global__ __launch_bounds__(SCAN_ONE_BLOCK) void k_scan_one(const int* __restrict__ in, int n, int* __restrict__ out,
                                                             ScanEnds E)
{
    __shared__ int lds[SCAN_ONE_BLOCK / 64 + 1];
    const int per = (n + SCAN_ONE_BLOCK - 1) / SCAN_ONE_BLOCK, base = (int)threadIdx.x * per;
    const int end = E.N.over() ? 0 : n;
    int v[SCAN_ONE_ITEMS], s = 0, m = 0;
#pragma unroll
    for (int i = 0; i < SCAN_ONE_ITEMS; i++) v[i] = i < per && base + i < end ? in[base + i] : 0;
#pragma unroll
    for (int i = 0; i < SCAN_ONE_ITEMS; i++) {
        s += v[i];
        m = max(m, v[i]);
    }
    int tot;
    int e = block_exclusive_scan(s, &tot, lds);
#pragma unroll
    for (int i = 0; i < SCAN_ONE_ITEMS; i++) {
        if (i < per && base + i < n) out[base + i] = e;
        e += v[i];
    }
    if (threadIdx.x == 0) {
        out[n] = tot;
        if (E.total_out) *E.total_out = tot;
    }
    if (E.max_out) {
        m = block_max(m, lds);
        if (threadIdx.x == 0) *E.max_out = m;
    }
}

// Longer ones: sums (and largest values) per tile of 1024, then each tile's
// scan behind the sum of the tiles before it, which its workgroup adds up
// itself up to SCAN_SELF tiles; beyond, one workgroup scans the sums between.
static constexpr int SCAN_SELF = 4096;

__global__ __launch_bounds__(SCAN_BLOCK) void k_scan_reduce(const int* __restrict__ in, int64_t n,
                                                            int* __restrict__ sums, int* __restrict__ maxs,
                                                            ScanEnds E)
{
    __shared__ int lds[SCAN_BLOCK / 64 + 1];
    if (E.N.over()) n = 0;
    int64_t base = (int64_t)blockIdx.x * SCAN_TILE + (int64_t)threadIdx.x * SCAN_ITEMS;
    int s = 0, m = 0;
#pragma unroll
    for (int i = 0; i < SCAN_ITEMS; i++)
        if (base + i < n) {
            s += in[base + i];
            m = max(m, in[base + i]);
        }
    int tot;
    block_exclusive_scan(s, &tot, lds);
    m = block_max(m, lds);
    if (threadIdx.x == 0) {
        sums[blockIdx.x] = tot;
        maxs[blockIdx.x] = m;
    }
}

// Single-block exclusive scan of the block sums (any length), in place.
__global__ __launch_bounds__(SCAN_BLOCK) void k_scan_sums(int* __restrict__ sums, int64_t nb)
{
    __shared__ int lds[SCAN_BLOCK / 64 + 1];
    int carry = 0;
    for (int64_t b = 0; b < nb; b += SCAN_BLOCK) {
        int64_t i = b + threadIdx.x;
        int v = i < nb ? sums[i] : 0;
        int tot;
        int e = block_exclusive_scan(v, &tot, lds);
        if (i < nb) sums[i] = e + carry;
        carry += tot;
    }
}

__global__ __launch_bounds__(SCAN_BLOCK) void k_scan_apply(const int* __restrict__ in, int64_t n,
                                                           const int* __restrict__ sums, int scanned,
                                                           const int* __restrict__ maxs, int* __restrict__ out,
                                                           ScanEnds E)
{
    __shared__ int lds[SCAN_BLOCK / 64 + 1];
    const bool over = E.N.over();
    int before = 0;
    if (scanned) {
        before = sums[blockIdx.x];
    } else {
        int p = 0;
        for (int b = threadIdx.x; b < (int)blockIdx.x; b += SCAN_BLOCK) p += sums[b];
        block_exclusive_scan(p, &before, lds);
    }
    int64_t base = (int64_t)blockIdx.x * SCAN_TILE + (int64_t)threadIdx.x * SCAN_ITEMS;
    int v[SCAN_ITEMS];
    int s = 0;
#pragma unroll
    for (int i = 0; i < SCAN_ITEMS; i++) {
        v[i] = base + i < n && !over ? in[base + i] : 0;
        s += v[i];
    }
    int tot;
    int e = block_exclusive_scan(s, &tot, lds) + before;
#pragma unroll
    for (int i = 0; i < SCAN_ITEMS; i++) {
        if (base + i < n) out[base + i] = e;
        e += v[i];
    }
    if (blockIdx.x == gridDim.x - 1 && threadIdx.x == 0) {
        out[n] = before + tot;
        if (E.total_out) *E.total_out = before + tot;
    }
    if (E.max_out && blockIdx.x == 0) {
        int m = 0;
        for (int b = threadIdx.x; b < (int)gridDim.x; b += SCAN_BLOCK) m = max(m, maxs[b]);
        m = block_max(m, lds);
        if (threadIdx.x == 0) *E.max_out = m;
    }
}

static int64_t scan_tmp_ints(int64_t n)
{
    return 2 * std::max<int64_t>(1, (n + SCAN_TILE - 1) / SCAN_TILE);
}

// out[0..n-1] = exclusive scan of in, out[n] = total, and what E asks for.
// tmp: scan_tmp_ints(n) ints of scratch (no allocation here, so the call can
// be captured into a graph).
static int scan_exclusive_tmp(const int* in, int* out, int64_t n, int* tmp, hipStream_t s, const ScanEnds& E)
{
    if (n <= SCAN_ONE) {
        hipLaunchKernelGGL(k_scan_one, dim3(1), dim3(SCAN_ONE_BLOCK), 0, s, in, (int)n, out, E);
    } else {
        const int64_t nb = (n + SCAN_TILE - 1) / SCAN_TILE;
        int *sums = tmp, *maxs = tmp + nb;
        hipLaunchKernelGGL(k_scan_reduce, dim3((unsigned)nb), dim3(SCAN_BLOCK), 0, s, in, n, sums, maxs, E);
        if (nb > SCAN_SELF) hipLaunchKernelGGL(k_scan_sums, dim3(1), dim3(SCAN_BLOCK), 0, s, sums, nb);
        hipLaunchKernelGGL(k_scan_apply, dim3((unsigned)nb), dim3(SCAN_BLOCK), 0, s, in, n, sums,
                           nb > SCAN_SELF ? 1 : 0, maxs, out, E);
    }
    HIPCHK(hipGetLastError());
    return D2BI_OK;
}

}  // namespace d2bi
