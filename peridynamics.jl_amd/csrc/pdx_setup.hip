// Context, body set-up and the bond system of libpdx.
//
// Bond system (reference: src/discretization/bond_system.jl:55-132, 142-176), all on the device:
//  - points are reordered along a Morton curve (radix sort, once) so that the neighbours of a
//    point are close in memory; every get/set maps back to the caller's order;
//  - the neighbour search runs over a cell list with cell size = horizon (the
//    GridNeighborhoodSearch of bond_system.jl:97-99); one wavefront per point counts the
//    neighbours, prefix sums give the rows, and a second pass fills the bonds of every point
//    ordered by internal index;
//  - the neighbour tables of the step kernels' blocks are built in LDS, one workgroup per block;
//  - the pair distance is formed as PointNeighbors does: pos_diff = x_i - x_j,
//    d2 = (p0*p0 + p1*p1) + p2*p2, accepted if d2 <= delta*delta, L = sqrt(d2), so that L
//    is bit-identical to the reference's Bond.length;
//  - precracks (predefined_cracks.jl:31-61, bond_system.jl:142-165, 249-267) are applied
//    inside the same passes: filtered bonds are never emitted, broken ones start inactive.
#include <algorithm>
#include <cmath>
#include <cstdarg>
#include <cstdlib>
#include <cstring>

#include "pdx_internal.h"

static const char *k_version = "pdx-mi355x 0.1.0 (gfx950)";

extern "C" const char *pdx_version(void) { return k_version; }

pdx_status pdx_fail(pdx_ctx *c, pdx_status st, const char *fmt, ...)
{
    if (c) {
        char buf[1024];
        va_list ap;
        va_start(ap, fmt);
        vsnprintf(buf, sizeof buf, fmt, ap);
        va_end(ap);
        c->err = buf;
    }
    return st;
}

extern "C" const char *pdx_last_error(const pdx_ctx *c)
{
    return c ? c->err.c_str() : "null context";
}

#define FREE(p)                                                                             \
    do {                                                                                    \
        if (p) (void)hipFree(p);                                                            \
        p = nullptr;                                                                        \
    } while (0)

static void free_bonds(pdx_ctx *c)
{
    FREE(c->slice_ptr);
    FREE(c->cnt);
    FREE(c->bw);
    FREE(c->bw16);
    FREE(c->pk);
    FREE(c->d_fp);
    FREE(c->halo_ptr);
    FREE(c->halo);
    c->lds_mode = false;
    c->halo_max = 0;
    FREE(c->L);
    FREE(c->Lf);
}

void pdx_free_all(pdx_ctx *c)
{
    pdx_nk_free(c);
    pdx_gnn_free(c);
    FREE(c->d_psets);
    FREE(c->d_pid);
    FREE(c->scf);
    FREE(c->scf32);
    FREE(c->mfactor);
    FREE(c->fd_pts);
    FREE(c->fd_src);
    FREE(c->dr_vh_old);
    FREE(c->dr_bint_old);
    FREE(c->dr_density);
    FREE(c->dr_part);
    FREE(c->rec[0]);
    FREE(c->rec[1]);
    FREE(c->Xr);
    FREE(c->u);
    FREE(c->vh);
    FREE(c->v);
    FREE(c->a);
    FREE(c->bint);
    FREE(c->bext);
    FREE(c->damage);
    FREE(c->nact);
    FREE(c->killed);
    FREE(c->pstate);
    FREE(c->defgrad);
    FREE(c->cauchy);
    FREE(c->d_perm);
    FREE(c->d_iperm);
    FREE(c->stage);
    FREE(c->bcslot);
    FREE(c->slot_src);
    FREE(c->bcvals);
    free_bonds(c);
    c->dev_bytes = 0;
    c->bonds_built = c->bonds_begun = false;
    c->bcvals_cap = 0;
}

extern "C" pdx_status pdx_create(pdx_ctx **out, int32_t device, int32_t precision)
{
    if (!out) return PDX_ERR_ARG;
    *out = nullptr;
    if (precision != PDX_FP64 && precision != PDX_MIXED) return PDX_ERR_ARG;
    int ndev = 0;
    if (hipGetDeviceCount(&ndev) != hipSuccess || ndev <= 0) return PDX_ERR_HIP;
    if (device < 0 || device >= ndev) return PDX_ERR_ARG;
    pdx_ctx *c = new pdx_ctx();
    c->device = device;
    c->precision = precision;
    if (const char *e = getenv("PDX_BB_UNROLL")) {
        const int v = atoi(e);
        if (v == 2 || v == 4) c->bb_unroll = v;
    }
    if (const char *e = getenv("PDX_BLOCK_POINTS")) c->block_points_env = atoi(e);
    if (const char *e = getenv("PDX_LDS_BUDGET")) c->lds_budget_env = atoi(e);
    if (hipSetDevice(device) != hipSuccess || hipStreamCreate(&c->stream) != hipSuccess ||
        hipEventCreate(&c->ev0) != hipSuccess || hipEventCreate(&c->ev1) != hipSuccess) {
        delete c;
        return PDX_ERR_HIP;
    }
    if (hipMalloc((void **)&c->d_flags, 8 * sizeof(unsigned long long)) != hipSuccess) {
        delete c;
        return PDX_ERR_OOM;
    }
    pdx_pin_open();
    *out = c;
    return PDX_OK;
}

extern "C" void pdx_destroy(pdx_ctx *c)
{
    if (!c) return;
    (void)hipSetDevice(c->device);
    if (c->stream) (void)hipStreamSynchronize(c->stream);
    pdx_export_free(c);
    pdx_pin_close(c);
    pdx_free_all(c);
    FREE(c->d_flags);
    (void)pdx_timed_flush(c);
    for (hipEvent_t e : c->evpool) (void)hipEventDestroy(e);
    if (c->open_ev) (void)hipEventDestroy(c->open_ev);
    if (c->ev0) (void)hipEventDestroy(c->ev0);
    if (c->ev1) (void)hipEventDestroy(c->ev1);
    if (c->stream) (void)hipStreamDestroy(c->stream);
    delete c;
}

extern "C" pdx_status pdx_synchronize(pdx_ctx *c)
{
    if (!c) return PDX_ERR_ARG;
    PDX_HIP(c, hipSetDevice(c->device));
    PDX_HIP(c, hipStreamSynchronize(c->stream));
    PDX_HIP(c, hipDeviceSynchronize());
    return PDX_OK;
}

extern "C" pdx_status pdx_set_points(pdx_ctx *c, int64_t n, const double *X, const double *vol,
                                     const uint8_t *fp)
{
    if (!c) return PDX_ERR_ARG;
    if (n <= 0 || !X || !vol) return pdx_fail(c, PDX_ERR_ARG, "invalid points (n=%lld)", (long long)n);
    if (n >= PDX_MAX_POINTS) return pdx_fail(c, PDX_ERR_UNSUPPORTED, "too many points");
    // all positions are looked at before the context changes: refused points leave the old ones in place
    double mn[3] = {INFINITY, INFINITY, INFINITY}, mx[3] = {-INFINITY, -INFINITY, -INFINITY};
    for (int64_t i = 0; i < n; i++)
        for (int d = 0; d < 3; d++) {
            const double x = X[3 * i + d];
            if (!std::isfinite(x)) return pdx_fail(c, PDX_ERR_ARG, "non-finite position");
            mn[d] = std::min(mn[d], x);
            mx[d] = std::max(mx[d], x);
        }
    PDX_HIP(c, hipSetDevice(c->device));
    PDX_HIP(c, hipStreamSynchronize(c->stream));
    pdx_free_all(c);
    c->n = n;
    c->nb = 0;
    c->X.assign(X, X + 3 * n);
    c->vol.assign(vol, vol + n);
    c->fail_permit.assign(n, 1);
    if (fp)
        for (int64_t i = 0; i < n; i++) c->fail_permit[i] = fp[i] ? 1 : 0;
    std::copy(mn, mn + 3, c->mn);
    std::copy(mx, mx + 3, c->mx);
    c->cracks.clear();
    c->n_src = 0;
    c->n_bcpts = 0;
    return PDX_OK;
}

extern "C" pdx_status pdx_set_material(pdx_ctx *c, int32_t kind, const pdx_params *p)
{
    if (!c || !p) return PDX_ERR_ARG;
    if (kind != PDX_BB && kind != PDX_OSB && kind != PDX_CPD)
        return pdx_fail(c, PDX_ERR_ARG, "unknown material kind %d", kind);
    if (!(p->delta > 0) || !(p->rho > 0))
        return pdx_fail(c, PDX_ERR_ARG, "horizon and rho have to be larger than zero");
    if (kind == PDX_CPD && p->zem != PDX_ZEM_SILLING && p->zem != PDX_ZEM_WAN)
        return pdx_fail(c, PDX_ERR_ARG, "unknown zero-energy-mode stabilisation %d", p->zem);
    if (kind == PDX_CPD && p->model != PDX_SVK && p->model != PDX_NHP && p->model != PDX_LINEAR_ELASTIC &&
        p->model != PDX_NEO_HOOKE)
        return pdx_fail(c, PDX_ERR_ARG, "unknown constitutive model %d", p->model);
    if (p->kernel < PDX_KERNEL_LINEAR || p->kernel > PDX_KERNEL_CUBIC_BSPLINE_NORM)
        return pdx_fail(c, PDX_ERR_ARG, "unknown influence function %d", p->kernel);
    if (kind == PDX_BB && p->kernel != PDX_KERNEL_LINEAR)
        return pdx_fail(c, PDX_ERR_ARG, "BBMaterial has no influence function");
    if (c->bonds_built && c->kind != kind)
        return pdx_fail(c, PDX_ERR_STATE, "material kind changed after the bonds were built");
    c->kind = kind;
    c->P = *p;
    return PDX_OK;
}

extern "C" pdx_status pdx_set_material_sets(pdx_ctx *c, int32_t kind, int32_t n_sets,
                                            const pdx_params *sets, const int32_t *point_set)
{
    if (!c || !sets || n_sets <= 0) return PDX_ERR_ARG;
    if (n_sets > PDX_MAX_PSETS) return pdx_fail(c, PDX_ERR_UNSUPPORTED, "at most %d parameter sets", PDX_MAX_PSETS);
    if (c->n <= 0) return pdx_fail(c, PDX_ERR_STATE, "pdx_set_points first");
    if (n_sets > 1 && !point_set) return PDX_ERR_ARG;
    PDX_TRY(pdx_set_material(c, kind, &sets[0]));
    c->psets.clear();
    c->pset_of.clear();
    if (n_sets == 1) return PDX_OK;
    if (kind == PDX_CPD)
        for (int32_t k = 1; k < n_sets; k++)
            if (sets[k].model != sets[0].model || sets[k].zem_cs != sets[0].zem_cs ||
                sets[k].maxdmg != sets[0].maxdmg || sets[k].zem != sets[0].zem)
                return pdx_fail(c, PDX_ERR_ARG, "the parameter sets of a CMaterial share its model, zem and maxdmg");
    for (int32_t k = 0; k < n_sets; k++) {
        if (!(sets[k].delta > 0) || !(sets[k].rho > 0))
            return pdx_fail(c, PDX_ERR_ARG, "horizon and rho have to be larger than zero");
        if (sets[k].delta != sets[0].delta)
            return pdx_fail(c, PDX_ERR_UNSUPPORTED, "the parameter sets of a body must share the horizon");
        if (sets[k].kernel != sets[0].kernel)
            return pdx_fail(c, PDX_ERR_ARG, "the parameter sets of a body share the material's influence function");
    }
    std::vector<uint8_t> of(c->n);
    for (int64_t i = 0; i < c->n; i++) {
        if (point_set[i] < 0 || point_set[i] >= n_sets)
            return pdx_fail(c, PDX_ERR_ARG, "parameter set of point %lld out of range", (long long)i);
        of[i] = (uint8_t)point_set[i];
    }
    c->psets.assign(sets, sets + n_sets);
    c->pset_of = of;
    return PDX_OK;
}

// device copies of the parameter sets and of each point's set (internal order)
static pdx_status upload_psets(pdx_ctx *c)
{
    if (!c->multi()) return PDX_OK;
    std::vector<pdx_pset> t(c->psets.size());
    for (size_t k = 0; k < t.size(); k++) {
        const pdx_params &q = c->psets[k];
        t[k] = {q.bc, q.epsc, q.epsc - 1e-11 * fabs(q.epsc), q.epsc + 1e-11 * fabs(q.epsc), q.rho,
                q.delta, q.G, q.K, q.lambda, q.mu, (q.zem_cs * q.bc) / q.delta, q.nu};
    }
    std::vector<uint8_t> pid(c->n);
    for (int64_t i = 0; i < c->n; i++) pid[c->iperm[i]] = c->pset_of[i];
    PDX_TRY(pdx_alloc(c, &c->d_psets, t.size()));
    PDX_TRY(pdx_alloc(c, &c->d_pid, c->n));
    PDX_HIP(c, hipMemcpy(c->d_psets, t.data(), sizeof(pdx_pset) * t.size(), hipMemcpyHostToDevice));
    PDX_HIP(c, hipMemcpy(c->d_pid, pid.data(), c->n, hipMemcpyHostToDevice));
    return PDX_OK;
}

extern "C" pdx_status pdx_add_precrack(pdx_ctx *c, int64_t na, const int32_t *a, int64_t nb,
                                       const int32_t *b, int32_t filter)
{
    if (!c) return PDX_ERR_ARG;
    if (c->bonds_built) return pdx_fail(c, PDX_ERR_STATE, "precracks must precede pdx_build_bonds");
    if ((int)c->cracks.size() >= PDX_MAX_CRACKS)
        return pdx_fail(c, PDX_ERR_UNSUPPORTED, "at most %d precracks", PDX_MAX_CRACKS);
    pdx_crack k;
    for (int64_t i = 0; i < na; i++) {
        if (a[i] < 0 || a[i] >= c->n) return pdx_fail(c, PDX_ERR_ARG, "precrack point out of range");
        k.a.push_back(a[i]);
    }
    for (int64_t i = 0; i < nb; i++) {
        if (b[i] < 0 || b[i] >= c->n) return pdx_fail(c, PDX_ERR_ARG, "precrack point out of range");
        k.b.push_back(b[i]);
    }
    k.filter = filter ? 1 : 0;
    c->cracks.push_back(k);
    return PDX_OK;
}

// ----------------------------------------------------------------------------------------
// Morton order: 63-bit keys (three quantised coordinates, bits interleaved), a stable radix sort
// of (key, caller index) eight bits a pass.  One wave sorts a run of keys per pass: it
// ranks 64 keys at a time by matching their digits over the wave, so the order inside a run is
// kept without a barrier.  Measured with the rest of the device set-up (see pdx_build_bonds).
// ----------------------------------------------------------------------------------------
// (256 to 2048 keys: as long as 512 runs remain, so that a small body's waves go through few rounds
// of 64 keys in series; at 6 k points a pass of 21.6 us came from 32 such rounds)
static int64_t rs_run(int64_t n)
{
    int64_t run = 256;
    while (run < 2048 && n > 512 * run) run *= 2;
    return run;
}

__device__ __forceinline__ uint64_t spread3(uint64_t v)
{
    v &= 0x1fffff;
    v = (v | v << 32) & 0x1f00000000ffffULL;
    v = (v | v << 16) & 0x1f0000ff0000ffULL;
    v = (v | v << 8) & 0x100f00f00f00f00fULL;
    v = (v | v << 4) & 0x10c30c30c30c30c3ULL;
    v = (v | v << 2) & 0x1249249249249249ULL;
    return v;
}

__global__ void k_morton_keys(int64_t n, const double *X, double3 mn, double s, uint64_t *key, int32_t *val)
{
    const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= n) return;
    const double m[3] = {mn.x, mn.y, mn.z};
    uint64_t q[3];
    for (int d = 0; d < 3; d++) {
        const double t = (X[3 * i + d] - m[d]) * s;
        q[d] = (uint64_t)fmin(fmax(t, 0.0), 2097151.0);
    }
    key[i] = spread3(q[0]) | spread3(q[1]) << 1 | spread3(q[2]) << 2;
    val[i] = (int32_t)i;
}

// digits of every run: cnt[digit * runs + run]
__global__ __launch_bounds__(64) void k_rs_hist(int64_t n, int run, int shift, const uint64_t *key, int32_t *cnt)
{
    __shared__ int32_t h[256];
    for (int d = threadIdx.x; d < 256; d += 64) h[d] = 0;
    __syncthreads();
    const int64_t b = (int64_t)blockIdx.x * run;
    for (int64_t k = b + threadIdx.x; k < b + run && k < n; k += 64)
        atomicAdd(&h[(key[k] >> shift) & 255], 1);
    __syncthreads();
    for (int d = threadIdx.x; d < 256; d += 64) cnt[(int64_t)d * gridDim.x + blockIdx.x] = h[d];
}

// exclusive sums over the runs of each digit (one workgroup per digit), and the digit's total
__global__ __launch_bounds__(256) void k_rs_scan(int runs, int32_t *cnt, int32_t *total)
{
    __shared__ int32_t sh[256];
    int32_t *c = cnt + (int64_t)blockIdx.x * runs;
    int32_t carry = 0;
    for (int k0 = 0; k0 < runs; k0 += 256) {
        const int k = k0 + threadIdx.x;
        const int32_t v = k < runs ? c[k] : 0;
        sh[threadIdx.x] = v;
        __syncthreads();
        for (int o = 1; o < 256; o <<= 1) {
            const int32_t a = (int)threadIdx.x >= o ? sh[threadIdx.x - o] : 0;
            __syncthreads();
            sh[threadIdx.x] += a;
            __syncthreads();
        }
        if (k < runs) c[k] = carry + sh[threadIdx.x] - v;
        carry += sh[255];
        __syncthreads();
    }
    if (threadIdx.x == 0) total[blockIdx.x] = carry;
}

__global__ __launch_bounds__(64) void k_rs_scatter(int64_t n, int run, int shift, const uint64_t *key, const int32_t *val,
                                                   const int32_t *cnt, const int32_t *total, uint64_t *key_out,
                                                   int32_t *val_out)
{
    __shared__ int32_t pos[256];
    const int lane = threadIdx.x;
    // first position of every digit: four digits per lane, then the sum over the lower lanes
    int32_t t[4], s = 0;
    for (int q = 0; q < 4; q++) {
        t[q] = s;
        s += total[4 * lane + q];
    }
    int32_t x = s;
    for (int o = 1; o < 64; o <<= 1) {
        const int32_t y = __shfl_up(x, o);
        if (lane >= o) x += y;
    }
    for (int q = 0; q < 4; q++)
        pos[4 * lane + q] = x - s + t[q] + cnt[(int64_t)(4 * lane + q) * gridDim.x + blockIdx.x];
    __syncthreads();
    const int64_t b = (int64_t)blockIdx.x * run;
    for (int64_t k0 = b; k0 < b + run && k0 < n; k0 += 64) {
        const int64_t k = k0 + lane;
        const bool in = k < n;
        const uint64_t v = in ? key[k] : 0;
        const int d = (int)((v >> shift) & 255);
        // the lanes with the same digit
        uint64_t same = __ballot(in);
        for (int bit = 0; bit < 8; bit++) {
            const uint64_t m = __ballot((d >> bit) & 1);
            same &= ((d >> bit) & 1) ? m : ~m;
        }
        const int before = __popcll(same & ((1ULL << lane) - 1ULL));
        int32_t p = 0;
        if (in) p = pos[d] + before;
        __syncthreads();  // (one wave: orders the reads of pos before its updates)
        if (in) {
            key_out[p] = v;
            val_out[p] = val[k];
            if (before == 0) pos[d] += __popcll(same);
        }
        __syncthreads();
    }
}

// exclusive sums of n int32 values as int64: runs of SCAN_RUN, then the run totals, then both
#define SCAN_RUN 4096
__global__ __launch_bounds__(256) void k_scan_runs(int64_t n, const int32_t *in, int64_t *total)
{
    __shared__ int64_t sh[4];
    const int64_t b = (int64_t)blockIdx.x * SCAN_RUN;
    int64_t s = 0;
    for (int64_t k = b + threadIdx.x; k < b + SCAN_RUN && k < n; k += 256) s += in[k];
    for (int o = 32; o > 0; o >>= 1) s += __shfl_xor(s, o);
    if ((threadIdx.x & 63) == 0) sh[threadIdx.x >> 6] = s;
    __syncthreads();
    if (threadIdx.x == 0) total[blockIdx.x] = (sh[0] + sh[1]) + (sh[2] + sh[3]);
}

// one workgroup: exclusive sums of the run totals in place, the grand total behind them
__global__ __launch_bounds__(1024) void k_scan_totals(int64_t runs, int64_t *total)
{
    __shared__ int64_t sh[1024];
    int64_t carry = 0;
    for (int64_t k0 = 0; k0 < runs; k0 += 1024) {
        const int64_t k = k0 + threadIdx.x;
        const int64_t v = k < runs ? total[k] : 0;
        sh[threadIdx.x] = v;
        __syncthreads();
        for (int o = 1; o < 1024; o <<= 1) {
            const int64_t a = (int)threadIdx.x >= o ? sh[threadIdx.x - o] : 0;
            __syncthreads();
            sh[threadIdx.x] += a;
            __syncthreads();
        }
        if (k < runs) total[k] = carry + sh[threadIdx.x] - v;
        carry += sh[1023];
        __syncthreads();
    }
    if (threadIdx.x == 0) total[runs] = carry;
}

__global__ __launch_bounds__(256) void k_scan_out(int64_t n, const int32_t *in, const int64_t *total, int64_t *out)
{
    __shared__ int64_t sh[256];
    const int64_t b = (int64_t)blockIdx.x * SCAN_RUN + (int64_t)threadIdx.x * (SCAN_RUN / 256);
    int64_t s = 0;
    for (int q = 0; q < SCAN_RUN / 256; q++) s += b + q < n ? in[b + q] : 0;
    sh[threadIdx.x] = s;
    __syncthreads();
    for (int o = 1; o < 256; o <<= 1) {
        const int64_t a = (int)threadIdx.x >= o ? sh[threadIdx.x - o] : 0;
        __syncthreads();
        sh[threadIdx.x] += a;
        __syncthreads();
    }
    int64_t x = total[blockIdx.x] + sh[threadIdx.x] - s;
    for (int q = 0; q < SCAN_RUN / 256; q++) {
        if (b + q >= n) break;
        out[b + q] = x;
        x += in[b + q];
    }
    if (blockIdx.x == gridDim.x - 1 && threadIdx.x == 0) out[n] = total[gridDim.x];
}

// scratch of one set-up, freed with it
struct setup_scratch {
    std::vector<void *> p;
    ~setup_scratch()
    {
        for (void *q : p) (void)hipFree(q);
    }
    template <class T>
    pdx_status get(pdx_ctx *c, T **out, size_t count)
    {
        *out = nullptr;
        const hipError_t e = hipMalloc((void **)out, std::max<size_t>(count * sizeof(T), 256));
        if (e != hipSuccess)
            return pdx_fail(c, PDX_ERR_OOM, "hipMalloc of %zu bytes failed: %s", count * sizeof(T), hipGetErrorString(e));
        p.push_back(*out);
        return PDX_OK;
    }
};

static inline dim3 grid256(int64_t m) { return dim3((unsigned)((m + 255) / 256)); }

// out[k] = in[0] + ... + in[k - 1], k = 0 .. n
static pdx_status scan_i32(pdx_ctx *c, setup_scratch &S, int64_t n, const int32_t *in, int64_t *out)
{
    const int64_t runs = std::max<int64_t>(1, (n + SCAN_RUN - 1) / SCAN_RUN);
    int64_t *total;
    PDX_TRY(S.get(c, &total, runs + 1));
    hipLaunchKernelGGL(k_scan_runs, dim3((unsigned)runs), dim3(256), 0, c->stream, n, in, total);
    hipLaunchKernelGGL(k_scan_totals, dim3(1), dim3(1024), 0, c->stream, runs, total);
    hipLaunchKernelGGL(k_scan_out, dim3((unsigned)runs), dim3(256), 0, c->stream, n, in, total, out);
    PDX_HIP(c, hipGetLastError());
    return PDX_OK;
}

__global__ void k_invert(int64_t n, const int32_t *perm, int32_t *iperm)
{
    const int64_t m = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (m < n) iperm[perm[m]] = (int32_t)m;
}

// perm and iperm on the device and the host, from the caller's positions on the device
static pdx_status morton_order(pdx_ctx *c, setup_scratch &S, const double *dX, const double mn[3], const double mx[3])
{
    const int64_t n = c->n;
    const double ext = std::max({mx[0] - mn[0], mx[1] - mn[1], mx[2] - mn[2], 1e-300});
    const int run = (int)rs_run(n);
    const int64_t runs = (n + run - 1) / run;
    uint64_t *key[2];
    int32_t *val[2], *cnt, *total;
    for (int q = 0; q < 2; q++) {
        PDX_TRY(S.get(c, &key[q], n));
        PDX_TRY(S.get(c, &val[q], n));
    }
    PDX_TRY(S.get(c, &cnt, 256 * runs));
    PDX_TRY(S.get(c, &total, 256));
    hipLaunchKernelGGL(k_morton_keys, grid256(n), dim3(256), 0, c->stream, n, dX, make_double3(mn[0], mn[1], mn[2]),
                       2097151.0 / ext, key[0], val[0]);
    for (int pass = 0; pass < 8; pass++) {
        const int a = pass & 1, b = a ^ 1;
        hipLaunchKernelGGL(k_rs_hist, dim3((unsigned)runs), dim3(64), 0, c->stream, n, run, 8 * pass, key[a], cnt);
        hipLaunchKernelGGL(k_rs_scan, dim3(256), dim3(256), 0, c->stream, (int)runs, cnt, total);
        hipLaunchKernelGGL(k_rs_scatter, dim3((unsigned)runs), dim3(64), 0, c->stream, n, run, 8 * pass, key[a], val[a],
                           cnt, total, key[b], pass == 7 ? c->d_perm : val[b]);
    }
    hipLaunchKernelGGL(k_invert, grid256(n), dim3(256), 0, c->stream, n, c->d_perm, c->d_iperm);
    PDX_HIP(c, hipGetLastError());
    c->perm.resize(n);
    c->iperm.resize(n);
    PDX_HIP(c, hipMemcpyAsync(c->perm.data(), c->d_perm, sizeof(int32_t) * n, hipMemcpyDeviceToHost, c->stream));
    PDX_HIP(c, hipMemcpyAsync(c->iperm.data(), c->d_iperm, sizeof(int32_t) * n, hipMemcpyDeviceToHost, c->stream));
    PDX_HIP(c, hipStreamSynchronize(c->stream));
    return PDX_OK;
}

// ----------------------------------------------------------------------------------------
// neighbour search kernels
// ----------------------------------------------------------------------------------------
struct search_args {
    int64_t n;
    const double4 *Xr;        // internal order
    const int32_t *pcell;     // 3 per point
    const int64_t *cell_start;
    const int32_t *cell_pts;
    int64_t gx, gy, gz;
    double r2;                // delta * delta
    const int32_t *perm;      // caller index of each internal point
    const uint16_t *cmask;    // crack membership (bit 2k: set a of crack k, 2k+1: set b)
    uint32_t filt_bits;       // bit 2k set: crack k filters its bonds
    const uint8_t *fp;        // fail_permit, internal order
    int32_t *counts;
    pdx_rows rows;
    const int32_t *cnt;
    uint32_t *bw;
    double *L;
    unsigned long long *flags;
};

// the points in internal order: records x|V (reference, both current buffers), failure permission,
// crack membership
__global__ void k_gather_points(int64_t n, const int32_t *perm, const double *X, const double *vol,
                                const uint8_t *fp_in, const uint16_t *cm_in, double4 *Xr, double4 *r0, double4 *r1,
                                uint8_t *fp, uint16_t *cm)
{
    const int64_t m = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (m >= n) return;
    const int64_t i = perm[m];
    const double4 x = make_double4(X[3 * i], X[3 * i + 1], X[3 * i + 2], vol[i]);
    Xr[m] = x;
    r0[m] = x;
    r1[m] = x;
    fp[m] = fp_in[i];
    if (cm) cm[m] = cm_in[i];
}

// cell of every point and the points per cell
__global__ void k_cells(int64_t n, const double4 *Xr, double3 mn, double cs, int64_t gx, int64_t gy, int64_t gz,
                        int32_t *pcell, int32_t *num)
{
    const int64_t m = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (m >= n) return;
    const double4 x = Xr[m];
    const int64_t qx = min(max((int64_t)floor((x.x - mn.x) / cs), (int64_t)0), gx - 1);
    const int64_t qy = min(max((int64_t)floor((x.y - mn.y) / cs), (int64_t)0), gy - 1);
    const int64_t qz = min(max((int64_t)floor((x.z - mn.z) / cs), (int64_t)0), gz - 1);
    pcell[3 * m] = (int32_t)qx;
    pcell[3 * m + 1] = (int32_t)qy;
    pcell[3 * m + 2] = (int32_t)qz;
    atomicAdd(&num[qx + gx * (qy + gy * qz)], 1);
}

// the points of every cell, in any order (the rows are sorted later); num counts down to zero
__global__ void k_cell_points(int64_t n, const int32_t *pcell, int64_t gx, int64_t gy, const int64_t *start,
                              int32_t *num, int32_t *pts)
{
    const int64_t m = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (m >= n) return;
    const int64_t cell = pcell[3 * m] + gx * (pcell[3 * m + 1] + gy * (int64_t)pcell[3 * m + 2]);
    pts[start[cell] + atomicSub(&num[cell], 1) - 1] = (int32_t)m;
}

// sum and maximum of the bond counts: out[0] += , out[1] = max
__global__ __launch_bounds__(256) void k_count_totals(int64_t n, const int32_t *cnt, unsigned long long *out)
{
    unsigned long long s = 0;
    int m = 0;
    for (int64_t k = (int64_t)blockIdx.x * 256 + threadIdx.x; k < n; k += (int64_t)gridDim.x * 256) {
        s += (unsigned long long)cnt[k];
        m = max(m, cnt[k]);
    }
    for (int o = 32; o > 0; o >>= 1) {
        s += __shfl_xor(s, o);
        m = max(m, __shfl_xor(m, o));
    }
    __shared__ unsigned long long sh[2][4];  // one pair of atomics per block
    if ((threadIdx.x & 63) == 0) {
        sh[0][threadIdx.x >> 6] = s;
        sh[1][threadIdx.x >> 6] = (unsigned long long)m;
    }
    __syncthreads();
    if (threadIdx.x == 0) {
        atomicAdd(&out[0], (sh[0][0] + sh[0][1]) + (sh[0][2] + sh[0][3]));
        atomicMax(&out[1], max(max(sh[1][0], sh[1][1]), max(sh[1][2], sh[1][3])));
    }
}

// slots of every slice: 64 per row group of its widest row
__global__ void k_slice_width(int64_t n, int64_t n_slices, pdx_rows rows, const int32_t *cnt, int32_t *width)
{
    const int64_t s = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (s >= n_slices) return;
    const int P = 64 >> rows.ls;
    int w = 0;
    for (int64_t m = P * s; m < min(n, P * s + P); m++) w = max(w, cnt[m]);
    width[s] = 64 * rows.groups(w);
}

// (A_i & B_j) | (B_i & A_j) per crack, at the even bit positions
__device__ __forceinline__ uint32_t crack_hits(uint32_t mi, uint32_t mj)
{
    uint32_t ai = mi & 0x5555u, bi = (mi >> 1) & 0x5555u;
    uint32_t aj = mj & 0x5555u, bj = (mj >> 1) & 0x5555u;
    return (ai & bj) | (bi & aj);
}

__device__ __forceinline__ double pair_d2(double4 xi, double4 xj)
{
    double p0 = xi.x - xj.x, p1 = xi.y - xj.y, p2 = xi.z - xj.z;
    return (p0 * p0 + p1 * p1) + p2 * p2;
}

__global__ __launch_bounds__(PDX_BLOCK) void k_count_bonds(search_args s)
{
    int64_t i = pdx_wave_point();
    if (i >= s.n) return;
    int lane = threadIdx.x & 63;
    double4 xi = s.Xr[i];
    int cx = s.pcell[3 * i], cy = s.pcell[3 * i + 1], cz = s.pcell[3 * i + 2];
    uint32_t mi = s.cmask ? s.cmask[i] : 0;
    int cnt = 0;
    const int64_t x0 = max(cx - 1, 0), x1 = min((int64_t)cx + 1, s.gx - 1);
    for (int z = cz - 1; z <= cz + 1; z++) {
        if (z < 0 || z >= s.gz) continue;
        for (int y = cy - 1; y <= cy + 1; y++) {
            if (y < 0 || y >= s.gy) continue;
            // the cells x - 1 .. x + 1 are one run of the cell list
            const int64_t row = s.gx * (y + s.gy * (int64_t)z);
            const int64_t e = s.cell_start[row + x1 + 1];
            for (int64_t k = s.cell_start[row + x0] + lane; k < e; k += 64) {
                int32_t j = s.cell_pts[k];
                if (j == i) continue;
                double d2 = pair_d2(xi, s.Xr[j]);
                if (d2 <= s.r2) {
                    if (sqrt(d2) < 2.220446049250313e-16) {
                        if (atomicExch(&s.flags[1], 1ULL) == 0ULL) {
                            s.flags[2] = (unsigned long long)s.perm[i];
                            s.flags[3] = (unsigned long long)s.perm[j];
                        }
                    }
                    uint32_t h = s.cmask ? crack_hits(mi, s.cmask[j]) : 0u;
                    if (!(h & s.filt_bits)) cnt++;
                }
            }
        }
    }
    cnt = pdx_wave_sum_i(cnt);
    if (lane == 0) s.counts[i] = cnt;
}

__global__ __launch_bounds__(PDX_BLOCK) void k_fill_bonds(search_args s)
{
    __shared__ __align__(16) int32_t cj[PDX_WAVES_PER_BLOCK][PDX_FILL_CAP + 4];
    int64_t i = pdx_wave_point();
    if (i >= s.n) return;
    int lane = threadIdx.x & 63;
    int w = threadIdx.x >> 6;
    double4 xi = s.Xr[i];
    int cx = s.pcell[3 * i], cy = s.pcell[3 * i + 1], cz = s.pcell[3 * i + 2];
    uint32_t mi = s.cmask ? s.cmask[i] : 0;
    const int64_t b0 = s.rows.row(i);
    const int want = s.cnt[i];                          // <= PDX_FILL_CAP, checked on the host
    int base = 0;
    const int64_t x0 = max(cx - 1, 0), x1 = min((int64_t)cx + 1, s.gx - 1);
    for (int z = cz - 1; z <= cz + 1; z++) {
        if (z < 0 || z >= s.gz) continue;
        for (int y = cy - 1; y <= cy + 1; y++) {
            if (y < 0 || y >= s.gy) continue;
            const int64_t row = s.gx * (y + s.gy * (int64_t)z);
            const int64_t st = s.cell_start[row + x0], e = s.cell_start[row + x1 + 1];
            for (int64_t k0 = st; k0 < e; k0 += 64) {
                int64_t k = k0 + lane;
                bool take = false;
                int32_t j = -1;
                if (k < e) {
                    j = s.cell_pts[k];
                    if (j != i) {
                        double d2 = pair_d2(xi, s.Xr[j]);
                        uint32_t h = s.cmask ? crack_hits(mi, s.cmask[j]) : 0u;
                        take = (d2 <= s.r2) && !(h & s.filt_bits);
                    }
                }
                uint64_t m = __ballot(take);
                int pos = base + (int)__popcll(m & ((1ULL << lane) - 1ULL));
                if (take && pos < PDX_FILL_CAP) cj[w][pos] = j;
                base += (int)__popcll(m);
            }
        }
    }
    const int cnt = min(base, want);
    if (lane < 4) cj[w][cnt + lane] = 0x7fffffff;  // the ranking reads four at a time
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
    // rows are ordered by the neighbour's internal (Morton) index, so that the lanes of a gather
    // read neighbouring records and the tiles of a table are met in order; pdx_get_bonds reorders
    // rows by caller index.  Two bonds per lane are ranked in one sweep over the row.
    for (int k = lane; k < cnt; k += 128) {
        const int32_t ja = cj[w][k], jb = k + 64 < cnt ? cj[w][k + 64] : 0x7fffffff;
        int ra = 0, rb = 0;
        for (int q = 0; q < cnt; q += 4) {
            const int4 v = *reinterpret_cast<const int4 *>(&cj[w][q]);
            ra += (v.x < ja ? 1 : 0) + (v.y < ja ? 1 : 0) + (v.z < ja ? 1 : 0) + (v.w < ja ? 1 : 0);
            rb += (v.x < jb ? 1 : 0) + (v.y < jb ? 1 : 0) + (v.z < jb ? 1 : 0) + (v.w < jb ? 1 : 0);
        }
#pragma unroll
        for (int u = 0; u < 2; u++) {
            if (k + 64 * u >= cnt) break;
            const int32_t j = u ? jb : ja;
            const double d2 = pair_d2(xi, s.Xr[j]);
            const uint32_t h = s.cmask ? crack_hits(mi, s.cmask[j]) : 0u;
            const uint32_t fpb = (s.fp[i] & s.fp[j]) ? PDX_BW_FP : 0u;
            const uint32_t act = (h & ~s.filt_bits) ? 0u : PDX_BW_ACT;  // broken at t = 0 by a precrack
            const int64_t b = s.rows.at(b0, u ? rb : ra);
            s.bw[b] = (uint32_t)j | act | fpb;
            s.L[b] = sqrt(d2);
        }
    }
}

__global__ void k_init_point_state(int64_t n, pdx_rows rows, const int32_t *cnt,
                                   const uint32_t *bw, int32_t *nact, double *damage)
{
    const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= n) return;
    const int64_t b0 = rows.row(i);
    int na = 0;
    for (int t = 0; t < cnt[i]; t++) na += (bw[rows.at(b0, t)] & PDX_BW_ACT) ? 1 : 0;
    nact[i] = na;
    // calc_damage!: 1 - n_active / n_neighbors (NaN for a point without bonds)
    damage[i] = 1.0 - (double)na / (double)cnt[i];
}

// Kernels over the bond slots.  A launch takes fewer than 2^32 threads, and a body of 37 M points at
// 3.015 spacings (8 M at 5.015) has more slots than that, so their threads go over the slots in
// strides; the grid covers bodies of up to 2^30 slots in one.
static inline dim3 slot_grid(int64_t slots)
{
    return dim3((unsigned)std::min<int64_t>((slots + 255) / 256, (int64_t)1 << 22));
}

#define PDX_SLOT_LOOP(k, n)                                                                               \
    for (int64_t k = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; k < (n); k += (int64_t)gridDim.x * blockDim.x)

__global__ void k_fill_value(int64_t n, double v, double *out)
{
    PDX_SLOT_LOOP(k, n) out[k] = v;
}

__global__ void k_L_to_float(int64_t nb, const double *L, float *Lf)
{
    PDX_SLOT_LOOP(k, nb) Lf[k] = (float)L[k];
}

// ----------------------------------------------------------------------------------------
// permuted transfers
// ----------------------------------------------------------------------------------------
// dev[m*stride + d] = stage[perm[m]*comps + d]
__global__ void k_scatter_in(int64_t n, int comps, int stride, const int32_t *perm,
                             const double *stage, double *dev)
{
    int64_t t = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (t >= n * comps) return;
    int64_t m = t / comps;
    int d = (int)(t - m * comps);
    dev[m * stride + d] = stage[(int64_t)perm[m] * comps + d];
}

// dst[t - t0] = dev[iperm[t / comps] * stride + t % comps]
__global__ void k_gather_out(int64_t t0, int64_t t1, int comps, int stride, const int32_t *iperm, const double *dev,
                             double *dst)
{
    const int64_t t = t0 + (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (t >= t1) return;
    const int64_t i = t / comps;
    const int d = (int)(t - i * comps);
    dst[t - t0] = dev[(int64_t)iperm[i] * stride + d];
}

pdx_status pdx_gather_range(pdx_ctx *c, const double *dev, int comps, int stride, int64_t t0, int64_t t1, double *dst)
{
    hipLaunchKernelGGL(k_gather_out, grid256(t1 - t0), dim3(256), 0, c->stream, t0, t1, comps, stride, c->d_iperm, dev, dst);
    PDX_HIP(c, hipGetLastError());
    return PDX_OK;
}

pdx_status pdx_upload_vec(pdx_ctx *c, const double *host, double *dev, int comps)
{
    int stride = comps;
    return pdx_upload_strided(c, host, dev, comps, stride);
}

pdx_status pdx_upload_strided(pdx_ctx *c, const double *host, double *dev, int comps, int stride)
{
    int64_t cnt = c->n * comps;
    PDX_HIP(c, hipMemcpyAsync(c->stage, host, sizeof(double) * cnt, hipMemcpyHostToDevice,
                              c->stream));
    int64_t blocks = (cnt + 255) / 256;
    hipLaunchKernelGGL(k_scatter_in, dim3(blocks), dim3(256), 0, c->stream, c->n, comps, stride,
                       c->d_perm, c->stage, dev);
    PDX_HIP(c, hipGetLastError());
    PDX_HIP(c, hipStreamSynchronize(c->stream));
    return PDX_OK;
}

// ----------------------------------------------------------------------------------------
// packed bonds
// ----------------------------------------------------------------------------------------
// bit patterns of the shortest and the longest active bond (positive doubles order as their bits
// do): range[0] starts at ~0, range[1] at 0
__global__ __launch_bounds__(256) void k_len_range(int64_t nb, const uint32_t *bw, const double *L,
                                                   unsigned long long *range)
{
    unsigned long long lo = ~0ULL, hi = 0ULL;
    for (int64_t b = (int64_t)blockIdx.x * 256 + threadIdx.x; b < nb; b += (int64_t)gridDim.x * 256) {
        if (!(bw[b] & PDX_BW_ACT)) continue;  // also the padding
        const unsigned long long v = (unsigned long long)__double_as_longlong(L[b]);
        lo = v < lo ? v : lo;
        hi = v > hi ? v : hi;
    }
    for (int o = 32; o > 0; o >>= 1) {
        const unsigned long long a = __shfl_xor(lo, o), b = __shfl_xor(hi, o);
        lo = a < lo ? a : lo;
        hi = b > hi ? b : hi;
    }
    // one pair of atomics per block: they all meet on one address (four pairs from each of 2048 blocks
    // took 0.2 to 0.33 ms)
    __shared__ unsigned long long sh[2][4];
    if ((threadIdx.x & 63) == 0) {
        sh[0][threadIdx.x >> 6] = lo;
        sh[1][threadIdx.x >> 6] = hi;
    }
    __syncthreads();
    if (threadIdx.x == 0) {
        for (int w = 1; w < 4; w++) {
            lo = sh[0][w] < lo ? sh[0][w] : lo;
            hi = sh[1][w] > hi ? sh[1][w] : hi;
        }
        atomicMin(&range[0], lo);
        atomicMax(&range[1], hi);
    }
}

// in place: the packed word of a slot takes its length's 8 bytes
__global__ void k_pack_bonds(int64_t nb, const uint16_t *w16, double *L, int shift, unsigned long long mask,
                             unsigned long long base)
{
    PDX_SLOT_LOOP(b, nb)
    {
        const uint32_t w = w16[b];
        const unsigned long long v = (unsigned long long)__double_as_longlong(L[b]) - base;
        L[b] = __longlong_as_double(
            (long long)((unsigned long long)(w & PDX_W16_SLOT) << shift | ((w & PDX_W16_ACT) ? v : mask)));
    }
}

// One 64-bit word per bond in place of the 16-bit word and the FP64 length (FP64 contexts with
// one parameter set): taken when the table slots and the span of the length patterns share 64
// bits, which the usual horizons do (3.015 spacings: 11 bits of slot, lengths within a factor of
// 4).  The words carry the bond state and take the place of the lengths in memory (12 bytes per
// slot with the 32-bit word, 14 unpacked); the passes that are not per step form a length again
// from the reference positions (pdx_ref_len).
static pdx_status pack_bonds(pdx_ctx *c)
{
    if (c->precision != PDX_FP64 || c->multi() || c->nb <= 0) return PDX_OK;
    unsigned long long *range = c->d_flags + 4, h[2] = {~0ULL, 0ULL};
    PDX_HIP(c, hipMemcpyAsync(range, h, sizeof h, hipMemcpyHostToDevice, c->stream));
    hipLaunchKernelGGL(k_len_range, dim3((unsigned)std::min<int64_t>((c->nb_alloc + 1023) / 1024, 2048)), dim3(256), 0,
                       c->stream, c->nb_alloc, c->bw, c->L, range);
    PDX_HIP(c, hipGetLastError());
    PDX_HIP(c, hipMemcpyAsync(h, range, sizeof h, hipMemcpyDeviceToHost, c->stream));
    PDX_HIP(c, hipStreamSynchronize(c->stream));
    int sb = 1;
    while ((1 << sb) < c->halo_max) sb++;
    const int shift = 64 - sb;
    const unsigned long long mask = (1ULL << shift) - 1;
    if (h[0] > h[1]) h[0] = h[1] = 0;  // no active bond
    if (h[1] - h[0] >= mask) return PDX_OK;
    c->pk_shift = shift;
    c->pk_mask = mask;
    c->pk_base = h[0];
    hipLaunchKernelGGL(k_pack_bonds, slot_grid(c->nb_alloc), dim3(256), 0, c->stream,
                       c->nb_alloc, c->bw16, c->L, shift, mask, h[0]);
    PDX_HIP(c, hipGetLastError());
    PDX_HIP(c, hipStreamSynchronize(c->stream));
    c->pk = reinterpret_cast<unsigned long long *>(c->L);
    c->L = nullptr;
    FREE(c->bw16);
    c->dev_bytes -= (int64_t)sizeof(uint16_t) * c->nb_alloc;
    return PDX_OK;
}

// ----------------------------------------------------------------------------------------
// Neighbour tables of the LDS-staged kernels: for every block of PB consecutive (Morton) points
// the sorted list of the points its bonds reach; every bond gets a 16-bit slot into its block's
// list.  One workgroup per block: the neighbours go into a hash table in LDS, its entries are
// compacted and sorted there, and the bonds look their slots up by bisection.  Run twice: the
// first run (WRITE = false) only counts.
// ----------------------------------------------------------------------------------------
#define HALO_T 512
#define HALO_HASH 16384
#define HALO_LIST (PDX_W16_SLOT + 1)  // longest table that the slots address

template <bool WRITE>
__global__ __launch_bounds__(HALO_T) void k_halo(int64_t n, int PB, pdx_rows rows, const int32_t *cnt,
                                                 const uint32_t *bw, int32_t *count, const int64_t *hptr,
                                                 int32_t *halo, uint16_t *w16)
{
    extern __shared__ int32_t lds[];
    int32_t *const hash = lds, *const list = lds + HALO_HASH;
    __shared__ int num, pos;
    const int64_t p0 = (int64_t)blockIdx.x * PB;
    const int P = 64 >> rows.ls, S = 1 << rows.ls, lane = threadIdx.x & 63;
    const int64_t s1 = (min(p0 + PB, n) + P - 1) / P;
    for (int q = threadIdx.x; q < HALO_HASH; q += HALO_T) hash[q] = -1;
    if (threadIdx.x == 0) num = pos = 0;
    __syncthreads();
    // lane -> point of the slice and its bonds: group g holds bond t(g) (pdx_rows::at)
    const int sub = lane & (S - 1), kk = sub >> 2, m = S >> 2;
    auto bond_no = [&](int g) { return 16 * ((g >> 2) * m + kk) + 4 * (g & 3) + (sub & 3); };
    for (int64_t s = p0 / P + (threadIdx.x >> 6); s < s1; s += HALO_T / 64) {
        const int64_t p = s * P + (lane >> rows.ls), b0 = rows.ptr[s];
        const int c = p < n ? cnt[p] : 0;
        const int ng = (int)((rows.ptr[s + 1] - b0) >> 6);
        for (int g = 0; g < ng; g++) {
            if (bond_no(g) >= c) continue;
            const int32_t j = (int32_t)(bw[b0 + (int64_t)g * 64 + lane] & PDX_BW_NBR);
            uint32_t h = ((uint32_t)j * 2654435761u) >> 18;
            // at most HALO_LIST entries and one more per thread go in, so a probe ends at j or a free cell
            while (true) {
                const int32_t e = hash[h];
                if (e == j) break;
                if (e == -1) {
                    if (*(volatile int *)&num > HALO_LIST) break;
                    const int32_t old = atomicCAS(&hash[h], -1, j);
                    if (old == -1) atomicAdd(&num, 1);
                    if (old == -1 || old == j) break;
                }
                h = (h + 1) & (HALO_HASH - 1);
            }
        }
    }
    __syncthreads();
    const int H = num;
    if (!WRITE) {
        if (threadIdx.x == 0) count[blockIdx.x] = H;
        return;
    }
    for (int q = threadIdx.x; q < HALO_HASH; q += HALO_T)
        if (hash[q] >= 0) list[atomicAdd(&pos, 1)] = hash[q];
    int np = 1;
    while (np < H) np <<= 1;
    __syncthreads();
    for (int q = H + (int)threadIdx.x; q < np; q += HALO_T) list[q] = 0x7fffffff;
    __syncthreads();
    for (int k = 2; k <= np; k <<= 1)
        for (int d = k >> 1; d > 0; d >>= 1) {
            for (int q = threadIdx.x; q < np / 2; q += HALO_T) {
                const int a = 2 * q - (q & (d - 1)), b = a + d;
                const int32_t x = list[a], y = list[b];
                if ((x > y) == ((a & k) == 0)) {
                    list[a] = y;
                    list[b] = x;
                }
            }
            __syncthreads();
        }
    int32_t *const out = halo + hptr[blockIdx.x];
    for (int q = threadIdx.x; q < H; q += HALO_T) out[q] = list[q];
    for (int64_t s = p0 / P + (threadIdx.x >> 6); s < s1; s += HALO_T / 64) {
        const int64_t p = s * P + (lane >> rows.ls), b0 = rows.ptr[s];
        const int c = p < n ? cnt[p] : 0;
        const int ng = (int)((rows.ptr[s + 1] - b0) >> 6);
        // the slots past the row's end repeat its last neighbour, not active
        const uint32_t last = c > 0 ? bw[rows.at(rows.row(p), c - 1)] & PDX_BW_NBR : 0u;
        for (int g = 0; g < ng; g++) {
            const int64_t b = b0 + (int64_t)g * 64 + lane;
            const uint32_t w = bond_no(g) < c ? bw[b] : last;
            const int32_t j = (int32_t)(w & PDX_BW_NBR);
            int lo = 0, hi = H;
            while (lo < hi) {
                const int mid = (lo + hi) >> 1;
                if (list[mid] < j) lo = mid + 1;
                else hi = mid;
            }
            w16[b] = c > 0 ? (uint16_t)(lo | ((w & PDX_BW_ACT) ? PDX_W16_ACT | PDX_W16_RACT : 0u) |
                                        ((w & PDX_BW_FP) ? PDX_W16_FP : 0u))
                           : (uint16_t)0;
        }
    }
}

// the largest of n counts
__global__ __launch_bounds__(256) void k_max_i32(int64_t n, const int32_t *in, unsigned long long *out)
{
    int m = 0;
    for (int64_t k = (int64_t)blockIdx.x * 256 + threadIdx.x; k < n; k += (int64_t)gridDim.x * 256) m = max(m, in[k]);
    for (int o = 32; o > 0; o >>= 1) m = max(m, __shfl_xor(m, o));
    if ((threadIdx.x & 63) == 0) atomicMax(out, (unsigned long long)m);
}

// Builds the tables and the 16-bit words; *ok = false (and no LDS layout) if a table does not fit.
static pdx_status build_halos(pdx_ctx *c, bool *ok)
{
    *ok = false;
    const int64_t n = c->n, PB = c->pb, nblk = (n + PB - 1) / PB;
    int lds = 0;
    PDX_HIP(c, hipDeviceGetAttribute(&lds, hipDeviceAttributeMaxSharedMemoryPerBlock, c->device));
    // 64 bytes of slack for the alignment pad of a trailing byte table.  A table longer than
    // what LDS holds is still served: the kernels stage it in tiles or stage what fits and read
    // the rest from global memory, so only the 13-bit slot field limits a table.
    c->lds_limit = std::min<int64_t>(lds, 160 * 1024) - 64;
    setup_scratch S;
    int32_t *count;
    PDX_TRY(S.get(c, &count, nblk));
    const size_t hl = sizeof(int32_t) * (HALO_HASH + HALO_LIST);
    hipLaunchKernelGGL(k_halo<false>, dim3((unsigned)nblk), dim3(HALO_T), hl, c->stream, n, (int)PB, c->rows(),
                       c->cnt, c->bw, count, nullptr, nullptr, nullptr);
    PDX_HIP(c, hipGetLastError());
    PDX_TRY(pdx_alloc(c, &c->halo_ptr, nblk + 1));
    PDX_TRY(scan_i32(c, S, nblk, count, c->halo_ptr));
    unsigned long long *mx = c->d_flags + 6, h[1] = {0};
    int64_t total = 0;
    PDX_HIP(c, hipMemcpyAsync(mx, h, sizeof h, hipMemcpyHostToDevice, c->stream));
    hipLaunchKernelGGL(k_max_i32, dim3((unsigned)std::min<int64_t>((nblk + 255) / 256, 256)), dim3(256), 0, c->stream,
                       nblk, count, mx);
    PDX_HIP(c, hipMemcpyAsync(h, mx, sizeof h, hipMemcpyDeviceToHost, c->stream));
    PDX_HIP(c, hipMemcpyAsync(&total, c->halo_ptr + nblk, sizeof total, hipMemcpyDeviceToHost, c->stream));
    PDX_HIP(c, hipStreamSynchronize(c->stream));
    // a longer table: the global-gather kernels
    if (h[0] > HALO_LIST) {
        FREE(c->halo_ptr);
        c->dev_bytes -= (int64_t)sizeof(int64_t) * (nblk + 1);
        return PDX_OK;
    }
    PDX_TRY(pdx_alloc(c, &c->bw16, c->nb_alloc));
    PDX_TRY(pdx_alloc(c, &c->halo, std::max<int64_t>(total, 1)));
    hipLaunchKernelGGL(k_halo<true>, dim3((unsigned)nblk), dim3(HALO_T), hl, c->stream, n, (int)PB, c->rows(),
                       c->cnt, c->bw, count, c->halo_ptr, c->halo, c->bw16);
    PDX_HIP(c, hipGetLastError());
    c->halo_max = (int32_t)h[0];
    c->halo_total = total;
    c->lds_mode = true;
    *ok = true;
    return pack_bonds(c);
}

// Points per block and lanes per point of the LDS-staged kernels (pdx_step.hip, with_cfg): 256 x 4,
// 128 x 4, 64 x 8 or 32 x 16.  A small body needs many small blocks (a 6400-point one is 25 blocks of
// 256 points on 256 CUs) and many lanes per point (its step is one chain of load latencies per
// lane); a large one wants the larger blocks' smaller neighbour tables per point.  Measured, us
// per step, the best of five runs of 100 or 200 steps (at 2 M points their mean is 1 % longer, single
// launches vary by 10 %), blocks of 256 / 128 / 64 / 32 points, 3.015 spacings:
//   BB FP64   6 k 14.9 / 10.3 /  7.7 /  6.6    14 k 17.5 / 12.0 /  9.1 /  9.0
//            25 k 17.8 / 12.2 / 12.5 / 13.0   100 k 31.4 / 30.7 / 30.8 / 35.3
//             2 M  569 /  530 /  628 /  762
//   CPD FP64  6 k  n/a / 27.9 / 21.7 / 18.5    14 k  n/a / 38.2 / 29.4 / 27.9
//            25 k  n/a / 40.4 / 39.1 / 46.5    54 k  n/a / 60.4 / 68.0 / 78.8
//           512 k  n/a /  450 /  580 /  762     2 M  n/a / 1731 / 2219 / 2965
// so the blocks are the largest that still give 160 of them, and those of 32 points, where twice as
// many cost little, hold until 64-point blocks number 256 (12 k to 16 k points, 64 against 32: BB
// 9.0 / 8.8, mixed BB 8.8 / 8.7, OSB 17.2 / 17.1, CPD 29.4 / 27.2; the load step of 14 k points
// 33.5 against 31.9 ms).  FP64 stops at 128 points, whose blocks share a CU two or three at a time (OSB
// at 2 M 1022 / 1029 / 1186 / 1446).  Horizons beyond about 4 spacings stop at 64 points, whose
// neighbour tables still fit a block's share of the LDS (5.015 spacings: BB at 121 k 215 / 174 / 160 /
// 163, OSB at 400 k 1050 / 935 / 918 / 968, CPD at 100 k n/a / 504 / 395 / 375, mixed BB 256 against 64
// points 54 / 52 at 54 k, 105 / 106 at 121 k, 327 / 295 at 400 k, 478 / 442 at 576 k, mixed OSB 932 / 893
// there; 4.015 spacings: CPD at 100 k n/a / 214 / 192 / 211).
// The mixed BB and OSB steps of bodies beyond a million points go to 256 points (340 against 361 and 647
// against 677 at 2 M, 200x200x50).  That line is coarse: four 128-point blocks share a CU where every table
// fits a quarter of its LDS (1279 entries), else three, and which it is depends on how the Morton
// curve folds into the body (BB, 256 against 128: 1 M points 164 / 157, 1.1 M 179 / 194, 1.3 M 214 / 208,
// 1.6 M 251 / 273, 1.7 M 224 / 219, 2.6 M 404 / 395; OSB 316 / 317, 339 / 360, 409 / 410, 479 / 507, 419 / 407,
// 779 / 788).
static void choose_blocks(pdx_ctx *c, bool lds)
{
    if (!lds) {
        c->cfg = -1;
        c->ls = 0;
        c->pb = PDX_BLOCK;
        return;
    }
    static const int pbs[4] = {256, 128, 64, 32}, lss[4] = {2, 2, 3, 4};
    int first = 1;
    if (c->nb > 180 * c->n) first = 2;
    else if (c->kind != PDX_CPD && c->precision == PDX_MIXED && c->n > 1000000) first = 0;
    int k = first;
    while (k < 3 && c->n < (int64_t)(k == 2 ? 256 : 160) * pbs[k]) k++;
    // PDX_BLOCK_POINTS: one of the four sizes whatever the body (no correspondence kernel has 256)
    for (int q = c->kind == PDX_CPD ? 1 : 0; q < 4; q++)
        if (c->block_points_env == pbs[q]) k = q;
    c->cfg = k;
    c->pb = pbs[k];
    c->ls = lss[k];
}

// the rows of the chosen layout: slice pointers, bond words and lengths
static pdx_status fill_rows(pdx_ctx *c, search_args &s)
{
    if (c->bw) c->dev_bytes -= (int64_t)(sizeof(uint32_t) + sizeof(double)) * c->nb_alloc;
    FREE(c->slice_ptr);
    FREE(c->bw);
    FREE(c->L);
    const int64_t n = c->n, n_slices = c->n_slices();
    setup_scratch S;
    int32_t *width;
    PDX_TRY(S.get(c, &width, n_slices));
    PDX_TRY(pdx_alloc(c, &c->slice_ptr, n_slices + 1));
    hipLaunchKernelGGL(k_slice_width, grid256(n_slices), dim3(256), 0, c->stream, n, n_slices, c->rows(), c->cnt, width);
    PDX_TRY(scan_i32(c, S, n_slices, width, c->slice_ptr));
    int64_t nba = 0;
    PDX_HIP(c, hipMemcpyAsync(&nba, c->slice_ptr + n_slices, sizeof nba, hipMemcpyDeviceToHost, c->stream));
    PDX_HIP(c, hipStreamSynchronize(c->stream));
    c->nb_alloc = nba;
    if (nba >= ((int64_t)1 << 40)) return pdx_fail(c, PDX_ERR_UNSUPPORTED, "too many bonds");
    PDX_TRY(pdx_alloc(c, &c->bw, nba));
    PDX_TRY(pdx_alloc(c, &c->L, nba));
    // padding slots: bond word 0, length 1
    PDX_HIP(c, hipMemsetAsync(c->bw, 0, sizeof(uint32_t) * nba, c->stream));
    if (nba > 0)
        hipLaunchKernelGGL(k_fill_value, slot_grid(nba), dim3(256), 0, c->stream, nba, 1.0, c->L);
    PDX_HIP(c, hipGetLastError());
    s.rows = c->rows();
    s.cnt = c->cnt;
    s.bw = c->bw;
    s.L = c->L;
    hipLaunchKernelGGL(k_fill_bonds, dim3((unsigned)pdx_wave_grid(n)), dim3(PDX_BLOCK), 0, c->stream, s);
    PDX_HIP(c, hipGetLastError());
    PDX_HIP(c, hipStreamSynchronize(c->stream));
    return PDX_OK;
}

// ----------------------------------------------------------------------------------------
// pdx_build_bonds.  The host takes part only to size allocations and to keep the point order (eight
// synchronisations, nine for a correspondence body).  A
// 576 k-point BB body of 61 M bonds: 8.6 ms (fill 1.5, tables 1.7, count 1.3, packing 0.5, sort 0.5
// ms of kernels, the rest allocations and the upload) against 0.27 s with the sort, the cell list
// and the tables on the host (the tables alone moved the 32-bit words to the host and back).
// ----------------------------------------------------------------------------------------
extern "C" pdx_status pdx_build_bonds(pdx_ctx *c, int64_t *n_bonds_out)
{
    if (!c) return PDX_ERR_ARG;
    if (c->n <= 0) return pdx_fail(c, PDX_ERR_STATE, "pdx_set_points first");
    if (c->kind < 0) return pdx_fail(c, PDX_ERR_STATE, "pdx_set_material first");
    PDX_HIP(c, hipSetDevice(c->device));
    const int64_t n = c->n;
    for (int d = 0; d < 3; d++)  // (the cells are counted from the extent)
        if (!std::isfinite(c->mx[d] - c->mn[d]))
            return pdx_fail(c, PDX_ERR_UNSUPPORTED, "the extent of the body is not a finite number");
    if (c->bonds_begun) {
        // again, or after a build that ended in an error and left arrays of its sizes behind (pdx_alloc
        // keeps what is there): drop everything but the points
        std::vector<pdx_crack> keep = c->cracks;
        pdx_free_all(c);
        c->cracks = keep;
    }
    c->bonds_begun = true;
    // cell list over the internal order, cell size = horizon
    double cs = c->P.delta;
    double *const mn = c->mn, *const mx = c->mx;
    for (;;) {
        double ncell = 1;
        for (int d = 0; d < 3; d++) ncell *= std::floor((mx[d] - mn[d]) / cs) + 1.0;
        if (ncell <= 8.0 * (double)n + 4096.0) break;
        cs *= 2.0;  // a coarser grid still finds every neighbour within the horizon
    }
    int64_t g[3];
    for (int d = 0; d < 3; d++) g[d] = (int64_t)std::floor((mx[d] - mn[d]) / cs) + 1;
    const int64_t ncell = g[0] * g[1] * g[2];
    // crack membership masks
    std::vector<uint16_t> cmask;
    uint32_t filt_bits = 0;
    if (!c->cracks.empty()) {
        cmask.assign(n, 0);
        for (size_t k = 0; k < c->cracks.size(); k++) {
            for (int32_t i : c->cracks[k].a) cmask[i] |= (uint16_t)(1u << (2 * k));
            for (int32_t i : c->cracks[k].b) cmask[i] |= (uint16_t)(1u << (2 * k + 1));
            if (c->cracks[k].filter) filt_bits |= 1u << (2 * k);
        }
    }
    // device buffers
    PDX_TRY(pdx_alloc(c, &c->rec[0], n));
    PDX_TRY(pdx_alloc(c, &c->rec[1], n));
    PDX_TRY(pdx_alloc(c, &c->Xr, n));
    PDX_TRY(pdx_alloc(c, &c->d_perm, n));
    PDX_TRY(pdx_alloc(c, &c->d_iperm, n));
    PDX_TRY(pdx_alloc(c, &c->stage, 9 * n));
    for (double **p : {&c->u, &c->vh, &c->v, &c->a, &c->bint, &c->bext})
        PDX_TRY(pdx_alloc(c, p, 3 * n));
    PDX_TRY(pdx_alloc(c, &c->damage, n));
    PDX_TRY(pdx_alloc(c, &c->nact, n));
    PDX_TRY(pdx_alloc(c, &c->killed, n));
    PDX_TRY(pdx_alloc(c, &c->bcslot, n));
    PDX_TRY(pdx_alloc(c, &c->d_fp, n));
    setup_scratch S;
    double *dX, *dV;
    uint8_t *dfp;
    uint16_t *dcm_in = nullptr, *d_cmask = nullptr;
    int32_t *d_pcell, *d_cell_pts, *d_num;
    int64_t *d_cell_start;
    PDX_TRY(S.get(c, &dX, 3 * n));
    PDX_TRY(S.get(c, &dV, n));
    PDX_TRY(S.get(c, &dfp, n));
    PDX_TRY(S.get(c, &d_pcell, 3 * n));
    PDX_TRY(S.get(c, &d_cell_pts, n));
    PDX_TRY(S.get(c, &d_num, ncell));
    PDX_TRY(S.get(c, &d_cell_start, ncell + 1));
    if (!cmask.empty()) {
        PDX_TRY(S.get(c, &dcm_in, n));
        PDX_TRY(S.get(c, &d_cmask, n));
        PDX_HIP(c, hipMemcpyAsync(dcm_in, cmask.data(), sizeof(uint16_t) * n, hipMemcpyHostToDevice, c->stream));
    }
    PDX_HIP(c, hipMemcpyAsync(dX, c->X.data(), sizeof(double) * 3 * n, hipMemcpyHostToDevice, c->stream));
    PDX_HIP(c, hipMemcpyAsync(dV, c->vol.data(), sizeof(double) * n, hipMemcpyHostToDevice, c->stream));
    PDX_HIP(c, hipMemcpyAsync(dfp, c->fail_permit.data(), n, hipMemcpyHostToDevice, c->stream));
    PDX_HIP(c, hipMemsetAsync(c->d_flags, 0, 8 * sizeof(unsigned long long), c->stream));
    PDX_HIP(c, hipMemsetAsync(d_num, 0, sizeof(int32_t) * ncell, c->stream));
    PDX_TRY(morton_order(c, S, dX, mn, mx));
    hipLaunchKernelGGL(k_gather_points, grid256(n), dim3(256), 0, c->stream, n, c->d_perm, dX, dV, dfp, dcm_in, c->Xr,
                       c->rec[0], c->rec[1], c->d_fp, d_cmask);
    const double3 mn3 = make_double3(mn[0], mn[1], mn[2]);
    hipLaunchKernelGGL(k_cells, grid256(n), dim3(256), 0, c->stream, n, c->Xr, mn3, cs, g[0], g[1], g[2], d_pcell, d_num);
    PDX_TRY(scan_i32(c, S, ncell, d_num, d_cell_start));
    hipLaunchKernelGGL(k_cell_points, grid256(n), dim3(256), 0, c->stream, n, d_pcell, g[0], g[1], d_cell_start, d_num,
                       d_cell_pts);
    PDX_HIP(c, hipGetLastError());
    // Each (Xr) record keeps the volume in .w for the bond passes; the reference record's
    // .w holds the volume too (only .xyz are read as the reference position).

    search_args s{};
    s.n = n;
    s.Xr = c->Xr;
    s.pcell = d_pcell;
    s.cell_start = d_cell_start;
    s.cell_pts = d_cell_pts;
    s.gx = g[0];
    s.gy = g[1];
    s.gz = g[2];
    s.r2 = c->P.delta * c->P.delta;
    s.perm = c->d_perm;
    s.cmask = d_cmask;
    s.filt_bits = filt_bits;
    s.fp = c->d_fp;
    PDX_TRY(pdx_alloc(c, &c->cnt, n));
    s.counts = c->cnt;
    s.flags = c->d_flags;
    hipLaunchKernelGGL(k_count_bonds, dim3((unsigned)pdx_wave_grid(n)), dim3(PDX_BLOCK), 0, c->stream, s);
    hipLaunchKernelGGL(k_count_totals, dim3((unsigned)std::min<int64_t>((n + 1023) / 1024, 256)), dim3(256), 0, c->stream, n,
                       c->cnt, c->d_flags + 4);
    PDX_HIP(c, hipGetLastError());
    unsigned long long hflags[8];
    PDX_HIP(c, hipMemcpyAsync(hflags, c->d_flags, sizeof hflags, hipMemcpyDeviceToHost, c->stream));
    PDX_HIP(c, hipStreamSynchronize(c->stream));
    if (hflags[1])
        return pdx_fail(c, PDX_ERR_DUPLICATE_POINT,
                        "point duplicate found! Point #%llu has a duplicate #%llu which will lead to NaNs",
                        hflags[2] + 1, hflags[3] + 1);
    const int64_t nb = (int64_t)hflags[4];
    if (hflags[5] > PDX_FILL_CAP)
        return pdx_fail(c, PDX_ERR_UNSUPPORTED, "a point has %d bonds (> %d)", (int)hflags[5], PDX_FILL_CAP);
    c->nb = nb;
    choose_blocks(c, !getenv("PDX_NO_LDS"));
    PDX_TRY(fill_rows(c, s));
    // the LDS-staged layout; tables it cannot address go to the global-gather layout
    if (c->ls > 0) {
        bool ok = false;
        PDX_TRY(build_halos(c, &ok));
        if (!ok) {
            choose_blocks(c, false);
            PDX_TRY(fill_rows(c, s));
        }
    }
    hipLaunchKernelGGL(k_init_point_state, dim3((unsigned)((n + 255) / 256)), dim3(256), 0,
                       c->stream, n, c->rows(), c->cnt, c->bw, c->nact, c->damage);
    PDX_HIP(c, hipGetLastError());
    // zero dynamic state
    for (double *p : {c->u, c->vh, c->v, c->a, c->bint, c->bext})
        PDX_HIP(c, hipMemsetAsync(p, 0, sizeof(double) * 3 * n, c->stream));
    PDX_HIP(c, hipMemsetAsync(c->killed, 0, n, c->stream));
    PDX_HIP(c, hipMemsetAsync(c->bcslot, 0xff, sizeof(int32_t) * n, c->stream));
    PDX_HIP(c, hipStreamSynchronize(c->stream));
    c->bext_nonzero = false;
    c->cur = 0;
    c->n_src = 0;
    c->n_bcpts = 0;
    // material state between the passes
    // OSB: the per-point pair of pass 1, then (LDS layout, one set) the own force part
    if (c->kind == PDX_OSB) PDX_TRY(pdx_alloc(c, &c->pstate, 5 * n));
    if (c->kind == PDX_CPD) {
        // Q per point; with ZEMWan also the stabilisation stiffness C_1 (15 numbers per point).
        // The LDS passes keep six more per point behind those: the own bond terms and
        // a = Q X + beta x (ZEMWan: Q X + C_1 x)
        PDX_TRY(pdx_alloc(c, &c->pstate, (c->P.zem == PDX_ZEM_WAN ? 21 : 15) * n));
        PDX_TRY(pdx_alloc(c, &c->defgrad, 9 * n));
        PDX_TRY(pdx_alloc(c, &c->cauchy, 9 * n));
        PDX_HIP(c, hipMemsetAsync(c->defgrad, 0, sizeof(double) * 9 * n, c->stream));
        PDX_HIP(c, hipMemsetAsync(c->cauchy, 0, sizeof(double) * 9 * n, c->stream));
        PDX_HIP(c, hipStreamSynchronize(c->stream));
    }
    // FP32 lengths for the global-gather mixed BB step (the LDS-staged steps take L = |D|)
    if (c->precision == PDX_MIXED && !c->lds_mode) {
        const int64_t nba = c->nb_alloc;
        PDX_TRY(pdx_alloc(c, &c->Lf, nba));
        hipLaunchKernelGGL(k_L_to_float, slot_grid(nba), dim3(256), 0, c->stream, nba, c->L, c->Lf);
        PDX_HIP(c, hipGetLastError());
    }
    PDX_TRY(upload_psets(c));
    if (c->kind == PDX_CPD && c->P.zem == PDX_ZEM_WAN && !c->lds_mode)
        return pdx_fail(c, PDX_ERR_UNSUPPORTED,
                        "ZEMWan needs the LDS-staged bond layout (a neighbour table did not fit)");
    if (c->multi() && !c->lds_mode)
        return pdx_fail(c, PDX_ERR_UNSUPPORTED,
                        "several parameter sets need the LDS-staged bond layout (a neighbour table did not fit)");
    if (c->corr && !c->lds_mode)
        return pdx_fail(c, PDX_ERR_UNSUPPORTED,
                        "the surface correction needs the LDS-staged bond layout (BB or OSB, neighbour tables that fit)");
    PDX_TRY(pdx_build_correction(c));
    c->bonds_built = true;
    if (n_bonds_out) *n_bonds_out = nb;
    return PDX_OK;
}

pdx_status pdx_caller_bond_slots(pdx_ctx *c, std::vector<int64_t> &slots)
{
    const int64_t n = c->n, nba = c->nb_alloc;
    const int64_t n_slices = c->n_slices();
    std::vector<int64_t> sp(n_slices + 1);
    std::vector<int32_t> cn(n);
    std::vector<uint32_t> w(nba);
    PDX_HIP(c, hipStreamSynchronize(c->stream));
    PDX_HIP(c, hipMemcpy(sp.data(), c->slice_ptr, sizeof(int64_t) * (n_slices + 1), hipMemcpyDeviceToHost));
    PDX_HIP(c, hipMemcpy(cn.data(), c->cnt, sizeof(int32_t) * n, hipMemcpyDeviceToHost));
    const pdx_rows hr{sp.data(), c->ls};
    PDX_HIP(c, hipMemcpy(w.data(), c->bw, sizeof(uint32_t) * nba, hipMemcpyDeviceToHost));
    slots.clear();
    std::vector<std::pair<int32_t, int64_t>> row;
    for (int64_t i = 0; i < n; i++) {
        const int64_t m = c->iperm[i];
        const int64_t b0 = hr.row(m);
        row.clear();
        for (int t = 0; t < cn[m]; t++) {
            const int64_t b = hr.at(b0, t);
            row.push_back({c->perm[w[b] & PDX_BW_NBR], b});
        }
        std::sort(row.begin(), row.end());
        for (auto &e : row) slots.push_back(e.second);
    }
    return PDX_OK;
}

extern "C" pdx_status pdx_get_bonds(pdx_ctx *c, int64_t *row_ptr, int32_t *nbr, double *L,
                                    uint8_t *fp, uint8_t *active)
{
    if (!c) return PDX_ERR_ARG;
    if (!c->bonds_built) return pdx_fail(c, PDX_ERR_STATE, "pdx_build_bonds first");
    const int64_t n = c->n, nba = c->nb_alloc;
    const int64_t n_slices = c->n_slices();
    std::vector<int64_t> sp(n_slices + 1);
    std::vector<int32_t> cn(n);
    std::vector<uint32_t> w(nba);
    std::vector<double> L_dev(L && c->L ? nba : 0);
    PDX_HIP(c, hipStreamSynchronize(c->stream));
    PDX_HIP(c, hipMemcpy(sp.data(), c->slice_ptr, sizeof(int64_t) * (n_slices + 1),
                         hipMemcpyDeviceToHost));
    PDX_HIP(c, hipMemcpy(cn.data(), c->cnt, sizeof(int32_t) * n, hipMemcpyDeviceToHost));
    const pdx_rows hr{sp.data(), c->ls};
    PDX_HIP(c, hipMemcpy(w.data(), c->bw, sizeof(uint32_t) * nba, hipMemcpyDeviceToHost));
    if (L && c->L) PDX_HIP(c, hipMemcpy(L_dev.data(), c->L, sizeof(double) * nba, hipMemcpyDeviceToHost));
    if (c->pk) {  // the packed words keep the bond state
        std::vector<unsigned long long> pk(nba);
        PDX_HIP(c, hipMemcpy(pk.data(), c->pk, sizeof(unsigned long long) * nba, hipMemcpyDeviceToHost));
        for (int64_t b = 0; b < nba; b++)
            w[b] = (w[b] & ~PDX_BW_ACT) | ((pk[b] & c->pk_mask) != c->pk_mask ? PDX_BW_ACT : 0u);
    } else if (c->lds_mode) {
        // the LDS-staged step keeps the bond state in the 16-bit words
        std::vector<uint16_t> w16(nba);
        PDX_HIP(c, hipMemcpy(w16.data(), c->bw16, sizeof(uint16_t) * nba, hipMemcpyDeviceToHost));
        for (int64_t b = 0; b < nba; b++)
            w[b] = (w[b] & ~PDX_BW_ACT) | ((w16[b] & PDX_W16_ACT) ? PDX_BW_ACT : 0u);
    }
    std::vector<uint8_t> killed(n, 0);
    if (c->kind == PDX_CPD)
        PDX_HIP(c, hipMemcpy(killed.data(), c->killed, n, hipMemcpyDeviceToHost));
    // caller order
    std::vector<int64_t> out_rp(n + 1, 0);
    for (int64_t i = 0; i < n; i++) {
        int64_t m = c->iperm[i];
        out_rp[i + 1] = out_rp[i] + cn[m];
    }
    if (row_ptr) std::memcpy(row_ptr, out_rp.data(), sizeof(int64_t) * (n + 1));
    // device rows are in Morton order of the neighbours; the caller's rows list neighbours
    // by ascending caller index (the reference's bond order within a grid cell)
    std::vector<std::pair<int32_t, int64_t>> row;
    for (int64_t i = 0; i < n; i++) {
        int64_t m = c->iperm[i];
        int64_t o = out_rp[i];
        row.clear();
        const int64_t b0 = hr.row(m);
        for (int t = 0; t < cn[m]; t++) {
            const int64_t b = hr.at(b0, t);
            row.push_back({c->perm[w[b] & PDX_BW_NBR], b});
        }
        std::sort(row.begin(), row.end());
        for (auto &e : row) {
            const int64_t b = e.second;
            if (nbr) nbr[o] = e.first;
            if (L) {
                if (c->L) {
                    L[o] = L_dev[b];
                } else {  // as the search formed it
                    const double *xi = &c->X[3 * i], *xj = &c->X[3 * (int64_t)e.first];
                    const double p0 = xi[0] - xj[0], p1 = xi[1] - xj[1], p2 = xi[2] - xj[2];
                    L[o] = std::sqrt((p0 * p0 + p1 * p1) + p2 * p2);
                }
            }
            if (fp) fp[o] = (w[b] & PDX_BW_FP) ? 1 : 0;
            if (active) active[o] = ((w[b] & PDX_BW_ACT) && !killed[m]) ? 1 : 0;
            o++;
        }
    }
    return PDX_OK;
}

// ----------------------------------------------------------------------------------------
// fields
// ----------------------------------------------------------------------------------------
pdx_status pdx_field_ptr(pdx_ctx *c, int field, double **p, int *comps, int *stride)
{
    *p = nullptr;
    *comps = 3;
    *stride = 3;
    switch (field) {
    case PDX_FIELD_POSITION: *p = (double *)c->rec[c->cur]; *stride = 4; break;
    case PDX_FIELD_DISPLACEMENT: *p = c->u; break;
    case PDX_FIELD_VELOCITY: *p = c->v; break;
    case PDX_FIELD_VELOCITY_HALF: *p = c->vh; break;
    case PDX_FIELD_ACCELERATION: *p = c->a; break;
    case PDX_FIELD_B_INT: *p = c->bint; break;
    case PDX_FIELD_B_EXT: *p = c->bext; break;
    case PDX_FIELD_DAMAGE: *p = c->damage; *comps = 1; *stride = 1; break;
    case PDX_FIELD_DEFGRAD: *p = c->defgrad; *comps = 9; *stride = 9; break;
    case PDX_FIELD_CAUCHY_STRESS: *p = c->cauchy; *comps = 9; *stride = 9; break;
    case PDX_FIELD_REF_POSITION: *p = (double *)c->Xr; *stride = 4; break;
    case PDX_FIELD_VOLUME: *p = ((double *)c->Xr) + 3; *comps = 1; *stride = 4; break;
    case PDX_FIELD_VELOCITY_HALF_OLD: *p = c->dr_vh_old; break;
    case PDX_FIELD_B_INT_OLD: *p = c->dr_bint_old; break;
    case PDX_FIELD_DENSITY_MATRIX: *p = c->dr_density; *comps = 1; *stride = 1; break;
    default: return pdx_fail(c, PDX_ERR_ARG, "unknown field %d", field);
    }
    if (!*p) return pdx_fail(c, PDX_ERR_ARG, "field %d is not held by this material", field);
    return PDX_OK;
}

__global__ void k_int_to_double(int64_t n, const int32_t *src, double *dst)
{
    int64_t k = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (k < n) dst[k] = (double)src[k];
}

__global__ void k_copy_xyz(int64_t n, const double4 *src, double4 *dst)
{
    int64_t k = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (k < n) dst[k] = src[k];
}

pdx_status pdx_field_comps(pdx_ctx *c, int field, int *comps)
{
    if (field == PDX_FIELD_N_ACTIVE_BONDS) {
        *comps = 1;
        return PDX_OK;
    }
    double *p;
    int stride;
    PDX_TRY(pdx_field_ptr(c, field, &p, comps, &stride));
    return PDX_OK;
}

pdx_status pdx_gather_field(pdx_ctx *c, int field, double *dst)
{
    double *p;
    int comps = 1, stride = 1;
    if (field == PDX_FIELD_N_ACTIVE_BONDS) {
        double *tmp = c->stage + 4 * c->n;  // second half of the staging buffer
        hipLaunchKernelGGL(k_int_to_double, dim3((c->n + 255) / 256), dim3(256), 0, c->stream,
                           c->n, c->nact, tmp);
        PDX_HIP(c, hipGetLastError());
        return pdx_gather_range(c, tmp, 1, 1, 0, c->n, dst);
    }
    PDX_TRY(pdx_field_ptr(c, field, &p, &comps, &stride));
    return pdx_gather_range(c, p, comps, stride, 0, c->n * comps, dst);
}

extern "C" pdx_status pdx_get_field(pdx_ctx *c, int32_t field, double *host)
{
    if (!c || !host) return PDX_ERR_ARG;
    if (!c->bonds_built) return pdx_fail(c, PDX_ERR_STATE, "pdx_build_bonds first");
    PDX_HIP(c, hipSetDevice(c->device));
    if (field == PDX_FIELD_N_ACTIVE_BONDS) {
        double *tmp = c->stage + 4 * c->n;  // second half of the staging buffer
        hipLaunchKernelGGL(k_int_to_double, dim3((c->n + 255) / 256), dim3(256), 0, c->stream,
                           c->n, c->nact, tmp);
        PDX_HIP(c, hipGetLastError());
        return pdx_download_vec(c, tmp, host, 1, 1);
    }
    double *p;
    int comps, stride;
    PDX_TRY(pdx_field_ptr(c, field, &p, &comps, &stride));
    if (field == PDX_FIELD_VOLUME) {
        // .w of the reference record
        return pdx_download_vec(c, p, host, 1, 4);
    }
    return pdx_download_vec(c, p, host, comps, stride);
}

extern "C" pdx_status pdx_set_field(pdx_ctx *c, int32_t field, const double *host)
{
    if (!c || !host) return PDX_ERR_ARG;
    if (!c->bonds_built) return pdx_fail(c, PDX_ERR_STATE, "pdx_build_bonds first");
    if (field == PDX_FIELD_REF_POSITION || field == PDX_FIELD_VOLUME ||
        field == PDX_FIELD_N_ACTIVE_BONDS || field == PDX_FIELD_DEFGRAD ||
        field == PDX_FIELD_CAUCHY_STRESS || field == PDX_FIELD_DENSITY_MATRIX)
        return pdx_fail(c, PDX_ERR_ARG, "field %d is read only", field);
    PDX_HIP(c, hipSetDevice(c->device));
    double *p;
    int comps, stride;
    PDX_TRY(pdx_field_ptr(c, field, &p, &comps, &stride));
    PDX_TRY(pdx_upload_strided(c, host, p, comps, stride));
    if (field == PDX_FIELD_B_EXT) {
        c->bext_nonzero = false;
        for (int64_t k = 0; k < 3 * c->n; k++)
            if (host[k] != 0.0) c->bext_nonzero = true;
    }
    return PDX_OK;
}

// ----------------------------------------------------------------------------------------
// stable time step: calc_timestep_point (bond_system.jl:269-277).  The device rows are in
// Morton order of the neighbours; the terms are ranked by the neighbour's caller index in
// LDS and summed in that order by one lane, so that the value equals the reference's bit
// for bit.
// ----------------------------------------------------------------------------------------
__global__ __launch_bounds__(PDX_BLOCK) void k_timestep(int64_t n, pdx_rows rows,
                                                         const int32_t *cnts,
                                                         const uint32_t *bw, const double *L,
                                                         const double4 *Xr, const int32_t *perm,
                                                         double bc, double rho,
                                                         const pdx_pset *psets, const uint8_t *pid,
                                                         double *dt)
{
    __shared__ double term[PDX_WAVES_PER_BLOCK][PDX_FILL_CAP];
    __shared__ int32_t key[PDX_WAVES_PER_BLOCK][PDX_FILL_CAP];
    const int64_t i = pdx_wave_point();
    if (i >= n) return;
    const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
    const int64_t b0 = rows.row(i);
    const int cnt = cnts[i];  // <= PDX_FILL_CAP (checked when built)
    const double4 Xi = Xr[i];
    if (psets) {  // the point's own parameter set (get_params(chunk, point_id))
        bc = psets[pid[i]].bc;
        rho = psets[pid[i]].rho;
    }
    for (int k = lane; k < cnt; k += 64) {
        const uint32_t j = bw[rows.at(b0, k)] & PDX_BW_NBR;
        key[w][k] = perm[j];
    }
    __builtin_amdgcn_fence(__ATOMIC_SEQ_CST, "wavefront");
    __builtin_amdgcn_wave_barrier();
    for (int k = lane; k < cnt; k += 64) {
        const int64_t b = rows.at(b0, k);
        const uint32_t j = bw[b] & PDX_BW_NBR;
        const int32_t kk = key[w][k];
        int rank = 0;
        for (int m = 0; m < cnt; m++) rank += (key[w][m] < kk) ? 1 : 0;
        const double4 Xj = Xr[j];
        term[w][rank] = Xj.w * bc / pdx_ref_len(L, b, Xi, Xj);
    }
    __builtin_amdgcn_fence(__ATOMIC_SEQ_CST, "wavefront");
    __builtin_amdgcn_wave_barrier();
    if (lane == 0) {
        double dtsum = 0.0;
        for (int k = 0; k < cnt; k++) dtsum += term[w][k];
        dt[i] = sqrt(2.0 * rho / dtsum);
    }
}

// minimum over each workgroup's share of v (NaN entries are passed over, as std::min does)
__global__ __launch_bounds__(256) void k_min(int64_t n, const double *v, double *out)
{
    __shared__ double sh[4];
    double m = INFINITY;
    for (int64_t k = (int64_t)blockIdx.x * 256 + threadIdx.x; k < n; k += (int64_t)gridDim.x * 256)
        m = v[k] < m ? v[k] : m;
    for (int o = 32; o > 0; o >>= 1) m = fmin(m, __shfl_xor(m, o));
    if ((threadIdx.x & 63) == 0) sh[threadIdx.x >> 6] = m;
    __syncthreads();
    if (threadIdx.x == 0) out[blockIdx.x] = fmin(fmin(sh[0], sh[1]), fmin(sh[2], sh[3]));
}

extern "C" pdx_status pdx_stable_timestep(pdx_ctx *c, double safety, double *dt_out)
{
    if (!c || !dt_out) return PDX_ERR_ARG;
    if (!c->bonds_built) return pdx_fail(c, PDX_ERR_STATE, "pdx_build_bonds first");
    if (!(safety > 0 && safety < 1))
        return pdx_fail(c, PDX_ERR_ARG, "`safety_factor` of VelocityVerlet has invalid value!");
    PDX_HIP(c, hipSetDevice(c->device));
    double *tmp = c->stage;
    hipLaunchKernelGGL(k_timestep, dim3((unsigned)pdx_wave_grid(c->n)), dim3(PDX_BLOCK), 0,
                       c->stream, c->n, c->rows(), c->cnt, c->bw, c->L, c->Xr, c->d_perm, c->P.bc,
                       c->P.rho, c->multi() ? c->d_psets : nullptr, c->multi() ? c->d_pid : nullptr, tmp);
    PDX_HIP(c, hipGetLastError());
    const int nb = (int)std::min<int64_t>((c->n + 255) / 256, 256);
    hipLaunchKernelGGL(k_min, dim3(nb), dim3(256), 0, c->stream, c->n, tmp, tmp + c->n);
    PDX_HIP(c, hipGetLastError());
    double dt[256];
    PDX_HIP(c, hipMemcpyAsync(dt, tmp + c->n, sizeof(double) * nb, hipMemcpyDeviceToHost, c->stream));
    PDX_HIP(c, hipStreamSynchronize(c->stream));
    double mn = INFINITY;
    for (int k = 0; k < nb; k++) mn = std::min(mn, dt[k]);
    *dt_out = mn * safety;
    return PDX_OK;
}

// ----------------------------------------------------------------------------------------
// velocity boundary conditions
// ----------------------------------------------------------------------------------------
extern "C" pdx_status pdx_set_velocity_bcs(pdx_ctx *c, int64_t npts, const int32_t *points,
                                           const int32_t *src, int64_t n_src)
{
    if (!c) return PDX_ERR_ARG;
    if (!c->bonds_built) return pdx_fail(c, PDX_ERR_STATE, "pdx_build_bonds first");
    if (npts < 0 || n_src < 0 || (npts > 0 && (!points || !src)))
        return pdx_fail(c, PDX_ERR_ARG, "invalid boundary condition table");
    PDX_HIP(c, hipSetDevice(c->device));
    std::vector<int32_t> slot(c->n, -1);
    std::vector<int32_t> ssrc(3 * std::max<int64_t>(npts, 1), -1);
    for (int64_t k = 0; k < npts; k++) {
        int32_t i = points[k];
        if (i < 0 || i >= c->n) return pdx_fail(c, PDX_ERR_ARG, "BC point out of range");
        if (slot[c->iperm[i]] >= 0) return pdx_fail(c, PDX_ERR_ARG, "BC point listed twice");
        slot[c->iperm[i]] = (int32_t)k;
        for (int d = 0; d < 3; d++) {
            int32_t sidx = src[3 * k + d];
            if (sidx < -1 || sidx >= n_src) return pdx_fail(c, PDX_ERR_ARG, "BC source out of range");
            ssrc[3 * k + d] = sidx;
        }
    }
    if (c->slot_src) {
        (void)hipFree(c->slot_src);
        c->slot_src = nullptr;
    }
    PDX_TRY(pdx_alloc(c, &c->slot_src, ssrc.size()));
    PDX_HIP(c, hipMemcpy(c->bcslot, slot.data(), sizeof(int32_t) * c->n, hipMemcpyHostToDevice));
    PDX_HIP(c, hipMemcpy(c->slot_src, ssrc.data(), sizeof(int32_t) * ssrc.size(),
                         hipMemcpyHostToDevice));
    c->n_bcpts = npts;
    c->n_src = n_src;
    return PDX_OK;
}

// force-density conditions on b_ext (forcedensity_bc! with f(t) or f(p, t),
// boundary_conditions.jl:559-575): dof 3 points[k] + d takes value src[3k + d] of the per-step
// row (the same rows as the velocity conditions, whose length pdx_set_velocity_bcs set)
extern "C" pdx_status pdx_set_force_density_bcs(pdx_ctx *c, int64_t npts, const int32_t *points,
                                                const int32_t *src)
{
    if (!c) return PDX_ERR_ARG;
    if (!c->bonds_built) return pdx_fail(c, PDX_ERR_STATE, "pdx_build_bonds first");
    if (npts < 0 || (npts > 0 && (!points || !src)))
        return pdx_fail(c, PDX_ERR_ARG, "invalid boundary condition table");
    PDX_HIP(c, hipSetDevice(c->device));
    std::vector<int32_t> pts(std::max<int64_t>(npts, 1), 0), ssrc(3 * std::max<int64_t>(npts, 1), -1);
    std::vector<uint8_t> seen(c->n, 0);
    for (int64_t k = 0; k < npts; k++) {
        const int32_t i = points[k];
        if (i < 0 || i >= c->n) return pdx_fail(c, PDX_ERR_ARG, "BC point out of range");
        if (seen[i]) return pdx_fail(c, PDX_ERR_ARG, "BC point listed twice");
        seen[i] = 1;
        pts[k] = c->iperm[i];
        for (int d = 0; d < 3; d++) {
            const int32_t sidx = src[3 * k + d];
            if (sidx < -1 || sidx >= c->n_src) return pdx_fail(c, PDX_ERR_ARG, "BC source out of range");
            ssrc[3 * k + d] = sidx;
        }
    }
    if (c->fd_pts) (void)hipFree(c->fd_pts);
    if (c->fd_src) (void)hipFree(c->fd_src);
    c->fd_pts = nullptr;
    c->fd_src = nullptr;
    PDX_TRY(pdx_alloc(c, &c->fd_pts, pts.size()));
    PDX_TRY(pdx_alloc(c, &c->fd_src, ssrc.size()));
    PDX_HIP(c, hipMemcpy(c->fd_pts, pts.data(), sizeof(int32_t) * pts.size(), hipMemcpyHostToDevice));
    PDX_HIP(c, hipMemcpy(c->fd_src, ssrc.data(), sizeof(int32_t) * ssrc.size(), hipMemcpyHostToDevice));
    c->n_fdpts = npts;
    if (npts > 0) c->bext_nonzero = true;
    return PDX_OK;
}

// b_ext of the constrained dofs from one row of condition values
__global__ void k_fd_bcs(pdx_fd_bcs fd)
{
    const int64_t t = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (t < 3 * fd.n) pdx_fd_dof(fd, t);
}

pdx_fd_bcs pdx_fd_table(const pdx_ctx *c, const double *bcv_row)
{
    pdx_fd_bcs fd{};
    if (c->n_fdpts > 0 && bcv_row) fd = {c->n_fdpts, c->fd_pts, c->fd_src, bcv_row, c->bext};
    return fd;
}

pdx_status pdx_apply_fd_bcs(pdx_ctx *c, const double *bcv_row)
{
    const pdx_fd_bcs fd = pdx_fd_table(c, bcv_row);
    if (fd.n <= 0) return PDX_OK;
    hipLaunchKernelGGL(k_fd_bcs, dim3((unsigned)((3 * fd.n + 255) / 256)), dim3(256), 0, c->stream, fd);
    PDX_HIP(c, hipGetLastError());
    return PDX_OK;
}

// ----------------------------------------------------------------------------------------
// instrumentation
// ----------------------------------------------------------------------------------------
extern "C" pdx_status pdx_set_profiling(pdx_ctx *c, int32_t enable)
{
    if (!c) return PDX_ERR_ARG;
    PDX_TRY(pdx_timed_flush(c));
    c->prof = enable != 0;
    c->ktime.clear();
    return PDX_OK;
}

static pdx_status take_event(pdx_ctx *c, hipEvent_t *e)
{
    if (!c->evpool.empty()) {
        *e = c->evpool.back();
        c->evpool.pop_back();
        return PDX_OK;
    }
    PDX_HIP(c, hipEventCreate(e));
    return PDX_OK;
}

// Launch timing with HIP events on the context's stream.  Events are only recorded here;
// they are read (and the stream waited for) in pdx_timed_flush, so timing does not
// serialise back-to-back launches.
pdx_status pdx_timed_begin(pdx_ctx *c)
{
    if (!c->prof) return PDX_OK;
    PDX_TRY(take_event(c, &c->open_ev));
    PDX_HIP(c, hipEventRecord(c->open_ev, c->stream));
    return PDX_OK;
}

pdx_status pdx_timed_end(pdx_ctx *c, const char *name)
{
    if (!c->prof || !c->open_ev) return PDX_OK;
    hipEvent_t b;
    PDX_TRY(take_event(c, &b));
    PDX_HIP(c, hipEventRecord(b, c->stream));
    c->pending.push_back({name, c->open_ev, b});
    c->open_ev = nullptr;
    if (c->pending.size() >= 4096) PDX_TRY(pdx_timed_flush(c));
    return PDX_OK;
}

pdx_status pdx_timed_flush(pdx_ctx *c)
{
    if (c->pending.empty()) return PDX_OK;
    PDX_HIP(c, hipEventSynchronize(c->pending.back().b));
    for (auto &t : c->pending) {
        float ms = 0;
        PDX_HIP(c, hipEventElapsedTime(&ms, t.a, t.b));
        auto &e = c->ktime[t.name];
        e.first += ms;
        e.second += 1;
        c->evpool.push_back(t.a);
        c->evpool.push_back(t.b);
    }
    c->pending.clear();
    return PDX_OK;
}

extern "C" pdx_status pdx_kernel_time(pdx_ctx *c, const char *name, double *avg_ms, int64_t *count)
{
    if (!c || !name) return PDX_ERR_ARG;
    PDX_TRY(pdx_timed_flush(c));
    auto it = c->ktime.find(name);
    if (it == c->ktime.end()) {
        if (avg_ms) *avg_ms = 0;
        if (count) *count = 0;
        return PDX_OK;
    }
    if (avg_ms) *avg_ms = it->second.second ? it->second.first / it->second.second : 0.0;
    if (count) *count = it->second.second;
    return PDX_OK;
}

extern "C" pdx_status pdx_info(pdx_ctx *c, int64_t *np, int64_t *nb, int64_t *bytes)
{
    if (!c) return PDX_ERR_ARG;
    if (np) *np = c->n;
    if (nb) *nb = c->nb;
    if (bytes) *bytes = c->dev_bytes;
    return PDX_OK;
}

extern "C" pdx_status pdx_layout(pdx_ctx *c, int32_t *lds_mode, int64_t *bond_slots,
                                 int64_t *halo_entries, int32_t *halo_max)
{
    if (!c) return PDX_ERR_ARG;
    if (!c->bonds_built) return pdx_fail(c, PDX_ERR_STATE, "pdx_build_bonds first");
    if (lds_mode) *lds_mode = c->lds_mode ? 1 : 0;
    if (bond_slots) *bond_slots = c->nb_alloc;
    if (halo_entries) *halo_entries = c->lds_mode ? c->halo_total : 0;
    if (halo_max) *halo_max = c->lds_mode ? c->halo_max : 0;
    return PDX_OK;
}

extern "C" int32_t pdx_bond_bytes(const pdx_ctx *c)
{
    if (!c || !c->bonds_built) return 0;
    return c->pk ? 8 : c->lds_mode ? 10 : 12;
}

extern "C" int32_t pdx_slice_points(const pdx_ctx *c) { return c && c->bonds_built ? 64 >> c->ls : 0; }

pdx_status pdx_reset_flags(pdx_ctx *c)
{
    unsigned long long init[2] = {~0ULL, 0ULL};
    PDX_HIP(c, hipMemcpyAsync(c->d_flags, init, sizeof init, hipMemcpyHostToDevice, c->stream));
    return PDX_OK;
}

pdx_status pdx_check_flags(pdx_ctx *c, int64_t *nan_step)
{
    unsigned long long h[2];
    PDX_HIP(c, hipMemcpyAsync(h, c->d_flags, sizeof h, hipMemcpyDeviceToHost, c->stream));
    PDX_HIP(c, hipStreamSynchronize(c->stream));
    if (nan_step) *nan_step = (h[0] == ~0ULL) ? -1 : (int64_t)h[0];
    return PDX_OK;
}
