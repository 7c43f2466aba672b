// Export pipeline: the device side of export_results / export_reference_results
// (src/core/threads_body_data_handler.jl:197-212) and _export_results (src/auxiliary/io.jl:157-167).
//
// pdx_export_begin gathers the requested fields of the current state into a device
// snapshot in the caller's point order (one kernel per field on the compute stream, so the
// snapshot is consistent with the step that just ended), then queues the copy of that
// snapshot into pinned host memory on a second stream.  It returns at once: the steps the
// caller launches next overlap with the copy, and the host writes the files of one export
// while the device computes the next ones.  Two slots alternate, so one export can be
// written out while the next is copied.
#include <algorithm>
#include <atomic>
#include <cstring>
#include <mutex>
#include <thread>

#include "pdx_internal.h"

// ----------------------------------------------------------------------------------------
// A field into the caller's memory.  The runtime's copy into pageable memory runs at the speed of
// one thread that takes the page faults of a fresh array and copies out of a staging buffer.  Here
// the gather into the caller's order writes straight into a pinned ring, over the bus, a slot per
// launch, and the calling thread with up to seven helpers carries the values over in pieces; the
// helpers touch the pages of their next piece while it is still under way.  24 MB into a new array:
// 6.6 ms in one piece by the runtime; the bus alone 0.47 ms (by the gather as by the copy engine;
// in slots of 2 MB with an event each 0.51 against the engine's 0.60, in slots of 512 KB 0.68 against
// 1.1); out of pinned memory with 1 / 2 / 4 / 8 threads 6.0 / 3.8 / 2.2 / 1.4 ms.  A single piece is
// copied by the calling thread alone (8 KB: 12 us, 26 us by the runtime).
// ----------------------------------------------------------------------------------------
#define PIN_PIECE ((size_t)512 << 10)

// The rings (16 MB of pinned memory) belong to the process, since to allocate one takes 0.4 ms and its
// first use another 0.1 to 1 ms of page faults: a call borrows a ring and gives it back, two are
// kept for the next calls of any thread, and the last context to go frees them.  While none is
// there, a context goes through the runtime's copy until that has carried PDX_PIN_RENT bytes (a call
// counts for 128 KB more), which is about when it has cost as much as a ring: a first pass over
// displacement, velocity and damage of 9 k points takes 110 us by the runtime, 550 with a new ring and
// 75 with one in use; of 512 k points 2.34, 2.38 and 0.91 ms.
// The gather writes a ring with a kernel's stores and host threads read it behind an event, so the
// memory is coherent by its own flag (and the events release to the system), not by the runtime's
// default, which the environment can change (HIP_HOST_COHERENT).
static std::mutex pin_mutex;
static int pin_contexts = 0;
static double *pin_idle[2] = {};

static double *pin_borrow(pdx_ctx *c, size_t bytes)
{
    {
        std::lock_guard<std::mutex> lock(pin_mutex);
        for (double *&p : pin_idle)
            if (p) {
                double *const r = p;
                p = nullptr;
                return r;
            }
    }
    c->pin_rent += bytes + ((size_t)128 << 10);
    if (c->pin_rent < PDX_PIN_RENT) return nullptr;
    void *p = nullptr;
    if (hipHostMalloc(&p, PDX_PIN_SLOTS * PDX_PIN_CHUNK, hipHostMallocPortable | hipHostMallocCoherent) != hipSuccess) {
        (void)hipGetLastError();
        return nullptr;
    }
    return (double *)p;
}

static void pin_return(double *r)
{
    if (!r) return;
    {
        std::lock_guard<std::mutex> lock(pin_mutex);
        for (double *&p : pin_idle)
            if (!p) {
                p = r;
                return;
            }
    }
    (void)hipHostFree(r);
}

struct pin_ring {
    double *p;
    pin_ring(pdx_ctx *c, size_t bytes) : p(pin_borrow(c, bytes)) {}
    ~pin_ring() { pin_return(p); }
};

void pdx_pin_open()
{
    std::lock_guard<std::mutex> lock(pin_mutex);
    pin_contexts++;
}

void pdx_pin_close(pdx_ctx *c)
{
    for (hipEvent_t &e : c->pin_ev) {
        if (e) (void)hipEventDestroy(e);
        e = nullptr;
    }
    std::lock_guard<std::mutex> lock(pin_mutex);
    if (--pin_contexts > 0) return;
    for (double *&p : pin_idle) {
        if (p) (void)hipHostFree(p);
        p = nullptr;
    }
}

static bool pin_events(pdx_ctx *c, int slots)
{
    for (int k = 0; k < slots; k++)
        if (!c->pin_ev[k] &&
            hipEventCreateWithFlags(&c->pin_ev[k], hipEventDisableTiming | hipEventReleaseToSystem) != hipSuccess) {
            c->pin_ev[k] = nullptr;
            (void)hipGetLastError();
            return false;
        }
    return true;
}

pdx_status pdx_download_vec(pdx_ctx *c, const double *dev, double *host, int comps, int stride)
{
    constexpr int64_t SLOT = PDX_PIN_CHUNK / sizeof(double), PIECE = PIN_PIECE / sizeof(double), PER = SLOT / PIECE;
    const int64_t cnt = c->n * comps;
    const int64_t nch = (cnt + SLOT - 1) / SLOT, npc = (cnt + PIECE - 1) / PIECE;
    const int slots = (int)std::min<int64_t>(nch, PDX_PIN_SLOTS);
    const pin_ring ring(c, sizeof(double) * cnt);
    if (!ring.p || !pin_events(c, npc > 1 ? slots : 0)) {
        PDX_TRY(pdx_gather_range(c, dev, comps, stride, 0, cnt, c->stage));
        PDX_HIP(c, hipMemcpyAsync(host, c->stage, sizeof(double) * cnt, hipMemcpyDeviceToHost, c->stream));
        PDX_HIP(c, hipStreamSynchronize(c->stream));
        return PDX_OK;
    }
    double *const pin = ring.p;
    if (npc == 1) {
        PDX_TRY(pdx_gather_range(c, dev, comps, stride, 0, cnt, pin));
        PDX_HIP(c, hipStreamSynchronize(c->stream));
        memcpy(host, pin, sizeof(double) * cnt);
        return PDX_OK;
    }
    // Chunk k passes through slot k % slots in PER pieces.  `ready` pieces have arrived, `next` is the
    // first one that nobody has taken, left[s] counts the pieces carried out of slot s.
    std::atomic<int64_t> ready{0}, next{0};
    std::atomic<int64_t> left[PDX_PIN_SLOTS] = {};
    std::atomic<bool> stop{false};
    auto carry = [&](int64_t k) {
        const int64_t s = (k / PER) % slots;
        memcpy(host + k * PIECE, pin + s * SLOT + (k % PER) * PIECE, sizeof(double) * std::min(PIECE, cnt - k * PIECE));
        left[s].fetch_add(1, std::memory_order_release);
    };
    auto helper = [&]() {
        for (int64_t k; (k = next.fetch_add(1)) < npc;) {
            volatile double *const h = host + k * PIECE;
            for (int64_t o = 0; o < std::min(PIECE, cnt - k * PIECE); o += 512) h[o] = 0.0;
            while (ready.load(std::memory_order_acquire) <= k) {
                if (stop.load()) return;
                std::this_thread::yield();
            }
            carry(k);
        }
    };
    pdx_status st = PDX_OK;
    int64_t issued = 0, arrived = 0;
    // every chunk whose slot is free goes on the stream
    auto issue = [&]() -> pdx_status {
        for (; issued < nch; issued++) {
            const int64_t s = issued % slots;
            if (left[s].load(std::memory_order_acquire) < issued / slots * PER) break;
            PDX_TRY(pdx_gather_range(c, dev, comps, stride, issued * SLOT, std::min(cnt, (issued + 1) * SLOT), pin + s * SLOT));
            PDX_HIP(c, hipEventRecord(c->pin_ev[s], c->stream));
        }
        return PDX_OK;
    };
    auto arrive = [&]() -> pdx_status {
        PDX_HIP(c, hipEventSynchronize(c->pin_ev[arrived % slots]));
        arrived++;
        ready.store(std::min(npc, arrived * PER), std::memory_order_release);
        return PDX_OK;
    };
    st = issue();
    const int64_t want = std::min<int64_t>(std::min<int64_t>(7, npc - 1), (int64_t)std::thread::hardware_concurrency() - 1);
    std::thread th[7];
    int nth = 0;
    try {
        for (; nth < want; nth++) th[nth] = std::thread(helper);
    } catch (...) {
        // no more threads to be had: those there are, and this one, do the work
    }
    while (st == PDX_OK && (arrived < nch || next.load() < npc)) {
        st = issue();
        if (st == PDX_OK && arrived < issued) {
            st = arrive();
            if (arrived < issued && nth > 0) continue;  // the next one first: the helpers wait for it
        }
        int64_t k = next.load();  // a piece that has arrived and that nobody has taken
        if (k < ready.load() && next.compare_exchange_strong(k, k + 1)) carry(k);
        else std::this_thread::yield();
    }
    if (st != PDX_OK) stop.store(true);
    for (int k = 0; k < nth; k++) th[k].join();
    if (st != PDX_OK) (void)hipStreamSynchronize(c->stream);  // the ring goes back idle
    return st;
}

#define PDX_EXPORT_MAX_FIELDS 16

void pdx_export_free(pdx_ctx *c)
{
    if (c->xstream) (void)hipStreamSynchronize(c->xstream);
    for (int s = 0; s < 2; s++) {
        if (c->xdev[s]) (void)hipFree(c->xdev[s]);
        if (c->xhost[s]) (void)hipHostFree(c->xhost[s]);
        if (c->xev_snap[s]) (void)hipEventDestroy(c->xev_snap[s]);
        if (c->xev_done[s]) (void)hipEventDestroy(c->xev_done[s]);
        c->xdev[s] = c->xhost[s] = nullptr;
        c->xev_snap[s] = c->xev_done[s] = nullptr;
        c->xcap[s] = 0;
    }
    if (c->xstream) (void)hipStreamDestroy(c->xstream);
    c->xstream = nullptr;
    c->xbegun = c->xwaited = 0;
}

static pdx_status export_init(pdx_ctx *c)
{
    if (c->xstream) return PDX_OK;
    // default priority, like the compute stream
    PDX_HIP(c, hipStreamCreateWithFlags(&c->xstream, hipStreamNonBlocking));
    for (int s = 0; s < 2; s++) {
        PDX_HIP(c, hipEventCreateWithFlags(&c->xev_snap[s], hipEventDisableTiming));
        PDX_HIP(c, hipEventCreateWithFlags(&c->xev_done[s], hipEventDisableTiming));
    }
    return PDX_OK;
}

extern "C" pdx_status pdx_export_begin(pdx_ctx *c, int32_t n_fields, const int32_t *fields, int64_t tag)
{
    if (!c || n_fields < 0 || (n_fields > 0 && !fields)) return PDX_ERR_ARG;
    if (n_fields > PDX_EXPORT_MAX_FIELDS)
        return pdx_fail(c, PDX_ERR_ARG, "at most %d fields per export", PDX_EXPORT_MAX_FIELDS);
    if (!c->bonds_built) return pdx_fail(c, PDX_ERR_STATE, "pdx_build_bonds first");
    if (c->xbegun - c->xwaited >= 2)
        return pdx_fail(c, PDX_ERR_STATE, "two exports are pending: pdx_export_wait first");
    PDX_HIP(c, hipSetDevice(c->device));
    PDX_TRY(export_init(c));
    const int s = (int)(c->xbegun & 1);
    std::vector<int64_t> off(n_fields + 1, 0);
    for (int k = 0; k < n_fields; k++) {
        int comps;
        PDX_TRY(pdx_field_comps(c, fields[k], &comps));
        off[k + 1] = off[k] + c->n * comps;
    }
    const size_t need = (size_t)std::max<int64_t>(off[n_fields], 1);
    if (need > c->xcap[s]) {
        if (c->xdev[s]) (void)hipFree(c->xdev[s]);
        if (c->xhost[s]) (void)hipHostFree(c->xhost[s]);
        c->xdev[s] = c->xhost[s] = nullptr;
        c->xcap[s] = 0;
        PDX_TRY(pdx_alloc(c, &c->xdev[s], need));
        PDX_HIP(c, hipHostMalloc((void **)&c->xhost[s], sizeof(double) * need, hipHostMallocDefault));
        c->xcap[s] = need;
    }
    for (int k = 0; k < n_fields; k++) PDX_TRY(pdx_gather_field(c, fields[k], c->xdev[s] + off[k]));
    PDX_HIP(c, hipEventRecord(c->xev_snap[s], c->stream));
    PDX_HIP(c, hipStreamWaitEvent(c->xstream, c->xev_snap[s], 0));
    if (off[n_fields] > 0)
        PDX_HIP(c, hipMemcpyAsync(c->xhost[s], c->xdev[s], sizeof(double) * off[n_fields],
                                  hipMemcpyDeviceToHost, c->xstream));
    PDX_HIP(c, hipEventRecord(c->xev_done[s], c->xstream));
    c->xfields[s].assign(fields, fields + n_fields);
    c->xoff[s] = off;
    c->xtag[s] = tag;
    c->xbegun++;
    return PDX_OK;
}

extern "C" pdx_status pdx_export_wait(pdx_ctx *c, int64_t *tag, int32_t *slot, const double **field_data)
{
    if (!c) return PDX_ERR_ARG;
    if (c->xwaited >= c->xbegun) return pdx_fail(c, PDX_ERR_STATE, "no export pending");
    PDX_HIP(c, hipSetDevice(c->device));
    const int s = (int)(c->xwaited & 1);
    PDX_HIP(c, hipEventSynchronize(c->xev_done[s]));
    if (tag) *tag = c->xtag[s];
    if (slot) *slot = s;
    if (field_data)
        for (size_t k = 0; k < c->xfields[s].size(); k++) field_data[k] = c->xhost[s] + c->xoff[s][k];
    c->xwaited++;
    return PDX_OK;
}
