// C ABI of the MAGIC step on MI355X (declared in include/magic_hip.h).
//
// A context owns the device-resident state of one grid: q and its backup
// (the reference's copyq3 work array), the background planes the step reads,
// the bc3 z-boundary density ratios, and the source-pass scratch planes.
// Everything runs on one HIP stream of default priority; every entry point
// returns after its work is complete.
#include <atomic>
#include <condition_variable>
#include <mutex>
#include <thread>
#include <unistd.h>

#include "ctx.h"

// ------------------------------------------------------ host transfers ---
// q crosses between the caller's host memory (pageable: a Fortran array)
// and the device through two page-locked bounce chunks shared by every
// context (one transfer at a time): a chunk's DMA runs while host threads
// copy the neighbouring chunk between the caller's memory and the other
// bounce chunk.  Bound by the link (57 GB/s) where the array is large; in a
// small one the first chunk's way in and the last one's way out show, and
// the start of threads did: chunks are an eighth of the transfer, 1 to 32
// MB, and the threads stay while a context is open.  Against chunks of 32 MB
// and threads started for each, set_q and get_q of 5.4 MB 0.28 and 0.28 -> 0.23
// and 0.20 ms, of 11.5 MB 0.43 and 0.43 -> 0.38 and 0.36, of 101 MB 2.35 and 2.32
// -> 2.2 and 2.1, of 756 MB 14.6 -> 14.5.
namespace {
constexpr size_t BOUNCE = size_t(32) << 20;   // bytes per bounce chunk, at most
constexpr int COPY_THREADS = 8;               // the calling thread among them
std::mutex bounce_mu;
char *bounce_buf[2] = {nullptr, nullptr};
hipEvent_t bounce_ev[2] = {nullptr, nullptr};

int bounce_setup()
{
    for (int k = 0; k < 2; k++) {
        if (!bounce_buf[k] && hipHostMalloc((void **)&bounce_buf[k], BOUNCE, hipHostMallocDefault) != hipSuccess)
            return MAGIC_ENOMEM;
        if (!bounce_ev[k]) HIPCHECK(hipEventCreateWithFlags(&bounce_ev[k], hipEventDisableTiming));
    }
    return MAGIC_OK;
}
size_t bounce_chunk(size_t bytes)
{
    const size_t c = ((bytes + 7) / 8 + 4095) & ~size_t(4095);
    return std::min(BOUNCE, std::max(size_t(1) << 20, c));
}

// Threads that copy with the calling one.  A job is cut into slices that each
// takes from one counter, so that a thread that wakes late holds nobody up;
// the counter's word also holds the job's number and its slices, so that
// whoever is given a valid slice holds the job's descriptor.  Calls are made under
// bounce_mu.  The threads start with the first job and end with the last
// context (pool_open, pool_close).
class CopyPool {
public:
    const pid_t pid = getpid();
    void copy(char *dst, const char *src, size_t n)
    {
        if (n < (size_t(1) << 20)) {
            memcpy(dst, src, n);
            return;
        }
        while (nth < COPY_THREADS - 1) {
            try {
                th[nth] = std::thread([this] { work(); });
            } catch (...) {   // no thread to be had: the others do its part
                break;
            }
            nth++;
        }
        // two slices a thread, of 256 KB at least
        const size_t part = std::max(size_t(256) << 10, (n / (2 * COPY_THREADS) + 4095) & ~size_t(4095));
        const uint64_t slices = (n + part - 1) / part, id = (state.load() >> 40) + 1;
        job = {dst, src, n, part};
        done.store(0, std::memory_order_relaxed);
        {
            std::lock_guard<std::mutex> lock(mu);
            state.store(id << 40 | slices << 20, std::memory_order_release);
        }
        if (asleep.load() > 0) cv.notify_all();
        while (take()) {}
        while (done.load(std::memory_order_acquire) < slices) std::this_thread::yield();
    }
    void end()
    {
        {
            std::lock_guard<std::mutex> lock(mu);
            stop = true;
        }
        cv.notify_all();
        for (int t = 0; t < nth; t++) th[t].join();
        nth = 0;
        stop = false;
    }

private:
    struct Job {
        char *dst;
        const char *src;
        size_t n, part;
    };
    static uint64_t left(uint64_t s) { return (s >> 20 & 0xfffff) > (s & 0xfffff); }
    // one slice of the current job; false: none left
    bool take()
    {
        if (!left(state.load(std::memory_order_acquire))) return false;
        const uint64_t s = state.fetch_add(1, std::memory_order_acq_rel);
        if (!left(s)) return false;
        const size_t o = (size_t)(s & 0xfffff) * job.part;
        memcpy(job.dst + o, job.src + o, std::min(job.part, job.n - o));
        done.fetch_add(1, std::memory_order_release);
        return true;
    }
    void work()
    {
        for (;;) {
            while (take()) {}
            // the next chunk follows within a fraction of a millisecond
            for (int n = 0; n < 2000 && !left(state.load(std::memory_order_relaxed)); n++) std::this_thread::yield();
            if (left(state.load())) continue;
            std::unique_lock<std::mutex> lock(mu);
            asleep++;
            cv.wait(lock, [this] { return stop || left(state.load()); });
            asleep--;
            if (stop) return;
        }
    }
    std::thread th[COPY_THREADS - 1];
    int nth = 0;
    Job job = {};
    std::atomic<uint64_t> state{0}, done{0};   // state: job's number, slices (20 bits), next slice (20 bits)
    std::atomic<int> asleep{0};
    bool stop = false;
    std::mutex mu;
    std::condition_variable cv;
};
CopyPool *pool = nullptr;
int pool_users = 0;

void pool_open()
{
    std::lock_guard<std::mutex> lock(bounce_mu);
    if (pool_users++ == 0) pool = new CopyPool;
}
void pool_close()
{
    std::lock_guard<std::mutex> lock(bounce_mu);
    if (--pool_users > 0) return;
    if (pool->pid != getpid()) return;   // a forked child: the threads are its parent's
    pool->end();
    delete pool;
    pool = nullptr;
}
}  // namespace

// host -> device (dev on the context's stream; returns with the copies queued)
static int upload(magic_ctx *c, void *dev, const void *host, size_t bytes)
{
    std::lock_guard<std::mutex> lock(bounce_mu);
    TRY(bounce_setup());
    const size_t chunk = bounce_chunk(bytes);
    for (size_t off = 0, i = 0; off < bytes; off += chunk, i++) {
        const size_t n = std::min(chunk, bytes - off);
        const int k = (int)(i & 1);
        HIPCHECK(hipEventSynchronize(bounce_ev[k]));   // the copy that last read this chunk is done
        pool->copy(bounce_buf[k], (const char *)host + off, n);
        HIPCHECK(hipMemcpyAsync((char *)dev + off, bounce_buf[k], n, hipMemcpyHostToDevice, c->stream));
        HIPCHECK(hipEventRecord(bounce_ev[k], c->stream));
    }
    // the bounce chunks are read until these copies run: wait before unlocking
    for (auto e : bounce_ev) HIPCHECK(hipEventSynchronize(e));
    return MAGIC_OK;
}

// device -> host (after the work queued on the context's stream)
static int download(magic_ctx *c, void *host, const void *dev, size_t bytes)
{
    std::lock_guard<std::mutex> lock(bounce_mu);
    TRY(bounce_setup());
    const size_t chunk = bounce_chunk(bytes), nchunk = (bytes + chunk - 1) / chunk;
    for (size_t i = 0; i <= nchunk; i++) {
        if (i < nchunk) {
            const int k = (int)(i & 1);
            HIPCHECK(hipMemcpyAsync(bounce_buf[k], (const char *)dev + i * chunk, std::min(chunk, bytes - i * chunk),
                                    hipMemcpyDeviceToHost, c->stream));
            HIPCHECK(hipEventRecord(bounce_ev[k], c->stream));
        }
        if (i > 0) {   // the previous chunk, while this one's copy runs
            const int k = (int)((i - 1) & 1);
            HIPCHECK(hipEventSynchronize(bounce_ev[k]));
            pool->copy((char *)host + (i - 1) * chunk, bounce_buf[k], std::min(chunk, bytes - (i - 1) * chunk));
        }
    }
    return MAGIC_OK;
}

extern "C" const char *magic_strerror(int s)
{
    switch (s) {
    case MAGIC_OK: return "ok";
    case MAGIC_ERHO: return "rho <= 0 in a Riemann problem";
    case MAGIC_EA2: return "a**2 <= 0 in a Roe average";
    case MAGIC_EBC: return "boundary condition needs MPI or a user routine (mthbc 0 or 4)";
    case MAGIC_EUNSUPPORTED: return "method or option not supported";
    case MAGIC_EARG: return "invalid argument";
    case MAGIC_EHIP: return "HIP runtime error";
    case MAGIC_ENOMEM: return "device allocation failed";
    default: return "unknown status";
    }
}


extern "C" int magic_create(int mx, int my, int mz, int meqn, int mbc, int maux, double xlower,
                            double ylower, double zlower, double dx, double dy, double dz,
                            magic_ctx **out)
{
    return magic_create_form(mx, my, mz, meqn, mbc, maux, xlower, ylower, zlower, dx, dy, dz,
                             MAGIC_FORM_FP64, out);
}

extern "C" int magic_create_form(int mx, int my, int mz, int meqn, int mbc, int maux, double xlower,
                                 double ylower, double zlower, double dx, double dy, double dz, int form,
                                 magic_ctx **out)
{
    if (!out) return MAGIC_EARG;
    *out = nullptr;
    if (form != MAGIC_FORM_FP64 && form != MAGIC_FORM_FP32P) return MAGIC_EARG;
    if (form == MAGIC_FORM_FP32P && mbc > 8) return MAGIC_EUNSUPPORTED;
    if (mx < 1 || my < 1 || mz < 1 || mbc < 2 || meqn < 5 || meqn > 10 || maux < 19) return MAGIC_EARG;
    if (!sweep_supported(meqn - 5)) return MAGIC_EUNSUPPORTED;
    if (mz > mx) {
        // conduct.f:86-91 writes S = mz-mx elements past each layer; the
        // device replays those writes after the in-row fills, which is the
        // reference's order only while the rows they land in come before
        // the rows that write them.
        const long long S = mz - mx, NX = mx + 2 * mbc, NY = my + 2 * mbc;
        if (2 * ((S - 1) / NX) + 1 >= NY) return MAGIC_EUNSUPPORTED;
    }
    magic_ctx *c = new magic_ctx();
    pool_open();
    c->form = form;
    c->mx = mx; c->my = my; c->mz = mz; c->meqn = meqn; c->mbc = mbc; c->maux = maux;
    c->xlower = xlower; c->ylower = ylower; c->zlower = zlower; c->dx = dx; c->dy = dy; c->dz = dz;
    c->d.mx = mx; c->d.my = my; c->d.mz = mz; c->d.mbc = mbc;
    c->d.NX = mx + 2 * mbc; c->d.NY = my + 2 * mbc; c->d.NZ = mz + 2 * mbc;
    c->P = c->d.P = (long long)c->d.NX * c->d.NY * c->d.NZ;
    const size_t P = (size_t)c->P;
    const size_t NXY = (size_t)c->d.NX * c->d.NY;
    bool ok = hipStreamCreateWithFlags(&c->stream, hipStreamNonBlocking) == hipSuccess;
    ok = ok && hipMalloc(&c->stage, P * meqn * sizeof(double)) == hipSuccess;
    ok = ok && hipMalloc(&c->dscal, 8 * sizeof(unsigned long long)) == hipSuccess;
    ok = ok && hipHostMalloc(&c->hscal, HSCAL_WORDS * sizeof(unsigned long long), hipHostMallocDefault) == hipSuccess;
    if (ok && form == MAGIC_FORM_FP32P) {
        const size_t NZ = (size_t)c->d.NZ;
        ok = hipMalloc(&c->q32, P * meqn * sizeof(float)) == hipSuccess &&
             hipMalloc(&c->qold32, P * meqn * sizeof(float)) == hipSuccess &&
             hipMalloc(&c->u32, 3 * P * sizeof(float)) == hipSuccess &&
             hipMalloc(&c->qt32, P * sizeof(float)) == hipSuccess &&
             hipMalloc(&c->ut32, P * sizeof(float)) == hipSuccess &&
             hipMalloc(&c->col32, NC32 * NZ * sizeof(float)) == hipSuccess &&
             hipMalloc(&c->bg64, NB64 * NZ * sizeof(double)) == hipSuccess;
        ok = ok && hipMemsetAsync(c->q32, 0, P * meqn * sizeof(float), c->stream) == hipSuccess &&
             hipMemsetAsync(c->qold32, 0, P * meqn * sizeof(float), c->stream) == hipSuccess &&
             hipMemsetAsync(c->u32, 0, 3 * P * sizeof(float), c->stream) == hipSuccess &&
             hipMemsetAsync(c->qt32, 0, P * sizeof(float), c->stream) == hipSuccess &&
             hipMemsetAsync(c->ut32, 0, P * sizeof(float), c->stream) == hipSuccess &&
             hipMemsetAsync(c->col32, 0, NC32 * NZ * sizeof(float), c->stream) == hipSuccess &&
             hipMemsetAsync(c->bg64, 0, NB64 * NZ * sizeof(double), c->stream) == hipSuccess &&
             hipStreamSynchronize(c->stream) == hipSuccess;
        if (!ok) {
            magic_destroy(c);
            (void)hipGetLastError();   // reported here; not left for the next launch check
            return MAGIC_ENOMEM;
        }
        *out = c;
        return MAGIC_OK;
    }
    ok = ok && hipMalloc(&c->q, P * meqn * sizeof(double)) == hipSuccess;
    ok = ok && hipMalloc(&c->qold, P * meqn * sizeof(double)) == hipSuccess;
    ok = ok && hipMalloc(&c->aux, P * NAUXP * sizeof(double)) == hipSuccess;
    ok = ok && hipMalloc(&c->zratio, 2 * mbc * NXY * sizeof(double)) == hipSuccess;
    ok = ok && hipMalloc(&c->u, 3 * P * sizeof(double)) == hipSuccess;
    ok = ok && hipMalloc(&c->qt, P * sizeof(double)) == hipSuccess;
    ok = ok && hipMalloc(&c->ut, P * sizeof(double)) == hipSuccess;
    ok = ok && hipMalloc(&c->col64, (size_t)NAUXP * c->d.NZ * sizeof(double)) == hipSuccess;
    if (ok) {
        ok = hipMemsetAsync(c->q, 0, P * meqn * sizeof(double), c->stream) == hipSuccess &&
             hipMemsetAsync(c->qold, 0, P * meqn * sizeof(double), c->stream) == hipSuccess &&
             hipMemsetAsync(c->aux, 0, P * NAUXP * sizeof(double), c->stream) == hipSuccess &&
             hipMemsetAsync(c->zratio, 0, 2 * mbc * NXY * sizeof(double), c->stream) == hipSuccess &&
             hipMemsetAsync(c->u, 0, 3 * P * sizeof(double), c->stream) == hipSuccess &&
             hipMemsetAsync(c->qt, 0, P * sizeof(double), c->stream) == hipSuccess &&
             hipMemsetAsync(c->ut, 0, P * sizeof(double), c->stream) == hipSuccess &&
             hipStreamSynchronize(c->stream) == hipSuccess;
    }
    if (!ok) {
        magic_destroy(c);
        (void)hipGetLastError();   // reported here; not left for the next launch check
        return MAGIC_ENOMEM;
    }
    *out = c;
    return MAGIC_OK;
}

extern "C" int magic_destroy(magic_ctx *c)
{
    if (!c) return MAGIC_OK;
    if (c->cstream) hipStreamSynchronize(c->cstream);   // a snapshot's copy out of stage
    if (c->stream) hipStreamSynchronize(c->stream);
    drain_timing(c);
    for (auto e : c->pool) hipEventDestroy(e);
    hipFree(c->q); hipFree(c->qold); hipFree(c->aux); hipFree(c->zratio); hipFree(c->stage);
    hipFree(c->u); hipFree(c->qt); hipFree(c->ut); hipFree(c->dscal);
    hipFree(c->q32); hipFree(c->qold32); hipFree(c->u32); hipFree(c->qt32); hipFree(c->ut32);
    hipFree(c->col32); hipFree(c->bg64); hipFree(c->col64); hipFree(c->sums_d);
    hipFree(c->largs); hipFree(c->lrun); hipFree(c->lone); hipFree(c->items);
    if (!c->parts_stage) hipFree(c->parts);
    if (c->hscal) hipHostFree(c->hscal);
    if (c->snap_conv) hipEventDestroy(c->snap_conv);
    if (c->snap_done) hipEventDestroy(c->snap_done);
    if (c->cstream) hipStreamDestroy(c->cstream);
    if (c->stream && c->own_stream) hipStreamDestroy(c->stream);
    pool_close();
    delete c;
    return MAGIC_OK;
}

extern "C" int magic_set_params(magic_ctx *c, const magic_params *p)
{
    if (!c || !p) return MAGIC_EARG;
    c->prm = *p;
    c->have_params = true;
    return MAGIC_OK;
}

// aux slots (1-based) of the ten background planes, in AX_ order
static const int AUX_SLOT[NAUXP] = {1, 2, 3, 4, 5, 11, 12, 17, 18, 19};

// FP32 form: the background must be one column at rest.  Keeps FP64
// columns of rho_bar, E_bar, gamma, R, aux17 and the background's own z jump
// of the well-balanced f-wave (p_bar(k) - p_bar(k-1) - .5 (rho_bar(k) +
// rho_bar(k-1)) aux17(k), p_bar = (gamma-1) E_bar as rpn3euX.f:166-169
// evaluates it for a state at rest; zero to FP64 rounding), which the
// form's FP64 Riemann solve and conversions read; float columns of nu and
// kappa for the diffusion passes; and the bc3 z factors per layer.  get(slot
// index, cell) returns the background value of a padded cell.
template <class F>
static int set_aux32(magic_ctx *c, F get, bool check_columns)
{
    const int NX = c->d.NX, NY = c->d.NY, NZ = c->d.NZ, mbc = c->mbc, mz = c->mz;
    std::vector<double> col((size_t)NAUXP * NZ);
    for (int kk = 0; kk < NZ; kk++) {
        const long long c0 = (long long)kk * NY * NX;
        for (int s = 0; s < NAUXP; s++) {
            const double v0 = get(s, c0);
            if ((s == AX_MX || s == AX_MY || s == AX_MZ) && v0 != 0.0) {
                fprintf(stderr, "magic_hip: FP32 form needs a background at rest (aux slot %d = %g)\n",
                        AUX_SLOT[s], v0);
                return MAGIC_EUNSUPPORTED;
            }
            if (check_columns)
                for (long long e = 0; e < (long long)NY * NX; e++)
                    if (get(s, c0 + e) != v0) {
                        fprintf(stderr, "magic_hip: FP32 form needs a background column (aux slot %d varies "
                                        "in layer %d)\n", AUX_SLOT[s], kk + 1 - mbc);
                        return MAGIC_EUNSUPPORTED;
                    }
            col[(size_t)s * NZ + kk] = v0;
        }
    }
    auto cv = [&](int s, int kk) { return col[(size_t)s * NZ + kk]; };
    std::vector<float> h((size_t)NC32 * NZ, 0.0f);
    std::vector<double> b64((size_t)NB64 * NZ, 0.0);
    for (int kk = 0; kk < NZ; kk++) {
        h[C32_NU * NZ + kk] = (float)cv(AX_NU, kk);
        h[C32_KAP * NZ + kk] = (float)cv(AX_KAP, kk);
        b64[B64_RHO * NZ + kk] = cv(AX_RHO, kk);
        b64[B64_E * NZ + kk] = cv(AX_E, kk);
        b64[B64_GAM * NZ + kk] = cv(AX_GAM, kk);
        b64[B64_R * NZ + kk] = cv(AX_R, kk);
        b64[B64_VG * NZ + kk] = cv(AX_VG, kk);
        if (kk > 0) {
            const double pb = (cv(AX_GAM, kk) - 1.0) * (cv(AX_E, kk) - 0.5 * 0.0 / cv(AX_RHO, kk));
            const double pa = (cv(AX_GAM, kk - 1) - 1.0) * (cv(AX_E, kk - 1) - 0.5 * 0.0 / cv(AX_RHO, kk - 1));
            b64[B64_RES * NZ + kk] = (pb - pa) - 0.5 * (cv(AX_RHO, kk) + cv(AX_RHO, kk - 1)) * cv(AX_VG, kk);
        }
    }
    for (int side = 0; side < 2; side++)
        for (int kbc = 1; kbc <= mbc; kbc++) {
            const int kg = side == 0 ? 1 - kbc : mz + kbc, kb = side == 0 ? 1 : mz;
            c->zr32.s[side][kbc - 1] = std::pow(cv(AX_RHO, kg + mbc - 1) / cv(AX_RHO, kb + mbc - 1), 0.5);
        }
    HIPCHECK(hipMemcpyAsync(c->col32, h.data(), h.size() * sizeof(float), hipMemcpyHostToDevice, c->stream));
    HIPCHECK(hipMemcpyAsync(c->bg64, b64.data(), b64.size() * sizeof(double), hipMemcpyHostToDevice,
                            c->stream));
    HIPCHECK(hipStreamSynchronize(c->stream));
    c->aux11_top = cv(AX_NU, mz + mbc - 1);
    c->aux12_top = cv(AX_KAP, mz + mbc - 1);
    c->have_aux = true;
    return MAGIC_OK;
}

// FP64 form: the ten slots as planes, the bc3 z factors per column.
template <class F>
static int set_aux64(magic_ctx *c, F get)
{
    const long long P = c->P;
    std::vector<double> h((size_t)P * NAUXP);
    for (int s = 0; s < NAUXP; s++) {
        double *dst = h.data() + (size_t)s * P;
        for (long long k = 0; k < P; k++) dst[k] = get(s, k);
    }
    HIPCHECK(hipMemcpyAsync(c->aux, h.data(), (size_t)P * NAUXP * sizeof(double), hipMemcpyHostToDevice,
                            c->stream));
    {   // layered background: every slot constant on each layer, bit for bit
        const long long NXY = (long long)c->d.NX * c->d.NY;
        const int NZ = c->d.NZ;
        bool layered = true;
        for (int s = 0; s < NAUXP && layered; s++)
            for (int k = 0; k < NZ && layered; k++) {
                const double *row = h.data() + (size_t)s * P + (size_t)k * NXY;
                for (long long e = 1; e < NXY; e++)
                    if (memcmp(row + e, row, sizeof(double)) != 0) {
                        layered = false;
                        break;
                    }
            }
        c->aux_layered = layered;
        if (layered) {
            std::vector<double> cols((size_t)NAUXP * NZ);
            for (int s = 0; s < NAUXP; s++)
                for (int k = 0; k < NZ; k++) cols[(size_t)s * NZ + k] = h[(size_t)s * P + (size_t)k * NXY];
            HIPCHECK(hipMemcpyAsync(c->col64, cols.data(), cols.size() * sizeof(double), hipMemcpyHostToDevice,
                                    c->stream));
            HIPCHECK(hipStreamSynchronize(c->stream));
        }
    }
    // bc3 z-face scale factors (aux(1,ghost)/aux(1,boundary))**0.5 in FP64
    // (bc3_mpi.f:560-573, 676-689), evaluated once on the host.
    const int NX = c->d.NX, NY = c->d.NY, mbc = c->mbc, mz = c->mz;
    const long long NXY = (long long)NX * NY;
    std::vector<double> zr((size_t)2 * mbc * NXY);
    const double *rho = h.data() + (size_t)AX_RHO * P;
    for (int side = 0; side < 2; side++)
        for (int kbc = 1; kbc <= mbc; kbc++)
            for (long long col = 0; col < NXY; col++) {
                const int kg = side == 0 ? 1 - kbc : mz + kbc;
                const int kb = side == 0 ? 1 : mz;
                const double g = rho[(long long)(kg + mbc - 1) * NXY + col];
                const double b = rho[(long long)(kb + mbc - 1) * NXY + col];
                zr[((size_t)side * mbc + (kbc - 1)) * NXY + col] = std::pow(g / b, 0.5);
            }
    HIPCHECK(hipMemcpyAsync(c->zratio, zr.data(), zr.size() * sizeof(double), hipMemcpyHostToDevice,
                            c->stream));
    HIPCHECK(hipStreamSynchronize(c->stream));
    // substep counts read the top cell of column (1,1): src3.f90:315, 319
    const long long c11 = ((long long)(mz + mbc - 1) * NY + (1 + mbc - 1)) * NX + (1 + mbc - 1);
    c->aux11_top = get(AX_NU, c11);
    c->aux12_top = get(AX_KAP, c11);
    c->have_aux = true;
    return MAGIC_OK;
}

extern "C" int magic_set_aux(magic_ctx *c, const double *aux)
{
    if (!c || !aux) return MAGIC_EARG;
    const int maux = c->maux;
    auto get = [&](int s, long long cell) { return aux[cell * maux + AUX_SLOT[s] - 1]; };
    if (c->form == MAGIC_FORM_FP32P) return set_aux32(c, get, true);
    return set_aux64(c, get);
}

extern "C" int magic_set_aux_column(magic_ctx *c, const double *col)
{
    if (!c || !col) return MAGIC_EARG;
    const int maux = c->maux;
    const long long NXY = (long long)c->d.NX * c->d.NY;
    auto get = [&](int s, long long cell) { return col[(cell / NXY) * maux + AUX_SLOT[s] - 1]; };
    if (c->form == MAGIC_FORM_FP32P) return set_aux32(c, get, false);
    return set_aux64(c, get);
}

// stage may be read by a snapshot's copy still in flight: the stream waits
// for it before anything writes stage
int stage_ready(magic_ctx *c)
{
    if (c->snap_pending) HIPCHECK(hipStreamWaitEvent(c->stream, c->snap_done, 0));
    return MAGIC_OK;
}

// q in the reference layout q(meqn, i, j, k), FP64, into stage (queued)
static int stage_q(magic_ctx *c)
{
    TRY(stage_ready(c));
    if (c->form == MAGIC_FORM_FP32P) {
        const int NZ = c->d.NZ;
        k32_pert_to_aos<<<padded_cells(c->d), cell_block(), 0, c->stream>>>(c->d, c->stage, c->q32, c->meqn,
                                                               c->bg64 + B64_RHO * NZ, c->bg64 + B64_E * NZ);
    } else {
        k_planes_to_aos<<<blocks(c->P, 256), 256, 0, c->stream>>>(c->stage, c->q, c->P, c->meqn);
    }
    return launch_check();
}

extern "C" int magic_set_q(magic_ctx *c, const double *q)
{
    if (!c || !q) return MAGIC_EARG;
    const size_t n = (size_t)c->P * c->meqn;
    TRY(stage_ready(c));
    if (c->form == MAGIC_FORM_FP32P) {
        if (!c->have_aux) return MAGIC_EARG;   // the perturbation needs the background
        const int NZ = c->d.NZ;
        TRY(upload(c, c->stage, q, n * sizeof(double)));
        k32_aos_to_pert<<<padded_cells(c->d), cell_block(), 0, c->stream>>>(c->d, c->q32, c->stage, c->meqn,
                                                               c->bg64 + B64_RHO * NZ, c->bg64 + B64_E * NZ);
        TRY(launch_check());
        HIPCHECK(hipMemcpyAsync(c->qold32, c->q32, n * sizeof(float), hipMemcpyDeviceToDevice, c->stream));
        HIPCHECK(hipStreamSynchronize(c->stream));
        return MAGIC_OK;
    }
    TRY(upload(c, c->stage, q, n * sizeof(double)));
    k_aos_to_planes<<<blocks(c->P, 256), 256, 0, c->stream>>>(c->q, c->stage, c->P, c->meqn);
    TRY(launch_check());
    HIPCHECK(hipMemcpyAsync(c->qold, c->q, n * sizeof(double), hipMemcpyDeviceToDevice, c->stream));
    HIPCHECK(hipStreamSynchronize(c->stream));
    return MAGIC_OK;
}

// qinit.f:74-82: q = aux(1:5) (fluid at rest on the background), tracers 0,
// on every cell including ghosts.
extern "C" int magic_qinit_rest(magic_ctx *c)
{
    if (!c || !c->have_aux) return MAGIC_EARG;
    const size_t P = (size_t)c->P, n = P * c->meqn;
    if (c->form == MAGIC_FORM_FP32P) {
        HIPCHECK(hipMemsetAsync(c->q32, 0, n * sizeof(float), c->stream));
        HIPCHECK(hipMemsetAsync(c->qold32, 0, n * sizeof(float), c->stream));
    } else {
        HIPCHECK(hipMemsetAsync(c->q, 0, n * sizeof(double), c->stream));
        HIPCHECK(hipMemcpyAsync(c->q, c->aux, 5 * P * sizeof(double), hipMemcpyDeviceToDevice, c->stream));
        HIPCHECK(hipMemcpyAsync(c->qold, c->q, n * sizeof(double), hipMemcpyDeviceToDevice, c->stream));
    }
    HIPCHECK(hipStreamSynchronize(c->stream));
    return MAGIC_OK;
}

extern "C" int magic_get_q(magic_ctx *c, double *q)
{
    if (!c || !q) return MAGIC_EARG;
    const size_t n = (size_t)c->P * c->meqn;
    TRY(stage_q(c));
    return download(c, q, c->stage, n * sizeof(double));
}

extern "C" int magic_snapshot_begin(magic_ctx *c, double *q, void **done)
{
    if (!c || !q || !done) return MAGIC_EARG;
    *done = nullptr;
    if (!c->cstream) {
        HIPCHECK(hipStreamCreateWithFlags(&c->cstream, hipStreamNonBlocking));
        HIPCHECK(hipEventCreateWithFlags(&c->snap_conv, hipEventDisableTiming));
        HIPCHECK(hipEventCreateWithFlags(&c->snap_done, hipEventDisableTiming));
    }
    const size_t n = (size_t)c->P * c->meqn;
    TRY(stage_q(c));
    HIPCHECK(hipEventRecord(c->snap_conv, c->stream));
    HIPCHECK(hipStreamWaitEvent(c->cstream, c->snap_conv, 0));
    HIPCHECK(hipMemcpyAsync(q, c->stage, n * sizeof(double), hipMemcpyDeviceToHost, c->cstream));
    HIPCHECK(hipEventRecord(c->snap_done, c->cstream));
    c->snap_pending = true;
    hipEvent_t ev = nullptr;
    HIPCHECK(hipEventCreateWithFlags(&ev, hipEventDisableTiming));
    if (hipEventRecord(ev, c->cstream) != hipSuccess) {
        hipEventDestroy(ev);
        return MAGIC_EHIP;
    }
    *done = ev;
    return MAGIC_OK;
}

extern "C" int magic_snapshot_wait(void *done)
{
    if (!done) return MAGIC_EARG;
    hipEvent_t ev = (hipEvent_t)done;
    const hipError_t e = hipEventSynchronize(ev);
    hipEventDestroy(ev);
    return e == hipSuccess ? MAGIC_OK : MAGIC_EHIP;
}

extern "C" int magic_host_alloc(size_t bytes, void **p)
{
    if (!p || bytes == 0) return MAGIC_EARG;
    *p = nullptr;
    return hipHostMalloc(p, bytes, hipHostMallocDefault) == hipSuccess ? MAGIC_OK : MAGIC_ENOMEM;
}

extern "C" int magic_host_free(void *p)
{
    if (p) HIPCHECK(hipHostFree(p));
    return MAGIC_OK;
}

// ------------------------------------------------------------- bc3 -------
static ZScale64 zscale(const magic_ctx *c, double)
{
    const double *A = c->aux;
    return {A + AX_RHO * c->P, A + AX_MX * c->P, A + AX_MY * c->P, A + AX_E * c->P, c->zratio, c->mbc,
            (long long)c->d.NX * c->d.NY};
}
static ZScale32 zscale(const magic_ctx *c, float) { return {c->zr32}; }
static int bc_z_apart(magic_ctx *c, double *q, int lo, int hi)
{
    const ZScale64 z = zscale(c, 0.0);
    k_bc_z<<<dim3(blocks(c->d.NX, 64), c->d.NY), 64, 0, c->stream>>>(c->d, q, c->meqn, lo, hi, z.aux1, z.aux2, z.aux3, z.aux5,
                                                                     z.zratio, GridGate{});
    return launch_check();
}
static int bc_z_apart(magic_ctx *c, float *q, int lo, int hi)
{
    k32_bc_z<<<dim3(blocks(c->d.NX, 64), c->d.NY), 64, 0, c->stream>>>(c->d, q, c->meqn, lo, hi, c->zr32, GridGate{});
    return launch_check();
}

// bc3 on q, with b4step3's clamp (CLAMP_BC) or diffuse's z ghosts (UVW_BC) in
// the same pass
template <typename T>
static int bc_launch(magic_ctx *c, T *q, const int *mthbc, int mode)
{
    for (int f = 0; f < 6; f++)
        if (mthbc[f] == 0 || mthbc[f] >= 4) return MAGIC_EBC;
    Span sp(c, TC_BC, 1);
    const Dims &d = c->d;
    Faces fc;
    for (int f = 0; f < 6; f++) fc.m[f] = mthbc[f] < 0 ? 0 : mthbc[f];
    // fewer layers than ghost layers: a mirrored or periodic z ghost can come
    // from the other side's ghosts, so the z faces follow in their own pass
    const bool apart = c->mz < c->mbc && (fc.m[4] != 0 || fc.m[5] != 0);
    const int lo = fc.m[4], hi = fc.m[5];
    if (apart) fc.m[4] = fc.m[5] = 0;
    const bool clamp = (mode & CLAMP_BC) != 0 && c->meqn > 5;
    const long long n = (long long)bc_lanes(d, 0) + bc_lanes(d, 1) + bc_lanes(d, 2) + (clamp ? bc_lanes(d, 3) : 0);
    k_bc<<<blocks(n, 256), 256, 0, c->stream>>>(d, q, c->meqn, fc, mode, zscale(c, T()), c->gate);
    TRY(launch_check());
    return apart ? bc_z_apart(c, q, lo, hi) : MAGIC_OK;
}
static int bc3_launch(magic_ctx *c, const int *mthbc, int mode = 0)
{
    return c->form == MAGIC_FORM_FP32P ? bc_launch(c, c->q32, mthbc, mode) : bc_launch(c, c->q, mthbc, mode);
}

extern "C" int magic_bc3(magic_ctx *c, const int mthbc[6])
{
    if (!c || !mthbc) return MAGIC_EARG;
    if (!c->have_aux) return MAGIC_EARG;
    TRY(bc3_launch(c, mthbc));
    HIPCHECK(hipStreamSynchronize(c->stream));
    return MAGIC_OK;
}

static int b4step3_launch(magic_ctx *c)
{
    if (c->meqn > 5) {
        Span sp(c, TC_OTHER, 1);
        if (c->form == MAGIC_FORM_FP32P) k_clamp<<<blocks(c->P, 256), 256, 0, c->stream>>>(c->q32, c->P, c->meqn, GridGate{});
        else k_clamp<<<blocks(c->P, 256), 256, 0, c->stream>>>(c->q, c->P, c->meqn, GridGate{});
        TRY(launch_check());
    }
    return MAGIC_OK;
}

extern "C" int magic_b4step3(magic_ctx *c)
{
    if (!c) return MAGIC_EARG;
    TRY(b4step3_launch(c));
    HIPCHECK(hipStreamSynchronize(c->stream));
    return MAGIC_OK;
}

// copyq3: q -> backup (to_backup) or backup -> q
static int copy_state(magic_ctx *c, bool to_backup)
{
    Span sp(c, TC_OTHER, 1);
    const size_t n = (size_t)c->P * c->meqn;
    if (c->form == MAGIC_FORM_FP32P) {
        HIPCHECK(hipMemcpyAsync(to_backup ? c->qold32 : c->q32, to_backup ? c->q32 : c->qold32,
                                n * sizeof(float), hipMemcpyDeviceToDevice, c->stream));
    } else {
        HIPCHECK(hipMemcpyAsync(to_backup ? c->qold : c->q, to_backup ? c->q : c->qold, n * sizeof(double),
                                hipMemcpyDeviceToDevice, c->stream));
    }
    return MAGIC_OK;
}

extern "C" int magic_backup(magic_ctx *c)
{
    if (!c) return MAGIC_EARG;
    TRY(copy_state(c, true));
    HIPCHECK(hipStreamSynchronize(c->stream));
    return MAGIC_OK;
}

extern "C" int magic_restore(magic_ctx *c)
{
    if (!c) return MAGIC_EARG;
    TRY(copy_state(c, false));
    HIPCHECK(hipStreamSynchronize(c->stream));
    return MAGIC_OK;
}

// ------------------------------------------------------------ step3 ------
__global__ void k_zero_scalars(unsigned long long *s)
{
    if (threadIdx.x < 8) s[threadIdx.x] = 0ull;
}

template <int NTR>
static int launch_sweep(magic_ctx *c, SweepArgs a, int *nl)
{
    if (a.n + 3 > 512) return MAGIC_EUNSUPPORTED;   // one workgroup per pencil
    const int NI = a.n + 3;
    const int threads = ((NI + 63) / 64) * 64;
    const size_t smem = (size_t)(7 + NTR) * NI * sizeof(double) + (size_t)NI * sizeof(int);
    for (int ca = 0; ca < 3; ca++)
        for (int cb = 0; cb < 3; cb++) {
            a.cA = ca;
            a.cB = cb;
            dim3 grid((unsigned)((a.nA + 1 - ca) / 3 + 1), (unsigned)((a.nB + 1 - cb) / 3 + 1));
            sweep_kernel<NTR><<<grid, threads, smem, c->stream>>>(a);
            TRY(launch_check());
            ++*nl;
        }
    return MAGIC_OK;
}

static bool use_tile()
{
    const char *e = getenv("MAGIC_SWEEP");
    return !(e && strcmp(e, "pencil") == 0);
}

static int sweep_dispatch(magic_ctx *c, const SweepArgs &a, int *nl)
{
    switch (ntracer(c)) {
    case 0: return launch_sweep<0>(c, a, nl);
    case 1: return launch_sweep<1>(c, a, nl);
    case 2: return launch_sweep<2>(c, a, nl);
    case 3: return launch_sweep<3>(c, a, nl);
    case 4: return launch_sweep<4>(c, a, nl);
    case 5: return launch_sweep<5>(c, a, nl);
    default: return MAGIC_EUNSUPPORTED;
    }
}

// Directional fields of the argument block: dir 0 = x-sweep
// (lib/step3.f:121-280, g = y, h = z), 1 = y-sweep (step3.f:289-450, g = z,
// h = x), 2 = z-sweep (step3.f:459-621, g = x, h = y, gravity on).
template <typename T>
static void dir_args(const magic_ctx *c, SweepArgsT<T> &a, int dir, double dt)
{
    const Dims &d = c->d;
    const long long NXY = (long long)d.NX * d.NY;
    const double dtdx = dt / c->dx, dtdy = dt / c->dy, dtdz = dt / c->dz;
    if (dir == 0) {
        a.comp[0] = 0; a.comp[1] = 1; a.comp[2] = 2; a.comp[3] = 3; a.comp[4] = 4;
        a.n = c->mx; a.nA = c->my; a.nB = c->mz;
        a.sN = 1; a.sA = d.NX; a.sB = NXY;
        a.gravity = 0; a.sweep = 1;
        a.dtdn = dtdx; a.fg = dtdy; a.fh = dtdz;
    } else if (dir == 1) {
        a.comp[0] = 0; a.comp[1] = 2; a.comp[2] = 3; a.comp[3] = 1; a.comp[4] = 4;
        a.n = c->my; a.nA = c->mz; a.nB = c->mx;
        a.sN = d.NX; a.sA = NXY; a.sB = 1;
        a.gravity = 0; a.sweep = 2;
        a.dtdn = dtdy; a.fg = dtdz; a.fh = dtdx;
    } else {
        a.comp[0] = 0; a.comp[1] = 3; a.comp[2] = 1; a.comp[3] = 2; a.comp[4] = 4;
        a.n = c->mz; a.nA = c->mx; a.nB = c->my;
        a.sN = NXY; a.sA = 1; a.sB = d.NX;
        a.gravity = 1; a.sweep = 3;
        a.dtdn = dtdz; a.fg = dtdx; a.fh = dtdy;
    }
}

// The increment buffer given back; the next sweep sets it up again
static void drop_parts(magic_ctx *c)
{
    if (!c->parts_stage) hipFree(c->parts);
    hipFree(c->items);
    c->parts = nullptr;
    c->parts_bytes = 0;
    c->parts_stage = false;
    c->items = nullptr;
}

// Buffers of the tiled sweeps for the context's shapes: argument blocks and
// run flags, the workgroups' blocks, and the increment buffer.  Where the
// device (or the caller) has no room for the whole grid's increments, the
// buffer holds a slab's, and the slabs are swept one after the other.
template <typename T>
static int sweep_setup(magic_ctx *c)
{
    if (!c->largs) {
        if (hipMalloc(&c->largs, 3 * sizeof(SweepArgsT<T>)) != hipSuccess ||
            hipMalloc(&c->lrun, 3 * sizeof(int *)) != hipSuccess || hipMalloc(&c->lone, sizeof(int)) != hipSuccess) {
            hipFree(c->largs); hipFree(c->lrun); hipFree(c->lone);
            c->largs = nullptr; c->lrun = nullptr; c->lone = nullptr;
            (void)hipGetLastError();
            return MAGIC_ENOMEM;
        }
        const int one = 1;
        const int *run[3] = {c->lone, c->lone, c->lone};
        HIPCHECK(hipMemcpy(c->lone, &one, sizeof(int), hipMemcpyHostToDevice));
        HIPCHECK(hipMemcpy(c->lrun, run, sizeof(run), hipMemcpyHostToDevice));
    }
    if (c->items && memcmp(c->item_shape, c->shape, sizeof(c->shape)) == 0) return MAGIC_OK;
    HIPCHECK(hipStreamSynchronize(c->stream));   // nothing reads the old lists or increments any more
    hipFree(c->items);
    c->items = nullptr;
    const Slabs<T> slabs(c, c->shape);
    const size_t least = slabs.least(), want = std::min(slabs.whole(), std::max(least, c->parts_room));
    if (c->parts_bytes < want) {
        drop_parts(c);
        size_t got = want;   // less room: narrower slabs, at last in the staging buffer, idle in a step
        while (hipMalloc(&c->parts, got) != hipSuccess) {
            (void)hipGetLastError();
            c->parts = nullptr;
            if (got == least) {
                if (stage_bytes(c) < least) return MAGIC_ENOMEM;
                c->parts = c->stage;
                c->parts_stage = true;
                got = stage_bytes(c);
                break;
            }
            got = std::max(least, got / 2);
        }
        c->parts_bytes = got;
    }
    c->slabs = slabs.within(c->parts_bytes);
    std::vector<int4> items;
    c->item_off.assign(1, 0);
    for (const Slab &slab : c->slabs)
        for (int dir = 0; dir < 3; dir++) {
            push_items(items, slabs.p[dir], dir, slab.lo[dir], slab.hi[dir], dir);
            c->item_off.push_back((int)items.size());
        }
    if (hipMalloc(&c->items, items.size() * sizeof(int4)) != hipSuccess) {
        (void)hipGetLastError();
        c->items = nullptr;
        return MAGIC_ENOMEM;
    }
    HIPCHECK(hipMemcpy(c->items, items.data(), items.size() * sizeof(int4), hipMemcpyHostToDevice));
    memcpy(c->item_shape, c->shape, sizeof(c->shape));
    return MAGIC_OK;
}

// The argument blocks of a slab's sweeps, and (scal) the step's reductions
// back to zero.  Launched before the sweeps on their stream.
template <typename T>
struct StepArgs {
    SweepArgsT<T> d[3];
};
template <typename T>
__global__ void k_put_step_args(SweepArgsT<T> *slots, StepArgs<T> a, unsigned long long *scal)
{
    if (threadIdx.x < 3) slots[threadIdx.x] = a.d[threadIdx.x];
    else if (scal && threadIdx.x >= 8 && threadIdx.x < 16) scal[threadIdx.x - 8] = 0ull;
}

// Argument blocks for step dt of slab s from base (state pointers and
// form-specific fields set), and the descriptors of the parts they fill
template <typename T>
static int put_step_args(magic_ctx *c, const SweepArgsT<T> &base, double dt, size_t s, StepParts<T> &sp)
{
    if (c->parts_stage) TRY(stage_ready(c));
    StepArgs<T> sa;
    const Slab &slab = c->slabs[s];
    sp.nc = c->meqn;
    T *next = (T *)c->parts;
    for (int dir = 0; dir < 3; dir++) {
        sa.d[dir] = base;
        sweep_geometry(c, dir, c->shape[dir], sa.d[dir], sp.d[dir]);
        sweep_factors(c, dir, dt, sa.d[dir]);
        next = parts_layout(sa.d[dir], sp.d[dir], dir, slab.lo[dir], slab.hi[dir], c->meqn, c->shape[dir], next);
    }
    k_put_step_args<T><<<1, 64, 0, c->stream>>>((SweepArgsT<T> *)c->largs, sa, s == 0 ? c->dscal : nullptr);
    return launch_check();
}

// One launch over the blocks of slab s and directions d0 .. d1-1 (of one shape)
template <typename T, bool PERT>
static int launch_tile(magic_ctx *c, size_t s, int d0, int d1)
{
    const void *fn = tile_fn<T, PERT>(ntracer(c), c->shape[d0]);
    if (!fn) return MAGIC_EARG;
    const SweepArgsT<T> *args = (const SweepArgsT<T> *)c->largs;
    const int *off = &c->item_off[3 * s];
    const int4 *items = c->items + off[d0];
    const int *const *run = c->lrun;
    void *kargs[] = {&args, &items, &run};
    Span sp(c, NTC, 1);
    const float blocks_ = (float)(off[d1] - off[d0]);
    for (int d = d0; d < d1; d++) sp.share[d] = (off[d + 1] - off[d]) / blocks_;
    HIPCHECK(hipLaunchKernel(fn, dim3((unsigned)(off[d1] - off[d0])), dim3(256), kargs, 0, c->stream));
    return MAGIC_OK;
}

// q += the increments of sp, the cells of slab s
template <typename T>
static int add_parts_launch(magic_ctx *c, T *q, const StepParts<T> &sp, const Slab &s)
{
    Span t(c, TC_OTHER, 1);
    k_add_parts<T><<<slab_cells(c->d, s), cell_block(), 0, c->stream>>>(c->d, q, sp, s.i0 + c->mbc - 1, s.i1 + c->mbc - 1, nullptr);
    return launch_check();
}

// The three sweeps of step3 (lib/step3.f:121-621) on argument block a, whose
// state pointers and form-specific fields are already set.  The sweeps only
// read a.qold and write their blocks' increments, so they are one launch
// (one per run of directions that share a tile shape); sp returns the
// increments, which add_parts or the source pass's conversion adds to q.
// In slabs, each slab's increments are added to q at once, the same sum for
// every cell, and sp is left empty.
template <typename T, bool PERT>
static int step3_sweeps(magic_ctx *c, const SweepArgsT<T> &a, T *q, double dt, StepParts<T> &sp)
{
    TRY(sweep_setup<T>(c));
    for (size_t s = 0; s < c->slabs.size(); s++) {
        TRY(put_step_args<T>(c, a, dt, s, sp));
        for (int d0 = 0, d1; d0 < 3; d0 = d1) {
            for (d1 = d0 + 1; d1 < 3 && c->shape[d1] == c->shape[d0];) d1++;
            TRY((launch_tile<T, PERT>(c, s, d0, d1)));
        }
        if (c->slabs.size() > 1) TRY(add_parts_launch(c, q, sp, c->slabs[s]));
    }
    if (c->slabs.size() > 1)
        for (auto &p : sp.d) p.base = nullptr;
    return MAGIC_OK;
}

// The FP64 form's one-workgroup-per-pencil kernel (MAGIC_SWEEP=pencil), which
// adds into q in nine colour launches per direction
static int pencil_sweeps(magic_ctx *c, const SweepArgs &a, double dt)
{
    for (int dir = 0; dir < 3; dir++) {
        Span sp(c, TC_SWX + dir, 0);
        SweepArgs d = a;
        dir_args(c, d, dir, dt);
        TRY(sweep_dispatch(c, d, &sp.n));
    }
    return MAGIC_OK;
}

// form-specific part of the argument block: state pointers, columns, scratch
static SweepArgsT<float> args32(magic_ctx *c)
{
    SweepArgsT<float> a;
    memset(&a, 0, sizeof(a));
    a.qold = c->qold32;
    a.qnew = c->q32;
    a.P = c->P;
    a.mbc = c->mbc;
    a.nspecadv = c->have_params ? c->prm.nspecadv : 0;
    a.cfl_bits = c->dscal;
    a.status = (int *)(c->dscal + 1);
    for (int m = 5; m < c->meqn; m++) a.comp[m] = m;
    const int NZ = c->d.NZ;
    a.crho = c->bg64 + B64_RHO * NZ;
    a.cE = c->bg64 + B64_E * NZ;
    a.cgam = c->bg64 + B64_GAM * NZ;
    a.cvg = c->bg64 + B64_VG * NZ;
    a.cres = c->bg64 + B64_RES * NZ;
    return a;
}

static SweepArgs args64(magic_ctx *c)
{
    SweepArgs a;
    memset(&a, 0, sizeof(a));
    a.qold = c->qold;
    a.qnew = c->q;
    a.gam = c->aux + AX_GAM * c->P;
    a.vgrav = c->aux + AX_VG * c->P;
    a.P = c->P;
    a.mbc = c->mbc;
    a.nspecadv = c->have_params ? c->prm.nspecadv : 0;
    a.cfl_bits = c->dscal;
    a.status = (int *)(c->dscal + 1);
    for (int m = 5; m < c->meqn; m++) a.comp[m] = m;
    return a;
}

// the pending increments of a step, added to q as a pass of their own
static int parts_flush(magic_ctx *c)
{
    if (!c->pending_parts) return MAGIC_OK;
    c->pending_parts = false;
    return c->form == MAGIC_FORM_FP32P ? add_parts_launch(c, c->q32, c->parts32, c->slabs[0])
                                       : add_parts_launch(c, c->q, c->parts64, c->slabs[0]);
}

// whether the sweeps leave their increments in the part buffer (known once
// sweep_setup has run) rather than in q
static bool form_tile(const magic_ctx *c) { return c->form == MAGIC_FORM_FP32P || use_tile(); }
static int setup_sweeps(magic_ctx *c)
{
    if (!form_tile(c)) return MAGIC_OK;
    return c->form == MAGIC_FORM_FP32P ? sweep_setup<float>(c) : sweep_setup<double>(c);
}
static bool sweeps_defer(const magic_ctx *c) { return form_tile(c) && c->slabs.size() == 1; }

static int scal_copy(magic_ctx *c)
{
    HIPCHECK(hipMemcpyAsync(c->hscal, c->dscal, 8 * sizeof(unsigned long long), hipMemcpyDeviceToHost, c->stream));
    return MAGIC_OK;
}

// The sweeps of one step and (without defer) the read-back of its reductions.  from_q: they
// read q itself (with deferred increments q does not change meanwhile);
// else the backup.  The increments end up in q, or with defer stay pending
// in the part buffer (c->pending_parts).
static int step3_launch(magic_ctx *c, double dt, bool from_q = false, bool defer = false)
{
    if (!form_tile(c)) {
        k_zero_scalars<<<1, 64, 0, c->stream>>>(c->dscal);
        TRY(launch_check());
        TRY(pencil_sweeps(c, args64(c), dt));
    } else if (c->form == MAGIC_FORM_FP32P) {
        SweepArgsT<float> a = args32(c);
        if (from_q) a.qold = c->q32;
        TRY((step3_sweeps<float, true>(c, a, c->q32, dt, c->parts32)));
        c->pending_parts = c->parts32.d[0].base != nullptr;
    } else {
        SweepArgs a = args64(c);
        if (from_q) a.qold = c->q;
        TRY((step3_sweeps<double, false>(c, a, c->q, dt, c->parts64)));
        c->pending_parts = c->parts64.d[0].base != nullptr;
    }
    if (defer) return MAGIC_OK;   // the source pass reports and adds the increments
    TRY(scal_copy(c));
    return parts_flush(c);
}

static int step3_finish(magic_ctx *c, double *cfl)
{
    HIPCHECK(hipStreamSynchronize(c->stream));
    double v;
    memcpy(&v, &c->hscal[0], sizeof(double));
    *cfl = v;
    const int *st = (const int *)(c->hscal + 1);
    if (st[0] != 0) {
        for (int k = 0; k < 4; k++) c->errloc[k] = st[1 + k];
        return st[0] == 1 ? MAGIC_ERHO : MAGIC_EA2;
    }
    return MAGIC_OK;
}

extern "C" int magic_step3(magic_ctx *c, double dt, double *cfl)
{
    if (!c || !cfl || !c->have_aux) return MAGIC_EARG;
    TRY(step3_launch(c, dt));
    int s = step3_finish(c, cfl);
    if (c->timing) drain_timing(c);
    return s;
}

// The end of a batch's scenario whose sweeps failed: q, which the attempt left
// as it was (its sweeps read it, nothing is added before the decision), becomes
// the backup, and the step's increments are added to it, as claw3 leaves a grid
// that fails.  Sweeping again costs a failed scenario one step; gates for it
// in the conversion cost every step (SGPRs spilt, or a wave fewer per SIMD).
int failed_step(magic_ctx *c, const int *shape, double dt)
{
    int keep[3];
    memcpy(keep, c->shape, sizeof(keep));
    memcpy(c->shape, shape, sizeof(keep));
    double cfl;
    int st = copy_state(c, true);
    if (st == MAGIC_OK) st = step3_launch(c, dt);
    if (st == MAGIC_OK) st = step3_finish(c, &cfl);
    memcpy(c->shape, keep, sizeof(keep));
    drop_parts(c);   // a scenario has no sweeps of its own otherwise
    return st == MAGIC_ERHO || st == MAGIC_EA2 ? MAGIC_OK : st;
}

// ------------------------------------------------------- tile shapes -----
extern "C" int magic_set_tile_shapes(magic_ctx *c, const int shapes[3])
{
    if (!c || !shapes || !shapes_valid(shapes)) return MAGIC_EARG;
    for (int k = 0; k < 3; k++) c->shape[k] = shapes[k];
    return MAGIC_OK;
}

extern "C" int magic_get_tile_shapes(magic_ctx *c, int shapes[3])
{
    if (!c || !shapes) return MAGIC_EARG;
    for (int k = 0; k < 3; k++) shapes[k] = c->shape[k];
    return MAGIC_OK;
}

extern "C" int magic_set_increment_room(magic_ctx *c, size_t bytes)
{
    if (!c) return MAGIC_EARG;
    HIPCHECK(hipStreamSynchronize(c->stream));
    c->parts_room = bytes ? bytes : ~size_t(0);
    drop_parts(c);
    return MAGIC_OK;
}

extern "C" int magic_set_sweep_overlap(magic_ctx *c, int) { return c ? MAGIC_OK : MAGIC_EARG; }

// Autotuner: every tile shape of every sweep direction is timed on this
// grid's current state (one untimed sweep, then reps timed ones, HIP events
// on the grid's stream) and the fastest shape of each direction is kept.
// The candidates read the backup copy and write only their increment
// blocks, so q does not change (the backup then holds it).
template <typename T, bool PERT>
static int tune_rounds(magic_ctx *c, const SweepArgsT<T> &a, double dt, int reps, TuneClock &clk)
{
    for (int r = 0; r <= reps; r++) {   // repetition 0 warms up and is not timed
        for (int sh = 0; sh < TILE_NSHAPE; sh++) {
            for (int k = 0; k < 3; k++) c->shape[k] = sh;
            TRY(sweep_setup<T>(c));
            StepParts<T> sp;
            const size_t n = c->slabs.size();
            if (n == 1) TRY(put_step_args<T>(c, a, dt, 0, sp));
            for (int dir = 0; dir < 3; dir++) {
                TRY(clk.mark(dir, sh, 0, c->stream));
                for (size_t s = 0; s < n; s++) {
                    if (n > 1) TRY(put_step_args<T>(c, a, dt, s, sp));
                    TRY((launch_tile<T, PERT>(c, s, dir, dir + 1)));
                }
                TRY(clk.mark(dir, sh, 1, c->stream));
            }
        }
        if (r > 0) TRY(clk.add_round());
    }
    return MAGIC_OK;
}

// The backup as the tuners time the sweeps on it: q with its ghost cells
// extrapolated.  After a step they hold the source pass's variables, which are no
// state: every interface there would report a failure, and the reports'
// atomics took 3 ms of a 4 ms sweep.
int tune_state(magic_ctx *c)
{
    static const int faces[6] = {1, 1, 1, 1, 1, 1};
    TRY(copy_state(c, true));
    return c->form == MAGIC_FORM_FP32P ? bc_launch(c, c->qold32, faces, 0) : bc_launch(c, c->qold, faces, 0);
}

// The backup a copy of q again, its ghosts too: after the tuners, whether
// they succeeded or not
int tune_done(magic_ctx *c) { return copy_state(c, true); }

extern "C" int magic_tune(magic_ctx *c, double dt, int reps, int shapes_out[3], float *ms_out)
{
    if (!c || !c->have_aux || !(dt > 0.0) || reps < 1) return MAGIC_EARG;
    if (!form_tile(c) || !sweep_supported(ntracer(c))) return MAGIC_EUNSUPPORTED;
    TuneClock clk;
    if (!clk.ok) return MAGIC_EHIP;
    const int keep[3] = {c->shape[0], c->shape[1], c->shape[2]};
    int st = tune_state(c);
    if (st == MAGIC_OK)
        st = c->form == MAGIC_FORM_FP32P ? tune_rounds<float, true>(c, args32(c), dt, reps, clk)
                                         : tune_rounds<double, false>(c, args64(c), dt, reps, clk);
    for (int k = 0; k < 3; k++) c->shape[k] = keep[k];
    const int sc = tune_done(c);
    TRY(st);
    TRY(sc);
    int best[3];
    clk.result(reps, best, ms_out);
    k_zero_scalars<<<1, 64, 0, c->stream>>>(c->dscal);   // the candidates' Courant numbers and reports
    TRY(launch_check());
    HIPCHECK(hipStreamSynchronize(c->stream));
    for (int k = 0; k < 3; k++) c->shape[k] = best[k];
    if (shapes_out)
        for (int k = 0; k < 3; k++) shapes_out[k] = best[k];
    return MAGIC_OK;
}

// ------------------------------------------------------------- src3 ------
// The substeps of the source pass after its conversion (src3.f90:341-376 with
// diffuse.f:37-210 and conduct.f:245-332): per substep the boundary pass with
// diffuse's z ghosts, the cross terms, and the directional passes of the
// velocities next to conduct's first substep; conduct's later substeps
// follow one by one.  q's planes keep the values before the cross terms,
// whose ghost layers the passes read (the reference's stale copy).  t5
// returns T' after the last substep: conduct leaves it in ut or qt, from
// where it goes back to q only between substeps.
template <typename T, bool COLC>
static int src3_substeps(magic_ctx *c, DiffArgs<T> a, const int *mthbc, int ndtr, double dtr, int ndtrc, double dtrc,
                         const T **t5)
{
    const Dims &d = c->d;
    const double fourthirds = 4.0 / 3.0;
    double dtdx2 = (dtr) / (c->dx * c->dx), dtdy2 = (dtr) / (c->dy * c->dy), dtdz2 = (dtr) / (c->dz * c->dz);
    for (int cc = 0; cc < 3; cc++) {   // diffuse.f:135-151
        if (cc == 0) {
            dtdx2 = fourthirds * dtdx2;
        } else if (cc == 1) {
            dtdy2 = fourthirds * dtdy2;
            dtdx2 = dtdx2 / fourthirds;
        } else {
            dtdz2 = fourthirds * dtdz2;
            dtdy2 = dtdy2 / fourthirds;
        }
        a.f[3 * cc] = (T)dtdx2; a.f[3 * cc + 1] = (T)dtdy2; a.f[3 * cc + 2] = (T)dtdz2;
    }
    a.f[9] = (T)((dtrc) / (c->dx * c->dx));
    a.f[10] = (T)((dtrc) / (c->dy * c->dy));
    a.f[11] = (T)((dtrc) / (c->dz * c->dz));
    a.S = c->mz > c->mx ? c->mz - c->mx : 0;
    a.kb = passes_kb(d);
    const double dtr32 = dtr / 6.0;
    const dim3 g4 = passes_grid(d, ndtrc > 0 ? 4 : 3), g1 = passes_grid(d, 1);
    const T *res = ndtrc <= 0 ? a.q + 4 * d.P : (ndtrc & 1) ? a.ut : a.qt;
    for (int nn = 1; nn <= ndtr; nn++) {
        TRY(bc_launch(c, a.q, mthbc, UVW_BC));
        Span sp(c, TC_SRC, 2 + (ndtrc > 1 ? ndtrc - 1 : 0) + (nn < ndtr ? 1 : 0));
        k_diff_cross<T, COLC, GridGate><<<diff_grid(d), cell_block(), 0, c->stream>>>(
            d, const_cast<T *>(a.u), a.q, a.nu, (T)(dtr32 / (c->dx * c->dy)), (T)(dtr32 / (c->dx * c->dz)),
            (T)(dtr32 / (c->dy * c->dz)), diff_kb(d), c->gate);
        TRY(launch_check());
        k_diff<T, COLC, GridGate><<<g4, cell_block(), 0, c->stream>>>(d, a, 1, c->gate);
        TRY(launch_check());
        for (int kk = 2; kk <= ndtrc; kk++) k_diff<T, COLC, GridGate><<<g1, cell_block(), 0, c->stream>>>(d, a, kk, c->gate);
        if (nn < ndtr && ndtrc > 0)
            k_copy_interior<<<interior_grid(d), cell_block(), 0, c->stream>>>(d, a.q + 4 * d.P, res, 1, c->gate);
        TRY(launch_check());
    }
    *t5 = ndtr > 0 ? res : a.q + 4 * d.P;
    return MAGIC_OK;
}

// The source pass of the FP32 form: the FP64 form's passes (below) on the
// perturbation planes, with nu and kappa as background columns.
static int src3_passes32(magic_ctx *c, const int *mthbc, int ndtr, double dtr, int ndtrc, double dtrc,
                         const Forcing &f)
{
    const Dims &d = c->d;
    const int NZ = d.NZ;
    const Col32 col = col32_of(c);
    {
        Span sp(c, TC_SRC, 1);
        if (!c->pending_parts) c->parts32.d[0].base = nullptr;
        // with pending increments the new state goes to the other buffer and
        // the old one stays behind as the backup
        float *to = c->pending_parts ? c->qold32 : c->q32;
        k32_src_convert<<<padded_cells(c->d), cell_block(), 0, c->stream>>>(d, c->q32, to, col, c->gate, c->parts32);
        TRY(launch_check());
        if (c->pending_parts) std::swap(c->q32, c->qold32);
        c->pending_parts = false;
    }
    const float *t5;
    const DiffArgs<float> a = {c->q32, c->u32, c->ut32, c->qt32, c->col32 + C32_NU * NZ, c->col32 + C32_KAP * NZ, {}, 0, 0};
    TRY((src3_substeps<float, true>(c, a, mthbc, ndtr, dtr, ndtrc, dtrc, &t5)));
    Span sp(c, TC_SRC, 1);
    k32_src_finish<<<interior_grid(d), cell_block(), 0, c->stream>>>(d, c->q32, t5, c->meqn, col, f, c->gate);
    return launch_check();
}

// The source pass of the FP64 form (src3.f90:203-634 with diffuse.f and
// conduct.f).  COL: the background (aux 1-5, 11, 12, 18, 19) is read from
// its columns, which hold the same values when it is constant on each layer.
template <bool COL>
static int src3_passes64(magic_ctx *c, const int *mthbc, int ndtr, double dtr, int ndtrc, double dtrc,
                         const Forcing &f)
{
    const Dims &d = c->d;
    const double *A = COL ? c->col64 : c->aux;
    const long long S = COL ? d.NZ : c->P;   // stride between slots
    const Aux ax = {A + AX_RHO * S, A + AX_MX * S, A + AX_MY * S, A + AX_MZ * S, A + AX_E * S, A + AX_R * S,
                    A + AX_GAM * S};
    {
        Span sp(c, TC_SRC, 1);
        if (!c->pending_parts) c->parts64.d[0].base = nullptr;
        // with pending increments the new state goes to the other buffer and
        // the old one stays behind as the backup
        double *to = c->pending_parts ? c->qold : c->q;
        k_src_convert<COL><<<padded_cells(d), cell_block(), 0, c->stream>>>(d, c->q, to, ax, c->gate, c->parts64);
        TRY(launch_check());
        if (c->pending_parts) std::swap(c->q, c->qold);
        c->pending_parts = false;
    }
    const double *t5;
    const DiffArgs<double> a = {c->q, c->u, c->ut, c->qt, A + AX_NU * S, A + AX_KAP * S, {}, 0, 0};
    TRY((src3_substeps<double, COL>(c, a, mthbc, ndtr, dtr, ndtrc, dtrc, &t5)));
    Span sp(c, TC_SRC, 1);
    k_src_finish<COL><<<interior_grid(d), cell_block(), 0, c->stream>>>(d, c->q, t5, c->meqn, ax, f, c->gate);
    return launch_check();
}

// Most launches of a source pass that claw3 queues behind the sweeps before
// it knows their Courant number.  They end at once in a rejected attempt, but
// each still takes 2-4 us, and the substeps of a dt far beyond the Courant
// limit may be any number; a pass of more launches than this hardly gains by
// the wait it saves (4-9 us).
constexpr double MAX_AHEAD = 32.0;
// About how many launches the source pass of a step dt takes, from its
// substep counts (src3.f90:314-322)
static double src_launches(const magic_ctx *c, double dt)
{
    const double dmin = std::min(std::min(c->dx, c->dy), c->dz), d2 = dmin * dmin;
    const double n = std::ceil((dt * (4.0 / 3.0) * c->aux11_top / d2) / 0.45);
    const double nc = n > 0.0 ? std::ceil((dt / n * c->aux12_top / d2) / 0.45) : 0.0;
    return 2.0 + n * (4.0 + nc);
}

static int src3_launch(magic_ctx *c, double t, double dt, const int *mthbc_in, int *ndtr_out,
                       int *ndtrc_out)
{
    const magic_params &p = c->prm;
    if (p.omega1 != 0.0) return MAGIC_EUNSUPPORTED;   // time-dependent wind (src3.f90:389-399)
    const int fm = (int)p.forcemth;
    if (!(p.forcemth == 0.0 || p.forcemth == 1.0 || p.forcemth == 3.0)) return MAGIC_EUNSUPPORTED;
    // substep counts: src3.f90:314-322
    double dmin = c->dx < c->dy ? c->dx : c->dy;
    dmin = dmin < c->dz ? dmin : c->dz;
    const double dxyzmin2 = dmin * dmin;
    const double difmax = (4.0 / 3.0) * c->aux11_top;
    const int ndtr = (int)std::ceil((dt * difmax / (dxyzmin2)) / 0.45);
    const double dtr = dt / ndtr;
    // no viscosity at the top: ndtr = 0 and the substep loop runs no pass
    // (src3.f90:341); the conduction count of an infinite dtr is then 0
    const int ndtrc = ndtr > 0 ? (int)std::ceil((dtr * c->aux12_top / (dxyzmin2)) / 0.45) : 0;
    const double dtrc = dtr / ndtrc;
    *ndtr_out = ndtr;
    *ndtrc_out = ndtrc;
    int mthbc[6];
    memcpy(mthbc, mthbc_in, sizeof(mthbc));
    mthbc[4] = -1;
    mthbc[5] = -1;
    Forcing f;
    f.forcemth = fm;
    f.t = t; f.dt = dt;
    f.xlower = c->xlower; f.ylower = c->ylower; f.zlower = c->zlower;
    f.dx = c->dx; f.dy = c->dy; f.dz = c->dz;
    f.amplitude = p.amplitude; f.xpos = p.xpos; f.ypos = p.ypos; f.zpos = p.zpos;
    f.xwidth = p.xwidth; f.ywidth = p.ywidth; f.zwidth = p.zwidth;
    f.tcenter = p.tcenter; f.twidth = p.twidth;
    f.omega = p.omega; f.propx = p.propx; f.propz = p.propz; f.vsrcx = p.vsrcx;
    f.tgauss = std::exp(-.5 * ((t - p.tcenter) * (t - p.tcenter) / (p.twidth * p.twidth)));
    if (c->form == MAGIC_FORM_FP32P) return src3_passes32(c, mthbc, ndtr, dtr, ndtrc, dtrc, f);
    return c->aux_layered ? src3_passes64<true>(c, mthbc, ndtr, dtr, ndtrc, dtrc, f)
                          : src3_passes64<false>(c, mthbc, ndtr, dtr, ndtrc, dtrc, f);
}

extern "C" int magic_src3(magic_ctx *c, double t, double dt, const int mthbc[6], int *ndtr, int *ndtrc)
{
    if (!c || !mthbc || !ndtr || !ndtrc || !c->have_aux || !c->have_params) return MAGIC_EARG;
    TRY(src3_launch(c, t, dt, mthbc, ndtr, ndtrc));
    HIPCHECK(hipStreamSynchronize(c->stream));
    if (c->timing) drain_timing(c);
    return MAGIC_OK;
}

// ------------------------------------------------------------ claw3 ------
// No source pass, or not the whole of one, ran behind a conversion: the state
// that it read is q again, the increments are still to be added, and its target
// is the backup.
static void take_back(magic_ctx *c)
{
    if (c->form == MAGIC_FORM_FP32P) std::swap(c->q32, c->qold32);
    else std::swap(c->q, c->qold);
    c->pending_parts = true;
}

extern "C" int magic_claw3(magic_ctx *c, double tstart, double *tend, double dtv[5], double cflv[4],
                           int nv[2], const int method[7], const int mthbc[6], double *log_dt,
                           double *log_cfl, int *log_acc, int maxlog, int *nlog)
{
    if (!c || !tend || !dtv || !cflv || !nv || !method || !mthbc) return MAGIC_EARG;
    if (!c->have_aux || !c->have_params) return MAGIC_EARG;
    if (method[0] != 1 || method[1] != 2 || method[2] != 22 || method[4] != 1 || method[5] != 0)
        return MAGIC_EUNSUPPORTED;
    if (cflv[1] > cflv[0]) return MAGIC_EARG;          // claw3_mpi.f:671-675
    double t = tstart, dt = dtv[0], cflmax = 0.0, dtmin = dt, dtmax = dt, cfl = 0.0;
    const int maxn = nv[0];
    int st = MAGIC_OK, nl = 0;
    nv[1] = 0;
    // With deferred increments the sweeps read q itself, which changes only in
    // an accepted step's source pass (into the other state buffer): the state
    // before the step needs no copy and a rejected step no restoring.  A
    // batch's grid keeps its buffers' places (its captured kernels hold them)
    // and takes the copying way.  A source pass of few launches is queued behind
    // the sweeps under their result's gate, and the host waits once per attempt.
    if (maxn > 0 && (st = setup_sweeps(c))) return st;
    const bool defer = sweeps_defer(c) && c->own_stream;
    for (int n = 1; n <= maxn; n++) {
        const double told = t;
        if (told + dt > *tend && tstart < *tend) dt = *tend - told;   // claw3_mpi.f:741
        for (;;) {
            if ((st = bc3_launch(c, mthbc, CLAMP_BC))) goto out;   // with b4step3
            if (!defer && (st = copy_state(c, true))) goto out;
            if ((st = step3_launch(c, dt, defer, defer))) goto out;
            int ss = MAGIC_OK, a, b;
            bool moved = false;   // the conversion's target is q already
            const bool ahead = defer && src_launches(c, dt) <= MAX_AHEAD;
            if (defer && !ahead && (st = scal_copy(c))) goto out;
            if (ahead) {
                const bool pending = c->pending_parts;
                c->gate = GridGate{c->dscal, c->hscal, cflv[0]};
                ss = src3_launch(c, told, dt, mthbc, &a, &b);   // claw3_mpi.f:900-905
                c->gate = GridGate{};
                moved = pending && !c->pending_parts;
                // a setting src3 refuses, before it launches anything: the step itself goes on
                if (ss && ss != MAGIC_EHIP && (st = scal_copy(c))) goto out;
            }
            st = ss == MAGIC_EHIP ? ss : step3_finish(c, &cfl);
            if (moved && (st || !(cfl <= cflv[0]))) take_back(c);
            if (st) goto out;
            t = told + dt;
            if (log_dt && nl < maxlog) {
                log_dt[nl] = dt;
                if (log_cfl) log_cfl[nl] = cfl;
                if (log_acc) log_acc[nl] = cfl <= cflv[0];
            }
            nl++;
            if (cfl <= cflv[0]) {                                  // claw3_mpi.f:861-886
                cflmax = cflmax > cfl ? cflmax : cfl;
                const bool pending = c->pending_parts;
                st = ahead ? ss : src3_launch(c, told, dt, mthbc, &a, &b);
                if (st && pending && !c->pending_parts) take_back(c);
                if (st) goto out;
                break;
            }
            t = told;
            c->pending_parts = false;   // the rejected step's increments are dropped with it
            if (!defer && (st = copy_state(c, false))) goto out;
            dt = dtv[1] < dt * cflv[1] / cfl ? dtv[1] : dt * cflv[1] / cfl;
        }
        if (cfl == 0.0) dt = dtv[1];                               // claw3_mpi.f:910-919
        else dt = dtv[1] < dt * cflv[1] / cfl ? dtv[1] : dt * cflv[1] / cfl;
        dtmin = dt < dtmin ? dt : dtmin;
        dtmax = dt > dtmax ? dt : dtmax;
        nv[1] = nv[1] + 1;
        if (t >= *tend) break;
    }
out:
    {
        // a step that stopped before its source pass still leaves its
        // increments in q and the state before it in the backup
        int sm = MAGIC_OK;
        if (c->pending_parts && (sm = copy_state(c, true)) == MAGIC_OK) sm = parts_flush(c);
        if (st == MAGIC_OK) st = sm;
    }
    hipStreamSynchronize(c->stream);
    if (c->timing) drain_timing(c);
    if (nlog) *nlog = nl < maxlog ? nl : maxlog;
    *tend = t;
    cflv[2] = cflmax;
    cflv[3] = cfl;
    dtv[2] = dtmin;
    dtv[3] = dtmax;
    dtv[4] = dt;
    return st;
}

extern "C" int magic_error_location(magic_ctx *c, int *sweep, int *i, int *j, int *k)
{
    if (!c) return MAGIC_EARG;
    if (sweep) *sweep = c->errloc[0];
    if (i) *i = c->errloc[1];
    if (j) *j = c->errloc[2];
    if (k) *k = c->errloc[3];
    return MAGIC_OK;
}

extern "C" int magic_timing_enable(magic_ctx *c, int on)
{
    if (!c) return MAGIC_EARG;
    hipStreamSynchronize(c->stream);
    drain_timing(c);
    c->timing = on != 0;
    return MAGIC_OK;
}

extern "C" int magic_timing_read(magic_ctx *c, double ms[6], long long launches[6])
{
    if (!c) return MAGIC_EARG;
    hipStreamSynchronize(c->stream);
    drain_timing(c);
    for (int k = 0; k < NTC; k++) {
        if (ms) ms[k] = c->ms[k];
        if (launches) launches[k] = c->launches[k];
    }
    return MAGIC_OK;
}

extern "C" int magic_timing_reset(magic_ctx *c)
{
    if (!c) return MAGIC_EARG;
    hipStreamSynchronize(c->stream);
    drain_timing(c);
    for (int k = 0; k < NTC; k++) {
        c->ms[k] = 0.0;
        c->launches[k] = 0;
    }
    return MAGIC_OK;
}
