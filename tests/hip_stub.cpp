// A HIP runtime without a device, preloaded by tests/test_host_control.py so
// that the library's host code (step control, allocation, error paths) runs on
// the CPU: device memory is host memory, streams are synchronous, kernels are
// looked up by name and do nothing but what the host's decisions hang on: the
// layout conversions of set_q and get_q, the reductions of a sweep (Courant
// numbers from a list the test sets), the mark that a source pass leaves in
// the state it writes, and the words that its last kernel hands to the host.
// A test can make the n-th launch of a kernel fail and bound device memory.
#include <cstdint>
#include <cstdlib>
#include <cstring>
#include <map>
#include <string>
#include <utility>
#include <vector>

namespace {
struct dim3 { uint32_t x, y, z; };
struct Config { dim3 g, b; size_t shared; void *stream; };
// Never destroyed: the library unregisters its kernels at the process's end
auto &names = *new std::map<const void *, std::string>;
auto &sizes = *new std::map<void *, size_t>;
auto &launched = *new std::vector<std::pair<std::string, dim3>>;
auto &courant = *new std::vector<double>;
auto &config = *new std::vector<Config>;
auto &log_text = *new std::string;
std::string fail_name;
int fail_after = -1, last_error = 0;
size_t room = ~size_t(0), used = 0, next_courant = 0;
double mark = 0.0;
uint64_t *scal = nullptr;

struct Gate { const uint64_t *scal; uint64_t *host; double limit; };   // GridGate (bc_src.h)
struct Dims { int mx, my, mz, mbc, NX, NY, NZ; long long P; };
double as_double(uint64_t v) { double d; memcpy(&d, &v, 8); return d; }
bool on(const Gate &g) { return !g.scal || (as_double(g.scal[0]) <= g.limit && *(const int *)(g.scal + 1) == 0); }

template <typename T>
void converted(void **a)   // k_src_convert<COL>(d, qin, q, aux, gate, sp)
{
    const Dims &d = *(const Dims *)a[0];
    T *q = *(T **)a[2];
    if (!on(*(const Gate *)a[4])) return;
    mark += 1.0;
    for (long long e = 0; e < 5 * d.P; e++) q[e] = (T)mark;
}
void run(const std::string &n, void **a)
{
    auto is = [&](const char *s) { return n.find(s) != std::string::npos; };
    if (is("k_aos_to_planes") || is("k_planes_to_aos")) {
        double *to = *(double **)a[0];
        const double *from = *(const double **)a[1];
        const long long P = *(const long long *)a[2];
        const int nc = *(const int *)a[3];
        for (long long c = 0; c < P; c++)
            for (int m = 0; m < nc; m++)
                if (is("k_aos")) to[m * P + c] = from[c * nc + m];
                else to[c * nc + m] = from[m * P + c];
    } else if (is("k_put_step_args")) {   // (slots, args, scal)
        if (!*(uint64_t **)a[2]) return;
        scal = *(uint64_t **)a[2];
        memset(scal, 0, 64);
        const double c = next_courant < courant.size() ? courant[next_courant++] : 0.5;
        memcpy(scal, &c, 8);
    } else if (is("13k_src_convert")) {
        converted<double>(a);
    } else if (is("k_src_finish")) {      // (d, q, t5, nc, aux, forcing, gate)
        const Gate &g = *(const Gate *)a[6];
        if (g.host) memcpy(g.host, g.scal, 64);
    }
}
}  // namespace

#pragma GCC visibility push(default)
extern "C" {
// ---- the test's side
void stub_courant(const double *c, int n) { courant.assign(c, c + n); next_courant = 0; }
void stub_fail(const char *name, int after) { fail_name = name; fail_after = after; }   // that many more succeed
void stub_room(size_t bytes) { room = bytes; }
size_t stub_used() { return used; }
void stub_clear() { launched.clear(); }
const char *stub_launches()   // "name gx gy gz" per launch (memory operations as names of their own)
{
    log_text.clear();
    for (auto &l : launched)
        log_text += l.first + " " + std::to_string(l.second.x) + " " + std::to_string(l.second.y) + " " + std::to_string(l.second.z) + "\n";
    return log_text.c_str();
}

// ---- the runtime's
void **__hipRegisterFatBinary(const void *) { static void *h; return &h; }
void __hipUnregisterFatBinary(void **) {}
void __hipRegisterFunction(void **, const void *f, char *, const char *name, unsigned, void *, void *, void *, void *, int *)
{
    names[f] = name;
}
void __hipRegisterVar(void **, void *, char *, char *, int, size_t, int, int) {}
int __hipPushCallConfiguration(dim3 g, dim3 b, size_t sh, void *s)
{
    config.push_back({g, b, sh, s});
    return 0;
}
int __hipPopCallConfiguration(dim3 *g, dim3 *b, size_t *sh, void **s)
{
    const Config c = config.back();
    config.pop_back();
    *g = c.g; *b = c.b; *sh = c.shared; *s = c.stream;
    return 0;
}
int hipLaunchKernel(const void *f, dim3 g, dim3, void **args, size_t, void *)
{
    const std::string &n = names[f];
    if (fail_after >= 0 && n.find(fail_name) != std::string::npos && fail_after-- == 0) return last_error = 719;
    launched.push_back({n, g});
    run(n, args);
    return 0;
}
int hipGetLastError() { const int e = last_error; last_error = 0; return e; }
const char *hipGetErrorString(int) { return "stub"; }
int hipGetDevice(int *d) { *d = 0; return 0; }
int hipDeviceGetAttribute(int *v, int, int) { *v = 256; return 0; }
int hipOccupancyMaxActiveBlocksPerMultiprocessor(int *n, const void *, int, size_t) { *n = 2; return 0; }
int hipMalloc(void **p, size_t n)
{
    if (used + n > room || !(*p = calloc(n ? n : 1, 1))) return last_error = 2;
    used += n;
    sizes[*p] = n;
    return 0;
}
int hipFree(void *p)
{
    if (!p) return 0;
    used -= sizes[p];
    sizes.erase(p);
    free(p);
    return 0;
}
int hipHostMalloc(void **p, size_t n, unsigned) { return (*p = calloc(n, 1)) ? 0 : 2; }
int hipHostFree(void *p) { free(p); return 0; }
int hipMemcpy(void *d, const void *s, size_t n, int) { memcpy(d, s, n); return 0; }
int hipMemcpyAsync(void *d, const void *s, size_t n, int kind, void *)
{
    if (kind == 3) launched.push_back({"copy", {0, 0, 0}});
    memcpy(d, s, n);
    return 0;
}
int hipMemsetAsync(void *d, int v, size_t n, void *) { memset(d, v, n); return 0; }
int hipStreamCreateWithFlags(void **s, unsigned) { *s = malloc(1); return 0; }
int hipStreamDestroy(void *s) { free(s); return 0; }
int hipStreamSynchronize(void *) { return 0; }
int hipStreamWaitEvent(void *, void *, unsigned) { launched.push_back({"wait", {0, 0, 0}}); return 0; }
int hipEventCreate(void **e) { *e = malloc(1); return 0; }
int hipEventCreateWithFlags(void **e, unsigned) { *e = malloc(1); return 0; }
int hipEventDestroy(void *e) { free(e); return 0; }
int hipEventRecord(void *, void *) { return 0; }
int hipEventSynchronize(void *) { return 0; }
int hipEventElapsedTime(float *ms, void *, void *) { *ms = 1.f; return 0; }
int hipGetSymbolAddress(void **, const void *) { return 1; }
int hipStreamBeginCapture(void *, int) { return 0; }
int hipStreamEndCapture(void *, void **g) { *g = malloc(1); return 0; }
int hipGraphInstantiate(void **e, void *, void **, char *, size_t) { *e = malloc(1); return 0; }
int hipGraphDestroy(void *g) { free(g); return 0; }
int hipGraphExecDestroy(void *e) { free(e); return 0; }
int hipGraphLaunch(void *, void *) { return 0; }
}
#pragma GCC visibility pop
