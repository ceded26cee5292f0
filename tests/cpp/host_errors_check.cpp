// host_errors_check.cpp -- the host side of the HIP library on a stand-in for
// the HIP runtime: memory is host memory, kernels do not run, and a named call
// fails on demand.  The program's own HIP functions come before the runtime's
// when the library given on the command line is loaded, so nothing here needs
// or touches a GPU.  What the host paths do with an error, and which launches
// they issue on which device, is checked without making a GPU fail.
//
//   host_errors_check LIBRARY CASE
//
// Prints the first check that does not hold and returns 1, otherwise returns 0.
#include "../../include/sphx.h"

#include <hip/hip_runtime_api.h>

#include <dlfcn.h>

#include <cstdio>
#include <cstdlib>
#include <cstring>
#include <map>
#include <string>
#include <vector>

namespace
{
struct Stream
{
    int device;
};
int g_device = 0;            // the calling thread's current device
int g_sync_error = 0;        // stream synchronizations that fail from now on
int g_uploads = 0;           // host-to-device copies
int g_other_device = 0;      // launches on a stream of a device that is not current
int g_captures = 0;          // stream captures begun
unsigned long long g_needed = 0; // what the next read of a single device word returns
std::map<const void *, std::string> g_names;
std::map<std::string, int> g_launches; // kernel -> launches
std::string g_record;                  // of this kernel's last launch:
unsigned g_workgroups = 0;
dim3 g_grid, g_block;
size_t g_lds;
hipStream_t g_stream;

int launches(const char *kernel)
{
    int n = 0;
    for (const auto &k : g_launches)
        if (k.first.find(kernel) != std::string::npos)
            n += k.second;
    return n;
}
} // namespace

#define OK(...)                                                                                                  \
    {                                                                                                            \
        __VA_ARGS__;                                                                                             \
        return hipSuccess;                                                                                       \
    }
extern "C" {
void **__hipRegisterFatBinary(const void *) { return new void *(nullptr); }
void __hipUnregisterFatBinary(void **) {}
void __hipRegisterFunction(void **, const void *host, char *, const char *name, unsigned, void *, void *, dim3 *,
                           dim3 *, int *)
{
    g_names[host] = name;
}
void __hipRegisterVar(void **, void *, char *, const char *, int, size_t, int, int) {}
hipError_t __hipPushCallConfiguration(dim3 g, dim3 b, size_t lds, hipStream_t s)
    OK(g_grid = g; g_block = b; g_lds = lds; g_stream = s)
hipError_t __hipPopCallConfiguration(dim3 *g, dim3 *b, size_t *lds, hipStream_t *s)
    OK(*g = g_grid; *b = g_block; *lds = g_lds; *s = g_stream)
hipError_t hipLaunchKernel(const void *f, dim3 g, dim3, void **, size_t, hipStream_t s)
{
    if (g.x == 0)
        return hipErrorInvalidConfiguration;
    ++g_launches[g_names[f]];
    if (g_names[f].find(g_record) != std::string::npos)
        g_workgroups = g.x;
    if (((Stream *)s)->device != g_device)
        ++g_other_device;
    return hipSuccess;
}
hipError_t hipFuncSetAttribute(const void *, hipFuncAttribute, int) OK()
hipError_t hipGetLastError(void) OK()
const char *hipGetErrorString(hipError_t) { return "the stand-in's error"; }
hipError_t hipGetDeviceCount(int *n) OK(*n = 2)
hipError_t hipSetDevice(int d) OK(g_device = d)
hipError_t hipGetSymbolAddress(void **p, const void *) OK(*p = std::calloc(1, 64))
hipError_t hipMalloc(void **p, size_t n) OK(*p = std::calloc(1, n))
hipError_t hipFree(void *p) OK(std::free(p))
hipError_t hipHostMalloc(void **p, size_t n, unsigned) OK(*p = std::calloc(1, n))
hipError_t hipHostFree(void *p) OK(std::free(p))
hipError_t hipMemcpyAsync(void *d, const void *s, size_t n, hipMemcpyKind k, hipStream_t)
{
    std::memcpy(d, s, n);
    g_uploads += k == hipMemcpyHostToDevice;
    if (k == hipMemcpyDeviceToHost && n == sizeof(g_needed) && g_needed)
    {
        std::memcpy(d, &g_needed, n);
        g_needed = 0;
    }
    return hipSuccess;
}
hipError_t hipMemsetAsync(void *d, int v, size_t n, hipStream_t) OK(std::memset(d, v, n))
hipError_t hipStreamCreateWithFlags(hipStream_t *s, unsigned) OK(*s = (hipStream_t) new Stream{g_device})
hipError_t hipStreamDestroy(hipStream_t s) OK(delete (Stream *)s)
hipError_t hipStreamGetDevice(hipStream_t s, hipDevice_t *d) OK(*d = ((Stream *)s)->device)
hipError_t hipStreamSynchronize(hipStream_t) { return g_sync_error ? hipErrorLaunchFailure : hipSuccess; }
hipError_t hipEventCreate(hipEvent_t *e) OK(*e = (hipEvent_t)std::calloc(1, 8))
hipError_t hipEventCreateWithFlags(hipEvent_t *e, unsigned) OK(*e = (hipEvent_t)std::calloc(1, 8))
hipError_t hipEventDestroy(hipEvent_t e) OK(std::free(e))
hipError_t hipEventRecord(hipEvent_t, hipStream_t) OK()
hipError_t hipEventSynchronize(hipEvent_t) OK()
hipError_t hipEventElapsedTime(float *ms, hipEvent_t, hipEvent_t) OK(*ms = 1.0f)
hipError_t hipStreamBeginCapture(hipStream_t, hipStreamCaptureMode) OK(++g_captures)
hipError_t hipStreamEndCapture(hipStream_t, hipGraph_t *g) OK(*g = (hipGraph_t)std::calloc(1, 8))
hipError_t hipGraphInstantiate(hipGraphExec_t *e, hipGraph_t, hipGraphNode_t *, char *, size_t)
    OK(*e = (hipGraphExec_t)std::calloc(1, 8))
hipError_t hipGraphDestroy(hipGraph_t g) OK(std::free(g))
hipError_t hipGraphExecDestroy(hipGraphExec_t e) OK(std::free(e))
hipError_t hipGraphLaunch(hipGraphExec_t, hipStream_t) OK()
}

namespace
{
void *g_lib;
#define API(name) ((decltype(&name))dlsym(g_lib, #name))

#define REQUIRE(cond)                                                                                            \
    do                                                                                                           \
    {                                                                                                            \
        if (!(cond))                                                                                             \
        {                                                                                                        \
            std::printf("line %d: %s (%s)\n", __LINE__, #cond, API(sphx_last_error)());                          \
            std::exit(1);                                                                                        \
        }                                                                                                        \
    } while (0)

// a fluid body of n particles with its cell list and inner relation, built
struct Scene
{
    sphx_context *ctx = nullptr;
    sphx_body *body = nullptr;
    sphx_cell_linked_list *cll = nullptr;
    sphx_relation *inner = nullptr;

    Scene(int device, int dim, int precision, uint32_t n)
    {
        REQUIRE(API(sphx_context_create)(device, &ctx) == SPHX_OK);
        body = make_body(dim, precision, SPHX_BODY_FLUID, n);
        const double lo[3] = {0, 0, 0}, up[3] = {1, 1, 1};
        REQUIRE(API(sphx_cell_linked_list_create)(body, lo, up, 0.026, 2, &cll) == SPHX_OK);
        REQUIRE(API(sphx_relation_create_inner)(body, cll, &inner) == SPHX_OK);
        REQUIRE(API(sphx_update_cell_linked_list)(cll) == SPHX_OK);
        REQUIRE(API(sphx_update_relation)(inner) == SPHX_OK);
    }
    sphx_body *make_body(int dim, int precision, int kind, uint32_t n)
    {
        sphx_body_desc d{};
        d.dim = dim;
        d.precision = precision;
        d.kind = kind;
        d.n_particles = n;
        d.spacing_ref = 0.01;
        d.h_spacing_ratio = 1.3;
        d.rho0 = 1.0;
        d.c0 = 10.0;
        sphx_body *b = nullptr;
        REQUIRE(API(sphx_body_create)(ctx, &d, &b) == SPHX_OK);
        return b;
    }
};

// a large write whose kernels fail says so
void large_write()
{
    Scene s(0, 2, SPHX_FP64, 1000000);
    std::vector<double> v(1000000, 1.0);
    REQUIRE(API(sphx_body_write)(s.body, SPHX_FIELD_PRESSURE, v.data(), v.size()) == SPHX_OK);
    g_sync_error = 1;
    REQUIRE(API(sphx_body_write)(s.body, SPHX_FIELD_PRESSURE, v.data(), v.size()) == SPHX_E_HIP);
    g_sync_error = 0;
    REQUIRE(API(sphx_body_write)(s.body, SPHX_FIELD_PRESSURE, v.data(), v.size()) == SPHX_OK);
}

// A batch whose options are changed between two steps: an error of the staging
// sets that the new options ask for is the call's, and the next step makes the
// batch's tables anew instead of going on with half of them
void options_error()
{
    Scene s(0, 3, SPHX_MIXED, 5000);
    sphx_batch *batch = nullptr;
    sphx_advection_config cfg{1.0, 0.25, 0.6, SPHX_RIEMANN_ACOUSTIC, SPHX_FLOW_FREE_SURFACE, 0, 0, 0.0, 0};
    sphx_batch_options o{0, 0, 1, 1u << 30, 1};
    REQUIRE(API(sphx_batch_create)(0, &batch) == SPHX_OK);
    REQUIRE(API(sphx_batch_set_options)(batch, &o) == SPHX_OK);
    REQUIRE(API(sphx_batch_add_scene)(batch, s.inner, nullptr, 0, s.cll, &cfg) == SPHX_OK);
    double t = 0.0;
    for (int k = 0; k < 2; ++k)
    {
        g_uploads = 0;
        REQUIRE(API(sphx_batch_advection_step)(batch, &t, nullptr, nullptr, nullptr) == SPHX_OK);
    }
    REQUIRE(g_uploads == 2 && launches("kb_stage_sets") == 0); // times and sort flags
    o.stage_min = 0;
    g_sync_error = 1;
    REQUIRE(API(sphx_batch_set_options)(batch, &o) == SPHX_E_HIP);
    g_sync_error = 0;
    g_uploads = 0;
    REQUIRE(API(sphx_batch_advection_step)(batch, &t, nullptr, nullptr, nullptr) == SPHX_OK);
    REQUIRE(g_uploads > 2 && launches("kb_stage_sets") == 1);
    REQUIRE(API(sphx_batch_destroy)(batch) == SPHX_OK);
}

// Options changed by a thread whose current device is another than the batch's:
// the staging sets are made on the batch's
void options_device()
{
    Scene s(1, 3, SPHX_MIXED, 5000);
    sphx_batch *batch = nullptr;
    sphx_advection_config cfg{1.0, 0.25, 0.6, SPHX_RIEMANN_ACOUSTIC, SPHX_FLOW_FREE_SURFACE, 0, 0, 0.0, 0};
    sphx_batch_options o{0, 0, 1, 1u << 30, 1};
    REQUIRE(API(sphx_batch_create)(1, &batch) == SPHX_OK);
    REQUIRE(API(sphx_batch_set_options)(batch, &o) == SPHX_OK);
    REQUIRE(API(sphx_batch_add_scene)(batch, s.inner, nullptr, 0, s.cll, &cfg) == SPHX_OK);
    double t = 0.0;
    REQUIRE(API(sphx_batch_advection_step)(batch, &t, nullptr, nullptr, nullptr) == SPHX_OK);
    REQUIRE(g_other_device == 0);
    const int before = launches("k_stage_sets");
    o.stage_min = 0;
    g_device = 0;
    REQUIRE(API(sphx_batch_set_options)(batch, &o) == SPHX_OK);
    REQUIRE(launches("k_stage_sets") == before + 1 && g_other_device == 0);
    REQUIRE(API(sphx_batch_destroy)(batch) == SPHX_OK);
}

// A caller that rebuilds a scene's lists between two batch steps and finds more
// neighbours than before: the lists get new memory, and the next step's tables
// hold its address
void regrown_lists()
{
    Scene s(0, 3, SPHX_FP64, 5000);
    sphx_batch *batch = nullptr;
    sphx_advection_config cfg{1.0, 0.25, 0.6, SPHX_RIEMANN_ACOUSTIC, SPHX_FLOW_FREE_SURFACE, 0, 0, 0.0, 0};
    sphx_batch_options o{0, 0, 1, 0, 1};
    REQUIRE(API(sphx_batch_create)(0, &batch) == SPHX_OK);
    REQUIRE(API(sphx_batch_set_options)(batch, &o) == SPHX_OK);
    REQUIRE(API(sphx_batch_add_scene)(batch, s.inner, nullptr, 0, s.cll, &cfg) == SPHX_OK);
    double t = 0.0;
    REQUIRE(API(sphx_batch_advection_step)(batch, &t, nullptr, nullptr, nullptr) == SPHX_OK);
    REQUIRE(API(sphx_update_relation)(s.inner) == SPHX_OK); // as wide as before
    g_uploads = 0;
    REQUIRE(API(sphx_batch_advection_step)(batch, &t, nullptr, nullptr, nullptr) == SPHX_OK);
    REQUIRE(g_uploads == 2); // times and sort flags
    g_needed = 200;
    REQUIRE(API(sphx_update_relation)(s.inner) == SPHX_OK);
    REQUIRE(g_needed == 0);
    g_uploads = 0;
    REQUIRE(API(sphx_batch_advection_step)(batch, &t, nullptr, nullptr, nullptr) == SPHX_OK);
    REQUIRE(g_uploads == 5); // and the three tables
    REQUIRE(API(sphx_batch_destroy)(batch) == SPHX_OK);
}

// Each value of tile_waves is a build of its own: for the few chunks of this
// batch four waves on one chunk, or two or four chunks with one wave each
void tile_waves()
{
    const char *kernel[] = {"kb_relation_tileILi2ELi1ELi4E", "kb_relation_tileILi2ELi2ELi1E",
                            "kb_relation_tileILi2ELi4ELi1E"};
    for (int k = 0; k < 3; ++k)
    {
        Scene s(0, 2, SPHX_MIXED, 5000);
        sphx_batch *batch = nullptr;
        sphx_advection_config cfg{1.0, 0.25, 0.6, SPHX_RIEMANN_ACOUSTIC, SPHX_FLOW_FREE_SURFACE, 0, 0, 0.0, 0};
        sphx_batch_options o{0, 0, 1 << k, 0, 1};
        REQUIRE(API(sphx_batch_create)(0, &batch) == SPHX_OK);
        REQUIRE(API(sphx_batch_set_options)(batch, &o) == SPHX_OK);
        REQUIRE(API(sphx_batch_add_scene)(batch, s.inner, nullptr, 0, s.cll, &cfg) == SPHX_OK);
        double t = 0.0;
        g_launches.clear();
        REQUIRE(API(sphx_batch_advection_step)(batch, &t, nullptr, nullptr, nullptr) == SPHX_OK);
        REQUIRE(launches("kb_relation_tile") == 1 && launches(kernel[k]) == 1);
        REQUIRE(API(sphx_batch_destroy)(batch) == SPHX_OK);
    }
}

// a few observers take a workgroup each, many share one (their lists are laid
// out for a thread each)
void observers()
{
    Scene s(0, 3, SPHX_FP64, 1000);
    for (uint32_t n : {1u, 100u, 32768u, 32769u, 1000000u})
    {
        sphx_body *o = s.make_body(3, SPHX_FP64, SPHX_BODY_OBSERVER, n);
        sphx_relation *r = nullptr;
        REQUIRE(API(sphx_relation_create_contact)(o, s.body, s.cll, &r) == SPHX_OK);
        REQUIRE(API(sphx_update_relation)(r) == SPHX_OK);
        std::vector<double> v(n);
        g_record = "k_interpolate";
        REQUIRE(API(sphx_interpolate_contact)(r, SPHX_FIELD_PRESSURE, v.data(), n) == SPHX_OK);
        REQUIRE(g_workgroups == (n <= 32768 ? n : (n + 63) / 64));
    }
}

// a scalar or velocity field up to a size is copied as it lies, without a kernel,
// if no dynamics was launched since the last wait or it is of floats (over 64 KB)
void array_copies()
{
    for (int precision : {SPHX_FP64, SPHX_MIXED})
        for (uint32_t n : {100u, 10000u, 100000u, 500000u, 2000000u})
        {
            Scene s(0, 3, precision, n);
            REQUIRE(API(sphx_context_synchronize)(s.ctx) == SPHX_OK);
            std::vector<double> v(3 * (size_t)n, 1.0);
            std::vector<uint32_t> id(n, 7u);
            const bool floats = precision == SPHX_MIXED;
            const size_t real = floats ? 4 : 8;
            for (bool busy : {false, true})
                for (bool write : {true, false})
                {
                    auto copied = [&](int field, void *host) {
                        if (busy)
                            REQUIRE(API(sphx_advection_step_setup)(s.body) == SPHX_OK);
                        g_launches.clear();
                        REQUIRE((write ? API(sphx_body_write)(s.body, field, host, n)
                                       : API(sphx_body_read)(s.body, field, host, n)) == SPHX_OK);
                        return launches("k_field_") == 0;
                    };
                    auto expected = [&](size_t bytes, size_t most, bool is_float) {
                        return bytes * n <= most << 10 && (!busy || (is_float && bytes * n > 65536));
                    };
                    REQUIRE(copied(SPHX_FIELD_PRESSURE, v.data()) ==
                            expected(real, write ? 4096 : floats ? 2048 : 1024, floats));
                    REQUIRE(copied(SPHX_FIELD_ORIGINAL_ID, id.data()) == expected(4, write ? 4096 : 1024, false));
                    REQUIRE(copied(SPHX_FIELD_VELOCITY, v.data()) == expected(4 * real, floats ? 2048 : 256, floats));
                    REQUIRE(!copied(SPHX_FIELD_POSITION, v.data()));
                }
        }
}
} // namespace

int main(int argc, char **argv)
{
    const std::map<std::string, void (*)()> cases = {
        {"large_write", large_write}, {"options_error", options_error}, {"options_device", options_device},
        {"regrown_lists", regrown_lists}, {"tile_waves", tile_waves}, {"observers", observers},
        {"array_copies", array_copies}};
    if (argc != 3 || !cases.count(argv[2]) || !(g_lib = dlopen(argv[1], RTLD_NOW)))
    {
        std::printf("usage: %s LIBRARY CASE\n", argv[0]);
        return 2;
    }
    cases.at(argv[2])();
    return 0;
}
