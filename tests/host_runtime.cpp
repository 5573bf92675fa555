// The engine's and the batch's host code (engine.cpp, batch.cpp,
// host_model.cpp) on a stand-in for the HIP runtime: device memory is host
// memory, streams and events only keep track of what has been waited for, and
// no kernel runs (an evolution launch reports a stop at its first generation).
// Allocations and launches are counted and can be made to fail, so that what
// the host does when they do can be checked without a device.
//
// Usage: host_runtime SCENARIO; prints what was wrong and exits with 1.
#include <hip/hip_runtime_api.h>

#include <cstdint>
#include <cstdio>
#include <cstdlib>
#include <cstring>
#include <map>
#include <new>
#include <set>
#include <string>
#include <vector>

#include "batch_kernels.hpp"
#include "deac_engine.h"
#include "init_kernels.hpp"
#include "kernels.hpp"
#include "pack_kernels.hpp"
#include "precision_kernels.hpp"
#include "split_kernels.hpp"

// ---------------------------------------------------------------- runtime

namespace {

struct Stream {
    bool pending = false;        // work that nothing has waited for
    std::set<Stream *> behind;   // streams whose work this one waits for
};
struct Event {
    std::set<Stream *> covers;
};

std::map<void *, size_t> live;   // device allocations
size_t live_bytes = 0;
long fail_malloc = 0;            // the n-th allocation from now on fails (1: the next), 0: none
long fail_launch = 0;            // likewise the launches
std::map<void *, unsigned> pinned;
std::set<Stream *> streams;
size_t host_largest = 0;         // largest single host allocation so far
long fail_new = 0;               // the n-th host allocation of the code under test fails, 0: none
thread_local int inside = 0;     // in the stand-in, whose own allocations do not count
struct Inside {
    Inside() { inside++; }
    ~Inside() { inside--; }
};

Stream *stream_of(hipStream_t s) { return reinterpret_cast<Stream *>(s); }
Event *event_of(hipEvent_t e) { return reinterpret_cast<Event *>(e); }

hipError_t last_error = hipSuccess;

hipError_t take_last_error()
{
    const hipError_t e = last_error;
    last_error = hipSuccess;
    return e;
}

// The launchers return the runtime's last error, whichever call left it.
hipError_t launch(hipStream_t s)
{
    if (last_error != hipSuccess) return take_last_error();
    if (fail_launch > 0 && --fail_launch == 0) return hipErrorLaunchFailure;
    if (s) stream_of(s)->pending = true;
    return hipSuccess;
}

bool anything_in_flight()
{
    for (Stream *s : streams)
        if (s->pending) return true;
    return false;
}

}  // namespace

void *operator new(size_t n)
{
    if (!inside) {
        if (n > host_largest) host_largest = n;
        if (fail_new > 0 && --fail_new == 0) throw std::bad_alloc();
    }
    if (void *p = std::malloc(n ? n : 1)) return p;
    throw std::bad_alloc();
}
void operator delete(void *p) noexcept { std::free(p); }
void operator delete(void *p, size_t) noexcept { std::free(p); }

extern "C" {
hipError_t hipGetDeviceCount(int *n) { return *n = 1, hipSuccess; }
hipError_t hipGetDevice(int *d) { return *d = 0, hipSuccess; }
hipError_t hipSetDevice(int) { return hipSuccess; }
hipError_t hipGetLastError() { return take_last_error(); }
hipError_t hipGetDeviceProperties(hipDeviceProp_t *p, int)
{
    *p = hipDeviceProp_t{};
    std::strcpy(p->gcnArchName, "gfx950:sramecc+:xnack-");
    p->multiProcessorCount = 256;
    return hipSuccess;
}
hipError_t hipMalloc(void **p, size_t n)
{
    const Inside own;
    if (fail_malloc > 0 && --fail_malloc == 0) return last_error = hipErrorOutOfMemory;
    if (!(*p = std::calloc(n, 1))) return hipErrorOutOfMemory;
    live[*p] = n;
    live_bytes += n;
    return hipSuccess;
}
hipError_t hipFree(void *p)
{
    if (!p) return hipSuccess;
    auto it = live.find(p);
    if (it == live.end()) return hipErrorInvalidValue;
    live_bytes -= it->second;
    live.erase(it);
    std::free(p);
    return hipSuccess;
}
hipError_t hipHostMalloc(void **p, size_t n, unsigned flags)
{
    const Inside own;
    *p = std::calloc(n, 1);
    pinned[*p] = flags;
    return hipSuccess;
}
hipError_t hipHostFree(void *p)
{
    pinned.erase(p);
    std::free(p);
    return hipSuccess;
}
hipError_t hipMemcpy(void *d, const void *s, size_t n, hipMemcpyKind) { return std::memcpy(d, s, n), hipSuccess; }
hipError_t hipMemcpyAsync(void *d, const void *s, size_t n, hipMemcpyKind, hipStream_t)
{
    return std::memcpy(d, s, n), hipSuccess;
}
hipError_t hipMemsetAsync(void *d, int v, size_t n, hipStream_t) { return std::memset(d, v, n), hipSuccess; }
hipError_t hipStreamCreateWithFlags(hipStream_t *s, unsigned)
{
    const Inside own;
    Stream *n = new Stream;
    streams.insert(n);
    *s = reinterpret_cast<hipStream_t>(n);
    return hipSuccess;
}
hipError_t hipStreamDestroy(hipStream_t s)
{
    streams.erase(stream_of(s));
    delete stream_of(s);
    return hipSuccess;
}
hipError_t hipStreamSynchronize(hipStream_t s)
{
    for (Stream *b : stream_of(s)->behind) b->pending = false;
    stream_of(s)->pending = false;
    return hipSuccess;
}
hipError_t hipStreamWaitEvent(hipStream_t s, hipEvent_t e, unsigned)
{
    const Inside own;
    for (Stream *b : event_of(e)->covers) stream_of(s)->behind.insert(b);
    return hipSuccess;
}
hipError_t hipEventCreateWithFlags(hipEvent_t *e, unsigned)
{
    const Inside own;
    *e = reinterpret_cast<hipEvent_t>(new Event);
    return hipSuccess;
}
hipError_t hipEventCreate(hipEvent_t *e) { return hipEventCreateWithFlags(e, 0); }
hipError_t hipEventDestroy(hipEvent_t e) { return delete event_of(e), hipSuccess; }
hipError_t hipEventRecord(hipEvent_t e, hipStream_t s)
{
    const Inside own;
    event_of(e)->covers = stream_of(s)->behind;
    event_of(e)->covers.insert(stream_of(s));
    return hipSuccess;
}
hipError_t hipEventSynchronize(hipEvent_t e)
{
    for (Stream *b : event_of(e)->covers) b->pending = false;
    return hipSuccess;
}
hipError_t hipEventElapsedTime(float *ms, hipEvent_t, hipEvent_t) { return *ms = 0.0f, hipSuccess; }
hipError_t hipStreamBeginCapture(hipStream_t, hipStreamCaptureMode) { return hipErrorNotSupported; }
hipError_t hipStreamEndCapture(hipStream_t, hipGraph_t *) { return hipErrorNotSupported; }
hipError_t hipGraphInstantiate(hipGraphExec_t *, hipGraph_t, hipGraphNode_t *, char *, size_t)
{
    return hipErrorNotSupported;
}
hipError_t hipGraphDestroy(hipGraph_t) { return hipSuccess; }
hipError_t hipGraphExecDestroy(hipGraphExec_t) { return hipSuccess; }
hipError_t hipGraphLaunch(hipGraphExec_t, hipStream_t) { return hipErrorNotSupported; }
}

// ---------------------------------------------------------------- kernels

namespace deac {

hipError_t launch_walk(const WalkArgs &, hipStream_t s) { return launch(s); }
hipError_t launch_mask(const MaskArgs &, const WalkArgs &, hipStream_t s) { return launch(s); }
hipError_t launch_ktile(const double *, double *, int, int, int, int, hipStream_t s) { return launch(s); }
hipError_t launch_evolve(const EvoArgs &a, const WalkArgs &, const MaskArgs &, hipStream_t s, hipEvent_t, hipEvent_t stop)
{
    if (a.ngen > 0) a.host_status[0] = 1;
    const hipError_t e = launch(s);
    if (stop) (void)hipEventRecord(stop, s);
    return e;
}
hipError_t launch_zero_u32(unsigned *, size_t, hipStream_t s) { return launch(s); }
int evolve_max_workgroups(int) { return 256; }

hipError_t launch_lane_tables(const LaneTabArgs &, int, hipStream_t s) { return launch(s); }
hipError_t launch_initial_population(const InitArgs &, hipStream_t s) { return launch(s); }
hipError_t launch_gather_best(const long *, size_t, const double *, int, const double *, double *, hipStream_t s)
{
    return launch(s);
}

hipError_t launch_pack_fp64(const PackArgs &, double, double *, hipStream_t s) { return launch(s); }
hipError_t launch_pack_fp32(const PackArgs &, float *, hipStream_t s) { return launch(s); }
hipError_t launch_pack_bf16x3(const PackArgs &, void *, void *, hipStream_t s) { return launch(s); }
hipError_t launch_pack_fp32_units(const PackArgs &, float *, hipStream_t s) { return launch(s); }
hipError_t launch_pack_transposed(const PackArgs &, int, int, double *, hipStream_t s) { return launch(s); }

hipError_t launch_split_trial(const EvoArgs &, int, int, void *, void *, int, hipStream_t s) { return launch(s); }
hipError_t launch_split_renorm(const EvoArgs &, hipStream_t s) { return launch(s); }
hipError_t launch_split_pack_fp64(const EvoArgs &, int, double *, int, int, hipStream_t s) { return launch(s); }
hipError_t launch_split_pack_fp32(const EvoArgs &, int, float *, int, int, hipStream_t s) { return launch(s); }
hipError_t launch_split_pack_bf16x3(const EvoArgs &, int, void *, void *, int, int, hipStream_t s) { return launch(s); }
hipError_t launch_split_fold(const EvoArgs &, hipStream_t s) { return launch(s); }
hipError_t launch_split_moments(const EvoArgs &, int, hipStream_t s) { return launch(s); }
hipError_t launch_split_select(const EvoArgs &, int, int, hipStream_t s) { return launch(s); }
hipError_t launch_split_model_select(const EvoArgs &, int, int, const float *, int, int, int, const int *, hipStream_t s)
{
    return launch(s);
}
hipError_t launch_split_iter(long *, long, hipStream_t s) { return launch(s); }
hipError_t launch_ks_fp64(const double *, const double *, double *, int, int, int, int, int, hipStream_t s, hipEvent_t,
                          hipEvent_t, const int *)
{
    return launch(s);
}
hipError_t launch_ks_fp32(const float *, const float *, float *, int, int, int, int, int, hipStream_t s, hipEvent_t,
                          hipEvent_t, const int *)
{
    return launch(s);
}
hipError_t launch_ks_bf16x3(const void *, const void *, const void *, const void *, float *, int, int, int, int, int,
                            hipStream_t s, hipEvent_t, hipEvent_t, const int *)
{
    return launch(s);
}

hipError_t launch_reduce_slices(const float *, float *, int, size_t, hipStream_t s, hipEvent_t, hipEvent_t)
{
    return launch(s);
}

static hipError_t batch_launch(const BatchDesc *d, int count, hipStream_t s)
{
    for (int i = 0; i < count; i++)
        for (int q = 0; q < d[i].Q && d[i].mode == 0; q++) {
            d[i].status[q][0] = 1;
            d[i].status[q][1] = d[i].gen0;
        }
    return launch(s);
}
hipError_t launch_batch(const BatchDesc *d, int n, int, int, int, hipStream_t s) { return batch_launch(d, n, s); }
hipError_t launch_batch_fold(const BatchDesc *d, int n, int, int, hipStream_t s) { return batch_launch(d, n, s); }
hipError_t launch_batch_mixed(const BatchDesc *d, int n, int, int, int, int, hipStream_t s)
{
    return batch_launch(d, n, s);
}
int batch_mixed_nq(int ntm, int) { return ntm <= 9 ? 9 : 0; }
hipError_t batch_scratch(int, double **p)
{
    const Inside own;
    static std::vector<double> scratch(kBatchScratchDoubles);
    return *p = scratch.data(), hipSuccess;
}
hipError_t batch_role_cycles_fp64(unsigned long long *, int) { return hipErrorNotSupported; }
hipError_t batch_role_cycles_mixed(unsigned long long *, int) { return hipErrorNotSupported; }

}  // namespace deac

// ---------------------------------------------------------------- scenarios

namespace {

int wrong = 0;
void expect(bool ok, const std::string &what)
{
    if (ok) return;
    std::printf("%s\n", what.c_str());
    wrong = 1;
}

struct Problem {
    std::vector<double> tau, isf, err, freq;
    deac_problem p{};
    Problem(size_t T, size_t G) : tau(T), isf(T), err(T), freq(G)
    {
        for (size_t t = 0; t < T; t++) {
            tau[t] = 0.37 * static_cast<double>(t) / static_cast<double>(T - 1);
            isf[t] = 1.0 - 0.5 * tau[t];
            err[t] = 0.01 * isf[t];
        }
        (void)deac_frequency_grid(G, 48.0, freq.data());
        p.number_of_timeslices = T;
        p.imaginary_time = tau.data();
        p.isf = isf.data();
        p.isf_error = err.data();
        p.genome_size = G;
        p.frequency = freq.data();
        p.temperature = 1.35;
        p.spectra_type = DEAC_BFULL;
        p.population_size = 8;
        p.first_moment = p.third_moment = -1.0;
        p.crossover_probability = p.differential_weight = 0.9;
        p.self_adapting_crossover_probability = p.self_adapting_differential_weight_probability = 0.1;
    }
};

// The kernel writes the status into pinned memory that the host reads after
// the dispatch's own event: memory that neither side may hold in a cache.
void status_memory()
{
    Problem q(9, 32);
    deac_handle *h = nullptr;
    expect(deac_create(&q.p, &h, nullptr) == DEAC_OK, "deac_create failed");
    expect(pinned.size() == 1, "one pinned allocation expected");
    for (auto &[ptr, flags] : pinned)
        expect((flags & hipHostMallocCoherent) != 0, "the status memory is not asked for as coherent");
    deac_destroy(h);
    expect(live.empty(), "device memory left after deac_destroy");
}

// A batch of n instances of one problem, and their outputs.
struct Batch {
    Problem q;
    deac_batch *h = nullptr;
    std::vector<uint64_t> rng;
    std::vector<deac_run_options> o;
    std::vector<deac_result> r;
    std::vector<std::vector<double>> out;
    Batch(size_t n, size_t T, size_t G, size_t generations) : q(T, G), rng(4 * n), o(n), r(n), out(5 * n)
    {
        const std::vector<deac_problem> p(n, q.p);
        expect(deac_batch_create(p.data(), n, &h, nullptr) == DEAC_OK, "deac_batch_create failed");
        const size_t len = deac_output_length(&q.p);
        for (size_t i = 0; i < n; i++) {
            deac_seed_state(i, &rng[4 * i]);
            o[i].number_of_generations = generations;
            o[i].track_stats = 1;
            for (int k = 0; k < 5; k++) out[5 * i + k].resize(k < 2 ? len : generations);
            r[i].dsf = out[5 * i].data();
            r[i].frequency = out[5 * i + 1].data();
            r[i].stats_mean = out[5 * i + 2].data();
            r[i].stats_minimum = out[5 * i + 3].data();
            r[i].stats_squared_mean = out[5 * i + 4].data();
        }
    }
    ~Batch() { deac_batch_destroy(h); }
    deac_status run() { return deac_batch_run(h, rng.data(), o.data(), r.data()); }
};

// Calls f with its first, second, ... host allocation failing until it gets by:
// every failure is a status, and leaves no more device memory than before.
template <class F>
void each_host_allocation(const char *what, F f)
{
    const size_t before = live_bytes;
    for (long k = 1; k < 100000; k++) {
        fail_new = k;
        deac_status st = DEAC_OK;
        bool thrown = false;
        try {
            st = f();
        } catch (...) {
            thrown = true;
        }
        const bool failed = fail_new == 0;
        fail_new = 0;
        expect(!thrown, std::string(what) + ": an exception left the entry point at allocation " + std::to_string(k));
        if (!failed) return expect(st == DEAC_OK, std::string(what) + ": fails by itself");
        // (a thread that cannot be started is done without)
        expect(st == DEAC_OK || st == DEAC_ERR_OUT_OF_MEMORY, std::string(what) + ": another status");
        if (st != DEAC_OK) expect(live_bytes <= before, std::string(what) + ": device memory left behind");
        if (wrong) return;
    }
    expect(false, std::string(what) + ": never got by");
}

void host_memory_runs_out()
{
    Problem q(20, 2048);  // its kernel matrix is built on two threads
    {
        deac_handle *h = nullptr;
        each_host_allocation("deac_create", [&] {
            deac_destroy(h);
            h = nullptr;
            return deac_create(&q.p, &h, nullptr);
        });
        const size_t len = deac_output_length(&q.p);
        std::vector<double> dsf(len), freq(len), mean(100);
        deac_result r{};
        r.dsf = dsf.data();
        r.frequency = freq.data();
        r.stats_mean = mean.data();
        for (int precision : {DEAC_PRECISION_FP64, DEAC_PRECISION_FP32}) {
            deac_run_options o{};
            o.number_of_generations = 100;
            o.track_stats = 1;
            o.ks_precision = precision;
            uint64_t first[4], rng[4];
            deac_seed_state(1, first);
            // (what a handle keeps is there before)
            std::memcpy(rng, first, sizeof rng);
            expect(deac_run(h, rng, &o, &r) == DEAC_OK, "deac_run failed");
            bool moved = false;
            each_host_allocation("deac_run", [&] {
                std::memcpy(rng, first, sizeof rng);
                const deac_status st = deac_run(h, rng, &o, &r);
                moved |= st != DEAC_OK && std::memcmp(rng, first, sizeof rng) != 0;
                return st;
            });
            expect(!moved, "deac_run: the random state of a run that failed has moved on");
        }
        deac_destroy(h);
    }
    each_host_allocation("deac_batch_create", [&] {
        deac_batch *h = nullptr;
        const deac_status st = deac_batch_create(&q.p, 1, &h, nullptr);
        deac_batch_destroy(h);
        return st;
    });
    {
        Batch b(3, 9, 64, 50);
        expect(b.run() == DEAC_OK, "deac_batch_run failed");
        each_host_allocation("deac_batch_run", [&] { return b.run(); });
        each_host_allocation("deac_batch_continue",
                             [&] {
                                 const long k = fail_new;
                                 fail_new = 0;
                                 (void)b.run();
                                 fail_new = k;
                                 return deac_batch_continue(b.h, b.rng.data(), b.o.data(), b.r.data());
                             });
        each_host_allocation("deac_batch_run_noalloc",
                             [&] { return deac_batch_run_noalloc(b.h, b.rng.data(), b.o.data(), b.r.data()); });
        each_host_allocation("deac_batch_tune",
                             [&] { return deac_batch_tune(b.h, b.rng.data(), b.o.data(), 10, nullptr); });
    }
    std::vector<double> genomes(5 * deac_genome_length(&q.p)), chi2(5);
    for (int precision : {DEAC_PRECISION_FP64, DEAC_PRECISION_FP32, DEAC_PRECISION_BF16X3})
        each_host_allocation("deac_model_isf", [&] {
            return deac_model_isf(&q.p, genomes.data(), 5, precision, nullptr, chi2.data(), nullptr, nullptr);
        });
    expect(live.empty(), "device memory left");
}

// A launch that fails in the middle of a run: nothing of the run is in flight when
// its status comes back, on whichever stream, and the next run is sound.
void launches_fail()
{
    Problem q[4] = {{9, 64}, {20, 64}, {40, 64}, {70, 64}};  // four kernel shapes
    std::vector<deac_problem> p;
    for (Problem &x : q) p.push_back(x.p);
    deac_batch *h = nullptr;
    expect(deac_batch_create(p.data(), p.size(), &h, nullptr) == DEAC_OK, "deac_batch_create failed");
    std::vector<double> out(8 * 127);
    std::vector<deac_run_options> o(4);
    std::vector<deac_result> r(4);
    std::vector<uint64_t> rng(16);
    for (size_t i = 0; i < 4; i++) {
        o[i].number_of_generations = 20;
        r[i].dsf = &out[2 * i * 127];
        r[i].frequency = r[i].dsf + 127;
    }
    for (int precision : {DEAC_PRECISION_FP64, DEAC_PRECISION_FP32})
        for (long k = 1;; k++) {
            for (size_t i = 0; i < 4; i++) {
                o[i].ks_precision = precision;
                deac_seed_state(i, &rng[4 * i]);
            }
            fail_launch = k;
            const deac_status st = deac_batch_run(h, rng.data(), o.data(), r.data());
            const bool failed = fail_launch == 0;
            fail_launch = 0;
            expect(!anything_in_flight(), "launch " + std::to_string(k) + " fails: work is left in flight");
            expect(st == (failed ? DEAC_ERR_DEVICE : DEAC_OK), "launch " + std::to_string(k) + ": another status");
            if (!failed) {
                expect(k > 8, "fewer launches than shapes");
                break;
            }
        }
    deac_batch_destroy(h);
}

// A first mixed-precision run for whose tiles the device memory does not last, or
// whose packing fails: each retry leaves as much as there was before.
void device_memory_runs_out()
{
    {
        Problem q(9, 64);
        for (long k = 1;; k++) {
            deac_handle *h = nullptr;
            fail_malloc = k;
            const deac_status st = deac_create(&q.p, &h, nullptr);
            const bool failed = fail_malloc == 0;
            fail_malloc = 0;
            expect(st == (failed ? DEAC_ERR_OUT_OF_MEMORY : DEAC_OK), "deac_create: another status");
            deac_destroy(h);
            expect(live.empty(), "deac_create: device memory left");
            h = nullptr;
            expect(deac_create(&q.p, &h, nullptr) == DEAC_OK, "no deac_create behind a failed allocation");
            deac_destroy(h);
            if (!failed) break;
        }
        deac_handle *h = nullptr;
        expect(deac_create(&q.p, &h, nullptr) == DEAC_OK, "deac_create failed");
        std::vector<double> out(2 * deac_output_length(&q.p));
        deac_run_options o{};
        o.number_of_generations = 50;
        o.track_stats = 1;
        deac_result r{};
        r.dsf = out.data();
        r.frequency = out.data() + out.size() / 2;
        for (int precision : {DEAC_PRECISION_FP64, DEAC_PRECISION_FP32, DEAC_PRECISION_BF16X3})
            for (long k = 1;; k++) {
                uint64_t rng[4];
                deac_seed_state(1, rng);
                o.ks_precision = precision;
                o.number_of_generations += 1;  // (longer statistics than there are)
                fail_malloc = k;
                const deac_status st = deac_run(h, rng, &o, &r);
                const bool failed = fail_malloc == 0;
                fail_malloc = 0;
                expect(st == (failed ? DEAC_ERR_OUT_OF_MEMORY : DEAC_OK), "deac_run: another status");
                deac_seed_state(1, rng);
                expect(deac_run(h, rng, &o, &r) == DEAC_OK, "no deac_run behind a failed allocation");
                if (!failed) break;
                if (precision != DEAC_PRECISION_FP64) {  // another precision's operands again
                    o.ks_precision = precision ^ 3;
                    deac_seed_state(1, rng);
                    expect(deac_run(h, rng, &o, &r) == DEAC_OK, "deac_run failed");
                }
            }
        deac_destroy(h);
    }
    for (int precision : {DEAC_PRECISION_FP32, DEAC_PRECISION_BF16X3})
        for (long *fail : {&fail_malloc, &fail_launch})
            for (long k = 1;; k++) {
                Batch b(1, 9, 64, 20);
                b.o[0].ks_precision = precision;
                const size_t before = live_bytes;
                bool failed = true;
                for (int retry = 0; retry < 3 && failed; retry++) {
                    *fail = k;
                    const deac_status st = b.run();
                    failed = *fail == 0;
                    *fail = 0;
                    expect(st == (!failed ? DEAC_OK : fail == &fail_malloc ? DEAC_ERR_OUT_OF_MEMORY : DEAC_ERR_DEVICE),
                           "failure " + std::to_string(k) + ": another status");
                    // (the run's own workspaces may come after its tiles)
                    if (failed && k == 1) expect(live_bytes == before, "a retry leaves device memory behind");
                    if (failed && fail == &fail_malloc && k <= 3)
                        expect(live_bytes == before, "a retry at allocation " + std::to_string(k) + " leaves " +
                                                         std::to_string(live_bytes - before) + " bytes behind");
                }
                expect(b.run() == DEAC_OK, "no run behind the failures");
                if (!failed) break;
            }
    expect(live.empty(), "device memory left");
}

// Long histories: neither the host nor the device keeps all instances' at once
// behind a run, and a long genome's best rows come back in pieces.
void long_histories()
{
    constexpr size_t kMuch = size_t(48) << 20;
    {
        Batch b(24, 9, 32, 1000000);  // 24 MB each, three histories
        const size_t before = live_bytes;
        host_largest = 0;
        expect(b.run() == DEAC_OK, "deac_batch_run failed");
        expect(host_largest < kMuch, "batch: one host allocation of " + std::to_string(host_largest) + " bytes");
        expect(live_bytes == before, "batch: " + std::to_string(live_bytes - before) + " bytes of device memory kept");
    }
    {
        Batch b(400, 3, 16384, 10);  // 105 MB of best rows
        host_largest = 0;
        expect(b.run() == DEAC_OK, "deac_batch_run failed");
        expect(host_largest < kMuch, "rows: one host allocation of " + std::to_string(host_largest) + " bytes");
    }
    Problem q(9, 32);
    deac_handle *h = nullptr;
    expect(deac_create(&q.p, &h, nullptr) == DEAC_OK, "deac_create failed");
    const size_t before = live_bytes, len = deac_output_length(&q.p), N = 4000000;
    std::vector<double> dsf(len), freq(len), mean(N);
    deac_run_options o{};
    o.number_of_generations = N;
    o.track_stats = 1;
    deac_result r{};
    r.dsf = dsf.data();
    r.frequency = freq.data();
    r.stats_mean = mean.data();
    uint64_t rng[4];
    deac_seed_state(1, rng);
    host_largest = 0;
    expect(deac_run(h, rng, &o, &r) == DEAC_OK, "deac_run failed");
    expect(host_largest < kMuch, "engine: one host allocation of " + std::to_string(host_largest) + " bytes");
    expect(live_bytes == before, "engine: " + std::to_string(live_bytes - before) + " bytes of device memory kept");
    deac_destroy(h);
}

}  // namespace

int main(int argc, char **argv)
{
    const std::map<std::string, void (*)()> scenarios = {
        {"status_memory", status_memory},
        {"long_histories", long_histories},
        {"host_memory_runs_out", host_memory_runs_out},
        {"launches_fail", launches_fail},
        {"device_memory_runs_out", device_memory_runs_out},
    };
    auto it = argc == 2 ? scenarios.find(argv[1]) : scenarios.end();
    if (it == scenarios.end()) return std::printf("no such scenario\n"), 2;
    it->second();
    return wrong;
}
