// C ABI of the DEAC engine (include/deac_engine.h): device memory, uploads,
// the batch schedule of the RNG walk / mask / evolution kernels, and the
// host-side epilogue (best member, output transform, final statistics).
#include <hip/hip_runtime_api.h>

#include <algorithm>
#include <cstdlib>
#include <cmath>
#include <cstring>
#include <memory>
#include <string>
#include <vector>

#include "deac_engine.h"
#include "host_model.hpp"
#include "init_kernels.hpp"
#include "kernels.hpp"
#include "ks_layout.hpp"
#include "pack_kernels.hpp"
#include "precision_kernels.hpp"
#include "split_kernels.hpp"

namespace {


struct DeviceBuffer {
    void *ptr = nullptr;
    size_t bytes = 0;
};

}  // namespace

struct deac_handle {
    deac::Model m;
    int device = 0;
    hipStream_t stream = nullptr;       // evolution
    hipStream_t draw_stream = nullptr;  // RNG walk, batches ahead of the evolution
    int MG = 0, TB = 0, stride = 0, rstride = 0, nwg = 0, maxwg = 0, chunk = 0, batch = 0;
    bool fixed_nwg = false;             // the number of workgroups is the user's
    std::vector<void *> allocations;
    double *kmat = nullptr, *ktile = nullptr, *nterm = nullptr, *fterm = nullptr, *tterm = nullptr, *obs = nullptr, *sig = nullptr;
    double *nfm_dt = nullptr;           // -1st-moment weights over tau (bdsf), or null
    double *pop0 = nullptr, *pop1 = nullptr, *fitness = nullptr, *cr_old = nullptr, *f_old = nullptr;
    double *emod = nullptr, *mom = nullptr;
    int *cur = nullptr;
    // Two buffer sets, used by batches of even and odd index: grid barrier
    // counter ([0]) and status ([4..6]) per set, and the batch's mask draws.
    // Three sets of the walk's records, four of its generation starts (see
    // the generation loop).
    unsigned *sync = nullptr;           // [2][kSyncWords]
    long *iter = nullptr;               // [2][4]: split loop generation counters, per buffer set
    int *host_status = nullptr;         // [3][4], pinned: status of the sets, then of the initial fitness
    deac::MemberCtl *ctl[3] = {};
    uint64_t *raw[2] = {};
    uint64_t *gen_start[4] = {};
    uint64_t *state = nullptr, *skip_rows = nullptr, *lane_tab = nullptr;
    uint64_t *tab1 = nullptr, *tab2 = nullptr, *skip_tab_dev = nullptr;  // wide walk
    uint64_t *columns = nullptr;        // matrices the lane tables are made of
    bool wide = false;
    uint64_t *init_start = nullptr;     // [P][4]: random state at each member's first initial draw
    std::vector<uint64_t> skip_tab;     // nibble table of T^Kc, host side
    double *stats = nullptr;            // statistics histories, kept between runs up to kStatsKept
    size_t stats_cap = 0;
    hipEvent_t ev0 = nullptr, ev1 = nullptr;
    // per set: walk start, walk end, mask end (fused path: the first batch's
    // masks between the first two), evolve start, evolve end (draws free),
    // status copied (split loop)
    hipEvent_t kev[3][7] = {};
    deac_run_profile last{};
    // Split loop: contraction operands of the precision it last ran at.
    struct Split {
        int precision = -1;
        deac::KsLayout y;
        void *A = nullptr, *Al = nullptr;  // kernel matrix (BF16X3: hi, lo)
        void *B = nullptr, *Bl = nullptr;  // genome operand
        float *part = nullptr;             // FP32 genome slices
        int *ex = nullptr;                 // per-row exponents
    } split;

    ~deac_handle()
    {
        if (stream) (void)hipStreamSynchronize(stream);
        if (draw_stream) (void)hipStreamSynchronize(draw_stream);
        for (void *p : allocations) (void)hipFree(p);
        if (host_status) (void)hipHostFree(host_status);
        if (ev0) (void)hipEventDestroy(ev0);
        if (ev1) (void)hipEventDestroy(ev1);
        for (auto &set : kev)
            for (hipEvent_t e : set)
                if (e) (void)hipEventDestroy(e);
        if (stream) (void)hipStreamDestroy(stream);
        if (draw_stream) (void)hipStreamDestroy(draw_stream);
    }

    template <class T>
    deac_status alloc(T *&out, size_t count)
    {
        void *p = nullptr;
        allocations.push_back(nullptr);  // its place, before there is anything to lose
        if (hipMalloc(&p, std::max<size_t>(count, 1) * sizeof(T)) != hipSuccess) {
            (void)hipGetLastError();
            allocations.pop_back();
            return DEAC_ERR_OUT_OF_MEMORY;
        }
        allocations.back() = p;
        out = static_cast<T *>(p);
        return DEAC_OK;
    }

    void release(void *&p)
    {
        if (!p) return;
        allocations.erase(std::find(allocations.begin(), allocations.end(), p));
        (void)hipFree(p);
        p = nullptr;
    }
};

namespace {

#define DEAC_TRY(expr)                         \
    do {                                       \
        const deac_status st_ = (expr);        \
        if (st_ != DEAC_OK) return st_;        \
    } while (0)
#define DEAC_HIP(expr)                         \
    do {                                       \
        if ((expr) != hipSuccess) {            \
            (void)hipGetLastError();           \
            return DEAC_ERR_DEVICE;            \
        }                                      \
    } while (0)

int round_up(int x, int m) { return (x + m - 1) / m * m; }

// Contraction operands of the split loop at `precision` (kept until another
// precision is asked for): the kernel matrix in the contraction's lane order,
// the genome operand and slice buffers for the population.
deac_status prepare_split(deac_handle *h, int precision)
{
    deac_handle::Split &sp = h->split;
    if (sp.precision == precision) return DEAC_OK;
    for (void **p : {&sp.A, &sp.Al, &sp.B, &sp.Bl, reinterpret_cast<void **>(&sp.part),
                     reinterpret_cast<void **>(&sp.ex)})
        h->release(*p);
    sp.precision = -1;
    const deac::Model &m = h->m;
    sp.y = deac::ks_layout(m, precision, m.P);
    const deac::KsLayout &y = sp.y;
    if (precision != DEAC_PRECISION_FP64) {
        DEAC_TRY(h->alloc(sp.part, static_cast<size_t>(y.slices) * y.mpad() * y.npad()));
        DEAC_TRY(h->alloc(sp.ex, y.T));
        DEAC_HIP(hipMemcpy(sp.ex, y.ex.data(), y.T * sizeof(int), hipMemcpyHostToDevice));
    }
    // K padded with -0.0 at FP64 (with genomes padded with +0.0 the padded
    // products are -0.0 and leave every chain exactly as it is), 0 otherwise
    const deac::PackArgs pk{h->kmat, sp.ex, static_cast<int>(y.T), static_cast<int>(y.L), y.Mt, static_cast<int>(y.Kb)};
    if (precision == DEAC_PRECISION_FP64) {
        double *a = nullptr, *b = nullptr;
        DEAC_TRY(h->alloc(a, y.a_count()));
        sp.A = a;
        DEAC_TRY(h->alloc(b, y.b_count()));
        sp.B = b;
        DEAC_HIP(deac::launch_pack_fp64(pk, -0.0, a, h->stream));
    } else if (precision == DEAC_PRECISION_FP32) {
        float *a = nullptr, *b = nullptr;
        DEAC_TRY(h->alloc(a, y.a_count()));
        sp.A = a;
        DEAC_TRY(h->alloc(b, y.b_count()));
        sp.B = b;
        DEAC_HIP(deac::launch_pack_fp32(pk, a, h->stream));
    } else {
        uint16_t *ah = nullptr, *al = nullptr, *bh = nullptr, *bl = nullptr;
        DEAC_TRY(h->alloc(ah, y.a_count()));
        sp.A = ah;
        DEAC_TRY(h->alloc(al, y.a_count()));
        sp.Al = al;
        DEAC_TRY(h->alloc(bh, y.b_count()));
        sp.B = bh;
        DEAC_TRY(h->alloc(bl, y.b_count()));
        sp.Bl = bl;
        DEAC_HIP(deac::launch_pack_bf16x3(pk, ah, al, h->stream));
    }
    sp.precision = precision;
    return DEAC_OK;
}

}  // namespace

extern "C" {

const char *deac_status_string(deac_status s)
{
    switch (s) {
    case DEAC_OK: return "success";
    case DEAC_ERR_INVALID_ARGUMENT: return "invalid argument";
    case DEAC_ERR_NO_DEVICE: return "no usable gfx950 device";
    case DEAC_ERR_OUT_OF_MEMORY: return "out of memory";
    case DEAC_ERR_DEVICE: return "device error";
    case DEAC_ERR_UNSUPPORTED: return "unsupported";
    }
    return "unknown status";
}

const char *deac_last_error_message(void) { return deac::last_message().c_str(); }

size_t deac_output_length(const deac_problem *p)
{
    if (!p) return 0;
    return (p->zero_temperature || p->spectra_type == DEAC_BDSF) ? p->genome_size : 2 * p->genome_size - 1;
}

void deac_seed_state(uint64_t seed, uint64_t state[4]) { deac::seed_state(seed, state); }

void deac_rng_advance(uint64_t state[4], uint64_t n)
{
    const deac::Gf2Matrix m = deac::transition_power(n);
    uint64_t out[4];
    m.apply(state, out);
    std::memcpy(state, out, sizeof out);
}

deac_status deac_frequency_grid(size_t G, double omega_max, double *f)
{
    if (G < 2 || !f) return DEAC_ERR_INVALID_ARGUMENT;
    const double d = omega_max / static_cast<double>(G - 1);  // deac.cpp:2121-2125
    for (size_t i = 0; i < G; i++) f[i] = static_cast<double>(i) * d;
    return DEAC_OK;
}

deac_status deac_create(const deac_problem *p, deac_handle **out, const char **message)
try {
    if (message) *message = nullptr;
    if (!p || !out) return DEAC_ERR_INVALID_ARGUMENT;
    *out = nullptr;
    const deac_status v = deac::validate(*p, deac::last_message());
    if (v != DEAC_OK) {
        if (message) *message = deac::last_message().c_str();
        return v;
    }

    int device = 0, count = 0;
    if (hipGetDeviceCount(&count) != hipSuccess || count == 0) {
        (void)hipGetLastError();
        return DEAC_ERR_NO_DEVICE;
    }
    DEAC_HIP(hipGetDevice(&device));
    hipDeviceProp_t prop;
    DEAC_HIP(hipGetDeviceProperties(&prop, device));
    if (std::strncmp(prop.gcnArchName, "gfx950", 6) != 0) return DEAC_ERR_NO_DEVICE;

    std::unique_ptr<deac_handle> own(new deac_handle());
    deac_handle *const h = own.get();
    h->m = deac::build_model(*p);
    h->device = device;
    const deac::Model &m = h->m;
    if (hipStreamCreateWithFlags(&h->stream, hipStreamNonBlocking) != hipSuccess ||
        hipStreamCreateWithFlags(&h->draw_stream, hipStreamNonBlocking) != hipSuccess)
        return DEAC_ERR_DEVICE;
    if (hipEventCreate(&h->ev0) != hipSuccess || hipEventCreate(&h->ev1) != hipSuccess) return DEAC_ERR_DEVICE;
    for (auto &set : h->kev)
        for (hipEvent_t &e : set)
            if (hipEventCreate(&e) != hipSuccess) return DEAC_ERR_DEVICE;
    // coherent: kernels write it (EvoArgs::host_status), the host reads it after a dispatch's own event
    if (hipHostMalloc(reinterpret_cast<void **>(&h->host_status), 12 * sizeof(int), hipHostMallocCoherent) !=
        hipSuccess) {
        h->host_status = nullptr;
        return DEAC_ERR_OUT_OF_MEMORY;
    }

    const int T = static_cast<int>(m.T), P = static_cast<int>(m.P), Kc = static_cast<int>(m.Kc);
    h->MG = (P + deac::kChainRows - 1) / deac::kChainRows;
    h->TB = (T + deac::kChainTau - 1) / deac::kChainTau;
    h->stride = round_up(Kc, deac::kChunk);
    h->rstride = round_up(Kc, 2);
    h->wide = deac::walk_is_wide(P, m.tau_cr, m.tau_f);
    h->chunk = round_up((Kc + 63) / 64, 2);
    // RNG batch: generations whose mask draws are buffered at once: 64 MiB per
    // buffer set, so that the evolution finds both sets in the 256 MB cache in
    // front of HBM (G = 4096, T = 65: 8 members 67.8 -> 65.7 ms for 2000
    // generations, 32 members 25.4 -> 24.0 for 600, against 256 MiB), but at
    // least 16 generations where 256 MiB hold them (a batch's launches and first
    // draws; long genomes of large populations would have 2 to 4).
    const size_t per_gen = static_cast<size_t>(P) * h->rstride * sizeof(uint64_t);
    const size_t most = (size_t(256) << 20) / per_gen;
    h->batch = static_cast<int>(std::clamp<size_t>(std::max((size_t(64) << 20) / per_gen, std::min<size_t>(16, most)), 1, 1024));

    const int maxwg = deac::evolve_max_workgroups(device);
    if (maxwg <= 0) return DEAC_ERR_DEVICE;
    h->maxwg = maxwg;
    // One workgroup per chain task or moment fold, which share a CU's L1 and
    // matrix cores otherwise, more where there is a trial phase (not
    // EvoArgs::fed) with over 1024 pairs of positions for each.  With a first
    // moment, 17 timeslices, us per generation: 16 members of 16384 positions 68.1
    // with the rule's 128 workgroups, 68.1 with 64, 72.0 with 32, 69.7 with 248; 40
    // members of 8192 43.9 with its 160, 47.4 with 48, 45.9 with 248; 8 members 37.7
    // with its 32, 38.9 with 12, 40.2 with 248.
    // One CU per XCD stays free for the walk: workgroups go to the XCDs in
    // turn, and one that found its XCD full would hold up the grid barriers
    // until the walk ends.
    const size_t trial_pairs = static_cast<size_t>(P) * h->stride / 2;
    const size_t folds = static_cast<size_t>(P) * (m.use_first + m.use_third);
    size_t tasks = static_cast<size_t>(h->MG) * h->TB + folds;
    if (m.bdsf) {
        // folds draw less memory than chains: four to a CU, once 64 have a CU
        // of their own (32 members, 65 timeslices, 4096 positions: 42.7 us per
        // generation with 64 workgroups, 49.8 with 160)
        tasks = static_cast<size_t>(P) * h->TB + folds;
        tasks = std::max(std::min<size_t>(tasks, 64), tasks / 4);
    }
    size_t nwg = std::max(tasks, trial_pairs / 1024);
    if (m.normalize && m.renormalize) nwg = std::max<size_t>(nwg, P);  // a workgroup renormalizes a member at a time
    // (the number of workgroups given from outside: always with a trial phase)
    h->fixed_nwg = std::getenv("DEAC_EVOLVE_WORKGROUPS") != nullptr;
    if (const char *user = std::getenv("DEAC_EVOLVE_WORKGROUPS")) nwg = std::max(std::atoi(user), 1);
    h->nwg = static_cast<int>(std::clamp<size_t>(nwg, 1, std::max(maxwg - 8, 1)));

    // Device buffers.
    const size_t pop_n = static_cast<size_t>(h->MG) * deac::kChainRows * h->stride;
    deac_status st = DEAC_OK;
    auto A = [&](auto *&ptr, size_t n) {
        if (st == DEAC_OK) st = h->alloc(ptr, n);
    };
    A(h->kmat, m.T * m.Kc);
    A(h->ktile, deac::ktile_doubles(h->TB, h->stride));
    A(h->obs, T);
    A(h->sig, T);
    A(h->pop0, 2 * pop_n);
    if (st == DEAC_OK) h->pop1 = h->pop0 + pop_n;
    A(h->cur, P);
    A(h->fitness, P);
    A(h->cr_old, static_cast<size_t>(P) * m.nsign);
    A(h->f_old, static_cast<size_t>(P) * m.nsign);
    A(h->emod, 2 * static_cast<size_t>(P) * T);
    A(h->mom, static_cast<size_t>(P) * 4);
    A(h->sync, 2 * deac::kSyncWords);
    A(h->iter, 8);
    for (deac::MemberCtl *&p : h->ctl) A(p, static_cast<size_t>(h->batch) * P);
    for (uint64_t *&p : h->raw) A(p, static_cast<size_t>(h->batch) * P * h->rstride);
    for (uint64_t *&p : h->gen_start) A(p, static_cast<size_t>(h->batch) * 4);
    A(h->state, 4);
    A(h->init_start, static_cast<size_t>(P) * 4);
    A(h->skip_rows, 256 * 4);
    constexpr size_t kTab = 64 * 16 * 4;  // words of a nibble table
    A(h->lane_tab, deac::kLaneTabWords);
    A(h->columns, deac::kLaneTabSets * 256 * 4);
    if (h->wide) {
        A(h->tab1, deac::kLaneTabWords);
        A(h->tab2, deac::kLaneTabWords);
        A(h->skip_tab_dev, kTab);
    }
    if (!m.nterm.empty()) A(h->nterm, Kc + 1);
    if (!m.fterm.empty()) A(h->fterm, Kc + 1);
    if (!m.tterm.empty()) A(h->tterm, Kc + 1);
    if (m.use_nfm) A(h->nfm_dt, T);
    if (st != DEAC_OK) return st;

    // Jump tables: T^(nsign*G) by rows for the serial walk and by nibbles for
    // the wide one, T^(l*chunk) by lanes for the mask generator, T^(l*c1) and
    // T^(l*(nsign*G+3)) for the wide walk.
    std::vector<uint64_t> rows(256 * 4);
    const deac::Gf2Matrix skip = deac::transition_power(static_cast<uint64_t>(Kc));
    deac::matrix_rows(skip, rows.data());
    h->skip_tab.resize(kTab);
    deac::nibble_table(skip, h->skip_tab.data());
    const int sets = h->wide ? 3 : 1;
    deac::LaneTabArgs la{};
    la.columns = h->columns;
    la.tab[0] = h->lane_tab;
    la.tab[1] = h->tab1;
    la.tab[2] = h->tab2;
    std::vector<deac::Gf2Matrix> steps{deac::transition_power(static_cast<uint64_t>(h->chunk))};
    if (h->wide) {
        steps.push_back(deac::transition_power(static_cast<uint64_t>(deac::walk_c1(P, m.nsign))));
        steps.push_back(deac::transition_power(static_cast<uint64_t>(Kc) + 3));
    }
    auto up = [&](void *dst, const void *src, size_t bytes) {
        if (st == DEAC_OK && hipMemcpy(dst, src, bytes, hipMemcpyHostToDevice) != hipSuccess) st = DEAC_ERR_DEVICE;
    };
    up(h->kmat, m.kernel.data(), m.T * m.Kc * sizeof(double));
    if (st == DEAC_OK && deac::launch_ktile(h->kmat, h->ktile, T, Kc, h->TB, h->stride, h->stream) != hipSuccess)
        st = DEAC_ERR_DEVICE;
    up(h->obs, m.isf.data(), m.T * sizeof(double));
    up(h->sig, m.err.data(), m.T * sizeof(double));
    up(h->skip_rows, rows.data(), rows.size() * sizeof(uint64_t));
    if (h->wide) up(h->skip_tab_dev, h->skip_tab.data(), h->skip_tab.size() * sizeof(uint64_t));
    up(h->columns, steps.data(), steps.size() * sizeof(deac::Gf2Matrix));
    if (st == DEAC_OK && deac::launch_lane_tables(la, sets, h->stream) != hipSuccess) st = DEAC_ERR_DEVICE;
    if (h->nterm) up(h->nterm, m.nterm.data(), m.Kc * sizeof(double));
    if (h->fterm) up(h->fterm, m.fterm.data(), m.Kc * sizeof(double));
    if (h->tterm) up(h->tterm, m.tterm.data(), m.Kc * sizeof(double));
    if (h->nfm_dt) up(h->nfm_dt, m.nfm_dt.data(), m.T * sizeof(double));
    // Populations: member-major rows of `stride` doubles for MG*4 members,
    // zero past Kc and past P.
    for (double *p : {h->pop0, h->pop1})
        if (st == DEAC_OK && hipMemsetAsync(p, 0, pop_n * sizeof(double), h->stream) != hipSuccess)
            st = DEAC_ERR_DEVICE;
    // Records: behind a stop, mask draws may run over records that no walk
    // has written (nothing reads those draws).
    for (deac::MemberCtl *p : h->ctl)
        if (st == DEAC_OK &&
            hipMemsetAsync(p, 0, static_cast<size_t>(h->batch) * P * sizeof(deac::MemberCtl), h->stream) != hipSuccess)
            st = DEAC_ERR_DEVICE;
    if (st != DEAC_OK) return st;
    *out = own.release();
    return DEAC_OK;
} catch (...) {
    return deac::caught();
}

void deac_destroy(deac_handle *h) { delete h; }

deac_status deac_last_run_profile(const deac_handle *h, deac_run_profile *profile)
{
    if (!h || !profile) return DEAC_ERR_INVALID_ARGUMENT;
    *profile = h->last;
    return DEAC_OK;
}

deac_status deac_run(deac_handle *h, uint64_t rng_state[4], const deac_run_options *o, deac_result *r)
try {
    if (!h || !rng_state || !o || !r || !r->dsf || !r->frequency) return DEAC_ERR_INVALID_ARGUMENT;
    if (o->number_of_generations < 2) {
        deac::last_message() = "number_of_generations must be at least 2";
        return DEAC_ERR_INVALID_ARGUMENT;
    }
    if (o->ks_precision != DEAC_PRECISION_FP64 && o->ks_precision != DEAC_PRECISION_FP32 &&
        o->ks_precision != DEAC_PRECISION_BF16X3) {
        deac::last_message() = "ks_precision must be DEAC_PRECISION_FP64, DEAC_PRECISION_FP32 or DEAC_PRECISION_BF16X3";
        return DEAC_ERR_INVALID_ARGUMENT;
    }
    if ((rng_state[0] | rng_state[1] | rng_state[2] | rng_state[3]) == 0) {
        // the all-zero state is a fixed point of xoshiro256+: every draw is 0
        // and the donor draws (deac.cpp:200-216) would never end
        deac::last_message() = "rng_state must not be all zero (a fixed point of xoshiro256+)";
        return DEAC_ERR_INVALID_ARGUMENT;
    }
    const deac::Model &m = h->m;
    const bool split = o->ks_precision != DEAC_PRECISION_FP64 || o->split_loop != 0;
    const size_t N = o->number_of_generations, P = m.P, Kc = m.Kc;
    const int nsign = m.nsign;
    hipStream_t s = h->stream;
    DEAC_HIP(hipSetDevice(h->device));
    if (split) DEAC_TRY(prepare_split(h, o->ks_precision));

    // Initial population and normalization (deac.cpp:430-603) on the device,
    // from the random state at each member's first draw; the state after the
    // last member is where the walk starts.
    deac::Xoshiro rng{{rng_state[0], rng_state[1], rng_state[2], rng_state[3]}};
    std::vector<uint64_t> starts(P * 4);
    for (size_t i = 0; i < P; i++) {
        std::memcpy(&starts[i * 4], rng.s, sizeof rng.s);
        deac::nibble_apply(h->skip_tab.data(), rng.s);
    }
    std::vector<int> cur(P, 0);
    std::vector<double> cr(P * nsign, m.cr0), fw(P * nsign, m.f0);  // deac.cpp:990-1032
    std::vector<double> fit(P), row(Kc);                            // for the results

    const bool track = o->track_stats != 0;
    std::vector<double> histories(track && 3 * N <= deac::kLongHistory ? 3 * N : 0);
    auto release_stats = [&]() {
        void *old = h->stats;
        h->stats = nullptr;
        h->stats_cap = 0;
        h->release(old);
    };
    if (track && h->stats_cap < 3 * N) {
        release_stats();
        DEAC_TRY(h->alloc(h->stats, 3 * N));
        h->stats_cap = 3 * N;
    }
    // (frees the histories of a long run behind it, whatever its outcome)
    struct AtReturn {
        decltype(release_stats) &release;
        const size_t &cap;
        ~AtReturn()
        {
            if (cap > deac::kStatsKept) release();
        }
    } at_return{release_stats, h->stats_cap};
    double *const stats = track ? h->stats : nullptr;

    DEAC_HIP(hipMemcpyAsync(h->init_start, starts.data(), starts.size() * sizeof(uint64_t), hipMemcpyHostToDevice, s));
    DEAC_HIP(hipMemcpyAsync(h->cur, cur.data(), P * sizeof(int), hipMemcpyHostToDevice, s));
    DEAC_HIP(hipMemcpyAsync(h->cr_old, cr.data(), cr.size() * sizeof(double), hipMemcpyHostToDevice, s));
    DEAC_HIP(hipMemcpyAsync(h->f_old, fw.data(), fw.size() * sizeof(double), hipMemcpyHostToDevice, s));
    DEAC_HIP(hipMemcpyAsync(h->state, rng.s, sizeof rng.s, hipMemcpyHostToDevice, s));
    deac::InitArgs ia{};
    ia.start = h->init_start;
    ia.pop = h->pop0;
    ia.tab = h->lane_tab;
    ia.nterm = m.normalize ? h->nterm : nullptr;
    ia.rows = static_cast<long>(P);
    ia.P = static_cast<int>(P);
    ia.G = static_cast<int>(m.G);
    ia.nsign = nsign;
    ia.stride = h->stride;
    ia.nsub = 64;
    ia.sublen = h->chunk;
    ia.lane_tab = true;
    ia.allow_neg = m.allow_negative;
    ia.zeroth = m.zeroth_moment;
    DEAC_HIP(deac::launch_initial_population(ia, s));

    deac::EvoArgs ea{};
    ea.P = static_cast<int>(P);
    ea.T = static_cast<int>(m.T);
    ea.G = static_cast<int>(m.G);
    ea.nsign = nsign;
    ea.Kc = static_cast<int>(Kc);
    ea.stride = h->stride;
    ea.MG = h->MG;
    ea.TB = h->TB;
    ea.by_tau = m.bdsf ? deac::evolve_by_tau(ea.P, 1, ea.TB) : deac::evolve_by_tau(ea.MG, deac::kChainRows, ea.TB);
    ea.use_first = m.use_first;
    ea.use_third = m.use_third;
    ea.renorm = m.normalize && m.renormalize;
    ea.allow_neg = m.allow_negative;
    ea.track_stats = track;
    ea.stop = o->stop_minimum_fitness;
    ea.zeroth = m.zeroth_moment;
    ea.first_moment = m.first_moment;
    ea.third_moment = m.third_moment;
    ea.third_moment_error = m.third_moment_error;
    ea.use_nfm = m.use_nfm;
    ea.nfm_value = m.nfm_value;
    ea.nfm_error = m.nfm_error;
    ea.nfm_dt = h->nfm_dt;
    ea.fold_ks = m.bdsf;
    ea.rstride = h->rstride;
    ea.local = deac::evolve_local(ea.P, ea.T, nsign, m.use_nfm);
    ea.fed = !h->fixed_nwg && deac::evolve_fed(ea, std::max(h->maxwg - 8, 1));
    ea.ktile = h->ktile;
    ea.nterm = h->nterm;
    ea.fterm = h->fterm;
    ea.tterm = h->tterm;
    ea.obs = h->obs;
    ea.sig = h->sig;
    ea.pop0 = h->pop0;
    ea.pop1 = h->pop1;
    ea.cur = h->cur;
    ea.fitness = h->fitness;
    ea.cr_old = h->cr_old;
    ea.f_old = h->f_old;
    ea.emod = h->emod;
    ea.mom = h->mom;
    ea.stats = stats;
    ea.stats_len = N;

    deac::WalkArgs wa{};
    wa.state = h->state;
    wa.skip_rows = h->skip_rows;
    wa.tab1 = h->tab1;
    wa.tab2 = h->tab2;
    wa.skip_tab = h->skip_tab_dev;
    wa.wide = h->wide;
    wa.c1 = deac::walk_c1(static_cast<int>(P), nsign);
    wa.P = static_cast<int>(P);
    wa.nsign = nsign;
    wa.mod_magic = ~UINT64_C(0) / P;
    wa.tau_cr = m.tau_cr;
    wa.tau_f = m.tau_f;
    deac::MaskArgs ma{};
    ma.lane_tab = h->lane_tab;
    ma.P = static_cast<int>(P);
    ma.Kc = static_cast<int>(Kc);
    ma.chunk = h->chunk;
    ma.rstride = h->rstride;

    // Generation loop: ii = 0 .. N-2 (deac.cpp:1138), in batches.  The launch
    // that evolves batch b also makes, on workgroups of its own, the mask draws
    // of batch b+1 and the walk of batch b+2 (two streams may share a hardware
    // queue and then run one after the other).  The evolution of b+1 is queued
    // before the host has read batch b's status.  Behind a stop it changes
    // nothing: the stop test sits at the top of a generation, so the fitnesses
    // it finds are those that stopped batch b, and it stops at its first
    // generation (its status and its statistics entry, past the stop, are
    // never read).  Batches start at 8 generations, so that the first masks,
    // which nothing hides, are few, and grow up to the buffer size by what
    // keeps the walk beside a batch, of the batch after the next, no longer
    // than the batch: by 1.1 for 8 members at G = 16 (walk 5.6 us a generation,
    // evolution 7; 200 generations 1.79 ms, 2.06 by 1.25), by at most a quarter.
    const double walk_us = h->wide ? 12.0 + 0.1 * static_cast<double>(P) : 0.7 * static_cast<double>(P);
    const double generation_us = 6.0 + 0.35 * (h->stride / deac::kChunk);  // at least
    const double grow = split ? 1.25 : std::clamp(std::sqrt(generation_us / walk_us), 1.1, 1.25);
    const size_t total = N - 1;
    std::vector<std::pair<size_t, int>> plan;  // first generation, generations
    for (size_t g = 0, len = std::min(8, h->batch); g < total;) {
        const int nb = static_cast<int>(std::min(len, total - g));
        plan.emplace_back(g, nb);
        g += static_cast<size_t>(nb);
        len = std::min(std::max(static_cast<size_t>(static_cast<double>(len) * grow), len + 1),
                       static_cast<size_t>(h->batch));
    }
    hipStream_t d = h->draw_stream;  // split loop: the draws of the next batch
    auto walk_args = [&](size_t b, const int *halt) {
        // four sets of generation starts: a stop in batch b is answered from
        // its set while the launch of b+1, queued behind, may walk b+3
        wa.gen_start = h->gen_start[b % 4];
        wa.ctl = h->ctl[b % 3];
        wa.halt = halt;
        wa.ngen = b < plan.size() ? plan[b].second : 0;
    };
    auto mask_args = [&](size_t b, const int *halt) {
        ma.ctl = h->ctl[b % 3];
        ma.raw = h->raw[b & 1];
        ma.halt = halt;
        ma.ngen = b < plan.size() ? plan[b].second : 0;
        // up to a workgroup per CU: a wavefront per SIMD, beside the evolution's
        ma.nwg = static_cast<int>(std::min<size_t>((static_cast<size_t>(ma.ngen) * P + 3) / 4, h->maxwg));
    };
    auto evolve = [&](size_t b) -> deac_status {
        const int k = static_cast<int>(b & 1);
        hipEvent_t *e = h->kev[k];
        unsigned *sy = h->sync + deac::kSyncWords * k;
        ea.ctl = h->ctl[b % 3];
        ea.raw = h->raw[k];
        ea.bar = sy;
        ea.status = reinterpret_cast<int *>(sy + 4);
        ea.host_status = h->host_status + 4 * k;
        ea.clear = h->sync + deac::kSyncWords * (k ^ 1);
        ea.xbar = sy + deac::kXcdSync;
        ea.gen0 = static_cast<long>(plan[b].first);
        ea.ngen = plan[b].second;
        mask_args(b + 1, ea.status);
        walk_args(b + 2, ea.status);
        std::fill_n(ea.host_status, 4, 0);  // read for batch b-2 by now
        DEAC_HIP(deac::launch_evolve(ea, wa, ma, s, e[4], e[5]));
        return DEAC_OK;
    };
    deac_run_profile prof{};
    size_t done = 0;          // generations evolved
    long stopped_at = -1;     // generation index of the stop, if any
    auto pipeline = [&]() -> deac_status {
        // Initial fitness (deac.cpp:857-976), on buffer set 1, with the first
        // walk beside it; then the first masks with the second walk.
        DEAC_HIP(deac::launch_zero_u32(h->sync, 2 * deac::kSyncWords, s));
        ea.init_mode = 1;
        ea.gen0 = 0;
        ea.ngen = 0;
        ea.bar = h->sync + deac::kSyncWords;
        ea.xbar = ea.bar + deac::kXcdSync;
        ea.status = reinterpret_cast<int *>(ea.bar + 4);
        ea.host_status = h->host_status + 8;
        ea.nwg = h->nwg;
        std::fill_n(ea.host_status, 4, 0);
        walk_args(0, nullptr);
        DEAC_HIP(deac::launch_evolve(ea, wa, deac::MaskArgs{}, s, nullptr, nullptr));
        ea.init_mode = 0;
        if (ea.fed) ea.nwg = ea.MG * ea.TB + 1;  // the last one keeps the statistics
        DEAC_HIP(hipEventRecord(h->ev0, s));
        mask_args(0, nullptr);
        walk_args(1, nullptr);
        DEAC_HIP(hipEventRecord(h->kev[0][0], s));
        DEAC_HIP(deac::launch_mask(ma, wa, s));
        DEAC_HIP(hipEventRecord(h->kev[0][1], s));
        DEAC_TRY(evolve(0));
        for (size_t b = 0; b < plan.size(); b++) {
            if (b + 1 < plan.size()) DEAC_TRY(evolve(b + 1));
            const int k = static_cast<int>(b & 1);
            hipEvent_t *e = h->kev[k];
            DEAC_HIP(hipEventSynchronize(e[5]));
            if (b == 0 && h->host_status[8 + 2]) return DEAC_ERR_DEVICE;  // initial fitness: barrier timeout
            float t_mask = 0, t_evo = 0;
            if (b == 0) DEAC_HIP(hipEventElapsedTime(&t_mask, e[0], e[1]));
            DEAC_HIP(hipEventElapsedTime(&t_evo, e[4], e[5]));
            prof.mask_ms += t_mask;
            prof.evolve_ms += t_evo;
            prof.evolve_launches += 1;
            const int *status = h->host_status + 4 * k;
            if (status[2]) return DEAC_ERR_DEVICE;  // a grid barrier timed out
            if (status[0]) {
                // RNG state at the top of the stopping generation
                stopped_at = static_cast<long>(plan[b].first) + status[1];
                uint64_t st4[4];
                DEAC_HIP(hipMemcpy(st4, h->gen_start[b % 4] + static_cast<size_t>(status[1]) * 4, sizeof st4,
                                   hipMemcpyDeviceToHost));
                std::memcpy(rng.s, st4, sizeof st4);
                done += static_cast<size_t>(status[1]);
                return DEAC_OK;
            }
            done += static_cast<size_t>(plan[b].second);
        }
        return DEAC_OK;
    };
    // The split loop: the same generations as separate kernels, batch by
    // batch on the plan above.  Batch b's draws (walk, then mask) run on the
    // draw stream while batch b-1 runs, into buffer set b%2; then, per
    // generation, top, trial, renormalization, the contraction at the chosen
    // precision, moments and selection run on the evolution stream.  One
    // status word serves the whole run: once a stop sets it, every kernel
    // queued behind (the rest of the batch and the next one) returns at once.
    // graphs of the split loop (per run: the kernel arguments hold this
    // run's buffers and options); DEAC_SPLIT_GRAPH sets the generations per
    // graph, 0 runs plain launches
    int graph_len = 8;
    if (const char *e = std::getenv("DEAC_SPLIT_GRAPH")) graph_len = std::max(0, std::atoi(e));
    hipGraphExec_t gexec[2] = {nullptr, nullptr};
    struct GraphFree {
        hipGraphExec_t *g;
        ~GraphFree()
        {
            for (int k = 0; k < 2; k++)
                if (g[k]) (void)hipGraphExecDestroy(g[k]);
        }
    } graph_free{gexec};
    auto split_loop = [&]() -> deac_status {
        const deac_handle::Split &sp = h->split;
        const deac::KsLayout &y = sp.y;
        const int Kb = static_cast<int>(y.Kb);
        ea.bar = h->sync;
        ea.status = reinterpret_cast<int *>(h->sync + 4);
        const int *halt = ea.status;
        // model ISF (and moment rows) of the contraction's genomes: the
        // current ones for the initial fitness, the trials otherwise; packed:
        // the genome operand is there already
        auto evaluate = [&](const deac::EvoArgs &a, int init, bool packed) -> deac_status {
            if (y.precision == DEAC_PRECISION_FP64 && a.fold_ks && !init) {
                DEAC_HIP(deac::launch_split_fold(a, s));
            } else if (y.precision == DEAC_PRECISION_FP64) {
                double *B = static_cast<double *>(sp.B);
                DEAC_HIP(deac::launch_split_pack_fp64(a, init, B, y.Nt, Kb, s));
                DEAC_HIP(deac::launch_ks_fp64(static_cast<const double *>(sp.A), B, a.emod, a.T, a.P, y.Mt, y.Nt,
                                              Kb, s, nullptr, nullptr, halt));
            } else {
                if (y.precision == DEAC_PRECISION_FP32) {
                    float *B = static_cast<float *>(sp.B);
                    if (!packed) DEAC_HIP(deac::launch_split_pack_fp32(a, init, B, y.Nt, Kb, s));
                    DEAC_HIP(deac::launch_ks_fp32(static_cast<const float *>(sp.A), B, sp.part, y.Mt, y.Nt, Kb,
                                                  y.kb_per_slice, y.slices, s, nullptr, nullptr, halt));
                } else {
                    if (!packed) DEAC_HIP(deac::launch_split_pack_bf16x3(a, init, sp.B, sp.Bl, y.Nt, Kb, s));
                    DEAC_HIP(deac::launch_ks_bf16x3(sp.A, sp.Al, sp.B, sp.Bl, sp.part, y.Mt, y.Nt, Kb, y.kb_per_slice,
                                                    y.slices, s, nullptr, nullptr, halt));
                }
            }
            if (a.use_first || a.use_third) DEAC_HIP(deac::launch_split_moments(a, init, s));
            return DEAC_OK;
        };
        auto select = [&](const deac::EvoArgs &a, int g, int init) -> deac_status {
            if (y.precision == DEAC_PRECISION_FP64)
                DEAC_HIP(deac::launch_split_select(a, g, init, s));
            else
                DEAC_HIP(deac::launch_split_model_select(a, g, init, sp.part, y.slices, static_cast<int>(y.npad()),
                                                         static_cast<int>(y.mpad()), sp.ex, s));
            return DEAC_OK;
        };
        // One generation g of a batch: top and trials, renormalization,
        // contraction, moments, selection; with a.iter, the generation comes
        // from the device counter, which they advance.
        auto one_generation = [&](const deac::EvoArgs &a, int g) -> deac_status {
            const bool fp64 = y.precision == DEAC_PRECISION_FP64, pack = !fp64 && !a.renorm;
            // with the top of generation g
            DEAC_HIP(deac::launch_split_trial(a, g, pack ? y.precision : DEAC_PRECISION_FP64, sp.B, sp.Bl, Kb, s));
            if (a.renorm) DEAC_HIP(deac::launch_split_renorm(a, s));
            DEAC_TRY(evaluate(a, 0, pack));
            DEAC_TRY(select(a, g, 0));
            return DEAC_OK;
        };
        // Graphs: the kernels of graph_len generations captured once per
        // buffer set and run, replayed for every full group of a batch's
        // generations (a launch per group instead of ~5 per generation);
        // the remainder of a batch runs as plain launches.  A capture the
        // runtime refuses leaves the run on plain launches.
        auto capture = [&](int k, const deac::EvoArgs &a) -> bool {
            hipGraph_t graph = nullptr;
            if (hipStreamBeginCapture(s, hipStreamCaptureModeThreadLocal) != hipSuccess) {
                (void)hipGetLastError();
                return false;
            }
            deac_status st = DEAC_OK;
            for (int r = 0; r < graph_len && st == DEAC_OK; r++) st = one_generation(a, 0);
            const hipError_t e = hipStreamEndCapture(s, &graph);
            bool ok = st == DEAC_OK && e == hipSuccess && graph;
            if (ok) ok = hipGraphInstantiate(&gexec[k], graph, nullptr, nullptr, 0) == hipSuccess;
            if (graph) (void)hipGraphDestroy(graph);
            if (!ok) {
                (void)hipGetLastError();
                gexec[k] = nullptr;
            }
            return ok;
        };
        // Initial fitness (deac.cpp:857-976).
        DEAC_HIP(deac::launch_zero_u32(h->sync, 8, s));
        DEAC_TRY(evaluate(ea, 1, false));
        DEAC_TRY(select(ea, 0, 1));
        DEAC_HIP(hipEventRecord(h->ev0, s));
        DEAC_HIP(hipStreamWaitEvent(d, h->ev0, 0));  // RNG state uploaded
        // Draws of batch b, into the buffers of batch b-2 once that is done.
        auto draw = [&](size_t b) -> deac_status {
            hipEvent_t *ev = h->kev[b % 3];
            walk_args(b, halt);
            mask_args(b, halt);
            wa.ctl = h->ctl[b & 1];  // (two sets, which the graphs hold)
            ma.ctl = h->ctl[b & 1];
            if (b >= 2) DEAC_HIP(hipStreamWaitEvent(d, h->kev[(b - 2) % 3][5], 0));
            DEAC_HIP(hipEventRecord(ev[0], d));
            DEAC_HIP(deac::launch_walk(wa, d));
            DEAC_HIP(hipEventRecord(ev[1], d));
            DEAC_HIP(deac::launch_mask(ma, deac::WalkArgs{}, d));
            DEAC_HIP(hipEventRecord(ev[2], d));
            return DEAC_OK;
        };
        auto generations = [&](size_t b) -> deac_status {
            const int k = static_cast<int>(b & 1);
            hipEvent_t *e = h->kev[b % 3];
            const int nb = plan[b].second;
            DEAC_HIP(hipStreamWaitEvent(s, e[2], 0));  // draws ready
            DEAC_HIP(hipEventRecord(e[3], s));
            ea.ctl = h->ctl[k];
            ea.raw = h->raw[k];
            ea.gen0 = static_cast<long>(plan[b].first);
            ea.ngen = nb;
            int g = 0;
            if (graph_len > 0 && nb >= graph_len) {
                deac::EvoArgs eg = ea;
                eg.iter = h->iter + 4 * k;
                DEAC_HIP(deac::launch_split_iter(eg.iter, eg.gen0, s));
                if (!gexec[k] && !capture(k, eg)) graph_len = 0;
                if (gexec[k]) {
                    for (; g + graph_len <= nb; g += graph_len) {
                        DEAC_HIP(hipGraphLaunch(gexec[k], s));
                        prof.graph_launches += 1;
                    }
                    for (; g < nb; g++) DEAC_TRY(one_generation(eg, 0));
                }
            }
            for (; g < nb; g++) DEAC_TRY(one_generation(ea, g));
            DEAC_HIP(hipEventRecord(e[5], s));
            DEAC_HIP(hipMemcpyAsync(h->host_status + 4 * k, h->sync + 4, 4 * sizeof(int), hipMemcpyDeviceToHost, s));
            DEAC_HIP(hipEventRecord(e[6], s));
            return DEAC_OK;
        };
        DEAC_TRY(draw(0));
        if (plan.size() > 1) DEAC_TRY(draw(1));
        DEAC_TRY(generations(0));
        for (size_t b = 0; b < plan.size(); b++) {
            // The draws are queued while batch b runs, ahead of batch b+1, whose
            // launches keep the host for most of a batch (behind them, or after
            // batch b, they left 0.2 ms between batches of 0.8 ms).
            if (b + 2 < plan.size()) DEAC_TRY(draw(b + 2));
            if (b + 1 < plan.size()) DEAC_TRY(generations(b + 1));
            const int k = static_cast<int>(b & 1);
            hipEvent_t *e = h->kev[b % 3];
            DEAC_HIP(hipEventSynchronize(e[6]));
            float t_walk = 0, t_mask = 0, t_evo = 0;
            DEAC_HIP(hipEventElapsedTime(&t_walk, e[0], e[1]));
            DEAC_HIP(hipEventElapsedTime(&t_mask, e[1], e[2]));
            DEAC_HIP(hipEventElapsedTime(&t_evo, e[3], e[5]));
            prof.walk_ms += t_walk;
            prof.mask_ms += t_mask;
            prof.evolve_ms += t_evo;
            prof.evolve_launches += 1;
            // the copy after batch b: a stop there, at generation status[1] of
            // the batch (later batches have not run, or returned at once)
            const int *status = h->host_status + 4 * k;
            if (status[0]) {
                stopped_at = static_cast<long>(plan[b].first) + status[1];
                uint64_t st4[4];
                DEAC_HIP(hipMemcpy(st4, h->gen_start[b % 4] + static_cast<size_t>(status[1]) * 4, sizeof st4,
                                   hipMemcpyDeviceToHost));
                std::memcpy(rng.s, st4, sizeof st4);
                done += static_cast<size_t>(status[1]);
                return DEAC_OK;
            }
            done += static_cast<size_t>(plan[b].second);
        }
        return DEAC_OK;
    };
    const deac_status ps = split ? split_loop() : pipeline();
    // nothing stays in flight past this call, whatever the outcome
    const bool drained = hipEventRecord(h->ev1, s) == hipSuccess && hipStreamSynchronize(s) == hipSuccess &&
                         hipStreamSynchronize(d) == hipSuccess;
    if (ps != DEAC_OK) return ps;
    if (!drained) {
        (void)hipGetLastError();
        return DEAC_ERR_DEVICE;
    }
    float ms = 0.0f;
    DEAC_HIP(hipEventElapsedTime(&ms, h->ev0, h->ev1));
    prof.loop_ms = ms;
    prof.generations = done;
    h->last = prof;
    if (stopped_at < 0) DEAC_HIP(hipMemcpy(rng.s, h->state, sizeof rng.s, hipMemcpyDeviceToHost));
    std::memcpy(rng_state, rng.s, sizeof rng.s);

    // Epilogue on the host (deac.cpp:1576-1685).
    DEAC_HIP(hipMemcpy(fit.data(), h->fitness, P * sizeof(double), hipMemcpyDeviceToHost));
    DEAC_HIP(hipMemcpy(cur.data(), h->cur, P * sizeof(int), hipMemcpyDeviceToHost));
    size_t generation = stopped_at >= 0 ? static_cast<size_t>(stopped_at) : N - 2;
    size_t best = 0;
    double minimum = fit[0];
    for (size_t i = 0; i < P; i++)
        if (fit[i] < minimum) {
            minimum = fit[i];
            best = i;
        }
    DEAC_HIP(hipMemcpy(row.data(), (cur[best] ? h->pop1 : h->pop0) + best * h->stride, Kc * sizeof(double),
                       hipMemcpyDeviceToHost));
    deac::output_transform(m, row.data(), r->dsf, r->frequency);

    if (track) {
        const size_t n = generation + 1;  // entries written
        double *const to[3] = {r->stats_mean, r->stats_minimum, r->stats_squared_mean};
        if (!histories.empty()) {
            DEAC_HIP(hipMemcpy(histories.data(), stats, 3 * N * sizeof(double), hipMemcpyDeviceToHost));
            for (int k = 0; k < 3; k++)
                if (to[k]) std::memcpy(to[k], &histories[k * N], n * sizeof(double));
        } else {
            for (int k = 0; k < 3; k++)
                if (to[k]) DEAC_HIP(hipMemcpy(to[k], stats + k * N, n * sizeof(double), hipMemcpyDeviceToHost));
        }
    }
    if (generation + 2 == N) {  // deac.cpp:1677-1685
        generation += 1;
        if (track) {
            if (r->stats_mean) r->stats_mean[generation] = deac::mean_of(fit.data(), P);
            if (r->stats_minimum) r->stats_minimum[generation] = minimum;
            if (r->stats_squared_mean) r->stats_squared_mean[generation] = deac::squared_mean_of(fit.data(), P);
        }
    }
    r->generation = generation;
    r->minimum_fitness = minimum;
    r->best_index = best;
    if (r->final_fitness) std::memcpy(r->final_fitness, fit.data(), P * sizeof(double));
    return DEAC_OK;
} catch (...) {
    return deac::caught();
}

}  // extern "C"
