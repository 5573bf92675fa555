// deac_model_isf: the model ISF E = K.S (deac.cpp:1385-1395) and the reduced
// chi^2 (deac.cpp:120-126, 1540-1542) of a stack of genomes at a chosen K.S
// precision -- the precision sweep of the K.S contraction.  FP64 is the
// engine's exact evaluation; FP32 and BF16X3 are the mixed-precision forms
// (K scaled per tau row by a power of two, FP32 accumulation), whose error
// against FP64 this entry point exists to measure.  chi^2 is FP64 in the
// reference's order at every precision.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <cmath>
#include <cstdint>
#include <cstring>
#include <string>
#include <vector>

#include "deac_engine.h"
#include "host_model.hpp"
#include "ks_layout.hpp"
#include "pack_kernels.hpp"
#include "precision_kernels.hpp"

namespace {


// Device buffers of one call, freed on every exit path.
struct Buffers {
    std::vector<void *> ptrs;
    ~Buffers()
    {
        for (void *p : ptrs) (void)hipFree(p);
    }
    template <class T>
    bool alloc(T *&out, size_t count)
    {
        void *p = nullptr;
        ptrs.push_back(nullptr);  // its place, before there is anything to lose
        if (hipMalloc(&p, count * sizeof(T)) != hipSuccess) {
            (void)hipGetLastError();
            ptrs.pop_back();
            return false;
        }
        ptrs.back() = p;
        out = static_cast<T *>(p);
        return true;
    }
};

// chi^2 / T in the reference's order: rounded squares added in tau order, the
// last one fused when T is odd (deac.cpp:120-126, 1540-1542).
double reduced_chi2(const deac::Model &m, const double *e)
{
    const size_t T = m.T;
    double acc = 0.0;
    for (size_t t = 0; t < T; t++) {
        const double d = (m.isf[t] - e[t]) / m.err[t];
        acc = ((T & 1) && t == T - 1) ? std::fma(d, d, acc) : acc + d * d;
    }
    return acc / static_cast<double>(T);
}

}  // namespace

#define PREC_HIP(call)                                  \
    do {                                                \
        if ((call) != hipSuccess) {                     \
            (void)hipGetLastError();                    \
            return DEAC_ERR_DEVICE;                     \
        }                                               \
    } while (0)

extern "C" size_t deac_genome_length(const deac_problem *p)
{
    if (!p) return 0;
    return (p->zero_temperature || p->spectra_type == DEAC_BDSF) ? p->genome_size : 2 * p->genome_size;
}

extern "C" deac_status deac_model_isf(const deac_problem *p, const double *genomes, size_t count, int precision,
                                      double *model_isf, double *chi2, double *kernel_ms, const char **message)
try {
    if (message) *message = nullptr;
    if (!p || !genomes || count == 0) return DEAC_ERR_INVALID_ARGUMENT;
    if (precision != DEAC_PRECISION_FP64 && precision != DEAC_PRECISION_FP32 && precision != DEAC_PRECISION_BF16X3) {
        deac::last_message() = "precision must be DEAC_PRECISION_FP64, DEAC_PRECISION_FP32 or DEAC_PRECISION_BF16X3";
        if (message) *message = deac::last_message().c_str();
        return DEAC_ERR_INVALID_ARGUMENT;
    }
    if (count > (1u << 24)) {
        deac::last_message() = "at most 2^24 genomes per call";
        if (message) *message = deac::last_message().c_str();
        return DEAC_ERR_UNSUPPORTED;
    }
    const deac_status v = deac::validate(*p, deac::last_message());
    if (v != DEAC_OK) {
        if (message) *message = deac::last_message().c_str();
        return v;
    }
    int devices = 0, device = 0;
    if (hipGetDeviceCount(&devices) != hipSuccess || devices == 0) {
        (void)hipGetLastError();
        return DEAC_ERR_NO_DEVICE;
    }
    PREC_HIP(hipGetDevice(&device));
    hipDeviceProp_t prop;
    PREC_HIP(hipGetDeviceProperties(&prop, device));
    if (std::strncmp(prop.gcnArchName, "gfx950", 6) != 0) return DEAC_ERR_NO_DEVICE;

    const deac::Model m = deac::build_model(*p);
    const deac::KsLayout y = deac::ks_layout(m, precision, count);
    const int T = static_cast<int>(m.T), N = static_cast<int>(count);
    const int Kb = static_cast<int>(y.Kb);
    std::vector<double> E(static_cast<size_t>(N) * T);

    hipStream_t s = nullptr;
    PREC_HIP(hipStreamCreateWithFlags(&s, hipStreamNonBlocking));
    struct StreamGuard {
        hipStream_t s;
        ~StreamGuard() { (void)hipStreamDestroy(s); }
    } sg{s};
    hipEvent_t e0 = nullptr, e1 = nullptr;
    PREC_HIP(hipEventCreate(&e0));
    PREC_HIP(hipEventCreate(&e1));
    struct EventGuard {
        hipEvent_t a, b;
        ~EventGuard()
        {
            (void)hipEventDestroy(a);
            (void)hipEventDestroy(b);
        }
    } eg{e0, e1};
    Buffers buf;
    const size_t asz = y.a_count(), bsz = y.b_count();

    // K and the genomes go up as they are and are packed on the device, the
    // genomes in blocks of whole tiles of at most about 256 MiB
    double *krows, *grows;
    const size_t L = y.L;
    const size_t block = std::min<size_t>(static_cast<size_t>(y.Nt) * 16,
                                          std::max<size_t>(1, (size_t(1) << 21) / L) * 16);
    if (!buf.alloc(krows, m.T * L) || !buf.alloc(grows, block * L)) return DEAC_ERR_OUT_OF_MEMORY;
    PREC_HIP(hipMemcpyAsync(krows, m.kernel.data(), m.T * L * sizeof(double), hipMemcpyHostToDevice, s));
    auto pack_genomes = [&](auto pack) -> deac_status {
        for (size_t n0 = 0; n0 < count; n0 += block) {
            const size_t n = std::min(block, count - n0);
            PREC_HIP(hipMemcpyAsync(grows, genomes + n0 * L, n * L * sizeof(double), hipMemcpyHostToDevice, s));
            const int tiles = static_cast<int>((n + 15) / 16);
            PREC_HIP(pack(deac::PackArgs{grows, nullptr, static_cast<int>(n), static_cast<int>(L), tiles, Kb},
                          n0 / 16 * y.Kb * 64 * y.per));
        }
        return DEAC_OK;
    };
    int *ex = nullptr;
    if (!y.ex.empty()) {
        if (!buf.alloc(ex, m.T)) return DEAC_ERR_OUT_OF_MEMORY;
        PREC_HIP(hipMemcpyAsync(ex, y.ex.data(), m.T * sizeof(int), hipMemcpyHostToDevice, s));
    }
    const deac::PackArgs pk{krows, ex, T, static_cast<int>(L), y.Mt, Kb};
    if (precision == DEAC_PRECISION_FP64) {
        double *dA, *dB, *dE;
        if (!buf.alloc(dA, asz) || !buf.alloc(dB, bsz) || !buf.alloc(dE, E.size())) return DEAC_ERR_OUT_OF_MEMORY;
        // -0.0 past K's rows and positions: with genomes padded with +0.0 the
        // padded products are -0.0 and leave every chain exactly as it is
        PREC_HIP(deac::launch_pack_fp64(pk, -0.0, dA, s));
        const deac_status st = pack_genomes(
            [&](const deac::PackArgs &a, size_t at) { return deac::launch_pack_fp64(a, 0.0, dB + at, s); });
        if (st != DEAC_OK) return st;
        PREC_HIP(deac::launch_ks_fp64(dA, dB, dE, T, N, y.Mt, y.Nt, Kb, s, e0, e1, nullptr));
        PREC_HIP(hipMemcpyAsync(E.data(), dE, E.size() * sizeof(double), hipMemcpyDeviceToHost, s));
        PREC_HIP(hipStreamSynchronize(s));
    } else {
        const size_t mn = y.mpad() * y.npad();
        float *part, *out;
        if (!buf.alloc(part, static_cast<size_t>(y.slices) * mn) || !buf.alloc(out, mn)) return DEAC_ERR_OUT_OF_MEMORY;
        if (precision == DEAC_PRECISION_FP32) {
            float *dA, *dB;
            if (!buf.alloc(dA, asz) || !buf.alloc(dB, bsz)) return DEAC_ERR_OUT_OF_MEMORY;
            PREC_HIP(deac::launch_pack_fp32(pk, dA, s));
            const deac_status st = pack_genomes(
                [&](const deac::PackArgs &a, size_t at) { return deac::launch_pack_fp32(a, dB + at, s); });
            if (st != DEAC_OK) return st;
            PREC_HIP(deac::launch_ks_fp32(dA, dB, part, y.Mt, y.Nt, Kb, y.kb_per_slice, y.slices, s, e0, nullptr,
                                          nullptr));
        } else {
            uint16_t *dAh, *dAl, *dBh, *dBl;
            if (!buf.alloc(dAh, asz) || !buf.alloc(dAl, asz) || !buf.alloc(dBh, bsz) || !buf.alloc(dBl, bsz))
                return DEAC_ERR_OUT_OF_MEMORY;
            PREC_HIP(deac::launch_pack_bf16x3(pk, dAh, dAl, s));
            const deac_status st = pack_genomes([&](const deac::PackArgs &a, size_t at) {
                return deac::launch_pack_bf16x3(a, dBh + at, dBl + at, s);
            });
            if (st != DEAC_OK) return st;
            PREC_HIP(deac::launch_ks_bf16x3(dAh, dAl, dBh, dBl, part, y.Mt, y.Nt, Kb, y.kb_per_slice, y.slices, s,
                                            e0, nullptr, nullptr));
        }
        PREC_HIP(deac::launch_reduce_slices(part, out, y.slices, mn, s, nullptr, e1));
        std::vector<float> E32(mn);
        PREC_HIP(hipMemcpyAsync(E32.data(), out, E32.size() * sizeof(float), hipMemcpyDeviceToHost, s));
        PREC_HIP(hipStreamSynchronize(s));
        const size_t Mpad = y.mpad();
        for (int n = 0; n < N; n++)
            for (int t = 0; t < T; t++)
                E[static_cast<size_t>(n) * T + t] =
                    std::ldexp(static_cast<double>(E32[static_cast<size_t>(n) * Mpad + t]), y.ex[t]);
    }
    if (kernel_ms) {
        float ms = 0.0f;
        PREC_HIP(hipEventElapsedTime(&ms, e0, e1));
        *kernel_ms = ms;
    }
    if (model_isf) std::memcpy(model_isf, E.data(), E.size() * sizeof(double));
    if (chi2)
        for (int n = 0; n < N; n++) chi2[n] = reduced_chi2(m, &E[static_cast<size_t>(n) * T]);
    return DEAC_OK;
} catch (...) {
    return deac::caught();
}
