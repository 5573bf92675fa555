// The split loop's launchers (split_kernels.hip, its host part) on a stand-in for
// the HIP runtime that records the launches: a dispatch holds fewer than 2^32
// threads, and the launches of one step cover what there is to do.
#include <cstdint>
#include <cstdio>
#include <map>
#include <string>
#include <vector>

#include "split_kernels.hpp"

namespace {

struct Launch {
    std::string kernel;
    size_t grid, block;
    int first;  // the kernel's last argument
};
std::vector<Launch> launches;
// (registered before this file's own globals are made)
std::map<const void *, std::string> &names()
{
    static std::map<const void *, std::string> m;
    return m;
}
dim3 grid_of, block_of;
int wrong = 0;

void expect(bool ok, const std::string &what)
{
    if (ok) return;
    std::printf("%s\n", what.c_str());
    wrong = 1;
}

int args_of(const std::string &kernel) { return kernel.find("split_fold") != std::string::npos ? 2 : 9; }

}  // namespace

extern "C" {
char fatbin;  // (no device code is looked at)
void **__hipRegisterFatBinary(const void *) { return reinterpret_cast<void **>(&fatbin); }
void __hipUnregisterFatBinary(void **) {}
void __hipRegisterFunction(void **, const void *host, char *, const char *name, unsigned, void *, void *, void *, void *,
                           int *)
{
    names()[host] = name;
}
hipError_t __hipPushCallConfiguration(dim3 g, dim3 b, size_t, hipStream_t) { return grid_of = g, block_of = b, hipSuccess; }
hipError_t __hipPopCallConfiguration(dim3 *g, dim3 *b, size_t *lds, hipStream_t *s)
{
    *g = grid_of;
    *b = block_of;
    *lds = 0;
    *s = nullptr;
    return hipSuccess;
}
hipError_t hipLaunchKernel(const void *host, dim3 g, dim3 b, void **args, size_t, hipStream_t)
{
    const std::string &name = names()[host];
    launches.push_back({name, static_cast<size_t>(g.x) * g.y * g.z, static_cast<size_t>(b.x) * b.y * b.z,
                        *static_cast<int *>(args[args_of(name) - 1])});
    return hipSuccess;
}
hipError_t hipGetLastError() { return hipSuccess; }
}

namespace {

void covers(const char *what, size_t items)
{
    size_t done = 0;
    for (const Launch &l : launches) {
        expect(l.grid * l.block <= UINT32_MAX, std::string(what) + ": a dispatch of " + std::to_string(l.grid * l.block) +
                                                   " threads");
        expect(static_cast<size_t>(l.first) == done, std::string(what) + ": starts at another item");
        done += l.grid;
    }
    expect(done == items, std::string(what) + ": " + std::to_string(done) + " of " + std::to_string(items) + " items");
    launches.clear();
}

}  // namespace

int main()
{
    deac::EvoArgs a{};
    for (int P : {4, 67000000, 70000000, 130000000})
        for (int T : {2, 257, 1024, 5000}) {
            a.P = P;
            a.T = T;
            a.TB = (T + 15) / 16;
            const std::string at = " P=" + std::to_string(P) + " T=" + std::to_string(T);
            (void)deac::launch_split_select(a, 0, 0, nullptr);
            covers(("select" + at).c_str(), P);
            for (int slices : {1, 9, 256}) {
                (void)deac::launch_split_model_select(a, 0, 0, nullptr, slices, 0, 0, nullptr, nullptr);
                covers(("model select" + at).c_str(), P);
            }
            if (static_cast<long>(P) * a.TB < INT32_MAX) {
                (void)deac::launch_split_fold(a, nullptr);
                covers(("fold" + at).c_str(), static_cast<size_t>(P) * a.TB);
            }
        }
    return wrong;
}
