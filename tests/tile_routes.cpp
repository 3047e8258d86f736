// Which kernel a product of packed vectors launches, on the host: the host code of csrc/macko_spmv_tile.hip and, in the place of
// the HIP runtime, functions that write down what would be launched.
//
// Reads lines "cols batch form n rows_1 entries_1 ... rows_n entries_n" (form 1: with a residual, 2: silu(gate) * up of two),
// prints "<kernel>:<workgroups>:<bytes of LDS>" of each launch, or "refused <code>".
#include <cxxabi.h>

#include <cstdio>
#include <cstdlib>
#include <map>
#include <string>
#include <vector>

#include "macko_spmv_tile.hip"

static std::map<const void *, std::string> &kernels()
{
    static std::map<const void *, std::string> all;
    return all;
}
static std::string launched, configuration;

extern "C" {
void **__hipRegisterFatBinary(const void *) { return nullptr; }
void __hipUnregisterFatBinary(void **) {}
void __hipRegisterFunction(void **, const void *function, char *, const char *name, unsigned, void *, void *, void *, void *, int *)
{
    char *plain = abi::__cxa_demangle(name, nullptr, nullptr, nullptr);
    std::string text = plain ? plain : name;
    std::free(plain);
    const size_t from = text.find("spmv_"), to = text.find('(', from == std::string::npos ? 0 : from);
    kernels()[function] = from == std::string::npos ? text : text.substr(from, to - from);
}
hipError_t __hipPushCallConfiguration(dim3 grid, dim3, size_t lds, hipStream_t)
{
    configuration = ":" + std::to_string(grid.x) + ":" + std::to_string(lds);
    return hipSuccess;
}
hipError_t __hipPopCallConfiguration(dim3 *, dim3 *, size_t *, hipStream_t *) { return hipSuccess; }
hipError_t hipLaunchKernel(const void *function, dim3, dim3, void **, size_t, hipStream_t)
{
    if (!launched.empty()) launched += " ";
    for (char c : kernels()[function])
        if (c != ' ') launched += c;
    launched += configuration;
    return hipSuccess;
}
hipError_t hipFuncSetAttribute(const void *, hipFuncAttribute, int) { return hipSuccess; }
hipError_t hipGetDevice(int *device)
{
    *device = 0;
    return hipSuccess;
}
hipError_t hipGetLastError(void) { return hipSuccess; }
}

namespace macko {
int device_info(DeviceInfo *out)
{
    *out = DeviceInfo{256, 160 * 1024};
    return 0;
}
}  // namespace macko

int main()
{
    void *somewhere = reinterpret_cast<void *>(uintptr_t{1} << 20);  // never read here
    int cols, batch, form, n;
    while (std::scanf("%d %d %d %d", &cols, &batch, &form, &n) == 4) {
        std::vector<macko_packed_matrix> all((size_t)n);
        for (macko_packed_matrix &m : all) {
            long long rows, entries;
            if (std::scanf("%lld %lld", &rows, &entries) != 2) return 1;
            m = {somewhere, somewhere, (const int32_t *)somewhere, somewhere, (int32_t)rows, entries, rows};
        }
        launched.clear();
        const macko_packed_matrix &m = all[0];
        const int rc = form == 2 && n == 2 ? macko_spmv_f16_packed_silu(&all[0], &all[1], somewhere, somewhere, cols, batch, nullptr)
                       : n > 1 ? macko_spmv_f16_packed_several(all.data(), n, somewhere, cols, batch, nullptr)
                             : macko_spmv_f16_packed(m.values, m.deltas, m.row_ptr, somewhere, form ? somewhere : nullptr, m.y, m.rows,
                                                     cols, m.padded_entries, batch, m.ldy, nullptr);
        if (rc != 0)
            std::printf("refused %d\n", rc);
        else
            std::printf("%s\n", launched.c_str());
    }
    return 0;
}
