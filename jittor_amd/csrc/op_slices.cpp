// What follows a product whose sum was cut into slices: the slices' float32 results added up (kernels/fold_slices.h), with the element-wise
// group that waits behind the product, if one does.
#include "common.h"
#include <mutex>
#include <unordered_map>

namespace mjt {

namespace {
std::mutex g_mu;
std::unordered_map<std::string, JitKernel*> g_kernels;
void forget() {   // the kernels belong to the run-time compiler's cache, which mjt_shutdown empties
    std::lock_guard<std::mutex> lock(g_mu);
    g_kernels.clear();
}
const bool g_registered = (at_shutdown(&forget), true);
}  // namespace

SliceFold::SliceFold(const void* part, void* y, int dtype, int64_t n, int64_t slices) {
    MJT_CHECK(slices >= 1 && slices <= 16 && (dtype == MJT_FLOAT32 || dtype == MJT_BFLOAT16 || dtype == MJT_FLOAT16), "slices of a sum: not covered");
    const int osz = dtype_size(dtype);
    int vs = 4;
    while (vs > 1 && (n % vs || (uintptr_t)y % (size_t)(vs * osz))) vs /= 2;
    ep = epilogue_code(vs, 3, dtype, n);
    if (!ep.on) check_no_epilogue();                              // (before anything is launched)
    const int out = dtype == MJT_BFLOAT16 ? 0 : dtype == MJT_FLOAT16 ? 1 : 2;
    std::ostringstream key;
    key << out << vs << "," << slices << ep.key;
    {
        std::lock_guard<std::mutex> lock(g_mu);
        auto it = g_kernels.find(key.str());
        k = it == g_kernels.end() ? nullptr : it->second;
    }
    if (!k) {
        std::ostringstream name;
        name << "mjt_fold_slices_" << mjt_dtype_name(dtype) << "_" << slices << "v" << vs << ep.suffix();
        k = jit_get(ep.defs + "#define ENTRY " + name.str() + "\n#define SLICES " + std::to_string(slices) + "\n#define VS " + std::to_string(vs) + "\n#define OUT " +
                        std::to_string(out) + "\n" + embedded_source("fold_slices.h") + "\n", name.str());
        std::lock_guard<std::mutex> lock(g_mu);
        g_kernels.emplace(key.str(), k);
    }
    args = {bits_of_ptr(part), bits_of_ptr(y), (uint64_t)(n / vs)};
    args.insert(args.end(), ep.words.begin(), ep.words.end());
    blocks = (n / vs + 255) / 256;
    MJT_CHECK(blocks < (int64_t(1) << 31), "slices of a sum: launch too large");
}

void SliceFold::launch() {
    epilogue_taken(ep);
    jit_launch(k, (unsigned)blocks, 1, 256, 0, args);
}

}  // namespace mjt
