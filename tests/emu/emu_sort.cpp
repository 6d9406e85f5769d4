// CPU emulation of the sort: tl_sort.hip built for the host over the HIP shim,
// one workgroup at a time with every lane a fiber, under AddressSanitizer.
// Every result is compared with std::sort and std::unique, over inputs that
// reach its paths: wide and narrow ranges, keys that repeat often, one key
// alone, keys in order and in reverse, and crowds with outliers.  Arguments: key
// type (u32, u64, i32, i64), then sizes.
#include "hip/hip_runtime.h"
#include "tree_layouts.h"
#include <algorithm>
#include <random>
#include <stdio.h>
#include <string>
#include <unistd.h>
#include <vector>

int emu_fallbacks, emu_large;   // runs that ended in the radix sort; large buckets

template <typename T>
static int run(tl_dtype dt, uint64_t n) {
    static const char *names[] = {"wide", "narrow", "heavy", "equal", "sorted", "reverse", "crowds"};
    std::mt19937_64 rng(n);
    int bad = 0;
    for (int d = 0; d < 7; d++) {
        std::vector<T> in(n);
        for (uint64_t i = 0; i < n; i++)
            in[i] = d == 0   ? (T)rng()
                    : d == 1 ? (T)(rng() % (n / 2 + 1)) - (T)(n / 4)
                    : d == 2 ? (rng() % 4 ? (T)77 : (T)(rng() % 100000))
                    : d == 3 ? (T)-5
                    : d == 4 ? (T)i
                    : d == 5 ? (T)(n - i)
                             : (T)((rng() % 8) << (8 * sizeof(T) - 5)) + (T)(rng() % 300);
        std::vector<T> want = in;
        std::sort(want.begin(), want.end());
        want.erase(std::unique(want.begin(), want.end()), want.end());
        T *a = (T *)malloc(n * sizeof(T));
        std::copy(in.begin(), in.end(), a);
        uint64_t m = 0;
        emu_fallbacks = emu_large = 0;
        const tl_status st = tl_sort_dedupe(a, n, dt, &m, nullptr, nullptr);
        const bool ok = st == TL_OK && m == want.size() && std::equal(want.begin(), want.end(), a);
        fprintf(stderr, "[emu-sort] %s dtype %d n=%llu: status %d, %llu of %zu distinct, %d fallback, %d large, %s\n",
                names[d], (int)dt, (unsigned long long)n, (int)st, (unsigned long long)m,
                want.size(), emu_fallbacks, emu_large, ok ? "right" : "WRONG");
        bad += !ok;
        free(a);
    }
    return bad;
}

int main(int argc, char **argv) {
    if (argc < 3) _exit(2);
    const std::string kind = argv[1];
    int bad = 0;
    for (int k = 2; k < argc; k++) {
        const uint64_t n = strtoull(argv[k], nullptr, 10);
        if (kind == "u32") bad += run<uint32_t>(TL_U32, n);
        if (kind == "u64") bad += run<uint64_t>(TL_U64, n);
        if (kind == "i32") bad += run<int32_t>(TL_I32, n);
        if (kind == "i64") bad += run<int64_t>(TL_I64, n);
    }
    fflush(stderr);
    _exit(bad ? 1 : 0);
}
