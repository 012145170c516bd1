// radial_basis under failing allocations and odd knot offsets (tests/test_radial_basis.py).
//   fail FILE     allocation k = 1, 2, .. throws until a call needs no more: prints the count
//   count FILE    prints the number of basis functions
//   empty         maps without knots, their table behind an unreadable page: prints the result
#include <sys/mman.h>

#include <atomic>
#include <cstdio>
#include <cstdlib>
#include <cstring>
#include <new>

#include "sfb_internal.h"

static std::atomic<long> g_left{-1};  // allocations until one throws (< 0: none)

void* operator new(std::size_t n)
{
    if (g_left.load() >= 0 && g_left.fetch_sub(1) == 0) throw std::bad_alloc();
    if (void* p = std::malloc(n)) return p;
    throw std::bad_alloc();
}
void operator delete(void* p) noexcept { std::free(p); }
void operator delete(void* p, std::size_t) noexcept { std::free(p); }

int main(int argc, char** argv)
{
    if (argc > 1 && !std::strcmp(argv[1], "empty")) {
        char* m = (char*)mmap(nullptr, 3 * 4096, PROT_READ | PROT_WRITE, MAP_PRIVATE | MAP_ANONYMOUS, -1, 0);
        if (m == (char*)MAP_FAILED || mprotect(m, 4096, PROT_NONE) || mprotect(m + 2 * 4096, 4096, PROT_NONE)) return 2;
        const double* x = (const double*)(m + 4096);
        const int64_t off[3] = {0, 0, 0}, end[2] = {512, 512};
        sfb::RadialBasis R;
        const bool a = sfb::radial_basis(2, off, x, x, x, &R, 4), b = sfb::radial_basis(1, end, x, x, x, &R, 4);
        std::printf("%d %d\n", a, b);
        return 0;
    }
    if (argc < 3) return 2;
    FILE* f = std::fopen(argv[2], "rb");
    if (!f) return 2;
    int64_t n[2];
    if (std::fread(n, 8, 2, f) != 2) return 2;
    std::vector<int64_t> off((size_t)n[0] + 1);
    std::vector<double> t(3 * (size_t)n[1]);
    if (std::fread(off.data(), 8, off.size(), f) != off.size() || std::fread(t.data(), 8, t.size(), f) != t.size()) return 2;
    std::fclose(f);
    const double *x = t.data(), *y = x + n[1], *ypp = y + n[1];
    if (!std::strcmp(argv[1], "count")) {
        sfb::RadialBasis R;
        const bool ok = sfb::radial_basis(n[0], off.data(), x, y, ypp, &R, 4);
        std::printf("%d %d\n", ok, R.nc);
        return 0;
    }
    for (long k = 0;; ++k) {
        sfb::RadialBasis R;
        g_left = k;
        const bool ok = sfb::radial_basis(n[0], off.data(), x, y, ypp, &R, 4);
        const bool reached = g_left.load() < 0;  // the k-th allocation was asked for
        g_left = -1;
        if (!reached) {
            std::printf("%ld %d %d\n", k, ok, R.nc);
            return 0;
        }
    }
}
