// place_check.cpp -- where the entries of a window's table of places lie
// (imexlb-1.0_amd/csrc/kernels.hpp), for tables on both sides of 2^32 entries.
//
//   place_check cells table ...      prints the table's first and last entry
#include <cstdio>
#include <cstdlib>

#include "kernels.hpp"

int main(int argc, char **argv)
{
    const uint32_t cells = uint32_t(std::atol(argv[1]));
    for (int k = 2; k < argc; ++k) {
        const int64_t base = imexlb::place_base(int32_t(std::atol(argv[k])), cells);
        std::printf("%lld %lld\n", (long long)base, (long long)(base + (8u * cells + (cells - 1u))));
    }
    return 0;
}
