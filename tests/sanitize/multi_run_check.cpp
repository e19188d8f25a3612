// multi_run_check.cpp -- how a run of steps is cut into launches of several
// (imexlb-1.0_amd/csrc/context.hpp), for every plan and length.
#include <cstdio>

#include "context.hpp"

int main()
{
    for (int halo : {3, 5, 7, 9})
        for (int least : {3, 5})
            for (int from : {4, 3 * halo + 1})
                for (int n = 0; n < 400; ++n) {
                    imexlb::MultiPlan m;
                    m.halo = halo;
                    m.least = least;
                    m.from = from;
                    const imexlb::MultiRun r = imexlb::multi_run(m, n);
                    std::printf("%d %d %d %d %d %d %d\n", halo, least, from, n, int(r.full), r.last, int(r.done));
                }
    return 0;
}
