// The tensor stage's face numbering (dgtd_amd/csrc/tensor_dev.hpp) against the
// face tables that set-up builds, orders 1-5, and against tables with two
// entries exchanged, which set-up refuses.  Run by tests/test_host_setup.py.
#include <cstdio>
#include <utility>

#include "../../dgtd_amd/csrc/hex.hpp"
#include "../../dgtd_amd/csrc/quad.hpp"
#include "../../dgtd_amd/csrc/tensor_dev.hpp"

int main()
{
    int bad = 0;
    for (int p = 1; p <= 5; ++p)
        for (int dim : {2, 3}) {
            std::vector<int> fmask = dim == 3 ? dgtd::build_refhex(p).Fmask : dgtd::build_refquad(p).Fmask;
            if (!dgtd::tensor_faces_match(dim, p, fmask)) ++bad, std::printf("dim %d order %d differs\n", dim, p);
            std::swap(fmask[0], fmask[1]);
            if (dgtd::tensor_faces_match(dim, p, fmask)) ++bad, std::printf("dim %d order %d: exchange missed\n", dim, p);
            fmask.pop_back();
            if (dgtd::tensor_faces_match(dim, p, fmask)) ++bad, std::printf("dim %d order %d: size missed\n", dim, p);
        }
    if (!bad) std::printf("OK\n");
    return bad != 0;
}
