// Prints what the launch arithmetic of gizmo_amd/csrc/gz_plan.h answers: one question per line of
// the standard input, one answer per line (tests/test_plan.py).
#include <cstdio>
#include <cstring>

#include "gz_plan.h"

int main()
{
    char what[32];
    while (std::scanf("%31s", what) == 1) {
        if (!std::strcmp(what, "stencil")) {
            long ncell;
            if (std::scanf("%ld", &ncell) != 1) return 1;
            std::printf("%u\n", gz::stencil_grid(ncell));
        } else {
            return 1;
        }
    }
    return 0;
}
