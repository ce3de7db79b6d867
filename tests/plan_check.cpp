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
        } else if (!std::strcmp(what, "force32") || !std::strcmp(what, "force64")) {
            long nrows;
            size_t room;
            if (std::scanf("%ld %zu", &nrows, &room) != 2) return 1;
            const gz::ForcePlan p = what[5] == '3' ? gz::force_plan<float>(nrows, room) : gz::force_plan<double>(nrows, room);
            std::printf("%d %d %zu\n", p.blocks, p.segment, p.bytes);
        } else {
            return 1;
        }
    }
    return 0;
}
