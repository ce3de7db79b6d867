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
        } else if (!std::strcmp(what, "by_row")) {
            // the groups, the rows still iterating, then the kinds of boxes: how many, particles and cells of one
            long ngroups, remaining, kinds;
            if (std::scanf("%ld %ld %ld", &ngroups, &remaining, &kinds) != 3) return 1;
            std::vector<gz::BoxCells> boxes;
            while (kinds-- > 0) {
                long count;
                gz::BoxCells one;
                if (std::scanf("%ld %ld %ld", &count, &one.particles, &one.cells) != 3) return 1;
                boxes.insert(boxes.end(), (size_t)count, one);
            }
            const double per_cell = gz::fullest_cells(boxes);
            std::printf("%d %.17g\n", gz::density_by_row(remaining, ngroups, per_cell), per_cell);
        } else if (!std::strcmp(what, "parts")) {
            long ngroups;
            if (std::scanf("%ld", &ngroups) != 1) return 1;
            std::printf("%u\n", gz::group_parts(ngroups));
        } else if (!std::strcmp(what, "lanes")) {
            long nrows;
            double share, even;
            if (std::scanf("%ld %lf %lf", &nrows, &share, &even) != 3) return 1;
            std::printf("%d\n", gz::force_by_lanes(nrows, share, even));
        } else {
            return 1;
        }
    }
    return 0;
}
