// Host check of the unfolded-image move arithmetic (walk_common.h) for noflux
// faces and voxel division, over every voxel and direction of small images:
// a noflux move turns around exactly where a walker in a face voxel would step
// outwards, and a sub-voxel address shifted by 3 bits per division is the
// undivided image's address of the walker's voxel, mirror reflection included.
// Also: the walker counts whose position sort fits its int item count.
#include <cstdio>
#include <cstdlib>

#include "../../randomwalk_nmr_amd/csrc/walk_common.h"

using namespace rwnmr;

static long fails = 0, checks = 0;
#define EXPECT(c, ...)                  \
    do {                                \
        ++checks;                       \
        if (!(c) && ++fails < 20)       \
            std::printf(__VA_ARGS__);   \
    } while (0)

int main()
{
    const uint32_t dims[][3] = {{2, 2, 2}, {8, 8, 8}, {16, 4, 2}, {5, 7, 3}, {3, 12, 2}, {9, 2, 6}};
    for (const auto &d : dims)
        for (uint32_t shift = 0; shift <= 2; ++shift) {
            ZLayout vox{}, sub{};
            EXPECT(zlayout_make(d[0], d[1], d[2], vox) == 1, "layout\n");
            EXPECT(zlayout_make(d[0] << shift, d[1] << shift, d[2] << shift, sub) == 1, "sub layout\n");
            EXPECT(sub.bits == vox.bits + 3u * shift, "bits\n");
            const uint32_t n[3] = {d[0] << shift, d[1] << shift, d[2] << shift};
            for (uint32_t z = 0; z < n[2]; ++z)
                for (uint32_t y = 0; y < n[1]; ++y)
                    for (uint32_t x = 0; x < n[0]; ++x) {
                        const uint32_t u[3] = {x, y, z};
                        const uint32_t A = zdeposit(x, sub.m[0]) | zdeposit(y, sub.m[1]) | zdeposit(z, sub.m[2]);
                        const uint32_t V = zdeposit(x >> shift, vox.m[0]) | zdeposit(y >> shift, vox.m[1]) |
                                           zdeposit(z >> shift, vox.m[2]);
                        EXPECT(A >> (3u * shift) == V, "voxel of sub-voxel\n");
                        for (uint32_t idx = 0; idx < 6; ++idx) {
                            const uint32_t r = zdir_residue(idx);
                            const int ax = move_axis(r);
                            int sg = move_sign(r);
                            const uint32_t g = u[ax] >> shift;
                            if ((sg < 0 && g == 0) || (sg > 0 && g == d[ax] - 1))
                                sg = -sg;
                            uint32_t v[3] = {x, y, z};
                            v[ax] = (uint32_t)((int)v[ax] + sg);
                            const uint32_t want =
                                zdeposit(v[0], sub.m[0]) | zdeposit(v[1], sub.m[1]) | zdeposit(v[2], sub.m[2]);
                            EXPECT(zmove_face(A, zdir_face(sub, idx, shift)) == want,
                                   "noflux %u,%u,%u shift %u at %u,%u,%u idx %u\n", d[0], d[1], d[2], shift, x, y, z,
                                   idx);
                        }
                    }
            // mirror: the folded sub-voxel coordinate falls in the folded voxel
            for (int a = 0; a < 3; ++a)
                for (int g = -3 * (int)n[a]; g < 3 * (int)n[a]; ++g) {
                    EXPECT(fold_mirror(g, (int)n[a]) >> shift == fold_mirror(g >> shift, (int)d[a]), "mirror fold\n");
                    EXPECT(mirror_flag(g, (int)n[a]) == mirror_flag(g >> shift, (int)d[a]), "mirror flag\n");
                    EXPECT(fold_periodic(g, (int)n[a]) >> shift == fold_periodic(g >> shift, (int)d[a]), "periodic\n");
                }
        }
    const uint64_t counts[] = {0ull, 1ull, 0x7FFFFFFFull, 0x80000000ull, 0xFFFFFFFFull, 0x100000000ull, 0x100000001ull};
    for (uint64_t n : counts)
        EXPECT(position_sort_takes(n) == (n < (1ull << 31)), "sort of %llu\n", (unsigned long long)n);
    std::printf("%ld checks, %ld failures\n", checks, fails);
    return fails ? 1 : 0;
}
