// Native check of how a frame is split over the device (march_lanes,
// batch_lanes, row_rotation and order_auto in pyvr_amd/csrc/hvr_rules.h): more
// rays never get more lanes, and the lines lie where the rules put them for
// 524,288 resident rays; the blocks of a frame in row order, rotated or not, are
// each dispatched once and stay in their class's rows; the ordering rule on both
// sides of each of its conditions, for one and for two lanes.  Exit status 0 on
// success.
#include <stdio.h>

#include <vector>

#include "hvr_rules.h"

using namespace hvr;

static int fails = 0;
#define CHECK(cond)                                                         \
    do {                                                                    \
        if (!(cond)) {                                                      \
            fprintf(stderr, "FAIL %s:%d: %s\n", __FILE__, __LINE__, #cond); \
            ++fails;                                                        \
        }                                                                   \
    } while (0)

int main()
{
    constexpr long long R = 524288;
    constexpr unsigned long long small = 8ull << 20, large = 1ull << 30;
    for (double steps : {100.0, 300.0, 700.0})
        for (bool skipping : {false, true})
            for (int texel : {1, 4, 8, 16})
                for (unsigned long long bytes : {small, large}) {
                    int before = 4;
                    for (long long rays = 1; rays < 4 * R; rays += 4099) {
                        const int lanes = march_lanes(rays, R, skipping, steps, texel, bytes);
                        CHECK(lanes == 1 || lanes == 2 || lanes == 4);
                        CHECK(lanes <= before);
                        before = lanes;
                    }
                    CHECK(before == 1);
                    CHECK(march_lanes(1, R, skipping, steps, texel, bytes) == 4);
                }
    // bricks stepped over: 4 lanes up to 3/8 of the resident rays, with long rays 7/8; 2 up to 9/4
    CHECK(march_lanes(3 * R / 8, R, true, 300, 8, small) == 4 && march_lanes(3 * R / 8 + 1, R, true, 300, 8, small) == 2);
    CHECK(march_lanes(7 * R / 8, R, true, 700, 8, small) == 4 && march_lanes(7 * R / 8 + 1, R, true, 700, 8, small) == 2);
    CHECK(march_lanes(9 * R / 4, R, true, 300, 8, small) == 2 && march_lanes(9 * R / 4 + 1, R, true, 300, 8, small) == 1);
    // none: by steps, texels and volume
    CHECK(march_lanes(5 * R / 16, R, false, 100, 8, small) == 4 && march_lanes(5 * R / 16 + 1, R, false, 100, 8, small) == 2);
    CHECK(march_lanes(9 * R / 16, R, false, 100, 8, large) == 2 && march_lanes(9 * R / 16 + 1, R, false, 100, 8, large) == 1);
    CHECK(march_lanes(3 * R / 8, R, false, 300, 8, small) == 4 && march_lanes(3 * R / 8 + 1, R, false, 300, 8, small) == 2);
    CHECK(march_lanes(R / 2, R, false, 700, 8, small) == 4 && march_lanes(R / 2 + 1, R, false, 700, 8, small) == 2);
    CHECK(march_lanes(3 * R / 4, R, false, 300, 8, small) == 2 && march_lanes(3 * R / 4 + 1, R, false, 300, 8, small) == 1);
    CHECK(march_lanes(3 * R / 2, R, false, 300, 16, small) == 2 && march_lanes(3 * R / 2 + 1, R, false, 300, 8, large) == 1);
    CHECK(march_lanes(3 * R / 4, R, false, 100, 2, small) == 4 && march_lanes(3 * R / 4 + 1, R, false, 700, 2, small) == 1);
    // batches
    for (double steps : {10.0, 63.0, 64.0, 255.0, 256.0, 511.0, 512.0, 1024.0, 5000.0}) {
        int before = 4;
        for (long long rays = 1; rays < 4 * R; rays += 4099) {
            const int lanes = batch_lanes(rays, R, steps);
            CHECK((lanes == 1 || lanes == 2 || lanes == 4) && lanes <= before);
            before = lanes;
        }
        CHECK(before == 1);
    }
    CHECK(batch_lanes(R / 10, R, 50) == 4 && batch_lanes(R / 10 + 1, R, 50) == 2 && batch_lanes(R / 4 + 1, R, 50) == 1);
    CHECK(batch_lanes(R / 4, R, 100) == 4 && batch_lanes(R / 4 + 1, R, 100) == 2 && batch_lanes(3 * R / 4 + 1, R, 100) == 1);
    CHECK(batch_lanes(3 * R / 8, R, 346) == 4 && batch_lanes(3 * R / 8 + 1, R, 346) == 2);
    CHECK(batch_lanes(5 * R / 4, R, 346) == 2 && batch_lanes(5 * R / 4 + 1, R, 346) == 1);
    CHECK(batch_lanes(7 * R / 4, R, 692) == 2 && batch_lanes(7 * R / 4 + 1, R, 692) == 1);
    CHECK(batch_lanes(9 * R / 4, R, 2000) == 2 && batch_lanes(9 * R / 4 + 1, R, 2000) == 1);

    // k_march's mapping in row order
    for (int ntx = 1; ntx <= 300; ++ntx) {
        const int rot = row_rotation(ntx);
        CHECK(rot >= 0 && rot < ntx);
        CHECK(ntx >= 16 || rot == 0);
        const int rows = 24, head = rows * ntx;
        std::vector<char> seen((size_t)head, 0);
        for (int b = 0; b < head; ++b) {
            const int j = b >> 3, row = j / ntx, logical = (row * 8 + (b & 7)) * ntx + (j + row * rot) % ntx;
            CHECK(logical >= 0 && logical < head && logical / ntx % 8 == (b & 7) && !seen[(size_t)logical]);
            if (logical >= 0 && logical < head) seen[(size_t)logical] = 1;
        }
    }
    CHECK(row_rotation(32) == 19 && row_rotation(64) == 19 && row_rotation(40) == 0);

    // 1024^2: 4096 blocks of one lane, 8192 of two; 692 or 346 or 173 steps
    CHECK(order_auto(4096, 1 << 20, R, true, 1, 346) && !order_auto(4096, 1 << 20, R, true, 1, 173));
    CHECK(!order_auto(2048, R, R, true, 1, 692) && order_auto(2049, R, R, true, 1, 692));   // all resident at once
    CHECK(order_auto(9 * 512, 9 * R / 4, R, true, 1, 692) && !order_auto(9 * 512 + 1, 9 * R / 4 + 1, R, true, 1, 692));
    CHECK(order_auto(9 * 512 + 1, 9 * R / 4 + 1, R, false, 1, 692) && !order_auto(9 * 512 + 1, 9 * R / 4 + 1, R, false, 1, 173));
    CHECK(order_auto(4096, 1 << 20, R, false, 1, 346) && !order_auto(2048, R, R, false, 1, 692));
    for (bool skipping : {false, true})
        CHECK(order_auto(8192, 1 << 20, R, skipping, 2, 692) && !order_auto(8192, 1 << 20, R, skipping, 2, 346));
    if (fails) return 1;
    printf("split ok\n");
    return 0;
}
