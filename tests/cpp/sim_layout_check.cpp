/*
 * sim_layout_check.cpp -- host-side check of the tile that a simulation is laid
 * out in, built from the library's host sources with g++ (no HIP) under
 * AddressSanitizer and UBSan: large networks with deep delays are laid out in
 * tiles of twice the caller's targets, and
 *
 *   1. only a valid tile is doubled, so that an invalid one is refused whatever
 *      the network's size.
 *
 * usage: sim_layout_check (prints "sim_layout_check ok")
 */
#include <stdint.h>
#include <stdio.h>

#include <string>
#include <vector>

#include "../../include/bsim_amd.h"
#include "../../bsim_amd/csrc/internal.h"
#include "../../bsim_amd/csrc/network.h"

thread_local std::string g_bsim_err;

static int fails = 0;
#define CHECK(c, ...)                                        \
    do {                                                     \
        if (!(c)) {                                          \
            fprintf(stderr, "FAIL %s:%d: ", __FILE__, __LINE__); \
            fprintf(stderr, __VA_ARGS__);                    \
            fprintf(stderr, "\n");                           \
            fails++;                                         \
        }                                                    \
    } while (0)

static void check_tile_rule()
{
    for (int64_t n : {100ll, 100000ll, 400000ll, 2000000ll})
        for (int32_t dmax : {1, 24, 25, 63})
            for (int32_t tile = -192; tile <= 4 * BSIM_MAX_TILE; tile++) {
                const int32_t lt = bsim::layout_tile(n, tile, dmax);
                const bool valid = tile > 0 && tile % BSIM_TILE_ALIGN == 0 && tile <= BSIM_MAX_TILE;
                const bool lvalid = lt > 0 && lt % BSIM_TILE_ALIGN == 0 && lt <= BSIM_MAX_TILE;
                CHECK(valid == lvalid && (lt == tile || lt == 2 * tile), "n %lld dmax %d: tile %d laid out in %d",
                      (long long)n, dmax, tile, lt);
            }
    CHECK(bsim::layout_tile(400000, 768, 25) == 1536, "large networks with deep delays");
}

int main()
{
    check_tile_rule();
    if (fails) {
        fprintf(stderr, "sim_layout_check: %d failure(s)\n", fails);
        return 1;
    }
    printf("sim_layout_check ok\n");
    return 0;
}
