/*
 * sim_layout_check.cpp -- host-side check of the tile that a simulation is laid
 * out in, built from the library's host sources with g++ (no HIP) under
 * AddressSanitizer and UBSan: large networks with deep delays are laid out in
 * tiles of twice the caller's targets, and
 *
 *   1. only a valid tile is doubled, so that an invalid one is refused whatever
 *      the network's size;
 *   2. where the groups of the larger tiles would receive too many synapses, the
 *      network is laid out in the caller's tile, and refused only if its groups
 *      do too.
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

static void check_group_limit()
{
    /* 342 tiles of 768; every neuron has two synapses from the first 64: 49,152 per group of 32 tiles */
    const int32_t n = 342 * 768, tile = 768, dmax = 30;
    bsim_network net;
    bsim::HostNet &h = net.net;
    const float row[bsim::kLifParams] = {0, 0, 0, 0.02f, 0.02f, 1e-3f, 5e-3f, 8e-3f, 1.0f, 0.5f, 5e-3f, 8e-3f};
    for (int32_t i = 0; i < n; i++) {
        h.kind.push_back((int8_t)BSIM_KIND_LIF);
        h.lif.insert(h.lif.end(), row, row + bsim::kLifParams);
        h.arr_off.push_back(0);
        h.bern_p.push_back(0u);
        h.bern_seed.push_back(0ull);
        h.bern_key.push_back(0u);
    }
    for (int32_t p = 0; p < 64; p++)
        for (int32_t i = p; i < 2 * n; i += 64) {
            h.pre.push_back(p);
            h.post.push_back(i % n);
            h.w.push_back(0.01f);
            h.d.push_back((float)dmax * 1e-4f);
            h.stype.push_back(0);
        }
    const struct {
        int64_t group_max;
        int rc;
        int32_t tile;
    } cases[] = {{bsim::kGroupSynapses, 0, 2 * tile}, {2 * 49152 + 1, 0, 2 * tile}, {2 * 49152, 0, tile},
                 {49152 + 1, 0, tile}, {49152, bsim::kGroupTooLarge, 0}};
    for (const auto &c : cases) {
        bsim::Layout L;
        std::string err;
        const int rc = bsim::build_sim_layout(h, 1e-4f, tile, dmax, L, err, c.group_max);
        CHECK(rc == c.rc, "limit %lld: %d (%s)", (long long)c.group_max, rc, err.c_str());
        if (rc != 0) {
            CHECK(err.find("use a smaller tile") != std::string::npos, "message: %s", err.c_str());
            continue;
        }
        CHECK(err.empty() && L.tile == c.tile && L.s == h.s() && (int64_t)L.syn_tgt.size() == h.s() &&
                  L.ntiles == (n + L.tile - 1) / L.tile && L.parts == bsim::default_parts(n, L.tile) &&
                  (int32_t)L.tile_rng.size() == L.ntiles + 1, "limit %lld: tile %d", (long long)c.group_max, L.tile);
    }
}

int main()
{
    check_tile_rule();
    check_group_limit();
    if (fails) {
        fprintf(stderr, "sim_layout_check: %d failure(s)\n", fails);
        return 1;
    }
    printf("sim_layout_check ok\n");
    return 0;
}
