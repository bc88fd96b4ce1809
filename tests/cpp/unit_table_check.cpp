/*
 * unit_table_check.cpp -- host-side check of the row tables as the step kernel
 * reads them, with a tile as one unit and as one unit per part, built from the
 * library's host sources with g++ (no HIP) under AddressSanitizer and UBSan:
 *
 *   for each unit, the sub-rows [entry, next entry) of its source chunks' rows,
 *   in order, hold exactly the synapses of the unit's targets, each target's in
 *   creation order; they ascend through the group's synapses, whose number the
 *   group's last entry holds; every entry read, and the one after it, exists.
 *
 * For networks with gaps between their sources, several segments per target,
 * more pres than a chunk, targets without a synapse, and for sweep networks
 * joined from parts.  usage: unit_table_check (prints "unit_table_check ok")
 */
#include <stdint.h>
#include <stdio.h>
#include <string.h>

#include <algorithm>
#include <functional>
#include <random>
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
            if (++fails > 20) exit(1);                       \
        }                                                    \
    } while (0)

static const float kDt = 1e-4f;

struct Syn {
    int32_t pre, d;
    float w;
};

static void check_tables(const bsim::Layout &L, const bsim::HostNet &h, const char *what)
{
    const int32_t n = L.n, U = L.tile / L.parts, D = L.dmax;
    std::vector<std::vector<Syn>> want((size_t)n), got((size_t)n);
    for (int64_t k = 0; k < h.s(); k++) {
        Syn s;
        s.pre = h.pre[k];
        const float *pd = &h.lif[(size_t)h.post[k] * bsim::kLifParams];
        CHECK(bsim::synapse_reset(h.w[k], h.d[k], h.stype[k] ? pd[11] : pd[10], kDt, &s.w, &s.d), "reset");
        want[(size_t)h.post[k]].push_back(s);
    }
    std::vector<int64_t> seen((size_t)L.s, 0);
    const int32_t units = (n + U - 1) / U;
    for (int32_t u = 0; u < units; u++) {
        const int32_t t = u / L.parts, part = u % L.parts;
        int64_t last = -1;              /* the end of the unit's sub-row before */
        for (int32_t ri = L.tile_rng[t]; ri < L.tile_rng[t + 1]; ri++) {
            const bsim_range &r = L.rng[ri];
            CHECK(r.lo % 64 == 0 && r.hi % 64 == 0 && r.hi - r.lo <= BSIM_CHUNK && r.lo >= 0 &&
                      (r.hi - 1) / 64 <= (n - 1) / 64, "%s: chunk [%d, %d)", what, r.lo, r.hi);
            for (int32_t p = r.lo; p < r.hi; p++)
                for (int32_t d = 1; d <= D; d++) {
                    const int64_t e = r.off_base + part + ((int64_t)(p - r.lo) * D + d - 1) * r.stride;
                    CHECK(e >= 0 && e + 1 < (int64_t)L.off_tab.size(), "%s: entry out of the table", what);
                    const uint32_t a = L.off_tab[e], b = L.off_tab[e + 1];
                    CHECK(a <= b && b <= L.tile_nsyn[t] && (int64_t)a >= last, "%s: sub-row %u..%u", what, a, b);
                    last = b;
                    for (uint32_t i = a; i < b; i++) {
                        const int64_t x = L.tile_base[t] + i;
                        const int32_t tgt = L.syn_tgt[x];
                        CHECK(tgt >= part * U && tgt < (part + 1) * U, "%s: target %d in part %d", what, tgt, part);
                        const int64_t id = (int64_t)t * L.tile + tgt;
                        CHECK(id < n, "%s: target past the last neuron", what);
                        if (id < n) got[(size_t)id].push_back(Syn{p, d, L.syn_w[x]});
                        seen[(size_t)x]++;
                    }
                }
        }
    }
    for (int64_t x = 0; x < L.s; x++) CHECK(seen[(size_t)x] == 1, "%s: synapse %lld in %lld sub-rows", what,
                                            (long long)x, (long long)seen[(size_t)x]);
    for (int32_t i = 0; i < n; i++) {
        bool same = want[i].size() == got[i].size();
        for (size_t k = 0; same && k < want[i].size(); k++)
            same = want[i][k].pre == got[i][k].pre && want[i][k].d == got[i][k].d &&
                   memcmp(&want[i][k].w, &got[i][k].w, 4) == 0;
        CHECK(same, "%s: inputs of neuron %d", what, i);
    }
    /* the group's last entry: where the next group's table, or the array, ends */
    for (int32_t t = 0; t < L.ntiles; t++) {
        if (t + 1 < L.ntiles && L.tile_base[t + 1] == L.tile_base[t] && L.tile_nsyn[t] > 0) continue;
        if (L.tile_rng[t] == L.tile_rng[t + 1]) continue;
        const bsim_range &r = L.rng[(size_t)L.tile_rng[t + 1] - 1];
        const int64_t end = r.off_base + ((int64_t)(r.hi - r.lo) * D - 1) * r.stride + L.parts;
        CHECK(end < (int64_t)L.off_tab.size() && L.off_tab[end] == L.tile_nsyn[t], "%s: end of the group of tile %d",
              what, t);
    }
}

static void add_lif(bsim::HostNet &h, int32_t n)
{
    const float row[bsim::kLifParams] = {0, 0, 0, 0.02f, 0.02f, 1e-3f, 5e-3f, 8e-3f, 1.0f, 0.5f, 5e-3f, 8e-3f};
    for (int32_t i = 0; i < n; i++) {
        h.kind.push_back((int8_t)BSIM_KIND_LIF);
        h.lif.insert(h.lif.end(), row, row + bsim::kLifParams);
        h.arr_off.push_back(h.arr_off.back());
        h.bern_p.push_back(0u);
        h.bern_seed.push_back(0ull);
        h.bern_key.push_back(0u);
    }
}

static void add_inert(bsim::HostNet &h, int32_t n)
{
    for (int32_t i = 0; i < n; i++) {
        h.kind.push_back((int8_t)BSIM_KIND_ARRAY);
        h.lif.insert(h.lif.end(), (size_t)bsim::kLifParams, 0.0f);
        h.arr_off.push_back(h.arr_off.back());
        h.bern_p.push_back(0u);
        h.bern_seed.push_back(0ull);
        h.bern_key.push_back(0u);
    }
}

/* runs: connections made in so many passes over ascending (pre, delay), each a
 * segment of every target it reaches; gap: pres in clusters so far apart */
static void check_net(int32_t n, int64_t syn, int32_t dmax, int32_t runs, int32_t gap, uint32_t seed, const char *what)
{
    std::mt19937 r(seed);
    bsim_network net;
    bsim::HostNet &h = net.net;
    add_lif(h, n);
    for (int32_t run = 0; run < runs; run++) {
        struct C {
            int32_t pre, d, post;
        };
        std::vector<C> c((size_t)(syn / runs));
        for (C &x : c) {
            x.pre = (int32_t)(r() % (uint32_t)n);
            if (gap) x.pre = x.pre / gap * gap + x.pre % 7;
            x.pre = std::min(x.pre, n - 1);
            x.d = 1 + (int32_t)(r() % (uint32_t)dmax);
            x.post = (int32_t)(r() % (uint32_t)n);
            if (x.post % 5 == 0) x.post = std::min(1, n - 1);            /* some targets have none */
        }
        std::stable_sort(c.begin(), c.end(), [](const C &a, const C &b) { return a.pre != b.pre ? a.pre < b.pre : a.d < b.d; });
        for (const C &x : c) {
            h.pre.push_back(x.pre);
            h.post.push_back(x.post);
            h.w.push_back(((int)(r() % 2000) - 800) * 1e-3f);
            h.d.push_back((float)x.d * kDt);
            h.stype.push_back((int8_t)(r() % 2));
        }
    }
    for (int32_t tile : {192, 768})
        for (int32_t parts : {1, BSIM_NWAVE}) {
            bsim::Layout L;
            std::string err;
            const int rc = bsim::build_layout(h, kDt, tile, L, err, 0, parts);
            CHECK(rc == 0, "%s: %s", what, err.c_str());
            if (rc != 0) continue;
            const std::string s = std::string(what) + " tile " + std::to_string(tile) + " parts " + std::to_string(parts);
            check_tables(L, h, s.c_str());
        }
}

static void check_chains(int32_t count, int64_t part_syn, int32_t tile, int32_t parts, uint32_t seed)
{
    std::mt19937 r(seed);
    std::vector<bsim_chain_params> p((size_t)count);
    for (auto &q : p) {
        memset(&q, 0, sizeof(q));
        q.npop = 2 + (int)(r() % 3);
        for (int i = 0; i < q.npop; i++) q.sizes[i] = 100 + (int)(r() % 500);
        q.fan_in = 10 + (int)(r() % 30);
        q.w0 = 0.6f;
        q.inh_frac = 0.2f;
        q.dmax = 6 + (int)(r() % 12);
        q.drive_rate_hz = 20.0f;
        q.n_drive = 100;
        q.drive_fan_in = 10;
        q.drive_w = 1.0f;
        q.seed = 1000 + r();
        q.tau_refrac = 2e-3f;
        q.ioff_lo = 14.5f;
        q.ioff_hi = 16.5f;
        q.tau_syn_E = 5e-3f;
        q.tau_syn_I = 10e-3f;
        q.v_thresh = 15.0f;
        q.dt = kDt;
    }
    int64_t nn = 0, ns = 0;
    int32_t dmax = 1;
    CHECK(bsim::chains_size(p.data(), count, &nn, &ns, &dmax) == 0, "chains_size");
    std::vector<uint16_t> tgt((size_t)ns);
    std::vector<float> w((size_t)ns);
    std::vector<int64_t> ends;
    auto upload = [&](const bsim::Layout &pl, int64_t s0) -> int {
        std::copy(pl.syn_tgt.begin(), pl.syn_tgt.end(), tgt.begin() + s0);
        std::copy(pl.syn_w.begin(), pl.syn_w.end(), w.begin() + s0);
        ends.push_back(s0 + (int64_t)pl.syn_tgt.size());
        return 0;
    };
    bsim::Layout J;
    std::vector<int32_t> first((size_t)count);
    std::string err;
    CHECK(bsim::build_chains_layout(p.data(), count, kDt, tile, dmax, part_syn, J, first.data(), err, upload, parts) == 0,
          "build_chains_layout: %s", err.c_str());
    CHECK(ends.size() >= 2, "expected several parts");
    J.syn_tgt = tgt;
    J.syn_w = w;
    /* the same network, each part padded to whole tiles */
    bsim_network one;
    int32_t c0 = 0;
    for (int64_t end : ends) {
        int32_t c1 = c0;
        int64_t syn = one.net.s(), a, b;
        int32_t d;
        while (c1 < count && syn < end) {
            CHECK(bsim::chains_size(&p[(size_t)c1], 1, &a, &b, &d) == 0, "chains_size");
            syn += b;
            c1++;
        }
        std::vector<int32_t> f((size_t)(c1 - c0));
        bsim_net_gen_chains(&one, &p[(size_t)c0], c1 - c0, f.data());
        add_inert(one.net, (tile - one.net.n() % tile) % tile);
        c0 = c1;
    }
    CHECK(c0 == count && J.parts == parts, "chains joined");
    check_tables(J, one.net, "joined chains");
}

int main()
{
    check_net(1000, 30000, 5, 1, 0, 1, "one range");
    check_net(5003, 40000, 3, 2, 1100, 2, "clusters of sources, two segments");
    check_net(9001, 60000, 7, 5, 0, 3, "more pres than a chunk, five segments");
    check_net(130, 500, 63, 3, 0, 4, "one tile");
    check_net(1, 9, 4, 2, 0, 5, "one neuron");
    for (int32_t parts : {1, BSIM_NWAVE}) {
        check_chains(7, 20000, 192, parts, 6);
        check_chains(5, 1, 384, parts, 7);
        check_chains(6, 40000, 768, parts, 8);
    }
    if (fails) {
        fprintf(stderr, "unit_table_check: %d failure(s)\n", fails);
        return 1;
    }
    printf("unit_table_check ok\n");
    return 0;
}
