// Checks of the resident solve's partition on the CPU (test_partition.py):
//   partition_check scenes CELLS,CELLS,... TARGET REAL DAMP FIXED CUS LDS
// builds Kuhn cubes of the given cells per edge as one batch, partitions it and
// checks every table the kernel reads against the tets and colours; prints
// "fits PATCHES LDS" or "does not fit".
//   partition_check memory
// lets the n-th allocation of a partition fail, for n = 1, 2, 4, ..., in whichever
// thread makes it: each must come out as std::bad_alloc.
#include <atomic>
#include <cstdio>
#include <cstdlib>
#include <cstring>
#include <new>
#include <set>
#include <string>

#include "resident.hpp"

using namespace avbd;

static std::atomic<long> allocations_left{-1};   // < 0: no limit
void* operator new(size_t n) {
    if (allocations_left.load() >= 0 && allocations_left.fetch_sub(1) <= 0) {
        allocations_left = 0;
        throw std::bad_alloc();
    }
    if (void* p = std::malloc(n ? n : 1)) return p;
    throw std::bad_alloc();
}
void operator delete(void* p) noexcept { std::free(p); }
void operator delete(void* p, size_t) noexcept { std::free(p); }

#define CHECK(c)                                              \
    do {                                                      \
        if (!(c)) {                                           \
            std::printf("line %d: %s\n", __LINE__, #c);      \
            std::exit(1);                                     \
        }                                                     \
    } while (0)

struct Batch {
    std::vector<HostNH> nh;
    std::vector<double> x;
    std::vector<uint32_t> scenes{0};
    std::vector<uint8_t> fixed;
    std::vector<HostGround> ground;
    std::vector<HostCos> cos;
    std::vector<HostRGround> rground;
    std::vector<HostJoint> joints;
    std::vector<HostJoint2> joints2;
    std::vector<int32_t> rot_of;
    HostModel model;
    ColorPlan plan;

    Batch(const std::vector<int>& cells, bool fix_top) {
        for (int n : cells) {
            const uint32_t base = scenes.back();
            const int m = n + 1;
            auto id = [&](const int* c) { return base + (uint32_t)((c[0] * m + c[1]) * m + c[2]); };
            for (int i = 0; i < m * m * m; i++)
                for (int v : {i / (m * m), i / m % m, i % m}) x.push_back(v / (double)n);
            const int paths[6][3] = {{0, 1, 2}, {0, 2, 1}, {1, 0, 2}, {1, 2, 0}, {2, 0, 1}, {2, 1, 0}};
            for (int i = 0; i < n * n * n; i++)
                for (auto& path : paths) {
                    int c[3] = {i / (n * n), i / n % n, i % n};
                    HostNH h{};
                    h.idx[0] = id(c);
                    for (int a = 0; a < 3; a++) {
                        c[path[a]]++;
                        h.idx[a + 1] = id(c);
                    }
                    nh.push_back(h);
                }
            scenes.push_back((uint32_t)(x.size() / 3));
        }
        const uint32_t n = scenes.back();
        fixed.assign(n, 0);
        for (uint32_t v = 0; v < n && fix_top; v++) fixed[v] = x[3 * v + 1] > 1 - 1e-9;
        rot_of.assign(n, -1);
        model.n = n;
        model.nh = &nh;
        model.ground = &ground;
        model.cos = &cos;
        model.rground = &rground;
        model.joints = &joints;
        model.joints2 = &joints2;
        model.fixed = &fixed;
        model.rot_of = &rot_of;
        model.scene_offsets = &scenes;
        build_color_plan(model, plan);
    }
};

static void check(const Batch& b, const ResidentLimits& lim, const ResidentPlan& out) {
    const uint32_t n = b.model.n, nc = b.plan.num_colors, words = lim.real_bytes == 8 ? 6 : 3;
    const size_t np = out.patches.size();
    std::vector<int> owner(n, -1);
    for (size_t q = 0; q < np; q++) {
        const ResidentPatch& p = out.patches[q];
        CHECK(p.first <= q && q < p.first + p.count && p.count <= lim.max_cluster);
        for (uint32_t k = 0; k < p.own; k++) {
            const uint32_t v = out.gid[p.gid_off + k];
            CHECK(v >= b.scenes[p.scene] && v < b.scenes[p.scene + 1] && owner[v] < 0);
            owner[v] = (int)q;
        }
    }
    for (uint32_t v = 0; v < n; v++) CHECK(owner[v] >= 0);   // every particle is owned once
    std::vector<uint32_t> slot_of(out.slots, ~0u);           // every halo copy has a slot of its own
    for (const ResidentPatch& p : out.patches)
        for (uint32_t k = p.own; k < p.local; k++) {
            CHECK(slot_of[p.slot + k - p.own] == ~0u);
            slot_of[p.slot + k - p.own] = out.gid[p.gid_off + k];
        }
    std::vector<std::set<uint32_t>> halo(np);
    uint64_t sent = 0, held = 0;
    for (size_t q = 0; q < np; q++) {
        const ResidentPatch& p = out.patches[q];
        const uint32_t bytes =
            resident_lds(p.own, p.items, p.local, p.tets, p.inc, p.targets, nc, lim.real_bytes, lim.damp, lim.ground).total;
        CHECK(bytes <= out.lds_bytes && out.lds_bytes <= lim.lds_bytes);
        const uint32_t *items = &out.col[p.col_off], *copies = items + nc + 1, *gid = &out.gid[p.gid_off];
        CHECK(items[0] == 0 && items[nc] == p.items && copies[0] == p.own && copies[nc] <= p.local);
        for (uint32_t c = 0; c < nc; c++) {
            CHECK(items[c] <= items[c + 1] && copies[c] <= copies[c + 1]);
            for (uint32_t k = items[c]; k < items[c + 1]; k++) {
                const uint32_t v = gid[k], inc = out.item[2 * (p.item_off + k)], to = out.item[2 * (p.item_off + k) + 1];
                const VItem& it = b.plan.item_of[v];
                CHECK(b.plan.item_kind[v] == 1 && b.plan.color[v] == c);
                CHECK((to & 0xffff) + (to >> 16) <= p.targets);
                for (uint32_t e = 0; e < to >> 16; e++) {   // sent to copies of itself
                    const uint32_t word = out.target[p.target_off + (to & 0xffff) + e];
                    CHECK(word % words == 0 && word / words < out.slots && slot_of[word / words] == v);
                }
                CHECK(inc >> 16 == it.inc_count && (inc & 0xffff) + it.inc_count <= p.inc);
                for (uint32_t e = 0; e < it.inc_count; e++) {   // the same incidences in the same order
                    const uint16_t* r = &out.inc[4 * (size_t)(p.inc_off + (inc & 0xffff) + e)];
                    CHECK((uint32_t)(r[3] >> 2) < p.tets);
                    const uint32_t t = out.tet[p.tet_off + (r[3] >> 2)];
                    CHECK((t << 2 | (r[3] & 3u)) == b.plan.inc[it.inc_begin + e]);
                    for (int j = 0; j < 3; j++)
                        CHECK(r[j] < p.local && gid[r[j]] == b.nh[t].idx[kEdgeCorner[r[3] & 3][j]]);
                }
            }
            for (uint32_t k = copies[c]; k < copies[c + 1]; k++) {
                const uint32_t v = gid[k];
                CHECK(b.plan.item_kind[v] == 1 && b.plan.color[v] == c && owner[v] != (int)q);
                CHECK(owner[v] >= (int)p.first && owner[v] < (int)(p.first + p.count));
                halo[q].insert(v);
            }
        }
        for (uint32_t k = copies[nc]; k < p.local; k++) CHECK(b.plan.item_kind[gid[k]] != 1);
        for (uint32_t t = 0; t < p.tets; t++)
            for (int a = 0; a < 4; a++) {
                const uint32_t l = out.tix[4 * (p.tet_off + t) + a];
                CHECK(l < p.local && gid[l] == b.nh[out.tet[p.tet_off + t]].idx[a]);
            }
        sent += p.targets;
        held += halo[q].size();
    }
    CHECK(sent == held);   // every copy is refreshed, none is sent to twice
    // A reader computes something from the copy that the owner waits for, so a word
    // is read before it is written again.
    for (size_t q = 0; q < np; q++)
        for (uint32_t v : halo[q]) {
            bool answered = false;
            for (uint32_t e = b.plan.static_off[v]; e < b.plan.static_off[v + 1] && !answered; e++) {
                const uint32_t u = b.plan.static_nb[e];
                answered = owner[u] == (int)q && b.plan.item_kind[u] == 1 && halo[owner[v]].count(u);
            }
            CHECK(answered);
        }
}

int main(int argc, char** argv) {
    if (argc == 2 && !std::strcmp(argv[1], "memory")) {
        for (const std::vector<int>& cells : {std::vector<int>{24}, std::vector<int>(24, 6)}) {
            const Batch b(cells, false);
            const ResidentLimits lim{4, false, true, 160 * 1024 - 1024, 256, 1000};
            ResidentPlan out;
            bool done = false;
            for (long n = 1; !done; n *= 2) {
                allocations_left = n;
                try {
                    CHECK(build_resident(b.model, b.plan, b.x.data(), lim, out));
                    done = allocations_left > 0;   // (a failure that a thread start met is made up for)
                } catch (const std::bad_alloc&) {
                }
                allocations_left = -1;
            }
            check(b, lim, out);
        }
        std::puts("every failure came out");
        return 0;
    }
    CHECK(argc == 9 && !std::strcmp(argv[1], "scenes"));
    std::vector<int> cells;
    for (const char* s = argv[2]; s; s = std::strchr(s, ',') ? std::strchr(s, ',') + 1 : nullptr) cells.push_back(std::atoi(s));
    const Batch b(cells, std::atoi(argv[6]) != 0);
    const ResidentLimits lim{(uint32_t)std::atoi(argv[4]), std::atoi(argv[5]) != 0, true, (uint32_t)std::atoi(argv[8]),
                             (uint32_t)std::atoi(argv[7]), (uint32_t)std::atoi(argv[3])};
    ResidentPlan out;
    if (!build_resident(b.model, b.plan, b.x.data(), lim, out)) {
        std::puts("does not fit");
        return 0;
    }
    check(b, lim, out);
    std::printf("fits %zu %u\n", out.patches.size(), out.lds_bytes);
}
