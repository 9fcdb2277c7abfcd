// resident_host.cpp -- partition of the scenes into patches for the resident
// solve (resident.hpp).
#include <algorithm>
#include <atomic>
#include <cmath>
#include <future>
#include <numeric>
#include <thread>

#include "resident.hpp"

namespace avbd {

namespace {

constexpr uint32_t NONE = 0xFFFFFFFFu;
// a thread of its own, or the caller's at get() when the system has none to give
constexpr std::launch kThreads = std::launch::async | std::launch::deferred;

// Recursive coordinate bisection: parts [0, parts) of the particles in
// idx[lo, hi), each cut along the longest side of the box so that the weight
// divides in proportion to the parts of the two sides.
void bisect(uint32_t* idx, uint32_t lo, uint32_t hi, uint32_t first, uint32_t parts, const double* pos,
            const uint32_t* weight, uint32_t base, uint32_t* part, uint32_t threads) {
    if (parts <= 1 || hi - lo <= 1) {
        for (uint32_t k = lo; k < hi; k++) part[idx[k]] = first;
        return;
    }
    double mn[3] = {1e300, 1e300, 1e300}, mx[3] = {-1e300, -1e300, -1e300};
    uint64_t total = 0;
    for (uint32_t k = lo; k < hi; k++) {
        const double* p = pos + 3 * (size_t)(base + idx[k]);
        for (int a = 0; a < 3; a++) {
            mn[a] = std::min(mn[a], p[a]);
            mx[a] = std::max(mx[a], p[a]);
        }
        total += weight[idx[k]];
    }
    int axis = 0;
    for (int a = 1; a < 3; a++)
        if (mx[a] - mn[a] > mx[axis] - mn[axis]) axis = a;
    // ties by index, so that the cut does not depend on the sort
    std::vector<std::pair<double, uint32_t>> key(hi - lo);
    for (uint32_t k = lo; k < hi; k++) key[k - lo] = {pos[3 * (size_t)(base + idx[k]) + axis], idx[k]};
    std::sort(key.begin(), key.end());
    for (uint32_t k = lo; k < hi; k++) idx[k] = key[k - lo].second;
    const uint32_t left = parts / 2;
    const uint64_t want = total * left / parts;
    uint64_t sum = 0;
    uint32_t cut = lo;
    while (cut < hi && sum + weight[idx[cut]] <= want) sum += weight[idx[cut++]];
    // the two sides touch different particles (a failure in either comes out of
    // get() or of this call, which then waits for the other)
    std::future<void> side;
    if (hi - lo > 4096 && threads > 1)
        side = std::async(kThreads, bisect, idx, lo, cut, first, left, pos, weight, base, part, threads / 2);
    else bisect(idx, lo, cut, first, left, pos, weight, base, part, 1);
    bisect(idx, cut, hi, first + left, parts - left, pos, weight, base, part, threads - threads / 2);
    if (side.valid()) side.get();
}

// Coordinates of the particles [lo, lo + n) along the edges of a tet: the two
// shortest that are not parallel, made orthogonal, and their normal.  A
// structured mesh is then cut along its cells however it is turned (cut along
// the world's axes, a turned 32^3 cube in FP64 had patches with up to a third more
// halo, did not always fit and was stepped at 30 instead of 14 us per
// iteration).  Rounded to a thousandth of an edge, so that a layer's particles tie
// and are cut in index order instead of by the last bits of the rotation.
std::vector<double> mesh_coordinates(const double* pos, uint32_t lo, uint32_t n, const uint32_t* corner) {
    double e[6][3], len[6];
    uint32_t order[6] = {0, 1, 2, 3, 4, 5}, k = 0;
    for (int a = 0; a < 4; a++)
        for (int b = a + 1; b < 4; b++, k++) {
            len[k] = 0;
            for (int c = 0; c < 3; c++) {
                e[k][c] = pos[3 * (size_t)corner[b] + c] - pos[3 * (size_t)corner[a] + c];
                len[k] += e[k][c] * e[k][c];
            }
            len[k] = std::sqrt(len[k]);
        }
    std::stable_sort(order, order + 6, [&](uint32_t a, uint32_t b) { return len[a] < len[b]; });
    double f[3][3] = {{1, 0, 0}, {0, 1, 0}, {0, 0, 1}};
    const double unit = len[order[0]];
    if (unit > 0) {
        for (int c = 0; c < 3; c++) f[0][c] = e[order[0]][c] / unit;
        for (uint32_t q = 1; q < 6; q++) {
            const double* v = e[order[q]];
            const double d = v[0] * f[0][0] + v[1] * f[0][1] + v[2] * f[0][2];
            const double w[3] = {v[0] - d * f[0][0], v[1] - d * f[0][1], v[2] - d * f[0][2]};
            const double m = std::sqrt(w[0] * w[0] + w[1] * w[1] + w[2] * w[2]);
            if (!(m > 0.1 * len[order[q]])) continue;
            for (int c = 0; c < 3; c++) f[1][c] = w[c] / m;
            for (int c = 0; c < 3; c++)
                f[2][c] = f[0][(c + 1) % 3] * f[1][(c + 2) % 3] - f[0][(c + 2) % 3] * f[1][(c + 1) % 3];
            break;
        }
    }
    const double scale = unit > 0 ? 1e3 / unit : 1.0;
    std::vector<double> x(3 * (size_t)n);
    for (uint32_t v = 0; v < n; v++)
        for (int a = 0; a < 3; a++) {
            double s = 0;
            for (int c = 0; c < 3; c++) s += f[a][c] * (pos[3 * (size_t)(lo + v) + c] - pos[3 * (size_t)lo + c]);
            x[3 * (size_t)v + a] = std::nearbyint(s * scale);
        }
    return x;
}

// One scene's patches (offsets relative to the scene's own arrays).
bool build_scene(const HostModel& m, const ColorPlan& plan, const double* pos, const ResidentLimits& lim,
                 uint32_t scene, uint32_t threads, ResidentPlan& out) {
    const uint32_t lo = (*m.scene_offsets)[scene], hi = (*m.scene_offsets)[scene + 1], n = hi - lo;
    if (n == 0) return true;
    const uint32_t colors = plan.num_colors;
    std::vector<uint32_t> weight(n), part(n), order(n);
    uint64_t total = 0;
    for (uint32_t v = 0; v < n; v++) {
        // an item costs its incidences and about eight more (reduction, solve)
        weight[v] = plan.item_kind[lo + v] == 1 ? plan.item_of[lo + v].inc_count + 8u : 1u;
        total += weight[v];
    }
    uint32_t parts = (uint32_t)std::min<uint64_t>((total + lim.target - 1) / lim.target, lim.max_cluster);
    parts = std::max(parts, 1u);
    std::vector<uint32_t> local(n, NONE), stamp(n, NONE);
    std::vector<uint32_t> tet_stamp, tet_local;
    std::vector<std::vector<uint32_t>> readers(n);   // halo slots holding a copy of the particle
    const auto& nh = *m.nh;
    uint32_t t0 = NONE, t1 = 0;   // the scene's tets lie in [t0, t1]
    for (uint32_t v = 0; v < n; v++)
        if (plan.item_kind[lo + v] == 1) {
            const VItem& it = plan.item_of[lo + v];
            for (uint32_t k = 0; k < it.inc_count; k++) {
                const uint32_t t = plan.inc[it.inc_begin + k] >> 2;
                t0 = std::min(t0, t);
                t1 = std::max(t1, t);
            }
        }
    const uint32_t n_tets = t0 == NONE ? 0 : t1 - t0 + 1;
    const uint32_t alone[4] = {lo, lo, lo, lo};
    const std::vector<double> x = mesh_coordinates(pos, lo, n, t0 == NONE ? alone : nh[t0].idx);
    while (true) {
        std::iota(order.begin(), order.end(), 0u);
        bisect(order.data(), 0, n, 0, parts, x.data(), weight.data(), 0, part.data(), threads);
        out = ResidentPlan{};
        std::vector<std::vector<uint32_t>> own(parts);
        for (uint32_t v = 0; v < n; v++) own[part[v]].push_back(v);
        tet_stamp.assign(n_tets, NONE);
        tet_local.assign(n_tets, 0);
        std::fill(stamp.begin(), stamp.end(), NONE);
        for (auto& r : readers) r.clear();
        bool fits = true;   // the LDS and the 16-bit local indices
        for (uint32_t q = 0; q < parts && fits; q++) {
            if (own[q].empty()) continue;
            auto colour_of = [&](uint32_t v) { return plan.item_kind[lo + v] == 1 ? plan.color[lo + v] : colors; };
            std::stable_sort(own[q].begin(), own[q].end(),
                             [&](uint32_t a, uint32_t b) { return colour_of(a) < colour_of(b); });
            ResidentPatch p{};
            p.scene = scene;
            p.own = (uint32_t)own[q].size();
            p.gid_off = (uint32_t)out.gid.size();
            p.tet_off = (uint32_t)out.tet.size();
            p.inc_off = (uint32_t)out.inc.size() / 4;
            p.item_off = (uint32_t)out.item.size() / 2;
            p.slot = out.slots;
            p.col_off = (uint32_t)out.col.size();
            std::vector<uint32_t> tets, halo;
            for (uint32_t k = 0; k < p.own; k++) {
                stamp[own[q][k]] = q;
                local[own[q][k]] = k;
            }
            for (uint32_t v : own[q]) {
                if (plan.item_kind[lo + v] != 1) break;
                const VItem& it = plan.item_of[lo + v];
                const uint32_t begin = (uint32_t)out.inc.size() / 4 - p.inc_off;
                fits = begin + it.inc_count <= 0xFFFFu && tets.size() + it.inc_count <= 0x4000u;
                if (!fits) break;
                out.item.push_back(begin | it.inc_count << 16);
                out.item.push_back(0);
                p.items++;
                for (uint32_t k = 0; k < it.inc_count; k++) {
                    const uint32_t code = plan.inc[it.inc_begin + k], t = code >> 2;
                    if (tet_stamp[t - t0] != q) {
                        tet_stamp[t - t0] = q;
                        tet_local[t - t0] = (uint32_t)tets.size();
                        tets.push_back(t);
                        for (uint32_t g : nh[t].idx) {
                            const uint32_t u = g - lo;
                            if (stamp[u] == q) continue;
                            stamp[u] = q;
                            halo.push_back(u);
                        }
                    }
                    // the particles' local indices are known once the halo is complete
                    for (int j = 0; j < 3; j++) out.inc.push_back(0);
                    out.inc.push_back((uint16_t)(tet_local[t - t0] << 2 | (code & 3u)));
                }
            }
            std::sort(halo.begin(), halo.end(), [&](uint32_t a, uint32_t b) {
                const uint32_t ca = colour_of(a), cb = colour_of(b);
                return ca < cb || (ca == cb && a < b);
            });
            p.local = p.own + (uint32_t)halo.size();
            p.tets = (uint32_t)tets.size();
            p.inc = (uint32_t)out.inc.size() / 4 - p.inc_off;
            if (p.local > 0xFFFFu) fits = false;
            if (!fits) break;
            for (uint32_t k = 0; k < halo.size(); k++) {
                local[halo[k]] = p.own + k;
                if (colour_of(halo[k]) < colors) readers[halo[k]].push_back(p.slot + k);
            }
            out.slots += (uint32_t)halo.size();
            for (uint32_t e = p.inc_off; e < p.inc_off + p.inc; e++) {
                const uint32_t code = out.inc[4 * (size_t)e + 3];
                for (int j = 0; j < 3; j++)
                    out.inc[4 * (size_t)e + j] = (uint16_t)local[nh[tets[code >> 2]].idx[kEdgeCorner[code & 3u][j]] - lo];
            }
            for (uint32_t v : own[q]) out.gid.push_back(lo + v);
            for (uint32_t v : halo) out.gid.push_back(lo + v);
            for (uint32_t t : tets) {
                out.tet.push_back(t);
                for (uint32_t g : nh[t].idx) out.tix.push_back((uint16_t)local[g - lo]);
            }
            // item and halo ranges per colour
            uint32_t k = 0;
            for (uint32_t c = 0; c <= colors; c++) {
                while (k < p.items && colour_of(own[q][k]) < c) k++;
                out.col.push_back(k);
            }
            k = 0;
            for (uint32_t c = 0; c <= colors; c++) {
                while (k < halo.size() && colour_of(halo[k]) < c) k++;
                out.col.push_back(p.own + k);
            }
            out.patches.push_back(p);
        }
        for (ResidentPatch& p : out.patches) {
            if (!fits) break;
            p.target_off = (uint32_t)out.target.size();
            for (uint32_t k = 0; k < p.items; k++) {
                const auto& r = readers[out.gid[p.gid_off + k] - lo];
                const uint32_t begin = (uint32_t)out.target.size() - p.target_off;
                fits = begin + r.size() <= 0xFFFFu;
                if (!fits) break;
                out.item[2 * (size_t)(p.item_off + k) + 1] = begin | (uint32_t)r.size() << 16;
                out.target.insert(out.target.end(), r.begin(), r.end());
            }
            p.targets = (uint32_t)out.target.size() - p.target_off;
            const uint32_t bytes = resident_lds(p.own, p.items, p.local, p.tets, p.inc, p.targets, colors,
                                                lim.real_bytes, lim.damp, lim.ground)
                                       .total;
            out.lds_bytes = std::max(out.lds_bytes, bytes);
            if (bytes > lim.lds_bytes) fits = false;
        }
        if (fits) return true;
        if (parts >= lim.max_cluster || parts >= n) return false;
        parts = std::min(lim.max_cluster, std::max(parts + 1, parts + parts / 5));
    }
}

}  // namespace

bool build_resident(const HostModel& m, const ColorPlan& plan, const double* pos, const ResidentLimits& lim,
                    ResidentPlan& out) {
    const uint32_t n_scenes = (uint32_t)m.scene_offsets->size() - 1;
    std::vector<ResidentPlan> scenes(n_scenes);
    std::atomic<uint32_t> next{0};
    std::atomic<bool> ok{true};
    const uint32_t cpus = std::max(1u, std::min(16u, std::thread::hardware_concurrency()));
    const uint32_t workers = std::min(n_scenes, cpus);
    auto work = [&] {
        for (uint32_t s; ok && (s = next++) < n_scenes;) {
            bool fits = false;
            try {
                fits = build_scene(m, plan, pos, lim, s, std::max(1u, cpus / workers), scenes[s]);
            } catch (...) {
                ok = false;   // the other threads stop
                throw;
            }
            if (!fits) ok = false;
        }
    };
    {
        std::vector<std::future<void>> pool;
        pool.reserve(workers);
        for (uint32_t w = 1; w < workers; w++) pool.push_back(std::async(kThreads, work));
        work();
        for (auto& t : pool) t.get();
    }
    if (!ok) return false;
    out = ResidentPlan{};
    const uint32_t words = lim.real_bytes == 8 ? 6u : 3u;   // per slot
    for (const ResidentPlan& s : scenes) {
        const uint32_t first = (uint32_t)out.patches.size(), count = (uint32_t)s.patches.size();
        for (ResidentPatch p : s.patches) {
            p.gid_off += (uint32_t)out.gid.size();
            p.tet_off += (uint32_t)out.tet.size();
            p.inc_off += (uint32_t)out.inc.size() / 4;
            p.item_off += (uint32_t)out.item.size() / 2;
            p.target_off += (uint32_t)out.target.size();
            p.slot += out.slots;
            p.col_off += (uint32_t)out.col.size();
            p.first = first;
            p.count = count;
            out.patches.push_back(p);
        }
        out.gid.insert(out.gid.end(), s.gid.begin(), s.gid.end());
        out.tet.insert(out.tet.end(), s.tet.begin(), s.tet.end());
        out.tix.insert(out.tix.end(), s.tix.begin(), s.tix.end());
        out.inc.insert(out.inc.end(), s.inc.begin(), s.inc.end());
        out.item.insert(out.item.end(), s.item.begin(), s.item.end());
        out.col.insert(out.col.end(), s.col.begin(), s.col.end());
        for (uint32_t t : s.target) out.target.push_back((t + out.slots) * words);
        out.slots += s.slots;
        out.lds_bytes = std::max(out.lds_bytes, s.lds_bytes);
        out.max_cluster = std::max(out.max_cluster, count);
    }
    return !out.patches.empty() && (uint64_t)out.slots * words < (1u << 28);
}

uint32_t resident_block(const ResidentPlan& plan, uint32_t colors, const ResidentLimits& lim, uint32_t lanes) {
    uint32_t most = 0;   // items of one colour in one patch
    for (const ResidentPatch& p : plan.patches)
        for (uint32_t c = 0; c < colors; c++)
            most = std::max(most, plan.col[p.col_off + c + 1] - plan.col[p.col_off + c]);
    return lim.real_bytes == 4 && lanes * most > 512 ? 1024u : 512u;
}

bool build_bundles(const HostModel& m, const ColorPlan& plan, BundlePlan& out) {
    const uint32_t n = m.n, nc = plan.num_colors;
    // connected components over rod elements and two-sided joints
    std::vector<uint32_t> root(n);
    std::iota(root.begin(), root.end(), 0u);
    auto find = [&](uint32_t v) {
        while (root[v] != v) v = root[v] = root[root[v]];
        return v;
    };
    auto join = [&](uint32_t a, uint32_t b) {   // the smaller index stays
        a = find(a);
        b = find(b);
        root[std::max(a, b)] = std::min(a, b);
    };
    for (const HostCos& e : *m.cos) join(e.idx[0], e.idx[1]);
    for (const HostJoint2& j : *m.joints2) join(j.p[0], j.p[1]);
    // components in order of their first particle, bundled within a scene until
    // a bundle has its share of the particles for 256 CUs, 128 at most (one to two
    // wavefronts per phase, as the largest rods have)
    std::vector<uint32_t> size(n, 0), bundle(n, NONE);
    for (uint32_t v = 0; v < n; v++) size[find(v)]++;
    const uint32_t share = std::max(1u, std::min(128u, n / 256u));
    uint32_t filled = 0, scene = 0, bundles = 0, last_scene = NONE;
    for (uint32_t v = 0; v < n; v++) {
        while (v >= (*m.scene_offsets)[scene + 1]) scene++;
        if (root[v] != v) {
            bundle[v] = bundle[find(v)];
            continue;
        }
        if (bundles == 0 || scene != last_scene || filled + size[v] > share) {
            bundles++;
            filled = 0;
        }
        last_scene = scene;
        filled += size[v];
        bundle[v] = bundles - 1;
    }
    std::vector<std::vector<uint32_t>> parts(bundles), joints(bundles);
    for (uint32_t v = 0; v < n; v++) parts[bundle[v]].push_back(v);
    const uint32_t first = (uint32_t)m.joints->size();   // two-sided records follow the one-sided ones
    for (uint32_t j = 0; j < m.joints2->size(); j++) joints[bundle[(*m.joints2)[j].p[0]]].push_back(first + j);
    out = BundlePlan{};
    out.n_bundles = bundles;
    out.n_colors = nc;
    uint32_t most = 1;   // threads a phase of a bundle can use
    for (uint32_t b = 0; b < bundles; b++) {
        out.part_off.push_back((uint32_t)out.parts.size());
        out.joint_off.push_back((uint32_t)out.joints.size());
        out.parts.insert(out.parts.end(), parts[b].begin(), parts[b].end());
        out.joints.insert(out.joints.end(), joints[b].begin(), joints[b].end());
        for (uint32_t c = 0; c < nc; c++) {
            out.item_off.push_back((uint32_t)out.items.size());
            for (uint32_t v : parts[b])
                if (plan.item_kind[v] == 2 && plan.color[v] == c) out.items.push_back(plan.oitem_of[v]);
            most = std::max(most, 2u * (uint32_t)(out.items.size() - out.item_off.back()));
        }
        out.item_off.push_back((uint32_t)out.items.size());
    }
    out.part_off.push_back((uint32_t)out.parts.size());
    out.joint_off.push_back((uint32_t)out.joints.size());
    out.block = (most + 63u) / 64u * 64u;
    return bundles > 0 && most <= 512u;
}

}  // namespace avbd
