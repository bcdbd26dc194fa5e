// The BVH builder (csrc/lbvh.hip with csrc/ploc.inc), compiled for the CPU and run on small scenes: every kernel's
// indexing is exercised under the host's memory checks (build with -fsanitize=address) and the finished structure is
// held against its invariants - before any of it runs on a GPU.  Test infrastructure; see hip/hip_runtime.h here.
#include "hip/hip_runtime.h"

#include "../../diff-surfel-tracing_amd/csrc/lbvh.hip"

#include <cstdio>
#include <random>
#include <set>

namespace {

struct Scene {
    std::vector<float> v;     // (4P,3)
    std::vector<int32_t> f;   // (2P,3)
    uint32_t P;
};

Scene make_scene(uint32_t P, int kind, uint32_t seed) {
    // kind 0: uniform cube, random orientations; 1: all centres at one point; 2: identical quads but a few; 3: some
    // quads with NaN / infinite corners; 4: a plane of overlapping quads plus a dense cluster
    Scene s;
    s.P = P;
    s.v.resize(12 * (size_t)P);
    s.f.resize(6 * (size_t)P);
    std::mt19937 rng(seed);
    std::uniform_real_distribution<float> U(-1.f, 1.f);
    std::normal_distribution<float> N(0.f, 1.f);
    float first[12];
    for (uint32_t g = 0; g < P; ++g) {
        float m[3] = {U(rng), U(rng), U(rng)};
        if (kind == 1) m[0] = m[1] = m[2] = 0.25f;
        if (kind == 4) {
            if (g % 3) m[2] = -1.f;
            else { m[0] = 0.3f + 0.05f * N(rng); m[1] = 0.05f * N(rng); m[2] = 0.05f * N(rng); }
        }
        float q[4] = {N(rng), N(rng), N(rng), N(rng)};
        if (kind == 4 && g % 3) { q[0] = 1.f; q[1] = q[2] = 0.f; q[3] = N(rng); }
        const float nq = std::sqrt(q[0] * q[0] + q[1] * q[1] + q[2] * q[2] + q[3] * q[3]);
        const float w = q[0] / nq, x = q[1] / nq, y = q[2] / nq, z = q[3] / nq;
        const float sx = std::exp(-3.5f + 0.5f * N(rng)), sy = std::exp(-3.5f + 0.5f * N(rng));
        const float u[3] = {(1 - 2 * (y * y + z * z)) * sx, 2 * (x * y + w * z) * sx, 2 * (x * z - w * y) * sx};
        const float t[3] = {2 * (x * y - w * z) * sy, (1 - 2 * (x * x + z * z)) * sy, 2 * (y * z + w * x) * sy};
        const float sa[4] = {-3, -3, 3, 3}, sb[4] = {3, -3, 3, -3};
        for (int k = 0; k < 4; ++k)
            for (int a = 0; a < 3; ++a) s.v[12 * (size_t)g + 3 * k + a] = m[a] + sa[k] * u[a] + sb[k] * t[a];
        if (g == 0) std::memcpy(first, &s.v[0], sizeof(first));
        if (kind == 2 && g + 40 < P) std::memcpy(&s.v[12 * (size_t)g], first, sizeof(first));
        if (kind == 3 && g % 97 == 5) s.v[12 * (size_t)g + (g % 12)] = (g % 2) ? NAN : INFINITY;
        if (kind == 3 && g % 211 == 7)
            for (int k = 0; k < 12; ++k) s.v[12 * (size_t)g + k] = NAN;
        for (int k = 0; k < 3; ++k) {
            s.f[6 * (size_t)g + k] = 4 * g + k;
            s.f[6 * (size_t)g + 3 + k] = 4 * g + 1 + k;
        }
    }
    return s;
}

int failures = 0;
#define CHECK(cond, ...)                                   \
    do {                                                   \
        if (!(cond)) {                                     \
            if (++failures < 20) {                         \
                std::printf("FAILED %s:%d: ", __FILE__, __LINE__); \
                std::printf(__VA_ARGS__);                  \
                std::printf("\n");                         \
            }                                              \
        }                                                  \
    } while (0)

struct Box { float lo[3], hi[3]; };
bool same_box(const float *lo, const float *hi, const Box &b) {
    for (int a = 0; a < 3; ++a)
        if (std::memcmp(&lo[a], &b.lo[a], 4) != 0 || std::memcmp(&hi[a], &b.hi[a], 4) != 0) return false;
    return true;
}

// The invariants the fit by look-up, the refit, the collapse and the walks rely on.  Returns the depth (nodes above the
// deepest leaf).
uint32_t check_structure(const dst_ctx &c, const Scene &s, const char *what) {
    const uint32_t n = c.n_leaves;
    CHECK(n == s.P, "%s: leaves", what);
    // every surfel exactly once, corners copied
    std::vector<int> seen(n, 0);
    std::vector<Box> lbox(n);
    for (uint32_t i = 0; i < n; ++i) {
        const DstLeaf &L = c.leaves[i];
        CHECK(L.g < n, "%s: leaf %u holds surfel %u", what, i, L.g);
        if (L.g >= n) continue;
        seen[L.g]++;
        {   // corner A and the edge vectors to B, C, D, as the fp32 differences of the corners
            const float *v = &s.v[12 * (size_t)L.g];
            float want[12];
            for (int a = 0; a < 3; ++a) {
                want[a] = v[a];
                for (int k = 1; k < 4; ++k) want[3 * k + a] = v[3 * k + a] - v[a];
            }
            CHECK(std::memcmp(L.A, want, 48) == 0, "%s: corner and edges of leaf %u", what, i);
        }
        float cc[4][3];
        std::memcpy(cc, &s.v[12 * (size_t)L.g], 48);
        float mag = 0.f;
        for (int k = 0; k < 4; ++k)
            for (int a = 0; a < 3; ++a)
                if (std::fabs(cc[k][a]) < INFINITY) mag = std::max(mag, std::fabs(cc[k][a]));
        const float pad = 4e-6f * mag;
        for (int a = 0; a < 3; ++a) {
            lbox[i].lo[a] = std::fmin(std::fmin(cc[0][a], cc[1][a]), std::fmin(cc[2][a], cc[3][a])) - pad;
            lbox[i].hi[a] = std::fmax(std::fmax(cc[0][a], cc[1][a]), std::fmax(cc[2][a], cc[3][a])) + pad;
        }
    }
    for (uint32_t g = 0; g < n; ++g) CHECK(seen[g] == 1, "%s: surfel %u appears %d times", what, g, seen[g]);
    if (n < 2) return 0;
    // walk from the root
    std::vector<int> node_seen(n - 1, 0), leaf_seen(n, 0);
    std::vector<Box> nbox(n - 1);
    std::vector<std::pair<uint32_t, uint32_t>> stack{{0u, 1u}};
    std::vector<uint32_t> order;
    uint32_t depth = 0;
    CHECK(c.node_parent[0] == DST_NO_PARENT, "%s: root parent", what);
    while (!stack.empty()) {
        auto [i, d] = stack.back();
        stack.pop_back();
        if (i + 1 >= n) { CHECK(false, "%s: node index %u", what, i); continue; }
        if (node_seen[i]++) { CHECK(false, "%s: node %u reached twice", what, i); continue; }
        order.push_back(i);
        depth = std::max(depth, d);
        const DstNode &nd = c.nodes[i];
        const uint32_t split = nd.c0 & ~DST_LEAF_BIT;
        CHECK(nd.first <= split && split < nd.last && nd.last < n, "%s: node %u range %u %u %u", what, i, nd.first, split, nd.last);
        CHECK((nd.c1 & ~DST_LEAF_BIT) == split + 1, "%s: node %u right child", what, i);
        CHECK(((nd.c0 & DST_LEAF_BIT) != 0) == (split == nd.first), "%s: node %u left leaf flag", what, i);
        CHECK(((nd.c1 & DST_LEAF_BIT) != 0) == (split + 1 == nd.last), "%s: node %u right leaf flag", what, i);
        CHECK(i == 0 || i == nd.first || i == nd.last, "%s: node %u is neither end of its range", what, i);
        const uint32_t cs[2] = {nd.c0, nd.c1};
        for (uint32_t w = 0; w < 2; ++w) {
            if (cs[w] & DST_LEAF_BIT) {
                const uint32_t j = cs[w] & ~DST_LEAF_BIT;
                if (j >= n) { CHECK(false, "%s: leaf index", what); continue; }
                CHECK(leaf_seen[j]++ == 0, "%s: leaf %u twice", what, j);
                CHECK(c.leaf_parent[j] == ((i << 1) | w), "%s: leaf %u parent", what, j);
            } else {
                if (cs[w] + 1 >= n) { CHECK(false, "%s: child index", what); continue; }
                CHECK(c.node_parent[cs[w]] == ((i << 1) | w), "%s: node %u parent", what, cs[w]);
                const DstNode &ch = c.nodes[cs[w]];
                CHECK(w == 0 ? (ch.first == nd.first && ch.last == split) : (ch.first == split + 1 && ch.last == nd.last),
                      "%s: child range of node %u", what, i);
                stack.push_back({cs[w], d + 1});
            }
        }
    }
    for (uint32_t i = 0; i + 1 < n; ++i) CHECK(node_seen[i] == 1, "%s: node %u reached %d times", what, i, node_seen[i]);
    for (uint32_t i = 0; i < n; ++i) CHECK(leaf_seen[i] == 1, "%s: leaf %u reached %d times", what, i, leaf_seen[i]);
    if (failures) return depth;
    // boxes: exact unions, bottom-up
    for (size_t k = order.size(); k-- > 0;) {
        const uint32_t i = order[k];
        const DstNode &nd = c.nodes[i];
        Box b[2];
        const uint32_t cs[2] = {nd.c0, nd.c1};
        for (int w = 0; w < 2; ++w) b[w] = (cs[w] & DST_LEAF_BIT) ? lbox[cs[w] & ~DST_LEAF_BIT] : nbox[cs[w]];
        CHECK(same_box(nd.lo0, nd.hi0, b[0]) && same_box(nd.lo1, nd.hi1, b[1]), "%s: boxes of node %u", what, i);
        for (int a = 0; a < 3; ++a) {
            nbox[i].lo[a] = std::fmin(b[0].lo[a], b[1].lo[a]);
            nbox[i].hi[a] = std::fmax(b[0].hi[a], b[1].hi[a]);
        }
    }
    // the wide nodes: from the root every leaf is reached once; a child's box is its binary node's (or leaf group's)
    if (n > DST_GROUP) {
        std::vector<int> hit(n, 0);
        struct Item { uint32_t ref, depth; };
        std::vector<Item> st{{0u, 1u}};
        uint32_t wdepth = 0, steps = 0;
        while (!st.empty() && steps++ < 4 * n) {
            Item it = st.back();
            st.pop_back();
            if (it.ref & DST_LEAF_BIT) {
                const uint32_t first = it.ref & DST_REF_FIRST_MASK, count = ((it.ref >> 28) & 7u) + 1u;
                CHECK(first + count <= n && count <= DST_GROUP, "%s: leaf group %u+%u", what, first, count);
                for (uint32_t q = 0; q < count && first + q < n; ++q) hit[first + q]++;
                continue;
            }
            if (it.ref + 1 >= n) { CHECK(false, "%s: wide index", what); continue; }
            wdepth = std::max(wdepth, it.depth);
            const DstWideNode &w = c.wide[it.ref];
            CHECK(w.count >= 2 && w.count <= DST_WIDE, "%s: wide node %u has %u children", what, it.ref, w.count);
            const DstNode &nd = c.nodes[it.ref];
            uint32_t at = nd.first;
            for (uint32_t k = 0; k < w.count && k < DST_WIDE; ++k) {
                const uint32_t r = w.ref[k];
                uint32_t f, l;
                if (r & DST_LEAF_BIT) { f = r & DST_REF_FIRST_MASK; l = f + ((r >> 28) & 7u); }
                else if (r + 1 < n) { f = c.nodes[r].first; l = c.nodes[r].last; }
                else { CHECK(false, "%s: wide child", what); continue; }
                CHECK(f == at, "%s: children of wide node %u are not in leaf order", what, it.ref);
                at = l + 1;
                Box u = lbox[f];
                for (uint32_t j = f + 1; j <= l && j < n; ++j)
                    for (int a = 0; a < 3; ++a) { u.lo[a] = std::fmin(u.lo[a], lbox[j].lo[a]); u.hi[a] = std::fmax(u.hi[a], lbox[j].hi[a]); }
                const float lo[3] = {w.lox[k], w.loy[k], w.loz[k]}, hi[3] = {w.hix[k], w.hiy[k], w.hiz[k]};
                CHECK(same_box(lo, hi, u), "%s: box of child %u of wide node %u", what, k, it.ref);
                st.push_back({r, it.depth + 1});
            }
            CHECK(at == nd.last + 1, "%s: wide node %u does not cover its range", what, it.ref);
        }
        for (uint32_t i = 0; i < n; ++i) CHECK(hit[i] == 1, "%s: leaf %u is in %d leaf groups", what, i, hit[i]);
        CHECK(3 * wdepth <= 126, "%s: wide hierarchy %u deep, the walks' stacks hold 128 entries", what, wdepth);
    }
    return depth;
}

void run_case(uint32_t P, int kind, bool agglomerate, uint32_t seed) {
    char what[128];
    std::snprintf(what, sizeof(what), "P=%u kind=%d %s", P, kind, agglomerate ? "agglomerated" : "morton");
    Scene s = make_scene(P, kind, seed);
    dst_ctx ctx;
    ctx.use_ploc = agglomerate;
    int rc = dst_lbvh_build(&ctx, s.v.data(), 4 * P, s.f.data(), P, true, nullptr);
    CHECK(rc == DST_OK, "%s: build returned %d (%s)", what, rc, ctx.err.c_str());
    if (rc != DST_OK) return;
    const uint32_t depth = check_structure(ctx, s, what);
    std::printf("%-40s depth %2u agglomerated %d refused %d key levels %d\n", what, depth, (int)ctx.agglomerated,
                (int)ctx.ploc_refused, ctx.fine_keys ? 2 : 1);
    CHECK(!agglomerate || P < 64 || ctx.agglomerated || ctx.ploc_refused, "%s: not agglomerated", what);
    CHECK(!ctx.agglomerated || ctx.hierarchy_depth == depth, "%s: reported depth %u", what, ctx.hierarchy_depth);
    // a refit on moved geometry keeps order and topology and fits the boxes again (both fits)
    std::vector<uint32_t> order(P);
    for (uint32_t i = 0; i < P; ++i) order[i] = ctx.leaves[i].g;
    Scene moved = s;
    std::mt19937 rng(seed + 1);
    std::normal_distribution<float> N(0.f, 0.1f);
    for (uint32_t g = 0; g < P; g += 2) {
        const float d[3] = {N(rng), N(rng), N(rng)};
        for (int k = 0; k < 4; ++k)
            for (int a = 0; a < 3; ++a) moved.v[12 * (size_t)g + 3 * k + a] += d[a];
    }
    rc = dst_lbvh_build(&ctx, moved.v.data(), 4 * P, nullptr, P, false, nullptr);
    CHECK(rc == DST_OK, "%s: refit returned %d", what, rc);
    check_structure(ctx, moved, what);
    for (uint32_t i = 0; i < P; ++i) CHECK(order[i] == ctx.leaves[i].g, "%s: refit moved leaf %u", what, i);
    if (P <= DST_STATIC_REFIT_MAX_SURFELS && P > 1) {   // the climbing fit with caller-provided counters
        std::vector<uint32_t> counters(P);
        rc = dst_lbvh_build(&ctx, s.v.data(), 4 * P, nullptr, P, false, nullptr, counters.data());
        CHECK(rc == DST_OK, "%s: climbing refit returned %d", what, rc);
        check_structure(ctx, s, what);
    }
    dst_lbvh_free(&ctx);
    std::free(ctx.bounds);
    std::free(ctx.core_box);
    std::free(ctx.bounds_host);
    std::free(ctx.ploc_host);
}

// ---- the rounds of the agglomeration, several to a launch on a window of the clusters, against rounds over all of them -------
struct Cluster { float lo, hi; uint32_t id, low, size; };   // a box (lo,lo,lo) .. (hi,hi,hi)
struct Merge { uint32_t c0, c1, size; };
bool operator==(const Merge &a, const Merge &b) { return a.c0 == b.c0 && a.c1 == b.c1 && a.size == b.size; }

void whole_round(std::vector<Cluster> &c, std::vector<Merge> &made) {
    const int n = (int)c.size();
    auto area = [&](int i, int j) {
        const float e = std::max(c[i].hi, c[j].hi) - std::min(c[i].lo, c[j].lo);
        return e * e + e * e + e * e;
    };
    std::vector<int> nn(n);
    for (int i = 0; i < n; ++i) {
        float best = INFINITY;
        nn[i] = i;
        for (int d = 1; d <= kPlocRadius; ++d) {
            const float up = i + d < n ? area(i, i + d) : INFINITY, down = i >= d ? area(i, i - d) : INFINITY;
            const bool lower = down < up || (down == up && i >= d && c[i - d].low * 2654435761u < c[i].low * 2654435761u);
            if ((lower ? down : up) < best) {
                best = lower ? down : up;
                nn[i] = lower ? i - d : i + d;
            }
        }
    }
    std::vector<Cluster> next;
    for (int i = 0; i < n; ++i) {
        const int j = nn[i];
        if (j == i || nn[j] != i) { next.push_back(c[i]); continue; }
        if (j < i) continue;
        const uint32_t node = c[j].low - 1u;
        made[node] = {c[i].id, c[j].id, c[i].size + c[j].size};
        next.push_back({std::min(c[i].lo, c[j].lo), std::max(c[i].hi, c[j].hi), node, c[i].low, made[node].size});
    }
    c.swap(next);
}

struct PlocTest {   // the buffers of ploc_hierarchy
    std::vector<float> box[2];
    std::vector<uint32_t> words[11];
    PlocBufs pb;
    explicit PlocTest(uint32_t n) {
        for (auto &b : box) b.assign(6 * (size_t)n, NAN);
        for (auto &w : words) w.assign(2 * (size_t)n + 64, 0xDEADBEEFu);
        pb.box[0] = box[0].data();
        pb.box[1] = box[1].data();
        uint32_t **to[] = {&pb.id[0], &pb.id[1], &pb.low[0], &pb.low[1], &pb.nn, &pb.pre, &pb.tc0, &pb.tc1, &pb.tsize, &pb.up, &pb.lpar};
        for (int k = 0; k < 11; ++k) *to[k] = words[k].data();
        pb.n_blocks = (n + ploc_own(4) - 1) / ploc_own(4);
        state.assign(kPlocStateWords + 2 * ((size_t)pb.n_blocks + 1), 0u);
        pb.state = state.data();
    }
    std::vector<uint32_t> state;
};

// `rounds`: 3 or 4 to a launch; 0: in turn
void check_rounds(std::vector<Cluster> c, int rounds, const char *what) {
    const uint32_t n = (uint32_t)c.size();
    PlocTest t(n);
    for (uint32_t i = 0; i < n; ++i) {
        for (int k = 0; k < 3; ++k) {
            t.box[0][6 * (size_t)i + k] = c[i].lo;
            t.box[0][6 * (size_t)i + 3 + k] = c[i].hi;
        }
        t.pb.id[0][i] = c[i].id = DST_LEAF_BIT | i;
        t.pb.low[0][i] = c[i].low = i;
        c[i].size = 1u;
    }
    t.state[0] = t.state[1] = n;
    int it = 0;
    for (; t.state[it & 1] > kPlocTail && it < 200; ++it) {
        const int r = rounds != 0 ? rounds : 3 + it % 2;
        const uint32_t own = ploc_own(r);
        if (r == 3) hipLaunchKernelGGL(k_ploc_rounds<3>, dim3((n + own - 1) / own), dim3(kPlocBlock), 0, nullptr, t.pb, it);
        else hipLaunchKernelGGL(k_ploc_rounds<4>, dim3((n + own - 1) / own), dim3(kPlocBlock), 0, nullptr, t.pb, it);
        hipLaunchKernelGGL(k_ploc_scan, dim3(1), dim3(kPlocBlock), 0, nullptr, t.pb, it, own);
    }
    hipLaunchKernelGGL(k_ploc_tail, dim3(1), dim3(kPlocBlock), 0, nullptr, t.pb, it);
    std::vector<Merge> want(n - 1);
    while (c.size() > 1) whole_round(c, want);
    uint32_t off = 0;
    for (uint32_t k = 0; k + 1 < n; ++k) off += Merge{t.pb.tc0[k], t.pb.tc1[k], t.pb.tsize[k]} == want[k] ? 0u : 1u;
    CHECK(off == 0u && t.state[0] == 1u && t.state[3] == n, "%s: %u of %u merges differ from rounds over all clusters", what, off, n - 1);
    std::printf("rounds %-40s %u clusters, %d launches, %u merges off\n", what, n, it, off);
}
void check_rounds(const std::vector<float> &at, int rounds, const char *what) {
    std::vector<Cluster> c;
    for (float t : at) c.push_back({t, t, 0u, 0u, 0u});
    check_rounds(c, rounds, what);
}

// The layout of `n` leaves over links of which one or two are not those of a hierarchy, though the counts at its root are: a
// build has to find out (state[4]), whatever the buffers held before.
void check_broken_links(uint32_t n) {
    const dim3 grid((n + kBlock - 1) / kBlock);
    for (int kind = 0; kind < 4; ++kind) {   // none; a leaf in another's place; a node in another's; a leaf on its sibling's side
        PlocTest t(n);
        std::mt19937 rng(3);
        for (uint32_t i = 0; i < n; ++i) {
            for (int k = 0; k < 6; ++k) t.box[0][6 * (size_t)i + k] = std::uniform_real_distribution<float>(0.f, 1.f)(rng) * (k % 3 == 0);
            for (int k = 0; k < 3; ++k) t.box[0][6 * (size_t)i + 3 + k] = t.box[0][6 * (size_t)i + k] + 0.01f;
            t.pb.id[0][i] = DST_LEAF_BIT | i;
            t.pb.low[0][i] = i;
        }
        t.state[0] = t.state[1] = n;
        hipLaunchKernelGGL(k_ploc_tail, dim3(1), dim3(kPlocBlock), 0, nullptr, t.pb, 0);
        const uint32_t root = t.state[2];
        if (kind == 1) t.pb.lpar[7] = t.pb.lpar[150];
        if (kind == 2) {   // two nodes of one size
            for (uint32_t a = 0, done = 0; a + 1 < n && !done; ++a)
                for (uint32_t b = a + 1; b + 1 < n && !done; ++b)
                    if (t.pb.tsize[a] == t.pb.tsize[b] && a != root && b != root) {
                        t.pb.up[2 * a] = t.pb.up[2 * b];
                        done = 1;
                    }
        }
        if (kind == 3) t.pb.lpar[20] ^= 1u;
        std::vector<uint32_t> in(n), out(n, 0xFFFFFFFFu), node_parent(n), leaf_parent(n);
        for (uint32_t i = 0; i < n; ++i) in[i] = (i * 77u) % n;
        for (uint32_t i = 0; i < n; ++i) out[i] = DST_LEAF_BIT | i;
        std::vector<DstNode> nodes(n - 1);
        hipLaunchKernelGGL(k_ploc_big_nodes, grid, dim3(kBlock), 0, nullptr, t.pb, n);
        hipLaunchKernelGGL(k_ploc_leaf_positions, grid, dim3(kBlock), 0, nullptr, t.pb, in.data(), out.data(), n);
        hipLaunchKernelGGL(k_ploc_node_numbers, grid, dim3(kBlock), 0, nullptr, t.pb, in.data(), out.data(), nodes.data(), n);
        hipLaunchKernelGGL(k_ploc_links, grid, dim3(kBlock), 0, nullptr, t.pb, nodes.data(), node_parent.data(), leaf_parent.data(), n);
        CHECK(t.state[0] == 1u && t.state[3] == n, "broken links %d: one cluster of %u", kind, n);
        CHECK((t.state[4] != 0u) == (kind != 0), "broken links %d: %u", kind, t.state[4]);
    }
}

// An order in which news travels as far as it can in four rounds: what lies 289 places beyond position `edge` (233 before
// it, `before`) decides about a merge of the cluster next to the edge.  Everything lies in tight groups of eight, each at a
// site of its own, that halve their number in every round; eight clusters a round merge across the edge (a merged cluster
// goes on in the lower one's place, so those beyond the edge lose eight, those before it none); and in every round there
// are three clusters eight places apart, a, b and c, of which b takes c where c is (still) alone, and a where not.
std::vector<float> far_reaching_order(uint32_t n, uint32_t edge, bool before) {
    const float in_group[8] = {0.f, 0.05f, 0.3f, 0.35f, 1.5f, 1.55f, 1.8f, 1.85f};
    uint32_t site = 0;
    std::vector<float> beyond, inside;   // places from the edge on, away from it and into the other side
    auto group = [&](std::vector<float> &to, uint32_t points, float where) {
        for (uint32_t k = 0; k < points; ++k) to.push_back(where + in_group[k]);
    };
    auto elsewhere = [&](std::vector<float> &to, uint32_t points) { group(to, points, 100.f * (float)(site++ % 60)); };
    const float home = 7000.f, a3 = home - 34.f, b3 = home - 25.f, a2 = home - 18.f, b2 = home - 12.f, a1 = home - 7.f, b1 = home - 3.f;
    if (before) {
        group(inside, 8, a3);
    } else {
        // the last eight clusters before the edge, the edge's side first; what they merge with beyond it in rounds 0, 1 and 2
        float u[8];
        for (int k = 0; k < 8; ++k) u[k] = k == 7 ? a3 : 6100.f + 100.f * (float)k;
        for (int k = 7; k >= 0; --k) inside.push_back(u[k]);
        for (int k = 0; k < 8; ++k) beyond.push_back(u[k] + 0.05f);
        for (int k = 0; k < 8; ++k) group(beyond, 2, u[k] + 0.3f);
        for (int k = 0; k < 8; ++k) group(beyond, 4, u[k] + 0.9f);
    }
    for (int k = 0; k < 15; ++k) {
        if (k == 7) group(beyond, 8, b3);
        else elsewhere(beyond, 8);
    }
    auto seven = [&](uint32_t points) {   // seven clusters of a round
        for (int k = 0; k < 3; ++k) elsewhere(beyond, 2 * points);
        elsewhere(beyond, points);
    };
    group(beyond, 4, a2);
    seven(4);
    group(beyond, 4, b2);
    seven(4);
    group(beyond, 2, a1);
    seven(2);
    group(beyond, 2, b1);
    seven(2);
    beyond.push_back(home);
    seven(1);
    beyond.push_back(home + 2.f);
    seven(1);
    beyond.push_back(home + 3.9f);
    std::vector<float> at(n);
    for (uint32_t i = 0; i < n; ++i) at[i] = 100.f * (float)((i / 8u) % 60) + 30.f + in_group[i % 8u];   // (all else)
    for (uint32_t k = 0; k < beyond.size(); ++k) at[before ? edge - 1u - k : edge + k] = beyond[k];
    for (uint32_t k = 0; k < inside.size(); ++k) at[before ? edge + k : edge - 1u - k] = inside[k];
    return at;
}

void check_windows() {
    char what[96];
    for (int before = 0; before < 2; ++before)
        for (uint32_t k = 1; k < 4; k += 2) {
            std::snprintf(what, sizeof(what), "four, far-reaching %s %u", before ? "before" : "beyond", k * ploc_own(4));
            check_rounds(far_reaching_order(3000, k * ploc_own(4), before != 0), 4, what);
            // three rounds: what the first of the four leaves, with the edge where it then lies
            bool found = false;
            for (uint32_t edge = 2 * k * ploc_own(3) - 24; !found && edge < 2 * k * ploc_own(3) + 24; ++edge) {
                std::vector<Cluster> c;
                for (float t : far_reaching_order(6000, edge, before != 0)) c.push_back({t, t, 0u, (uint32_t)c.size(), 1u});
                std::vector<Merge> made(c.size());
                whole_round(c, made);
                uint32_t at = 0;
                while (c[at].low < edge) ++at;
                found = at == k * ploc_own(3);
                if (!found) continue;
                std::snprintf(what, sizeof(what), "three, far-reaching %s %u", before ? "before" : "beyond", at);
                check_rounds(c, 3, what);
            }
            CHECK(found, "no order with an edge at %u", k * ploc_own(3));
        }
    std::mt19937 rng(5);
    for (uint32_t n : {1025u, 2900u, 5000u}) {
        for (int kind = 0; kind < 3; ++kind) {   // even, clustered, equal
            std::vector<float> at(n);
            for (float &t : at) {
                t = std::uniform_real_distribution<float>(0.f, 1000.f)(rng);
                if (kind == 1) t = std::round(t / 50.f) * 50.f + std::exp2(-(float)(rng() % 12u)) * t / 100.f;
                if (kind == 2) t = std::round(t / 200.f);
            }
            for (int rounds : {0, 3, 4}) check_rounds(at, rounds, kind == 0 ? "even" : (kind == 1 ? "clustered" : "equal"));
        }
    }
}

}  // namespace

int main(int argc, char **argv) {
    std::setvbuf(stdout, nullptr, _IONBF, 0);
    if (argc == 4) {   // one case: surfels, kind of scene, agglomerate
        run_case((uint32_t)std::atoi(argv[1]), std::atoi(argv[2]), std::atoi(argv[3]) != 0, 1);
        std::printf(failures ? "FAILED: %d checks\n" : "ALL OK\n", failures);
        return failures ? 1 : 0;
    }
    check_windows();
    check_broken_links(200);
    check_broken_links(900);   // with big nodes
    const bool quick = argc > 1 && std::string(argv[1]) == "quick";
    const uint32_t sizes[] = {1, 2, 3, 63, 64, 65, 100, 1024, 1025, 2500, 5000};
    for (uint32_t P : {kPlocBig, kPlocBig + 1, kPlocBig + 2}) run_case(P, 0, true, 11 + P);   // the root the one big node
    for (int agg = 1; agg >= 0; --agg) {
        for (uint32_t P : sizes) {
            if (quick && P > 2500) continue;
            run_case(P, 0, agg != 0, 11 + P);
        }
        run_case(3000, 1, agg != 0, 5);
        run_case(3000, 2, agg != 0, 6);
        run_case(3000, 3, agg != 0, 7);
        run_case(4000, 4, agg != 0, 8);
        if (!quick) run_case(110000, 0, agg != 0, 9);   // range table of two workgroups; three rounds to a launch, then four
    }
    std::printf(failures ? "FAILED: %d checks\n" : "ALL OK\n", failures);
    return failures ? 1 : 0;
}
