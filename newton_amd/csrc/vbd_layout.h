// Host-side "pass layout" for the color-pass kernel (built once per model in vbd_create).
//
// For every color, the color's vertices (in color-group order) are cut into
// batches: runs of at most max_v consecutive vertices whose element counts sum
// to at most cap (the work-group shape: 256 lanes -> cap 256, max_v 21; 128
// lanes -> cap 128, max_v 10) and whose elements touch at most cap distinct
// vertices.  A batch is one workgroup, and lane t evaluates item t: all
// triangle items of the batch, then all bending-edge items (first those whose
// vertex lies opposite the hinge edge, then those on it: the two run different
// code), then all tet items, then the springs, each carrying the canonical row (the position of that
// contribution in its vertex's serial sum: the vertex's triangles in CSR order,
// then its edges, then its tets) and the vertex's local slot in the element.
//
// Storage is by fixed slots, so a lane finds its item, and its share of the
// batch's vertex list, from the batch number alone, in the same round trip as
// the batch header: item t of batch b is item_rec[b * cap + t]; the wider part
// of a triangle (tet, spring) record sits in an array with one slot for each
// lane that holds that kind in any batch ([tri_lo, tri_hi) and so on), or, for
// passes of every kind, in the slots of the widest kind.  Slots
// that a batch does not use are never used.  Items name their vertices by 8-bit
// slots of the batch's vertex list (the batch's own vertices first), whose
// positions the work-group stages in LDS: a hinge item is 16 bytes, and a
// position is gathered once per batch instead of once per element.
//
// Values of an element that no step changes are evaluated here once, in single
// precision and the kernels' expression order: lambda + mu, the rest ratio
// alpha = 1 + mu / (lambda + mu), a tet's rest volume, stiffness * rest length.
//
// Elements the reference's solve skips are left out: triangles and tets with
// mu <= 0 and lambda <= 0, edges with ke <= 0 (particle_vbd_kernels.py:2636,
// :2658, :2679), and boundary hinges (o0 or o1 == -1), whose contribution is
// an exact zero (:682-683).  Inactive particles (flag bit 0 clear or mass 0)
// get no items.  A vertex with more than cap items, or whose elements touch
// more than list_cap(cap) vertices, goes to the "slow" list, handled by the generic
// kernel that walks the CSR in chunks.
//
// Springs (particle_vbd_kernels.py:1733-1783) join the batch as items of their
// own: each active endpoint of a spring gets one item, in spring-index order
// per vertex, whose row follows the vertex's element rows (the solve adds them
// to the contact sum, after the contacts).  A spring whose endpoints share a
// color cannot be evaluated inside the pass (the other endpoint moves during
// it); its items are evaluated by a pre-pass over the color into global rows
// ("pre items") and the pass item only points at its row.
#pragma once

#include <algorithm>
#include <cmath>
#include <cstdint>
#include <cstring>
#include <string>
#include <vector>

namespace vbd_layout {

constexpr int kLayoutCap = 256;  // static items (rows) per batch of the 256-lane shape
constexpr int kLayoutMaxV = 21;  // vertices per batch of the 256-lane shape (12 component lanes each)

// record widths in 32-bit words
constexpr int kItemWords = 4;    // vertex slots (4 x 8 bits) | item_meta | two words by kind:
                                 //   triangle: area -   hinge: rest_angle ke*rest_length
                                 //   tet: mu lambda+mu  spring: pre_row rest_length
constexpr int kTriWords = 8;     // D00 D01 D10 D11 | mu lambda+mu alpha kd
constexpr int kTetWords = 12;    // Dm^-1 (9) rest_volume alpha kd
constexpr int kSpringWords = 2;  // ke kd
constexpr int kBatchWords = 4;   // vbegin nv static_rows batch_flags
constexpr int kVertWords = 4;    // v row_start nrows (local | active << 16 | nsprings << 17)
// Distinct vertices of a batch: its own and their elements' others (a regular cloth's batch has 7 to 9 for each
// of its own, so the lanes fill first); the work-group stages that many positions in LDS, and a smaller bound
// lets more work-groups share a CU.
constexpr int list_cap(int cap) { return cap <= 192 ? 128 : 192; }
// batch block: header (kBatchWords) then max_v vertex records (unused ones zero),
// fixed size so a workgroup reads its header and vertex records in one round trip
inline int block_words(int max_v) { return kBatchWords + max_v * kVertWords; }  // a multiple of 4 words

// batch_flags.  They follow the damping coefficients, which a rebuild may switch from or to zero under a captured graph:
// in the batch header they are data of the layout, not arguments of the launch.
enum BatchFlags {
    kPrevAll = 1,      // some item reads previous positions of the listed vertices (damping, springs)
    kHingeDamped = 2,  // some hinge has kd > 0 (hinge_damp is read)
};

enum ItemKind { kNone = 0, kTri = 1, kHinge = 2, kTet = 3, kSpring = 5 };
// row (9 bits) | slot in the element << 9 (2 bits) | damped << 11 | kind << 12
inline int32_t item_meta(int row, int slot, bool damped, int kind) {
    return (int32_t)(row | (slot << 9) | ((damped ? 1 : 0) << 11) | (kind << 12));
}

struct HostModel {
    int N = 0, T = 0, E = 0, K = 0;
    std::vector<float> mass;
    std::vector<int32_t> flags;
    std::vector<int32_t> tri_idx, edge_idx, tet_idx;
    std::vector<float> tri_pose, tri_mat, tri_area;
    std::vector<float> edge_rest, edge_len, edge_bend;
    std::vector<float> tet_pose, tet_mat;
    std::vector<int32_t> adj_tri, adj_tri_off, adj_edge, adj_edge_off, adj_tet, adj_tet_off;
    std::vector<int32_t> color_off, color_particles;
    int S = 0;
    std::vector<int32_t> spring_idx;
    std::vector<float> spring_rest, spring_ke, spring_kd;
    bool self_contact = false;  // of the solver: decides the kinds of a pass (kinds_of_pass)
};

// Lanes [lo, hi) that hold one kind of item in any batch (empty when lo == hi).
struct LaneRange {
    int lo = 0, hi = 0;
    int count() const { return hi - lo; }
    void cover(int b, int e) {
        if (e <= b) return;
        if (hi == lo) {
            lo = b;
            hi = e;
        } else {
            lo = std::min(lo, b);
            hi = std::max(hi, e);
        }
    }
    bool operator==(const LaneRange& o) const { return lo == o.lo && hi == o.hi; }
};

// What a launch is given besides the arrays; equal shapes may be exchanged under a captured graph.
struct PassShape {
    LaneRange tri, hinge, tet, spring;  // tet: of every kind with a record where they share an array
    int list_stride = 0;  // entries of a batch's vertex list
    // Two corners of some edge or triangle share a color (elements without stiffness are not part of the coloring
    // graph): a pass moves one corner of their edge/face contacts while another's entry reads it, so those entries'
    // rows are evaluated before the pass.
    bool shared_corners = false;
    bool operator==(const PassShape& o) const {
        return tri == o.tri && hinge == o.hinge && tet == o.tet && spring == o.spring &&
               list_stride == o.list_stride && shared_corners == o.shared_corners;
    }
};

namespace pass_kinds {
// Element kinds a pass holds.  Every contribution of a cloth pass (triangles, hinges, springs, contacts with
// shapes) has a Hessian that is symmetric bit for bit, so its rows hold 9 numbers instead of 12: less LDS
// (more work-groups per CU) and fewer lanes in the sums.  Tet and self-contact Hessians are symmetric
// only up to rounding.
constexpr int kClothKinds = 0, kClothSpringKinds = 1, kTetKinds = 2, kAllKinds = 3;
// Added to the kinds of a context whose contacts include edge/face records.  A pass evaluates those itself, their
// corners read from memory and in parts when they outnumber the rows; a kernel of their rows took 8.5 us before each
// pass (256x256 cloth on moving bodies, substep 988 -> 716 us).  That kernel, k_contact_rows, serves models whose
// edges or faces hold corners of one color, where the pass itself moves what the entries read.  Kept apart from the
// other passes: compiled into them it cost their occupancy (substeps of 512 cloth worlds 1,160 -> 1,354 us, of a
// 256x256 cloth 395 -> 437 us).
constexpr int kEdgeFace = 4;
// Added for self-contact, whose rows k_sc_rows evaluates (contacts crowd in a few batches: evaluated in the pass, it
// took 39 us instead of 12 and 11 of the rows kernel).
constexpr int kSelfRows = 8;
// What the pass is compiled for.
constexpr int kInstantiated[] = {
    kClothKinds, kClothSpringKinds, kTetKinds, kAllKinds, kClothKinds + kEdgeFace, kClothSpringKinds + kEdgeFace,
    kTetKinds + kEdgeFace, kAllKinds + kEdgeFace, kClothKinds + kSelfRows, kAllKinds + kSelfRows,
    kClothKinds + kSelfRows + kEdgeFace, kAllKinds + kSelfRows + kEdgeFace};
}  // namespace pass_kinds

// The kinds a layout's passes run with.
inline int kinds_of_pass(const PassShape& sh, bool full_surface, bool self_contact) {
    using namespace pass_kinds;
    const bool cloth = sh.tri.count() + sh.hinge.count() > 0;
    const bool tet = sh.tet.count() > 0, spring = sh.spring.count() > 0;
    int kinds = tet ? kTetKinds : (spring ? kClothSpringKinds : kClothKinds);
    if ((tet && (cloth || spring)) || (self_contact && (tet || spring))) kinds = kAllKinds;
    return kinds + (full_surface ? kEdgeFace : 0) + (self_contact ? kSelfRows : 0);
}

struct PassLayout {
    std::vector<int32_t> fast_color_off;  // [C+1] into batch records
    std::vector<int32_t> slow_color_off;  // [C+1] into slow_pos
    std::vector<int32_t> batch_blk;       // [B * block_words(max_v)]: header + vertex records
    int cap = kLayoutCap, max_v = kLayoutMaxV, blk_words = block_words(kLayoutMaxV);
    PassShape shape;
    std::vector<int32_t> vert_rec;        // [N * kVertWords], indexed by color position
    std::vector<int32_t> item_rec;        // [B * cap * kItemWords]
    std::vector<int32_t> list;            // [B * list_stride] vertex list of each batch, its first again past its end
    std::vector<int32_t> tri_rec, tet_rec, spr_rec;  // [B * range.count() * words]
    std::vector<int32_t> hinge_damp;      // [B * hinge.count()] kd * rest_length (float bits)
    std::vector<int32_t> slow_pos;        // color positions of oversized vertices
    std::vector<int32_t> pre_item;        // [P, 2] (spring, endpoint) of same-color spring items
    std::vector<int32_t> pre_color_off;   // [C+1] into pre_item
    std::vector<int32_t> slow_spr_off;    // [slow + 1] into slow_spr
    std::vector<int32_t> slow_spr;        // [*, 4] (spring, endpoint, pre_row or -1, 0) of slow vertices
    int64_t fast_items = 0;
};

inline int32_t fbits(float f) {
    int32_t i;
    std::memcpy(&i, &f, 4);
    return i;
}

// lambda + mu and the rest ratio alpha of a stable Neo-Hookean element (particle_vbd_kernels.py:76-292, :502-632)
inline float lame_sum(float mu, float lambda) { return lambda + mu; }
inline float rest_ratio(float mu, float lambda) {
    const float l_nh = lame_sum(mu, lambda);
    const float l_safe = (l_nh < 0.0f ? -1.0f : 1.0f) * std::fmax(std::fabs(l_nh), 1.0e-6f);
    return 1.0f + mu / l_safe;
}
// 1 / (6 det Dm^-1), determinant as row0 . (row1 x row2)
inline float rest_volume(const float* m) {
    const float cx = m[4] * m[8] - m[5] * m[7], cy = m[5] * m[6] - m[3] * m[8], cz = m[3] * m[7] - m[4] * m[6];
    return 1.0f / ((m[0] * cx + m[1] * cy + m[2] * cz) * 6.0f);
}

// Lanes an item range takes when ranges start on wave (64-lane) boundaries.
inline int wave_align(int n) { return (n + 63) & ~63; }

// Builds the layout; returns an empty string or an error message.
// aligned: each kind's items start on a wave boundary of the work-group (a wave then evaluates one
// kind only); the batch's lane budget counts the padded ranges.
inline std::string build_pass_layout(const HostModel& m, PassLayout& L, int cap = kLayoutCap,
                                     int max_v = kLayoutMaxV, bool aligned = false) {
    const int N = m.N;
    const int C = (int)m.color_off.size() - 1;
    std::vector<char> active((size_t)N), tri_ok((size_t)m.T), edge_ok((size_t)m.E), tet_ok((size_t)m.K);
    for (int v = 0; v < N; ++v) active[v] = (m.flags[v] & 1) && m.mass[v] != 0.0f;
    for (int t = 0; t < m.T; ++t) tri_ok[t] = m.tri_mat[5 * t] > 0.0f || m.tri_mat[5 * t + 1] > 0.0f;
    for (int e = 0; e < m.E; ++e)
        edge_ok[e] = m.edge_bend[2 * e] > 0.0f && m.edge_idx[4 * e] != -1 && m.edge_idx[4 * e + 1] != -1;
    for (int k = 0; k < m.K; ++k) tet_ok[k] = m.tet_mat[3 * k] > 0.0f || m.tet_mat[3 * k + 1] > 0.0f;
    std::vector<int32_t> color_of((size_t)N, -1);
    for (int c = 0; c < C; ++c)
        for (int k = m.color_off[c]; k < m.color_off[c + 1]; ++k) color_of[m.color_particles[k]] = c;
    auto same = [&](int a, int b) { return a >= 0 && a < N && b >= 0 && b < N && color_of[a] == color_of[b]; };
    bool shared_corners = false;
    for (int t = 0; t < m.T && !shared_corners; ++t) {
        const int32_t* c = &m.tri_idx[3 * (size_t)t];
        shared_corners = same(c[0], c[1]) || same(c[1], c[2]) || same(c[2], c[0]);
    }
    for (int e = 0; e < m.E && !shared_corners; ++e)
        shared_corners = same(m.edge_idx[4 * (size_t)e + 2], m.edge_idx[4 * (size_t)e + 3]);
    // per-vertex spring items in spring-index order: 2 * spring + endpoint
    std::vector<int32_t> vs_off((size_t)N + 1, 0), vs_item;
    for (int s = 0; s < m.S; ++s)
        for (int e = 0; e < 2; ++e) {
            int v = m.spring_idx[2 * s + e];
            if (v < 0 || v >= N) return "spring_indices out of range";
            ++vs_off[v + 1];
        }
    for (int v = 0; v < N; ++v) vs_off[v + 1] += vs_off[v];
    vs_item.assign((size_t)vs_off[N], 0);
    {
        std::vector<int32_t> fill(vs_off.begin(), vs_off.end() - 1);
        for (int s = 0; s < m.S; ++s)
            for (int e = 0; e < 2; ++e) vs_item[fill[m.spring_idx[2 * s + e]]++] = 2 * s + e;
    }
    auto same_color = [&](int s) { return color_of[m.spring_idx[2 * s]] == color_of[m.spring_idx[2 * s + 1]]; };

    auto count_ok = [&](const std::vector<int32_t>& vals, const std::vector<int32_t>& off, const std::vector<char>& ok,
                        int v) {
        if (off.empty()) return 0;
        int c = 0;
        for (int p = off[v]; p < off[v + 1]; p += 2) c += ok[vals[p]] ? 1 : 0;
        return c;
    };
    // hinges by the vertex's place: opposite the edge (slots 0, 1) or on it (slots 2, 3)
    std::vector<int32_t> ntri((size_t)N, 0), nopp((size_t)N, 0), nedge((size_t)N, 0), ntet((size_t)N, 0), nspr((size_t)N, 0);
    for (int v = 0; v < N; ++v) {
        if (!active[v]) continue;
        if (m.T > 0) ntri[v] = count_ok(m.adj_tri, m.adj_tri_off, tri_ok, v);
        if (m.E > 0) {
            nedge[v] = count_ok(m.adj_edge, m.adj_edge_off, edge_ok, v);
            for (int p = m.adj_edge_off[v]; p < m.adj_edge_off[v + 1]; p += 2)
                nopp[v] += edge_ok[m.adj_edge[p]] && m.adj_edge[p + 1] < 2;
        }
        if (m.K > 0) ntet[v] = count_ok(m.adj_tet, m.adj_tet_off, tet_ok, v);
        nspr[v] = vs_off[v + 1] - vs_off[v];
    }
    L = PassLayout();
    L.cap = cap;
    L.max_v = max_v;
    L.blk_words = block_words(max_v);
    L.shape.shared_corners = shared_corners;
    L.vert_rec.assign((size_t)N * kVertWords, 0);
    L.fast_color_off.assign((size_t)C + 1, 0);
    L.slow_color_off.assign((size_t)C + 1, 0);
    L.pre_color_off.assign((size_t)C + 1, 0);
    L.slow_spr_off.push_back(0);
    // pre rows of same-color spring items, per color in color-position order
    std::vector<int32_t> pre_row((size_t)vs_off[N], -1);
    for (int c = 0; c < C; ++c) {
        L.pre_color_off[c] = (int32_t)(L.pre_item.size() / 2);
        for (int k = m.color_off[c]; k < m.color_off[c + 1]; ++k) {
            int v = m.color_particles[k];
            if (!active[v]) continue;
            for (int p = vs_off[v]; p < vs_off[v + 1]; ++p) {
                int s = vs_item[p] >> 1;
                if (!same_color(s)) continue;
                pre_row[p] = (int32_t)(L.pre_item.size() / 2);
                L.pre_item.push_back(s);
                L.pre_item.push_back(vs_item[p] & 1);
            }
        }
    }
    L.pre_color_off[C] = (int32_t)(L.pre_item.size() / 2);
    // fn(kind, element, slot, vertices of the element, their count) over v's items in canonical order
    auto for_items = [&](int v, auto&& fn) {
        if (!active[v]) return;
        if (m.T > 0)
            for (int p = m.adj_tri_off[v]; p < m.adj_tri_off[v + 1]; p += 2)
                if (tri_ok[m.adj_tri[p]]) fn(kTri, m.adj_tri[p], m.adj_tri[p + 1], &m.tri_idx[3 * (size_t)m.adj_tri[p]], 3);
        if (m.E > 0)
            for (int p = m.adj_edge_off[v]; p < m.adj_edge_off[v + 1]; p += 2)
                if (edge_ok[m.adj_edge[p]])
                    fn(kHinge, m.adj_edge[p], m.adj_edge[p + 1], &m.edge_idx[4 * (size_t)m.adj_edge[p]], 4);
        if (m.K > 0)
            for (int p = m.adj_tet_off[v]; p < m.adj_tet_off[v + 1]; p += 2)
                if (tet_ok[m.adj_tet[p]]) fn(kTet, m.adj_tet[p], m.adj_tet[p + 1], &m.tet_idx[4 * (size_t)m.adj_tet[p]], 4);
        for (int p = vs_off[v]; p < vs_off[v + 1]; ++p)
            fn(kSpring, p, vs_item[p] & 1, &m.spring_idx[2 * (size_t)(vs_item[p] >> 1)], 2);
    };

    // lane ranges of a batch: triangles, opposite hinges, edge hinges, tets, springs
    constexpr int kLanes = 5;

    // ---- the batches: greedy runs of a color's vertices that fit one work-group
    struct Batch {
        int vb, nv;
        int n[kLanes];     // items of each lane range
        bool one_hinge_range;
        int list_begin;    // into L.list while the runs are found
        int list_count;
    };
    std::vector<Batch> batches;
    std::vector<int32_t> lists;                       // vertex lists, one after another
    std::vector<int32_t> stamp((size_t)N, -1), slot_of((size_t)N, 0);
    PassShape& sh = L.shape;
    auto align = [&](int n) { return aligned ? wave_align(n) : n; };
    // First lane of each range and, at [kLanes], the lanes of all.  A vertex with more kinds than an aligned work-group
    // has waves (a spring on a cloth with 192 lanes, a cloth with 128) gets its hinges in one range, both forms in a
    // wave: on the generic path it would take ten times as long (256x256 cloth with springs, 192 aligned lanes,
    // substep 483 us, 6,900 us).
    struct Starts {
        int at[kLanes + 1];
    };
    auto starts = [&](const int* n, bool one_hinge_range) {
        Starts s{};
        for (int i = 0; i < kLanes; ++i)
            s.at[i + 1] = s.at[i] + align(n[i]);
        if (one_hinge_range) {
            const int saved = align(n[1]) + align(n[2]) - align(n[1] + n[2]);
            s.at[2] = s.at[1] + n[1];
            for (int i = 3; i <= kLanes; ++i) s.at[i] -= saved;
        }
        return s;
    };
    for (int c = 0; c < C; ++c) {
        L.fast_color_off[c] = (int32_t)batches.size();
        L.slow_color_off[c] = (int32_t)L.slow_pos.size();
        int k = m.color_off[c];
        const int kend = m.color_off[c + 1];
        while (k < kend) {
            const int id = (int)batches.size();
            Batch b{};
            b.vb = k;
            b.list_begin = (int)lists.size();
            std::vector<int32_t> seen;  // distinct vertices so far (own and neighbours)
            auto meet = [&](int v) {
                if (stamp[v] == id) return;
                stamp[v] = id;
                seen.push_back(v);
            };
            while (k < kend && b.nv < max_v) {
                const int v = m.color_particles[k];
                const int add[kLanes] = {ntri[v], nopp[v], nedge[v] - nopp[v], ntet[v], nspr[v]};
                int n[kLanes];
                for (int i = 0; i < kLanes; ++i) n[i] = b.n[i] + add[i];
                if (b.nv == 0 && starts(n, false).at[kLanes] > cap) b.one_hinge_range = true;
                if (starts(n, b.one_hinge_range).at[kLanes] > cap) break;
                const size_t before = seen.size();
                meet(v);
                for_items(v, [&](int, int, int, const int32_t* e, int n) {
                    for (int i = 0; i < n; ++i) meet(e[i]);
                });
                if ((int)seen.size() > list_cap(cap)) {
                    for (size_t i = before; i < seen.size(); ++i) stamp[seen[i]] = -1;
                    seen.resize(before);
                    break;
                }
                for (int i = 0; i < kLanes; ++i) b.n[i] += add[i];
                ++b.nv;
                ++k;
            }
            if (b.nv == 0) {  // oversized vertex: generic kernel
                const int v0 = m.color_particles[k];
                L.slow_pos.push_back(k);
                if (active[v0])
                    for (int p = vs_off[v0]; p < vs_off[v0 + 1]; ++p) {
                        const int32_t r[4] = {vs_item[p] >> 1, vs_item[p] & 1, pre_row[p], 0};
                        L.slow_spr.insert(L.slow_spr.end(), r, r + 4);
                    }
                L.slow_spr_off.push_back((int32_t)(L.slow_spr.size() / 4));
                ++k;
                continue;
            }
            // the batch's own vertices first, then the others in the order they were met
            for (int v : seen) slot_of[v] = -1;
            for (int s = 0; s < b.nv; ++s) {
                lists.push_back(m.color_particles[b.vb + s]);
                slot_of[m.color_particles[b.vb + s]] = s;
            }
            for (int v : seen)
                if (slot_of[v] < 0) lists.push_back(v);
            b.list_count = (int)lists.size() - b.list_begin;
            sh.list_stride = std::max(sh.list_stride, b.list_count);
            const Starts first = starts(b.n, b.one_hinge_range);
            LaneRange* ranges[kLanes] = {&sh.tri, &sh.hinge, &sh.hinge, &sh.tet, &sh.spring};
            for (int i = 0; i < kLanes; ++i) ranges[i]->cover(first.at[i], first.at[i] + b.n[i]);
            batches.push_back(b);
        }
    }
    L.fast_color_off[C] = (int32_t)batches.size();
    L.slow_color_off[C] = (int32_t)L.slow_pos.size();

    // ---- the records
    const size_t B = batches.size();
    sh.list_stride = (sh.list_stride + 3) & ~3;
    // A pass of every kind reads one record a lane, of any kind, from the array of the widest: an array a kind, it read
    // the slots of each in every batch (cloth of 128x128 and eight tet cubes, substep 285 us, 271 us so).
    const bool shared_rec = (kinds_of_pass(sh, false, m.self_contact) & 3) == pass_kinds::kAllKinds;
    if (shared_rec) {
        sh.tet.cover(sh.tri.lo, sh.tri.hi);
        sh.tet.cover(sh.spring.lo, sh.spring.hi);
    }
    L.batch_blk.assign(B * (size_t)L.blk_words, 0);
    L.item_rec.assign(B * (size_t)cap * kItemWords, 0);
    L.list.assign(B * (size_t)sh.list_stride, 0);
    L.tri_rec.assign(shared_rec ? 0 : B * (size_t)sh.tri.count() * kTriWords, 0);
    L.tet_rec.assign(B * (size_t)sh.tet.count() * kTetWords, 0);
    L.spr_rec.assign(shared_rec ? 0 : B * (size_t)sh.spring.count() * kSpringWords, 0);
    L.hinge_damp.assign(B * (size_t)sh.hinge.count(), 0);
    for (size_t bi = 0; bi < B; ++bi) {
        const Batch& b = batches[bi];
        const int32_t* list = &lists[(size_t)b.list_begin];
        std::memcpy(&L.list[bi * (size_t)sh.list_stride], list, sizeof(int32_t) * (size_t)b.list_count);
        for (int i = b.list_count; i < sh.list_stride; ++i) L.list[bi * (size_t)sh.list_stride + i] = list[0];
        for (int i = 0; i < b.list_count; ++i) slot_of[list[i]] = i;
        const Starts first = starts(b.n, b.one_hinge_range);
        int lane[kLanes];
        for (int i = 0; i < kLanes; ++i) lane[i] = first.at[i];
        int32_t* head = &L.batch_blk[bi * (size_t)L.blk_words];
        int row = 0, flags = 0;
        for (int s = 0; s < b.nv; ++s) {
            const int v = m.color_particles[b.vb + s];
            const int nr = ntri[v] + nedge[v] + ntet[v];
            int32_t* vr = &L.vert_rec[(size_t)(b.vb + s) * kVertWords];
            vr[0] = v;
            vr[1] = row;
            vr[2] = nr;
            vr[3] = s | ((active[v] ? 1 : 0) << 16) | (nspr[v] << 17);
            std::memcpy(head + kBatchWords + s * kVertWords, vr, sizeof(int32_t) * kVertWords);
            for_items(v, [&](int kind, int e, int slot, const int32_t* who, int n) {
                const int which = kind == kTri ? 0 : (kind == kHinge ? 1 + (slot >> 1) : (kind == kTet ? 3 : 4));
                const int t = lane[which]++;
                int32_t* r = &L.item_rec[(bi * (size_t)cap + t) * kItemWords];
                uint32_t slots = 0;
                for (int i = 0; i < n; ++i) slots |= (uint32_t)slot_of[who[i]] << (8 * i);
                r[0] = (int32_t)slots;
                bool damped = false;
                auto record = [&](std::vector<int32_t>& own, const LaneRange& range, int words) {
                    return shared_rec ? &L.tet_rec[(bi * (size_t)sh.tet.count() + (t - sh.tet.lo)) * kTetWords]
                                      : &own[(bi * (size_t)range.count() + (t - range.lo)) * words];
                };
                if (kind == kTri) {
                    const float* mat = &m.tri_mat[5 * (size_t)e];
                    int32_t* w = record(L.tri_rec, sh.tri, kTriWords);
                    for (int q = 0; q < 4; ++q) w[q] = fbits(m.tri_pose[4 * (size_t)e + q]);
                    w[4] = fbits(mat[0]);
                    w[5] = fbits(lame_sum(mat[0], mat[1]));
                    w[6] = fbits(rest_ratio(mat[0], mat[1]));
                    w[7] = fbits(mat[2]);
                    r[2] = fbits(m.tri_area[e]);
                    damped = mat[2] > 0.0f;
                } else if (kind == kHinge) {
                    const float* bend = &m.edge_bend[2 * (size_t)e];
                    r[2] = fbits(m.edge_rest[e]);
                    r[3] = fbits(bend[0] * m.edge_len[e]);
                    damped = bend[1] > 0.0f;
                    if (damped) flags |= kHingeDamped;
                    L.hinge_damp[bi * (size_t)sh.hinge.count() + (t - sh.hinge.lo)] = fbits(bend[1] * m.edge_len[e]);
                } else if (kind == kTet) {
                    const float* mat = &m.tet_mat[3 * (size_t)e];
                    const float* dm = &m.tet_pose[9 * (size_t)e];
                    int32_t* w = record(L.tet_rec, sh.tet, kTetWords);
                    for (int q = 0; q < 9; ++q) w[q] = fbits(dm[q]);
                    w[9] = fbits(rest_volume(dm));
                    w[10] = fbits(rest_ratio(mat[0], mat[1]));
                    w[11] = fbits(mat[2]);
                    r[2] = fbits(mat[0]);
                    r[3] = fbits(lame_sum(mat[0], mat[1]));
                    damped = mat[2] > 0.0f;
                } else {  // e indexes vs_item
                    const int sp = vs_item[e] >> 1;
                    int32_t* w = record(L.spr_rec, sh.spring, kSpringWords);
                    w[0] = fbits(m.spring_ke[sp]);
                    w[1] = fbits(m.spring_kd[sp]);
                    r[2] = pre_row[e];
                    r[3] = fbits(m.spring_rest[sp]);
                    damped = true;  // a spring always reads its endpoints' previous positions
                }
                if (damped) flags |= kPrevAll;
                r[1] = item_meta(row, slot, damped, kind);
                ++row;
            });
        }
        head[0] = b.vb;
        head[1] = b.nv;
        head[2] = row;
        head[3] = flags;
        L.fast_items += row;
    }
    return std::string();
}

}  // namespace vbd_layout
