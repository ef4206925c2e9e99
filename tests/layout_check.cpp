// Checks a color-pass layout (vbd_layout.h) against the mesh it was built from; driven by test_pass_layout.py.
// Returns 0, or the line of the first check that failed.
#include "../newton_amd/csrc/vbd_layout.h"

#define CHECK(c) \
    do {         \
        if (!(c)) return __LINE__; \
    } while (0)

using namespace vbd_layout;

#define MODEL_ARGS                                                                                                    \
    int N, int T, int E, int K, int S, int C, const float *mass, const int *flags, const int *tri,                   \
        const float *tri_mat, const int *edge, const float *bend, const int *tet, const float *tet_mat,              \
        const int *at_off, const int *at, const int *ae_off, const int *ae, const int *ak_off, const int *ak,        \
        const int *spring, const int *color_off, const int *color_particles
#define MODEL_NAMES                                                                                                    \
    N, T, E, K, S, C, mass, flags, tri, tri_mat, edge, bend, tet, tet_mat, at_off, at, ae_off, ae, ak_off, ak, spring, \
        color_off, color_particles

static HostModel host_model(MODEL_ARGS) {
    HostModel m;
    m.N = N, m.T = T, m.E = E, m.K = K, m.S = S;
    m.mass.assign(mass, mass + N);
    m.flags.assign(flags, flags + N);
    m.tri_idx.assign(tri, tri + 3 * T);
    m.tri_mat.assign(tri_mat, tri_mat + 5 * T);
    m.tri_pose.resize(4 * (size_t)T);
    m.tri_area.resize(T);
    for (int t = 0; t < T; ++t) m.tri_area[t] = (float)t;  // names the element an item came from
    m.edge_idx.assign(edge, edge + 4 * E);
    m.edge_bend.assign(bend, bend + 2 * E);
    m.edge_len.assign(E, 1.0f);
    m.edge_rest.resize(E);
    for (int e = 0; e < E; ++e) m.edge_rest[e] = (float)e;
    m.tet_idx.assign(tet, tet + 4 * K);
    m.tet_mat.assign(tet_mat, tet_mat + 3 * K);
    m.tet_pose.assign(9 * (size_t)K, 0.0f);
    for (int k = 0; k < K; ++k) m.tet_pose[9 * (size_t)k + 1] = (float)k;
    if (T) m.adj_tri_off.assign(at_off, at_off + N + 1), m.adj_tri.assign(at, at + at_off[N]);
    if (E) m.adj_edge_off.assign(ae_off, ae_off + N + 1), m.adj_edge.assign(ae, ae + ae_off[N]);
    if (K) m.adj_tet_off.assign(ak_off, ak_off + N + 1), m.adj_tet.assign(ak, ak + ak_off[N]);
    m.spring_idx.assign(spring, spring + 2 * S);
    m.spring_rest.resize(S);
    for (int s = 0; s < S; ++s) m.spring_rest[s] = (float)s;
    m.spring_ke.resize(S);
    m.spring_kd.resize(S);
    for (int s = 0; s < S; ++s) m.spring_ke[s] = 2.0f + s, m.spring_kd[s] = 0.5f + s;
    m.color_off.assign(color_off, color_off + C + 1);
    m.color_particles.assign(color_particles, color_particles + N);
    return m;
}

// v: the model's arrays in HostModel order; stats: {batches, slow vertices, items, list stride}
extern "C" int check_layout(MODEL_ARGS, int cap, int max_v, int aligned, long long* stats) {
    const HostModel m = host_model(MODEL_NAMES);
    PassLayout L;
    if (!build_pass_layout(m, L, cap, max_v, aligned != 0).empty()) return -1;

    const int B = L.fast_color_off[C];
    const PassShape& sh = L.shape;
    CHECK((int)L.fast_color_off.size() == C + 1 && (int)L.slow_color_off.size() == C + 1);
    CHECK(L.batch_blk.size() == (size_t)B * L.blk_words && L.item_rec.size() == (size_t)B * cap * kItemWords);
    CHECK(L.list.size() == (size_t)B * sh.list_stride && sh.list_stride <= list_cap(cap) && sh.tri.lo == 0);
    CHECK(sh.tri.hi <= cap && sh.hinge.hi <= cap && sh.tet.hi <= cap && sh.spring.hi <= cap);
    // records of every kind share one array when a pass holds every kind
    const bool shared = (kinds_of_pass(sh, false, false) & 3) == pass_kinds::kAllKinds;
    CHECK(!shared || (L.tri_rec.empty() && L.spr_rec.empty()));
    if (shared) CHECK(sh.tet.hi >= sh.tri.hi && sh.tet.hi >= sh.spring.hi && (sh.tri.count() == 0 || sh.tet.lo == 0));
    std::vector<int> color_of(N);
    for (int c = 0; c < C; ++c)
        for (int k = color_off[c]; k < color_off[c + 1]; ++k) color_of[color_particles[k]] = c;
    std::vector<char> done(N, 0);
    long long items = 0;
    for (int c = 0; c < C; ++c)
        for (int b = L.fast_color_off[c]; b < L.fast_color_off[c + 1]; ++b) {
            const int32_t* h = &L.batch_blk[(size_t)b * L.blk_words];
            const int vb = h[0], nv = h[1], nrows = h[2];
            CHECK(nv >= 1 && nv <= max_v && vb >= color_off[c] && vb + nv <= color_off[c + 1]);
            CHECK(nrows <= cap);
            const int32_t* list = &L.list[(size_t)b * sh.list_stride];
            const int count = sh.list_stride;
            CHECK(count >= nv);
            for (int i = 0; i < count; ++i) CHECK(list[i] >= 0 && list[i] < N);
            // the batch's first vertex: do its kinds, each on a wave boundary, fit the work-group?
            int lanes = 0;
            {
                const int v = h[kBatchWords], active = (flags[v] & 1) && mass[v] != 0.0f;
                int n[5] = {0, 0, 0, 0, 0};
                if (T && active)
                    for (int p = at_off[v]; p < at_off[v + 1]; p += 2)
                        n[0] += tri_mat[5 * at[p]] > 0.0f || tri_mat[5 * at[p] + 1] > 0.0f;
                if (E && active)
                    for (int p = ae_off[v]; p < ae_off[v + 1]; p += 2)
                        n[1 + ae[p + 1] / 2] += bend[2 * ae[p]] > 0.0f && edge[4 * ae[p]] >= 0 && edge[4 * ae[p] + 1] >= 0;
                if (K && active)
                    for (int p = ak_off[v]; p < ak_off[v + 1]; p += 2)
                        n[3] += tet_mat[3 * ak[p]] > 0.0f || tet_mat[3 * ak[p] + 1] > 0.0f;
                for (int sp = 0; sp < 2 * S && active; ++sp) n[4] += spring[sp] == v;
                for (int k : n) lanes += aligned ? (k + 63) / 64 * 64 : k;
            }
            const bool one_hinge_range = lanes > cap;
            std::vector<int> row_owner(nrows, -1), row_kind(nrows, 0), row_elem(nrows, -1), row_slot(nrows, -1);
            for (int t = 0; t < cap; ++t) {
                const int32_t* r = &L.item_rec[((size_t)b * cap + t) * kItemWords];
                const int kind = r[1] >> 12, row = r[1] & 0x1ff, slot = (r[1] >> 9) & 3;
                if (kind == kNone) continue;
                ++items;
                CHECK(row < nrows && row_kind[row] == 0);
                int elem = -1, n = 0;
                const int32_t* who = nullptr;
                float f;
                if (kind == kTri) {
                    CHECK(t < sh.tri.hi);
                    std::memcpy(&f, &r[2], 4);
                    elem = (int)f, n = 3, who = &m.tri_idx[3 * (size_t)elem];
                    const int32_t* w = shared ? &L.tet_rec[((size_t)b * sh.tet.count() + t - sh.tet.lo) * kTetWords]
                                              : &L.tri_rec[((size_t)b * sh.tri.count() + t) * kTriWords];
                    CHECK(w[4] == fbits(m.tri_mat[5 * (size_t)elem]) && w[7] == fbits(m.tri_mat[5 * (size_t)elem + 2]));
                } else if (kind == kHinge) {
                    CHECK(t >= sh.hinge.lo && t < sh.hinge.hi);
                    std::memcpy(&f, &r[2], 4);
                    elem = (int)f, n = 4, who = &m.edge_idx[4 * (size_t)elem];
                } else if (kind == kTet) {
                    CHECK(t >= sh.tet.lo && t < sh.tet.hi);
                    std::memcpy(&f, &L.tet_rec[((size_t)b * sh.tet.count() + t - sh.tet.lo) * kTetWords + 1], 4);
                    elem = (int)f, n = 4, who = &m.tet_idx[4 * (size_t)elem];
                } else {
                    CHECK(kind == kSpring && t >= sh.spring.lo && t < sh.spring.hi);
                    std::memcpy(&f, &r[3], 4);
                    elem = (int)f, n = 2, who = &m.spring_idx[2 * (size_t)elem];
                    const int32_t* w = shared ? &L.tet_rec[((size_t)b * sh.tet.count() + t - sh.tet.lo) * kTetWords]
                                              : &L.spr_rec[((size_t)b * sh.spring.count() + t - sh.spring.lo) * kSpringWords];
                    CHECK(w[0] == fbits(m.spring_ke[elem]) && w[1] == fbits(m.spring_kd[elem]));
                }
                if (aligned) {  // a wave evaluates one kind, and one form of a hinge, only
                    const int32_t* first = &L.item_rec[((size_t)b * cap + (t & ~63)) * kItemWords];
                    CHECK(first[1] >> 12 == kind);
                    if (kind == kHinge && !one_hinge_range) CHECK((first[1] >> 10 & 1) == slot >> 1);
                }
                for (int i = 0; i < n; ++i) {
                    const int at_slot = (uint32_t)r[0] >> (8 * i) & 0xff;
                    CHECK(at_slot < count && list[at_slot] == who[i]);
                }
                row_kind[row] = kind;
                row_elem[row] = elem;
                row_slot[row] = slot;
                row_owner[row] = who[slot];
            }
            int next = 0;
            for (int s = 0; s < nv; ++s) {
                const int32_t* vr = h + kBatchWords + kVertWords * s;
                const int v = vr[0];
                CHECK(v == color_particles[vb + s] && list[s] == v && !done[v] && vr[1] == next);
                done[v] = 1;
                const bool active = (flags[v] & 1) && mass[v] != 0.0f;
                CHECK((vr[3] & 0xffff) == s && ((vr[3] >> 16) & 1) == (active ? 1 : 0));
                // rows in canonical order: the CSR's triangles, hinges, tets, then the springs by index
                int r = next;
                auto expect = [&](int kind, int elem, int slot) {
                    if (!active) return true;
                    const bool ok = r < nrows && row_kind[r] == kind && row_elem[r] == elem && row_slot[r] == slot &&
                                    row_owner[r] == v;
                    ++r;
                    return ok;
                };
                if (T)
                    for (int p = at_off[v]; p < at_off[v + 1]; p += 2)
                        if (tri_mat[5 * at[p]] > 0.0f || tri_mat[5 * at[p] + 1] > 0.0f)
                            CHECK(expect(kTri, at[p], at[p + 1]));
                if (E)
                    for (int p = ae_off[v]; p < ae_off[v + 1]; p += 2)
                        if (bend[2 * ae[p]] > 0.0f && edge[4 * ae[p]] >= 0 && edge[4 * ae[p] + 1] >= 0)
                            CHECK(expect(kHinge, ae[p], ae[p + 1]));
                if (K)
                    for (int p = ak_off[v]; p < ak_off[v + 1]; p += 2)
                        if (tet_mat[3 * ak[p]] > 0.0f || tet_mat[3 * ak[p] + 1] > 0.0f)
                            CHECK(expect(kTet, ak[p], ak[p + 1]));
                CHECK(vr[2] == r - next);
                const int elements = r;
                for (int sp = 0; sp < S; ++sp)
                    for (int e = 0; e < 2; ++e)
                        if (spring[2 * sp + e] == v) CHECK(expect(kSpring, sp, e));
                CHECK(vr[3] >> 17 == r - elements);
                next = r;
            }
            CHECK(next == nrows);
        }
    for (int k : L.slow_pos) {
        CHECK(!done[color_particles[k]]);
        done[color_particles[k]] = 1;
    }
    for (int v = 0; v < N; ++v) CHECK(done[v]);
    CHECK(items == L.fast_items);
    stats[0] = B, stats[1] = (long long)L.slow_pos.size(), stats[2] = items, stats[3] = sh.list_stride;
    return 0;
}

// Layouts that differ in damping only, zero or not, may be written over one another under a captured graph: the same
// array sizes, batch ranges and launch arguments; the batch flags tell what each batch reads.
extern "C" int check_damping_edit(MODEL_ARGS, int cap, int max_v, int aligned) {
    const HostModel base = host_model(MODEL_NAMES);
    PassLayout L[4];
    for (int i = 0; i < 4; ++i) {
        HostModel m = base;
        for (int t = 0; t < T; ++t) m.tri_mat[5 * (size_t)t + 2] = i & 1 ? 0.5f : 0.0f;
        for (int k = 0; k < K; ++k) m.tet_mat[3 * (size_t)k + 2] = i & 1 ? 0.5f : 0.0f;
        for (int e = 0; e < E; ++e) m.edge_bend[2 * (size_t)e + 1] = i & 2 ? 0.25f : 0.0f;
        if (!build_pass_layout(m, L[i], cap, max_v, aligned != 0).empty()) return -1;
    }
    for (int i = 1; i < 4; ++i) {
        CHECK(L[i].shape == L[0].shape && L[i].batch_blk.size() == L[0].batch_blk.size());
        CHECK(L[i].item_rec.size() == L[0].item_rec.size() && L[i].list == L[0].list);
        CHECK(L[i].tri_rec.size() == L[0].tri_rec.size() && L[i].tet_rec.size() == L[0].tet_rec.size());
        CHECK(L[i].hinge_damp.size() == L[0].hinge_damp.size() && L[i].spr_rec.size() == L[0].spr_rec.size());
        CHECK(L[i].fast_color_off == L[0].fast_color_off && L[i].slow_color_off == L[0].slow_color_off);
    }
    const int B = L[0].fast_color_off[C];
    for (int i = 0; i < 4; ++i)
        for (int b = 0; b < B; ++b) {
            int want = 0;
            for (int t = 0; t < cap; ++t) {
                const int meta = L[i].item_rec[((size_t)b * cap + t) * kItemWords + 1], kind = meta >> 12;
                const bool hinge = kind == kHinge && (i & 2), other = (kind == kTri || kind == kTet) && (i & 1);
                CHECK((meta >> 11 & 1) == (hinge || other || kind == kSpring));
                want |= hinge ? kPrevAll | kHingeDamped : (other || kind == kSpring ? kPrevAll : 0);
            }
            CHECK(L[i].batch_blk[(size_t)b * L[i].blk_words + 3] == want);
        }
    return 0;
}

// 1 when two corners of some edge or triangle share a color, 0 when not
extern "C" int shares_corners(MODEL_ARGS, int cap, int max_v, int aligned) {
    const HostModel m = host_model(MODEL_NAMES);
    PassLayout L;
    if (!build_pass_layout(m, L, cap, max_v, aligned != 0).empty()) return -1;
    return L.shape.shared_corners ? 1 : 0;
}

// Every combination of element ranges and contact kinds has a compiled pass that holds its kinds.
extern "C" int check_kinds() {
    using namespace pass_kinds;
    for (int mask = 0; mask < 64; ++mask) {
        PassShape sh;
        if (mask & 1) sh.tri.cover(0, 10);
        if (mask & 2) sh.hinge.cover(10, 20);
        if (mask & 4) sh.tet.cover(20, 30);
        if (mask & 8) sh.spring.cover(30, 40);
        const int kinds = kinds_of_pass(sh, mask & 16, mask & 32), elems = kinds & 3;
        bool found = false;
        for (int k : kInstantiated) found = found || k == kinds;
        CHECK(found);
        CHECK(!(mask & 3) || elems != kTetKinds);
        CHECK(!(mask & 4) || elems == kTetKinds || elems == kAllKinds);
        CHECK(!(mask & 8) || elems == kClothSpringKinds || elems == kAllKinds);
        CHECK(((kinds & kEdgeFace) != 0) == ((mask & 16) != 0) && ((kinds & kSelfRows) != 0) == ((mask & 32) != 0));
    }
    return 0;
}
