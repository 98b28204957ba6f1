// CPU checks of host parts of libBaryTree_gpu.so that the C ABI does not show:
// the interaction lists' order and the cover check of the near field's items.
// Test infrastructure only; compiled by tests/test_host_checks.py.
#include <cmath>
#include <cstdio>
#include <string>
#include <vector>

#include "../barytree_amd/csrc/bt_host.h"
#include "../barytree_amd/csrc/bt_solver.h"

using namespace bt;

namespace {

// The reference's walks (interaction_lists.c:464-533, 537-748) in one thread.
void pc_walk(Lists &L, int key, const Tree &k, const Tree &s, int node, const Params &prm)
{
    const double dx = k.xmid[key] - s.xmid[node], dy = k.ymid[key] - s.ymid[node], dz = k.zmid[key] - s.zmid[node];
    const double dist = std::sqrt(dx * dx + dy * dy + dz * dz);
    if (s.radius[node] + k.radius[key] < dist * prm.theta && s.radius[node] != 0.0 &&
        prm.size_check_factor * prm.P < s.numpar[node]) {
        L.approx[key].push_back(node);
    } else if (s.nchild[node] == 0) {
        L.pp[key].push_back(node);
    } else {
        for (int i = 0; i < s.nchild[node]; i++) pc_walk(L, key, k, s, s.child[8 * node + i], prm);
    }
}

void cc_walk(Lists &L, const Tree &s, int sn, const Tree &t, int tn, const Params &prm)
{
    const int small = (int)(prm.size_check_factor * prm.P);
    const double dx = t.xmid[tn] - s.xmid[sn], dy = t.ymid[tn] - s.ymid[sn], dz = t.zmid[tn] - s.zmid[sn];
    const double dist = std::sqrt(dx * dx + dy * dy + dz * dz);
    if (s.radius[sn] + t.radius[tn] < dist * prm.theta) {
        const bool ss = s.numpar[sn] <= small, ts = t.numpar[tn] <= small;
        (ss && ts ? L.pp : ss ? L.cc_cp : ts ? L.cc_pc : L.approx)[tn].push_back(sn);
        return;
    }
    const bool tleaf = t.nchild[tn] == 0, sleaf = s.nchild[sn] == 0;
    if (tleaf && sleaf) {
        L.pp[tn].push_back(sn);
    } else if (sleaf || (!tleaf && s.numpar[sn] < t.numpar[tn])) {
        for (int i = 0; i < t.nchild[tn]; i++) cc_walk(L, s, sn, t, t.child[8 * tn + i], prm);
    } else {
        for (int i = 0; i < s.nchild[sn]; i++) cc_walk(L, s, s.child[8 * sn + i], t, tn, prm);
    }
}

bool make_tree(Tree &t, int n, const double *x, const double *y, const double *z, int leaf, bool leaves_only)
{
    Particles p;
    p.n = n;
    p.x.assign(x, x + n); p.y.assign(y, y + n); p.z.assign(z, z + n);
    p.q.assign(n, 0.0);
    p.order.resize(n);
    for (int i = 0; i < n; i++) p.order[i] = i;
    return build_tree(t, p, leaf, leaves_only).empty();
}

}  // namespace

// Lists of sources n, targets m against the plain walks, entry by entry in
// order; returns the number of lists that differ, -1 on a tree error, and the
// number of keys.
extern "C" int check_lists(int cc, int n, const double *sx, const double *sy, const double *sz, int m,
                           const double *tx, const double *ty, const double *tz, double theta, int degree, int leaf,
                           int *keys)
{
    Params prm;
    prm.theta = theta; prm.degree = degree; prm.P = (degree + 1) * (degree + 1) * (degree + 1);
    prm.size_check_factor = 1.0;
    Tree s, t;
    if (!make_tree(s, n, sx, sy, sz, leaf, false) || !make_tree(t, m, tx, ty, tz, leaf, !cc)) return -1;
    Lists got, want;
    for (auto *v : {&want.pp, &want.approx, &want.cc_pc, &want.cc_cp}) v->resize(t.n);
    if (cc) {
        make_cc_lists(got, s, t, prm);
        cc_walk(want, s, 0, t, 0, prm);
    } else {
        make_pc_lists(got, s, t, prm);
        for (int k = 0; k < t.n; k++) pc_walk(want, k, t, s, 0, prm);
        got.cc_pc.resize(t.n);
        got.cc_cp.resize(t.n);
    }
    *keys = t.n;
    int bad = 0;
    for (int k = 0; k < t.n; k++)
        bad += (got.pp[k] != want.pp[k]) + (got.approx[k] != want.approx[k]) + (got.cc_pc[k] != want.cc_pc[k]) +
               (got.cc_cp[k] != want.cc_cp[k]);
    return bad;
}

// check_items on two keys (targets 0..299 with ranges of 5 and 7 sources,
// targets 300..309 with none) and one more (310..319, 4 sources), whole and
// with one part missing or doubled.  Returns the number of the first case with
// the wrong verdict, 0 if none.
extern "C" int check_cover()
{
    WorkCSR near;
    near.key = {3, 4, 5};
    near.tbeg = {0, 300, 310};
    near.tcnt = {300, 10, 10};
    near.seg_off = {0, 2, 2, 3};
    near.seg_beg = {0, 5, 20};
    near.seg_cnt = {5, 7, 4};
    const std::vector<int> off = {0, 2, 2, 3};
    const std::vector<btk::Tile> tiles = {{0, 0, 256, 0}, {0, 256, 44, 0}, {2, 310, 10, 0}};
    const long long pairs = 300 * 12 + 10 * 4;
    if (!check_items(near, off, tiles, pairs).empty()) return 1;
    if (check_items(near, off, tiles, pairs - 10 * 4).empty()) return 2;               // an item's pairs missing
    if (check_items(near, {0, 1, 1, 2}, tiles, pairs).empty()) return 3;               // a slot missing
    if (check_items(near, off, {tiles[0], tiles[1]}, pairs).empty()) return 4;         // a key not reduced
    if (check_items(near, off, {tiles[0], tiles[2]}, pairs).empty()) return 5;         // targets left out
    if (check_items(near, off, {tiles[0], tiles[1], tiles[1], tiles[2]}, pairs).empty()) return 6;  // twice
    if (check_items(near, off, {tiles[0], tiles[1], {1, 300, 10, 0}, tiles[2]}, pairs).empty()) return 7;
    if (check_items(near, {0, 2, 2}, tiles, pairs).empty()) return 8;
    return 0;
}
