// The Kuhn triangulation of TetrahedronMesh.from_box: corners, tetrahedra and
// neighbour offsets as compile-time constants.
#pragma once
#include "common.hpp"

namespace fa {

// TetrahedronMesh.from_box (tetrahedron_mesh.py:1017-1086) numbers node
// (ix, iy, iz) as (ix (ny+1) + iy) (nz+1) + iz, cube (cx, cy, cz) as
// (cx ny + cy) nz + cz, and cell 6 cube + t, the Kuhn tetrahedron t over the
// cube corners box_kuhn(t, v).  The cells around a node in ascending order are
// those of the cubes (ix - a, iy - b, iz - c) in the order (a, b, c) = (1,1,1),
// (1,1,0), ..., (0,0,0), and in each the tetrahedra that hold the node's corner,
// ascending t.
// offsets of corner k as bit masks over k (corners 1, 2, 5, 6 have x + 1;
// 2, 3, 6, 7 have y + 1; 4-7 have z + 1): branch-free for a runtime k
constexpr int box_cdx(int k) { return (0x66 >> k) & 1; }
constexpr int box_cdy(int k) { return (0xCC >> k) & 1; }
constexpr int box_cdz(int k) { return (k >> 2) & 1; }
constexpr int box_corner_of(int a, int b, int c) {
    return c == 0 ? (a == 0 ? (b == 0 ? 0 : 3) : (b == 0 ? 1 : 2)) : (a == 0 ? (b == 0 ? 4 : 7) : (b == 0 ? 5 : 6));
}
constexpr int box_kuhn(int t, int v) {
    constexpr int K[6][4] = {{0, 1, 2, 6}, {0, 5, 1, 6}, {0, 4, 5, 6}, {0, 7, 4, 6}, {0, 3, 7, 6}, {0, 2, 3, 6}};
    return K[t][v];
}
// local index of corner k in tetrahedron t, or -1
constexpr int box_local(int t, int k) {
    return box_kuhn(t, 0) == k ? 0 : box_kuhn(t, 1) == k ? 1 : box_kuhn(t, 2) == k ? 2 : box_kuhn(t, 3) == k ? 3 : -1;
}
// accumulator slot of offset (dx, dy, dz): rank among the 15 offsets in
// lexicographic order, -1 for an offset that is no Kuhn edge
constexpr int box_slot(int dx, int dy, int dz) {
    constexpr int S[27] = {0, 1, -1, 2, 3, -1, -1, -1, -1, 4, 5, -1, 6, 7, 8, -1, 9, 10,
                           -1, -1, -1, -1, 11, 12, -1, 13, 14};
    return S[(dx + 1) * 9 + (dy + 1) * 3 + (dz + 1)];
}
constexpr int BOX_SLOTS = 15;

// Kuhn tetrahedra as paths: the corners of tetrahedron t, ordered by their
// number of +1 offsets, run from corner 0 to corner 6 one axis at a time.
// box_pos: path position of local vertex v; box_axis: the axis of path step
// p (1..3); box_sign: orientation of the local vertex order (the sign of
// det(o1 - o0, o2 - o0, o3 - o0) on the unit cube)
constexpr int box_pos(int t, int v) {
    return box_cdx(box_kuhn(t, v)) + box_cdy(box_kuhn(t, v)) + box_cdz(box_kuhn(t, v));
}
constexpr int box_corner_at(int t, int p) {
    return box_pos(t, 0) == p ? box_kuhn(t, 0)
           : box_pos(t, 1) == p ? box_kuhn(t, 1)
           : box_pos(t, 2) == p ? box_kuhn(t, 2)
                                : box_kuhn(t, 3);
}
constexpr int box_axis(int t, int p) {
    return box_cdx(box_corner_at(t, p)) != box_cdx(box_corner_at(t, p - 1))   ? 0
           : box_cdy(box_corner_at(t, p)) != box_cdy(box_corner_at(t, p - 1)) ? 1
                                                                               : 2;
}
constexpr int box_off(int t, int v, int d) {
    return (d == 0 ? box_cdx(box_kuhn(t, v)) : d == 1 ? box_cdy(box_kuhn(t, v)) : box_cdz(box_kuhn(t, v))) -
           (d == 0 ? box_cdx(box_kuhn(t, 0)) : d == 1 ? box_cdy(box_kuhn(t, 0)) : box_cdz(box_kuhn(t, 0)));
}
constexpr int box_sign(int t) {
    return box_off(t, 1, 0) * (box_off(t, 2, 1) * box_off(t, 3, 2) - box_off(t, 2, 2) * box_off(t, 3, 1)) -
           box_off(t, 1, 1) * (box_off(t, 2, 0) * box_off(t, 3, 2) - box_off(t, 2, 2) * box_off(t, 3, 0)) +
           box_off(t, 1, 2) * (box_off(t, 2, 0) * box_off(t, 3, 1) - box_off(t, 2, 1) * box_off(t, 3, 0));
}

// tab[((k * nmax + i) * 6 + t) * nq + q]: factor k of a separable expression at
// point q of tetrahedron t in the cubes of index i along its dimension, nmax the
// largest of nx, ny, nz; axes: nx + ny + nz + 3 grid-line coordinates
int launch_box_sep_table(int nx, int ny, int nz, const double* node_wide, const void* sep, int nq, double* axes,
                         double* tab, hipStream_t s);

}  // namespace fa
