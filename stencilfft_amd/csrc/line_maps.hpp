// line_maps.hpp -- host side of the natural-order line passes and of the layout
// converters: their address maps for every (N, P, B).
#pragma once

#include "kernels.hpp"

namespace zm {

// ---------------------------------------------------------------------------
// Address maps of the natural-order line passes (line_pass.hpp).  With lower-
// case names for the log2 of N, P, B, L, VEC, .. a rank slab holds 2^(d l)
// elements and rank ids run col, row, depth; a line's index lambda counts, from
// its lowest bits, the position y its tile runs along, the untouched index e
// (3D) and the rank coordinates off the axis.
//
// Between the y and the z pass of a tiled 3D transform a slab holds [row]
// [depth][col] instead of [depth][row][col]: a z tile then reads runs L
// elements apart like a y tile, where runs L^2 apart (512 KB at 512^3) cost
// the inverse pass 11% (0.409 -> 0.368 ms, FP32).
// ---------------------------------------------------------------------------
struct NatMaps {
    const Geo& g;
    int d, lvp, lm, slab;
    explicit NatMaps(const Geo& geo)
        : g(geo), d(geo.dims), lvp(geo.lvec - geo.lp), lm(geo.lb + geo.lp), slab(geo.dims * geo.ll) {}

    int member(int axis) const { return slab + axis * g.lp; }  // shift of the axis's own rank coordinate
    // lambda -> line base: y at shift `ys`, e at `es`, the ranks off `axis`
    BitMap<4> lines(int axis, int ys, int es) const {
        const int lo = member(axis == 0 ? 1 : 0), hi = member(axis == 2 ? 1 : 2);
        if (d == 2) return {{bit_field(0, g.ll, ys), bit_field(g.ll, g.lp, lo), {}, {}}};
        return {{bit_field(0, g.ll, ys), bit_field(g.ll, g.ll, es), bit_field(2 * g.ll, g.lp, lo),
                 bit_field(2 * g.ll + g.lp, g.lp, hi)}};
    }
    // rows: the lines of a pass on its reciprocal (or packed) side
    BitMap<4> row_lines(int axis, bool tiled) const {
        const bool swapped = axis == 2 || (axis == 1 && tiled && d == 3);
        return swapped ? lines(axis, 2 * g.ll, g.ll) : lines(axis, g.ll, 2 * g.ll);
    }
    // reciprocal row: k = k1 + VEC k2 -> k1 % VP + k2 VP of member k1 / VP
    BitMap<3> row(int axis) const {
        return {{bit_field(0, lvp, 0), bit_field(lvp, g.lp, member(axis)), bit_field(g.lvec, lm, lvp)}};
    }
    // memory-order element of the P rank rows of a packed line, and its sample n
    BitMap<3> packed(int axis) const { return {{bit_field(0, g.ll, 0), bit_field(g.ll, g.lp, member(axis)), {}}}; }
    BitMap<3> packed_to_n() const {
        return {{bit_field(0, g.lvec, lm), bit_field(g.lvec, g.lb, 0), bit_field(g.ll, g.lp, g.lb)}};
    }
    // tile (before the repack): sample n = jj M + gm B + j in local index
    // jj B + j of member gm, L elements apart
    BitMap<4> tile_lines(int axis) const { return lines(axis, 0, 2 * g.ll); }
    BitMap<3> tile(int axis) const {
        return {{bit_field(0, g.lb, g.ll), bit_field(g.lb, g.lp, member(axis)), bit_field(lm, g.lvec, g.lb + g.ll)}};
    }
    // frequency of an axis off the last one, by lambda: its rank coordinate is
    // at bit `rank`, its local (reciprocal) index at bit `local`
    BitMap<3> frequency(int local, int rank) const {
        return {{bit_field(local, lvp, 0), bit_field(local + lvp, g.ll - lvp, g.lvec), bit_field(rank, g.lp, lvp)}};
    }
    // frequencies of axis 0 and (3D) axis 1 of the last axis's lines: the rows
    // of the y pass are kx; the rows of the z pass are kc (e) and kr (y)
    BitMap<3> frequency0() const { return d == 2 ? frequency(0, g.ll) : frequency(g.ll, 2 * g.ll); }
    BitMap<3> frequency1() const { return d == 2 ? BitMap<3>{} : frequency(0, 2 * g.ll + g.lp); }
    // global row plane N + row of an x pass -> row base
    BitMap<6> global_rows() const {
        BitMap<6> m{};
        for (int axis = 1; axis < d; axis++) {
            const int at = (axis - 1) * g.ln, local = axis * g.ll;
            m.f[3 * axis - 3] = bit_field(at, g.lb, local);
            m.f[3 * axis - 2] = bit_field(at + g.lb, g.lp, member(axis));
            m.f[3 * axis - 1] = bit_field(at + lm, g.lvec, local + g.lb);
        }
        return m;
    }
    // both ends of pass `kind` along `axis`
    void ends(LinePass kind, int axis, bool tiled, LinePassArgs* a) const {
        const BitMap<4> rl = row_lines(axis, tiled), tl = tile_lines(axis);
        const BitMap<3> rn = row(axis), tn = tile(axis), pn = packed(axis);
        const bool tin = kind == LP_TILE_FWD || kind == LP_TILE_SPEC, tout = kind == LP_TILE_INV || kind == LP_TILE_SPEC;
        const bool lap = kind == LP_ROW_LAP2 || kind == LP_ROW_LAP3;
        const bool pin = kind == LP_ROW_FWD || kind == LP_ROW_SPEC || lap, pout = kind == LP_ROW_INV || kind == LP_ROW_SPEC;
        a->in_l = tin ? tl : rl;
        a->in_n = tin ? tn : pin ? pn : rn;
        a->out_l = tout ? tl : rl;
        a->out_n = tout ? tn : pout ? pn : rn;
        a->pk = packed_to_n();
        if (lap) a->rows = global_rows();
    }
};

// natural <-> packed conversion in tiles of 2^ltile elements (spectral.hip)
struct ConvertArgs {
    BitMap<6> nat;    // q -> natural index
    BitMap<13> pk;    // q -> packed index
    BitMap<3> order;  // tile element in the packed side's order (jj, r, rows) -> q
    int ltile, lfield;
};

// log2 of the elements of a converter tile (spectral.hip): 8 KB
template <typename T>
constexpr int kConvertTile = sizeof(T) == 8 ? 9 : 10;

inline ConvertArgs convert_args(const Geo& g, int le) {
    ConvertArgs a{};
    const int d = g.dims, lm = g.lb + g.lp, slab = d * g.ll;
    a.lfield = d * g.ln;
    a.ltile = le < a.lfield ? le : a.lfield;
    // bits of the tile: r and jj whole with rows above where they fit, else
    // about half of the tile each
    int lr = lm, lj = g.lvec;
    while (lr + lj > a.ltile) {
        if (lr > lj) lr--;
        else lj--;
    }
    const int lrow = a.ltile - lr - lj, nrow = (d - 1) * g.ln;
    a.order = {{bit_field(0, lj, lr), bit_field(lj, lr, 0), bit_field(lj + lr, lrow, lj + lr)}};
    // q from its lowest bit: the tile's r, jj, rows, then the rest of each
    int q = 0, fn = 0, fp = 0;
    auto nat = [&](int nbits, int to) { a.nat.f[fn++] = bit_field(q, nbits, to); };
    // bits [lo, hi) of a quantity whose bits [from, to) sit at `at` + from ..
    auto packed = [&](int lo, int hi, int from, int to, int at) {
        const int l = lo > from ? lo : from, h = hi < to ? hi : to;
        if (l < h) a.pk.f[fp++] = bit_field(q + l - lo, h - l, at + l - from);
    };
    auto put_r = [&](int lo, int hi) {  // gm B + j -> j VEC, member rank gm
        nat(hi - lo, lo);
        packed(lo, hi, 0, g.lb, g.lvec);
        packed(lo, hi, g.lb, lm, slab);
        q += hi - lo;
    };
    auto put_j = [&](int lo, int hi) {
        nat(hi - lo, lm + lo);
        packed(lo, hi, 0, g.lvec, 0);
        q += hi - lo;
    };
    auto put_rows = [&](int lo, int hi) {  // (row in block, rank, block) of rows, then planes
        nat(hi - lo, g.ln + lo);
        for (int axis = 1; axis < d; axis++) {
            const int at = (axis - 1) * g.ln, local = axis * g.ll;
            packed(lo, hi, at, at + g.lb, local);
            packed(lo, hi, at + g.lb, at + lm, slab + axis * g.lp);
            packed(lo, hi, at + lm, at + g.ln, local + g.lb);
        }
        q += hi - lo;
    };
    put_r(0, lr), put_j(0, lj), put_rows(0, lrow);
    put_r(lr, lm), put_j(lj, g.lvec), put_rows(lrow, nrow);
    return a;
}

}  // namespace zm
