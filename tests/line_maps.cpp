// Checks the address maps of the line passes (csrc/line_maps.hpp) against the
// layout algebra (csrc/maps.hpp), over every valid (N, P, B) up to a size:
// each end of each pass is a permutation of the field, the packed and tile ends
// hold sample n of the line where the real-space maps put it, the row end holds
// frequency k where the reciprocal maps do, the passes chain (what one writes as
// rows the next reads as tiles), and a multiplier's maps give the lines'
// frequencies.  The converters' maps are checked the same way.  Prints the
// number of shapes.
#include <cstdio>
#include <vector>

#include "../stencilfft_amd/csrc/line_maps.hpp"
#include "../stencilfft_amd/csrc/maps.hpp"

using namespace zm;

static int lg(int x) {
    int r = 0;
    while ((1 << r) < x) r++;
    return r;
}

template <int K>
static int at(const BitMap<K>& m, int v) {
    int r = 0;
    for (int i = 0; i < K; i++) r += ((v >> m.f[i].from) & m.f[i].mask) << m.f[i].to;
    return r;
}

static bool fail(const char* what, int d, int n, int p, int b, int axis) {
    std::printf("%s: dims %d N %d P %d B %d axis %d\n", what, d, n, p, b, axis);
    return false;
}

// A slab element of the layout an axis pass finds: rank coordinates (did, rid,
// cid) and local (depth, row, col).
struct Where {
    int did, rid, cid, ld, lr, lc;
};
static int addr(const Geo& g, const Where& w) {
    const int id = (w.did * g.p + w.rid) * g.p + w.cid;
    return id * (int)g.local + (w.ld * g.l + w.lr) * g.l + w.lc;
}

static bool check(int d, int n, int p, int b) {
    Geo g{};
    g.dims = d, g.n = n, g.p = p, g.b = b, g.l = n / p, g.vec = g.l / b, g.vp = g.vec / p, g.m = b * p;
    g.ln = lg(n), g.lp = lg(p), g.lb = lg(b), g.ll = lg(g.l), g.lvec = lg(g.vec);
    g.local = d == 3 ? g.l * g.l * g.l : g.l * g.l;
    g.field = d == 3 ? n * n * n : n * n;
    const MapShape ms = make_map_shape(n, p, b);
    const NatMaps m(g);
    const int lines = d == 3 ? n * n : n, L = g.l;
    // frequencies of the other axes for the last axis's lines
    for (int lam = 0; lam < lines; lam++) {
        const int y = lam & (L - 1), e = (lam >> g.ll) & (L - 1);
        const int o = lam >> ((d - 1) * g.ll), cid = o & (p - 1), rid = o >> g.lp;
        if (at(m.frequency0(), lam) != recip_to_freq(ms, cid, d == 2 ? y : e)) return fail("frequency 0", d, n, p, b, d - 1);
        if (d == 3 && at(m.frequency1(), lam) != recip_to_freq(ms, rid, y)) return fail("frequency 1", d, n, p, b, 2);
    }
    // global rows of the Laplacian pass
    for (int gl = 0; gl < lines; gl++) {
        Where w{};
        global_row_to_local(ms, gl % n, &w.rid, &w.lr);
        global_row_to_local(ms, gl / n, &w.did, &w.ld);
        if (d == 2) w.did = w.ld = 0;
        if (at(m.global_rows(), gl) != addr(g, w)) return fail("global rows", d, n, p, b, 0);
    }
    for (int tiled = 0; tiled < 2; tiled++)
        for (int axis = 0; axis < d; axis++)
            for (int kind = LP_ROW_FWD; kind <= LP_ROW_SPEC; kind++) {
                const bool tile_kind = kind >= LP_TILE_FWD && kind <= LP_TILE_SPEC;
                if (tile_kind && (!tiled || axis == 0)) continue;
                if (!tile_kind && tiled && axis > 0) continue;
                LinePassArgs a{};
                m.ends((LinePass)kind, axis, tiled, &a);
                std::vector<char> in(g.field), out(g.field);
                for (int lam = 0; lam < lines; lam++) {
                    // the line's coordinates: y, e, and the ranks off the axis
                    const int y = lam & (L - 1), e = d == 3 ? (lam >> g.ll) & (L - 1) : 0;
                    const int o = lam >> ((d - 1) * g.ll), o0 = o & (p - 1), o1 = o >> g.lp;
                    for (int i = 0; i < n; i++) {
                        const int ai = at(a.in_l, lam) + at(a.in_n, i), ao = at(a.out_l, lam) + at(a.out_n, i);
                        if (ai < 0 || ai >= g.field || in[ai]++) return fail("input end", d, n, p, b, axis);
                        if (ao < 0 || ao >= g.field || out[ao]++) return fail("output end", d, n, p, b, axis);
                        // ranks: the axis's own coordinate r, the others from o
                        auto ranks = [&](int r, Where* w) {
                            w->cid = axis == 0 ? r : o0;
                            w->rid = axis == 1 ? r : axis == 0 ? o0 : o1;
                            w->did = axis == 2 ? r : d == 3 ? o1 : 0;
                        };
                        // rows of a line after (before) its transform: 2D [y]; 3D
                        // x and untiled y [e][y], tiled y and z [y][e]
                        auto row = [&](int pos, Where* w) {
                            const bool swapped = d == 3 && (axis == 2 || (axis == 1 && tiled));
                            w->lc = pos;
                            w->lr = swapped ? e : y;
                            w->ld = d == 3 ? (swapped ? y : e) : 0;
                        };
                        auto is_row = [&](int addr_) {  // frequency i
                            int r, pos;
                            freq_to_recip(ms, i, &r, &pos);
                            Where w;
                            ranks(r, &w), row(pos, &w);
                            return addr(g, w) == addr_;
                        };
                        auto is_tile = [&](int addr_) {  // sample i, slabs [e][sample][y]
                            int r, li;
                            global_row_to_local(ms, i, &r, &li);
                            Where w;
                            ranks(r, &w);
                            w.lc = y, w.lr = li, w.ld = e;
                            return addr(g, w) == addr_;
                        };
                        auto is_packed = [&](int addr_) {  // memory order, sample pk(i)
                            int r, lc;
                            global_col_to_local(ms, at(a.pk, i), &r, &lc);
                            Where w;
                            ranks(r, &w), row(lc, &w);
                            return addr(g, w) == addr_;
                        };
                        const bool tin = kind == LP_TILE_FWD || kind == LP_TILE_SPEC;
                        const bool tout = kind == LP_TILE_INV || kind == LP_TILE_SPEC;
                        const bool pin = kind == LP_ROW_FWD || kind == LP_ROW_SPEC;
                        const bool pout = kind == LP_ROW_INV || kind == LP_ROW_SPEC;
                        if (!(tin ? is_tile(ai) : pin ? is_packed(ai) : is_row(ai)))
                            return fail("input layout", d, n, p, b, axis);
                        if (!(tout ? is_tile(ao) : pout ? is_packed(ao) : is_row(ao)))
                            return fail("output layout", d, n, p, b, axis);
                    }
                }
            }
    // converters: tiles of several sizes, larger than the field among them
    for (int le : {8, 11, 12}) {
        const ConvertArgs a = convert_args(g, le);
        std::vector<char> seen(g.field);
        for (int q = 0; q < g.field; q++) {
            const int nat = at(a.nat, q), pk = at(a.pk, q);
            if (nat < 0 || nat >= g.field || seen[nat]++) return fail("natural side", d, n, p, b, 0);
            const int gc = nat % n, gr = nat / n % n, gd = nat / n / n;
            Where w{};
            global_col_to_local(ms, gc, &w.cid, &w.lc);
            global_row_to_local(ms, gr, &w.rid, &w.lr);
            if (d == 3) global_row_to_local(ms, gd, &w.did, &w.ld);
            if (addr(g, w) != pk) return fail("packed side", d, n, p, b, 0);
        }
        std::vector<char> slot(1 << a.ltile);
        for (int e = 0; e < 1 << a.ltile; e++) {
            const int s = at(a.order, e);
            if (s < 0 || s >= 1 << a.ltile || slot[s]++) return fail("tile order", d, n, p, b, 0);
        }
    }
    return true;
}

int main() {
    int shapes = 0;
    for (int d = 2; d <= 3; d++)
        for (int n = 16; n <= (d == 2 ? 256 : 32); n *= 2)
            for (int p = 1; p * p <= n; p *= 2)
                for (int b = 1; p * p * b <= n; b *= 2, shapes++)
                    if (!check(d, n, p, b)) return 1;
    std::printf("%d shapes\n", shapes);
    return 0;
}
