// The address maps as the library launches them, beside those of line_maps.cpp:
// the converters with the tile size of their kernel, and the ends of the
// Laplacian row passes (packed input, row output, lines as global rows), against
// the layout algebra (csrc/maps.hpp).  Prints the number of shapes.
#include <cstdio>
#include <vector>

#include "../stencilfft_amd/csrc/line_maps.hpp"
#include "../stencilfft_amd/csrc/maps.hpp"

using namespace zm;

template <int K>
static int at(const BitMap<K>& m, int v) {
    int r = 0;
    for (int i = 0; i < K; i++) r += ((v >> m.f[i].from) & m.f[i].mask) << m.f[i].to;
    return r;
}

static int lg(int x) {
    int r = 0;
    while ((1 << r) < x) r++;
    return r;
}

static bool fail(const char* what, const Geo& g) {
    std::printf("%s: dims %d N %d P %d B %d\n", what, g.dims, g.n, g.p, g.b);
    return false;
}

// real-space index of global (plane, row, column)
static int real_index(const Geo& g, const MapShape& ms, int gd, int gr, int gc) {
    int cid, rid, did = 0, lc, lr, ld = 0;
    global_col_to_local(ms, gc, &cid, &lc);
    global_row_to_local(ms, gr, &rid, &lr);
    if (g.dims == 3) global_row_to_local(ms, gd, &did, &ld);
    return ((did * g.p + rid) * g.p + cid) * (int)g.local + (ld * g.l + lr) * g.l + lc;
}

static bool check(int d, int n, int p, int b) {
    Geo g{};
    g.dims = d, g.n = n, g.p = p, g.b = b, g.l = n / p, g.vec = g.l / b, g.vp = g.vec / p, g.m = b * p;
    g.ln = lg(n), g.lp = lg(p), g.lb = lg(b), g.ll = lg(g.l), g.lvec = lg(g.vec);
    g.local = d == 3 ? g.l * g.l * g.l : g.l * g.l;
    g.field = d == 3 ? n * n * n : n * n;
    const MapShape ms = make_map_shape(n, p, b);

    // converters: every element, each tile a permutation of its slots, and the
    // element in slot order where the tile's own bits say (kernel: bits(order,
    // slot), then the packed map of it)
    for (int le : {kConvertTile<float>, kConvertTile<double>}) {
        const ConvertArgs a = convert_args(g, le);
        std::vector<char> seen(g.field);
        for (int q = 0; q < g.field; q++) {
            const int nat = at(a.nat, q);
            if (nat < 0 || nat >= g.field || seen[nat]++) return fail("natural side", g);
            if (real_index(g, ms, nat / n / n, nat / n % n, nat % n) != at(a.pk, q)) return fail("packed side", g);
        }
        const int tile = 1 << a.ltile;
        if (a.ltile != (le < a.lfield ? le : a.lfield)) return fail("tile size", g);
        for (int base = 0; base < g.field; base += tile) {
            std::vector<char> slot(tile);
            for (int e = 0; e < tile; e++) {
                const int s = at(a.order, e);
                if (s < 0 || s >= tile || slot[s]++) return fail("tile order", g);
                if (at(a.pk, base) + at(a.pk, s) != at(a.pk, base + s)) return fail("tile base", g);
                if (at(a.nat, base) + at(a.nat, e) != at(a.nat, base + e)) return fail("tile base", g);
            }
        }
    }

    // Laplacian passes: line = global row (plane N + row)
    const NatMaps m(g);
    LinePassArgs lp{}, fwd{};
    m.ends(d == 2 ? LP_ROW_LAP2 : LP_ROW_LAP3, 0, true, &lp);
    m.ends(LP_ROW_FWD, 0, true, &fwd);
    const int lines = d == 3 ? n * n : n;
    std::vector<char> in(g.field), out(g.field);
    for (int gl = 0; gl < lines; gl++)
        for (int e = 0; e < n; e++) {
            // memory-order element e is sample pk(e) of the row
            const int ai = at(lp.rows, gl) + at(lp.in_n, e), ao = at(lp.rows, gl) + at(lp.out_n, e);
            if (ai < 0 || ai >= g.field || in[ai]++) return fail("Laplacian input", g);
            if (ao < 0 || ao >= g.field || out[ao]++) return fail("Laplacian output", g);
            if (ai != real_index(g, ms, gl / n, gl % n, at(lp.pk, e))) return fail("Laplacian sample", g);
            // frequency e of the line: rank column and position of the
            // reciprocal map, in the local row that the line was read from
            int cid, pos, rc, lc;
            freq_to_recip(ms, e, &cid, &pos);
            global_col_to_local(ms, 0, &rc, &lc);
            const int row0 = real_index(g, ms, gl / n, gl % n, 0) - rc * (int)g.local - lc;
            if (ao != row0 + cid * (int)g.local + pos) return fail("Laplacian frequency", g);
        }
    // the lines are those of the plain x pass in another order, on both ends
    std::vector<char> base(g.field);
    for (int lam = 0; lam < lines; lam++) base[at(fwd.in_l, lam)] |= 1, base[at(fwd.out_l, lam)] |= 2;
    for (int gl = 0; gl < lines; gl++)
        if (base[at(lp.rows, gl)] != 3) return fail("Laplacian lines", g);
    for (int e = 0; e < n; e++)
        if (at(lp.in_n, e) != at(fwd.in_n, e) || at(lp.out_n, e) != at(fwd.out_n, e)) return fail("Laplacian ends", g);
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
