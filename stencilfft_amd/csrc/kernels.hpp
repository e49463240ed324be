// kernels.hpp -- launch interface between the host plan (plan.cpp) and the
// gfx950 kernels (fft.hip, stencil.hip, spectral.hip).
#pragma once

#include <hip/hip_runtime.h>

#include "common.hpp"

namespace zm {

// fused line kernel: lines of one exchange axis
struct LineArgs {
    int sg;               // world-rank stride between members of the exchange group
    int lines_per_group;  // L^(dims-1) local rows per rank
    int lpb;              // lines per workgroup
};

// two-stage kernels: rank rows
struct StageArgs {
    int sg;             // world-rank stride between members of the exchange group
    int rows_per_rank;  // L^(dims-1)
    int rpb;            // rows per workgroup
    int ndep;           // depth slices of a slot (1 in 2D, L in 3D)
};

constexpr int REPACK_TX = 32;
constexpr int REPACK_TY = 32;

struct RepackArgs {
    int64_t ei, eo;  // stride of the untouched index on the x/y side and on the packed side
    int64_t sxi;     // stride of x on the x/y side (y has stride 1)
    int64_t syo;     // stride of y on the packed side (pack(x) has stride 1)
    int ecount;      // extent of the untouched index
    int tx, ty;      // tile extents (<= REPACK_TX, REPACK_TY)
};

template <typename T>
hipError_t launch_line(const Cx<T>* in, Cx<T>* out, const Geo& g, const LineArgs& a, const Cx<T>* tw, int batch,
                       bool fwd, bool compute, double scale, hipStream_t stream);
template <typename T>
hipError_t launch_stage_a(const Cx<T>* in, Cx<T>* out, const Geo& g, const StageArgs& a, const Cx<T>* tw, int batch,
                          bool fwd, bool compute, double scale, hipStream_t stream);
template <typename T>
hipError_t launch_stage_b(const Cx<T>* in, Cx<T>* out, const Geo& g, const StageArgs& a, const Cx<T>* tw, int batch,
                          bool fwd, bool compute, hipStream_t stream);
template <typename T>
hipError_t launch_repack(const Cx<T>* in, Cx<T>* out, const Geo& g, const RepackArgs& a, int batch, bool fwd,
                         hipStream_t stream);

// compile-time specialised fused line pass (line_fast.hip)
template <typename T>
bool fast_line_supported(int vec, int m);
template <typename T>
int fast_line_occupancy(int vec, int m, bool fwd, bool mf, bool lapx);
// whether the plain passes of both directions are built for this (VEC, M) pair
// (beside the fused Laplacian, below, the forward one is)
template <typename T>
bool fast_line_plain(int vec, int m, bool mf);
// whether the fused Laplacian + x pass (lapx) exists for this (VEC, M) pair
// in `dims` dimensions with block size `b`
template <typename T>
bool fast_line_lapx(int vec, int m, bool mf, int dims, int b);
// log2 of the lines per group of the specialised pass for N = vec * m
int fast_line_lapx_lines_log2(int vec, int m);
// mf: radix-16 passes as split-precision FP16 MFMA GEMMs (FP32 only).
// lapx (forward x pass, fast_line_lapx): transform `scale` times the 5-point
// (2D) / 7-point (3D) Laplacian of the input (the fused Laplacian + forward
// transform).  3D: grid_x = (N / lines per group) row tiles times the number
// of plane chunks, which must divide N.
template <typename T>
hipError_t launch_line_fast(const Cx<T>* in, Cx<T>* out, const Geo& g, const LineArgs& a, const Cx<T>* tables,
                            int batch, bool fwd, double scale, int grid_x, bool mf, bool lapx, hipStream_t stream);
// entries of the specialised pass's table
int line_table_entries(int vec, int m);

// A bit permutation v -> sum over fields of ((v >> from) & mask) << to.
struct BitField {
    int from, mask, to;
};
template <int K>
struct BitMap {
    BitField f[K];
};
inline BitField bit_field(int from, int nbits, int to) { return BitField{from, (1 << nbits) - 1, to}; }
template <int K>
__device__ __forceinline__ int bits(const BitMap<K>& m, int v) {
    int r = 0;
#pragma unroll
    for (int i = 0; i < K; i++) r += ((v >> m.f[i].from) & m.f[i].mask) << m.f[i].to;
    return r;
}

// Line passes over natural-order lines (line_pass.hpp).  A line has an index
// lambda in [0, N^(d-1)); a workgroup takes 2^lines of consecutive ones.  Each
// end of the pass places element n of line lambda at bits(l, lambda) +
// bits(n, n) of the field; a packed end maps the memory-order element e of a
// line's rank rows there instead, and `pk` maps e to its sample n.
struct LinePassArgs {
    BitMap<4> in_l, out_l;
    BitMap<3> in_n, out_n, pk;
    BitMap<6> rows;  // Laplacian passes: global row (plane N + row) -> row base, for both ends
    int lgroups;    // log2 of the line groups per field
    int groups;     // line groups of the whole batch
    int xcd;        // consecutive groups on one XCD
    int64_t field;  // elements per field
};

// A spectral multiplier between the two transforms of a pass: f0, f1 map
// lambda to the frequencies of the other axes (axis 0 first; f1 in 3D only).
struct SpectralArgs {
    int kind, conj, dims;
    double p0, p1, kscale;
    BitMap<3> f0, f1;
    const double* half_sin;  // sin(pi s / N), s the signed wavenumber of f < N
    const double* factor;    // device value times the multiplier (null: 1)
};

// kinds of line pass: the two ends and the direction
enum LinePass {
    LP_ROW_FWD = 0,    // packed -> row
    LP_ROW_INV = 1,    // row -> packed
    LP_TILE_FWD = 2,   // tile -> row
    LP_TILE_INV = 3,   // row -> tile
    LP_TILE_SPEC = 4,  // tile -> multiplier -> tile
    LP_ROW_SPEC = 5,   // packed -> multiplier -> packed
    LP_ROW_LAP2 = 6,   // 5-point Laplacian of packed -> row
    LP_ROW_LAP3 = 7    // 7-point Laplacian of packed -> row
};
// the radix passes of a line and the size of their twiddle table: for each pass
// p >= 1 of radix R after NS = the product of the radices before it, W_{NS R}^(jm r)
// at r NS + jm, one pass after the other
struct LineRadices {
    int np, entries;
    int lr[7];  // log2 of the radices
};
struct LinePassInfo {
    int lines_log2;  // log2 of the lines per workgroup; -1: not built
    bool loop;       // workgroups loop over groups (else one group each)
    LineRadices radices;
};
// Lines of 2^ln points; small: the variant for fields with few line groups;
// radix16: the split with the largest radices, where it differs.
struct LinePassSize {
    int ln;
    bool small, radix16;
};
template <typename T>
LinePassInfo line_pass_info(LinePass kind, const LinePassSize& size);
// workgroups per CU (0: the query failed), the grid of the looping passes
template <typename T>
int line_pass_occupancy(LinePass kind, const LinePassSize& size);
template <typename T>
hipError_t launch_line_pass(LinePass kind, const LinePassSize& size, const Cx<T>* in, Cx<T>* out, const LinePassArgs& a,
                            const Cx<T>* tables, double scale, const SpectralArgs& sp, int grid, hipStream_t stream);

// stencils: E = element type (T or Cx<T>)
enum StencilOp { OP_LAPLACE = 0, OP_DX4 = 1, OP_DY4 = 2, OP_DZ4 = 3 };
template <typename T>
hipError_t launch_stencil(const void* in, void* out, const Geo& g, int batch, StencilOp op, bool complex_elems,
                          double coef, bool negate, hipStream_t stream);

// out += alpha * coef * Laplacian(in)
template <typename T>
hipError_t launch_laplace_add(const Cx<T>* in, Cx<T>* out, const Geo& g, int batch, double coef, double alpha,
                              hipStream_t stream);

// The tables of a plan, computed in FP64 and rounded to its precision; null: not
// wanted.
template <typename T>
struct PlanTables {
    int n;
    Cx<T>* tw;                // exp(-2 pi i t / n), t < n
    Cx<T>* line;              // the specialised pass's (line_fast.hip), of `line_entries`
    int line_entries, line_s;
    Cx<T>* nat[2];            // the row and the tile passes' (line_pass.hpp)
    LineRadices radices[2];
    double* half_sin;         // sin(pi s / n), s the signed wavenumber of f < n
};
template <typename T>
hipError_t launch_plan_tables(const PlanTables<T>& t, hipStream_t stream);

// r -= g over n elements; *norm2 = sum |r|^2 (FP64 partial sums in `partials`)
constexpr int kNormBlocks = 2048;
template <typename T>
hipError_t launch_residual_norm(Cx<T>* r, const Cx<T>* g, int64_t n, double* partials, T* norm2, hipStream_t stream);

// reciprocal-space multiplier
template <typename T>
hipError_t launch_spectral(const Cx<T>* in, Cx<T>* out, const Geo& g, int batch, int kind, double p0, double p1,
                           double kscale, bool conj, const double* factor, hipStream_t stream);

// index tables and natural <-> packed conversion
hipError_t launch_index_table(int64_t* out, const Geo& g, bool reciprocal, hipStream_t stream);
template <typename T>
hipError_t launch_natural_packed(const Cx<T>* in, Cx<T>* out, const Geo& g, int batch, bool to_packed,
                                 hipStream_t stream);

}  // namespace zm
