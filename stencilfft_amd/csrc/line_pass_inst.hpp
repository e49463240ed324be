// line_pass_inst.hpp -- instances and dispatch of the natural-order line
// passes for one storage precision; included by line_pass_f32.hip and
// line_pass_f64.hip, which compile in parallel.
#pragma once

#include "line_pass.hpp"

namespace zm {
namespace lp {

constexpr size_t kLdsLimit = 160 * 1024;

// Row and tile passes of 2^LN-point lines: log2 of the elements per thread and
// of the lines per workgroup (and of the lines in the small variant), mode;
// -1 lines: not built.  RADIX16: the alternative split of a plan that prefers
// the largest radices (LinePassSize::radix16).
//
// Elements per thread: 8, whose radices of 8 need the fewest registers per value
// in flight, up to the N where a line would then take a fourth radix pass or more
// than 1024 threads; fewer for lines of 16 points, 32 where a 2048-point tile of
// eight lines needs them.
// Lines per workgroup, against half and twice as many (512 MB of fields, P = 2 and
// 8, forward and inverse, time over the table's):
//   rows   half 0.95-1.10, mostly 1.00; twice 0.98-1.07, at N = 512 FP64 1.07-1.12:
//          about 1024 to 4096 elements, several workgroups per CU.
//   tiles  half FP32 1.0-1.4 (runs of 64 bytes instead of 128), FP64 1.0-1.3 and at
//          N = 2048 both 1.3-2.3 (runs of 32); twice 0.90-1.03 up to N = 256 and
//          1.03-1.12 at N = 512, where it leaves a CU one workgroup, and beyond
//          that LDS is full.
// Mode, the other one: ONCE for N <= 512 (LOOP 1.03-1.27, N = 512 0.98-1.21), LOOP
// where the tile leaves a CU one workgroup, N >= 1024 (ONCE in FP32 1.00-1.12, FP64
// 0.98-1.02).  Rows loop at N = 2048 FP64 only: one field forward 55-59 us against
// 59-63, eight 443-478 against 433-465.
template <typename T, int LN, bool RADIX16>
struct Split {
    static constexpr int row_ept = 4, row = -1, row_small = -1, tile_ept = 4, tile = -1, tile_small = -1;
    static constexpr Mode row_mode = ONCE, tile_mode = ONCE;
};
#define ZM_SPLIT(T, LN, R16, RE, RL, RS, RM, TE, TL, TS, TM)                   \
    template <>                                                                \
    struct Split<T, LN, R16> {                                                 \
        static constexpr int row_ept = RE, row = RL, row_small = RS;           \
        static constexpr Mode row_mode = RM;                                   \
        static constexpr int tile_ept = TE, tile = TL, tile_small = TS;        \
        static constexpr Mode tile_mode = TM;                                  \
    };

constexpr bool is_lap(int kind) { return kind == LP_ROW_LAP2 || kind == LP_ROW_LAP3; }
constexpr bool is_row(int kind) {
    return kind == LP_ROW_FWD || kind == LP_ROW_INV || kind == LP_ROW_SPEC || is_lap(kind);
}

// the same radix passes, and so the same twiddle table
constexpr bool same_radices(const LineRadices& a, const LineRadices& b) {
    if (a.np != b.np || a.entries != b.entries) return false;
    for (int p = 0; p < a.np; p++)
        if (a.lr[p] != b.lr[p]) return false;
    return true;
}

template <typename T, int LN, bool R16, int KIND, bool SMALL>
struct Inst {
    using S = Split<T, LN, R16>;
    static constexpr bool ROWS = is_row(KIND);
    static constexpr int LNP = LN, LLP = ROWS ? (SMALL ? S::row_small : S::row) : (SMALL ? S::tile_small : S::tile);
    // multiplier tiles with at most 512 threads (256 VGPRs), on the tile passes'
    // tables
    static constexpr int LEPT0 = ROWS ? S::row_ept : S::tile_ept;
    static constexpr int LEPT = KIND == LP_TILE_SPEC && LN + LLP - LEPT0 > 9 ? LN + LLP - 9 : LEPT0;
    // row multipliers only where no tile is built (FP64 N = 8192 spills)
    static constexpr bool built =
        LLP >= 0 && (KIND != LP_ROW_SPEC || (S::tile < 0 && !(sizeof(T) == 8 && LN == 13))) &&
        (!is_lap(KIND) || LN <= (KIND == LP_ROW_LAP2 ? 11 : 10)) &&
        // five rows of 16 FP64 values per thread spill
        !(KIND == LP_ROW_LAP3 && sizeof(T) == 8 && LEPT > 3);
    static constexpr int DIR = KIND == LP_TILE_SPEC || KIND == LP_ROW_SPEC ? SPEC
                               : KIND == LP_ROW_INV || KIND == LP_TILE_INV ? INV
                                                                           : FWD;
    static constexpr Mode MODE = SMALL || DIR == SPEC || is_lap(KIND) ? ONCE : ROWS ? S::row_mode : S::tile_mode;
    static constexpr int IN = KIND == LP_ROW_LAP2                          ? LAP2
                              : KIND == LP_ROW_LAP3                         ? LAP3
                              : KIND == LP_ROW_FWD || KIND == LP_ROW_SPEC   ? PACKED
                              : KIND == LP_ROW_INV || KIND == LP_TILE_INV ? ROW
                                                                          : TILE;
    static constexpr int OUT = KIND == LP_ROW_INV || KIND == LP_ROW_SPEC    ? PACKED
                               : KIND == LP_ROW_FWD || KIND == LP_TILE_FWD || is_lap(KIND) ? ROW
                                                                           : TILE;
    using K = Line<T, LN, LLP < 0 ? 4 : LLP, LEPT>;
    static_assert(!built || same_radices(Radices<LN, LEPT>::list(), Radices<LN, LEPT0>::list()), "the table of the row or tile passes");
    static constexpr size_t lds() {
        static_assert(K::lds_bytes() <= kLdsLimit, "LDS");
        return K::lds_bytes();
    }
    static const void* fn() { return (const void*)&line_pass_kernel<T, LN, LLP, LEPT, IN, OUT, DIR, MODE>; }
    static hipError_t prepare() {
        if (lds() <= 65536) return hipSuccess;
        return hipFuncSetAttribute(fn(), hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds());
    }
};

template <typename T, typename Op>
auto with_line_pass(int kind, const LinePassSize& size, Op&& op) {
#define ZM_LP3(LN, R16, KIND, SM)                                                 \
    if constexpr (Inst<T, LN, R16, KIND, SM>::built) {                            \
        if (size.ln == LN && size.radix16 == R16 && kind == KIND && size.small == SM) \
            return op.template run<Inst<T, LN, R16, KIND, SM>>();                 \
    }
#define ZM_LP2(LN, R16, KIND) ZM_LP3(LN, R16, KIND, false) ZM_LP3(LN, R16, KIND, true)
#define ZM_LP1(LN, KIND) ZM_LP2(LN, false, KIND) ZM_LP2(LN, true, KIND)
#define ZM_LP(LN)                                                                                 \
    ZM_LP1(LN, LP_ROW_FWD) ZM_LP1(LN, LP_ROW_INV) ZM_LP1(LN, LP_TILE_FWD) ZM_LP1(LN, LP_TILE_INV) \
    ZM_LP1(LN, LP_TILE_SPEC) ZM_LP1(LN, LP_ROW_SPEC) ZM_LP1(LN, LP_ROW_LAP2) ZM_LP1(LN, LP_ROW_LAP3)
    ZM_LP(4) ZM_LP(5) ZM_LP(6) ZM_LP(7) ZM_LP(8) ZM_LP(9) ZM_LP(10) ZM_LP(11) ZM_LP(12) ZM_LP(13)
#undef ZM_LP
#undef ZM_LP1
#undef ZM_LP2
#undef ZM_LP3
    return op.none();
}

struct InfoOp {
    template <typename I>
    LinePassInfo run() {
        return LinePassInfo{I::LLP, I::MODE != ONCE, I::K::list()};
    }
    LinePassInfo none() { return LinePassInfo{-1, false, {}}; }
};

struct OccupancyOp {
    template <typename I>
    int run() {
        int blocks = 0;
        if (I::prepare() != hipSuccess ||
            hipOccupancyMaxActiveBlocksPerMultiprocessor(&blocks, I::fn(), I::K::NT, I::lds()) != hipSuccess)
            return 0;
        return blocks;
    }
    int none() { return 0; }
};

template <typename T>
struct LaunchOp {
    const Cx<T>* in;
    Cx<T>* out;
    const LinePassArgs& a;
    const Cx<T>* tables;
    T scale;
    const SpectralArgs& sp;
    int grid;
    hipStream_t stream;
    template <typename I>
    hipError_t run() {
        const hipError_t e = I::prepare();
        if (e != hipSuccess) return e;
        hipLaunchKernelGGL((line_pass_kernel<T, I::LNP, I::LLP, I::LEPT, I::IN, I::OUT, I::DIR, I::MODE>),
                           dim3((unsigned)grid), dim3(I::K::NT), I::lds(), stream, in, out, a, tables, scale, sp);
        return hipGetLastError();
    }
    hipError_t none() { return hipErrorInvalidValue; }
};

}  // namespace lp

template <typename T>
LinePassInfo line_pass_info(LinePass kind, const LinePassSize& size) {
    return lp::with_line_pass<T>((int)kind, size, lp::InfoOp{});
}
template <typename T>
int line_pass_occupancy(LinePass kind, const LinePassSize& size) {
    return lp::with_line_pass<T>((int)kind, size, lp::OccupancyOp{});
}
template <typename T>
hipError_t launch_line_pass(LinePass kind, const LinePassSize& size, const Cx<T>* in, Cx<T>* out, const LinePassArgs& a,
                            const Cx<T>* tables, double scale, const SpectralArgs& sp, int grid, hipStream_t stream) {
    return lp::with_line_pass<T>((int)kind, size,
                                 lp::LaunchOp<T>{in, out, a, tables, (T)scale, sp, grid, stream});
}

}  // namespace zm
