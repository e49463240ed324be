// plan.hip -- host side of the C ABI declared in include/stencilfft.h: shape
// validation, plans (twiddle tables, kernel-path choice, scratch), the stage
// sequences of the forward / inverse transforms, stencils and index maps.
#include <hip/hip_runtime.h>

#include <cmath>
#include <cstdint>
#include <cstdlib>
#include <mutex>
#include <new>
#include <vector>

#include "../../include/stencilfft.h"
#include "kernels.hpp"
#include "line_maps.hpp"
#include "maps.hpp"

using zm::Geo;

struct zm_plan {
    zm_shape shape;
    zm_dims dims;
    zm_precision precision;
    int batch;
    unsigned flags;
    int device;
    Geo geo;
    // the plan's tables, one allocation holding in its precision what its passes
    // read: tw = exp(-2 pi i t / N), t < N; and those below
    void* tables;
    void* tw;
    bool two_stage;
    int lpb;  // lines per workgroup of the fused line kernel
    int rpb;  // rank rows per workgroup of the two-stage kernels
    void* own_scratch;
    size_t scratch_bytes;
    // compile-time specialised line pass (line_fast.hip): grids, 0 where the
    // plan does not use it
    bool fast;
    void* ltab;  // per-line twiddle tables (W_S, W_N two-level)
    int fast_grid_fwd, fast_grid_inv;
    int fast_grid_lapx;  // the fused Laplacian + x pass
    // natural-order line passes (line_pass.hpp) by axis; grid 0: not used
    struct NatPass {
        zm::LinePass kind;
        zm::LinePassSize size;
        int grid;
        const void* tables;
        zm::LinePassArgs args;
    };
    NatPass nat_fwd[3], nat_inv[3];
    NatPass nat_lap;       // the x pass of the Laplacian (grid 0: not used)
    NatPass nat_spec;      // the last axis forward, a spectral multiplier, and back
    bool tiled;            // the passes after the first axis hold the repacks
    void* nat_tables[2];  // twiddles of the row and of the tile passes
    double* half_sin;      // sin(pi s / N) by frequency
    // per-stage timing (zm_timing_*)
    bool timing;
    struct Timed {
        int stage;
        hipEvent_t start, stop;
        bool own_start;  // start is this entry's own event, not the previous launch's stop
        bool own_stop;   // false: a stage that ran inside the previous launch (start == stop, no time of its own)
    };
    std::vector<Timed> timed;
    hipEvent_t last_stop;  // completion event of the previous timed launch
    hipStream_t last_stream;
};

namespace {

// Runs `launch` (returning hipError_t) and, when the plan records per-stage
// timing, records one event after it on `stream`.  A launch's time is the
// interval from the previous timed launch's completion event on the same
// stream (or from an event recorded just before it, for the first launch on
// a stream) to its own: one event per launch, so back-to-back launches are
// timed without doubling the events in the queue.
template <typename F>
hipError_t timed_launch(zm_plan* p, int stage, hipStream_t stream, F&& launch, bool record = true) {
    if (!p->timing || !record) return launch();
    zm_plan::Timed t{stage, nullptr, nullptr, false, true};
    hipError_t e = hipSuccess;
    if (p->last_stop && p->last_stream == stream) {
        t.start = p->last_stop;
    } else {
        e = hipEventCreate(&t.start);
        if (e == hipSuccess) e = hipEventRecord(t.start, stream);
        t.own_start = true;
    }
    if (e == hipSuccess) e = hipEventCreate(&t.stop);
    if (e == hipSuccess) e = launch();
    if (e == hipSuccess) e = hipEventRecord(t.stop, stream);
    if (e == hipSuccess) {
        p->timed.push_back(t);
        p->last_stop = t.stop;
        p->last_stream = stream;
    } else {
        if (t.own_start && t.start) (void)hipEventDestroy(t.start);
        if (t.stop) (void)hipEventDestroy(t.stop);
    }
    return e;
}

// A stage that ran inside the launch just timed: counted, with no time of its
// own (the launch's stage holds it).
void timed_inside(zm_plan* p, int stage, bool record) {
    if (p->timing && record && p->last_stop)
        p->timed.push_back(zm_plan::Timed{stage, p->last_stop, p->last_stop, false, false});
}

void drop_timing(zm_plan* p) {
    for (auto& t : p->timed) {
        if (t.own_start) (void)hipEventDestroy(t.start);
        if (t.own_stop) (void)hipEventDestroy(t.stop);
    }
    p->timed.clear();
    p->last_stop = nullptr;
    p->last_stream = nullptr;
}

}  // namespace

// ---------------------------------------------------------------------------
// Scratch of zm_forward_noalloc: a file-scope device array, one copy on every
// GPU the library runs on, resident until the process ends.  In host code the
// name `scratch` is only a stand-in for the symbol, never a device address:
// zm_plan_create looks up the current device's copy once with
// hipGetSymbolAddress, and every use goes through that per-device address.
// ---------------------------------------------------------------------------
namespace noalloc {

static __device__ __align__(256) unsigned char scratch[ZM_NOALLOC_SCRATCH_BYTES];

constexpr int kMaxDevices = 64;
std::mutex mu;
bool looked_up[kMaxDevices];
void* addr[kMaxDevices];  // this device's copy of `scratch`, or null if the lookup failed

// Called by zm_plan_create with `device` current.
void resolve(int device) {
    if (device < 0 || device >= kMaxDevices) return;
    std::lock_guard<std::mutex> lock(mu);
    if (looked_up[device]) return;
    void* ptr = nullptr;
    if (hipGetSymbolAddress(&ptr, HIP_SYMBOL(scratch)) != hipSuccess) ptr = nullptr;
    addr[device] = ptr;
    looked_up[device] = true;
}

void* device_copy(int device) {
    if (device < 0 || device >= kMaxDevices) return nullptr;
    std::lock_guard<std::mutex> lock(mu);
    return looked_up[device] ? addr[device] : nullptr;
}

}  // namespace noalloc

namespace {

bool is_pow2(int x) { return x > 0 && (x & (x - 1)) == 0; }

int ilog2(int x) {
    int r = 0;
    while ((1 << r) < x) r++;
    return r;
}

zm::MapShape map_shape(const zm_shape* s) { return zm::make_map_shape(s->n, s->p, s->b); }

size_t elem_bytes(zm_precision p) { return p == ZM_FP64 ? sizeof(double2) : sizeof(float2); }

zm_status launch_status(hipError_t e) { return e == hipSuccess ? ZM_OK : ZM_ERR_LAUNCH; }

#define ZM_TRY(expr)                              \
    do {                                          \
        zm_status _st = (expr);                   \
        if (_st != ZM_OK) return _st;             \
    } while (0)

int ipow(int a, int e) {
    int r = 1;
    while (e-- > 0) r *= a;
    return r;
}

// Workgroup size targets (elements held in LDS per workgroup).
constexpr int kLineTarget = 4096;
constexpr int kStageTarget = 4096;
constexpr size_t kMaxLds = 160 * 1024;
static_assert(ZM_NORM_PARTIALS == zm::kNormBlocks, "partial sums of zm_residual_norm");

// FP64 lines of 256 points run as 16 x 16 on at most two ranks per axis, the
// radices of the VEC = M = 16 pass that these plans ran before, and as 8 x 8 x 4
// on more, where 16 x 16 stores runs of 16 / P values in its last pass: P = 4
// 0.357 against 0.300 ms, P = 8 0.820 against 0.290.
// On P <= 2 the choice keeps the rounding that the gradient check of the 256^3
// rollout was set for: the noise of its central difference (two losses' rounding
// over 2 eps) is 6.1e-7 with 16 x 16 and 1.00e-6, its bar, with 8 x 8 x 4.  It is
// neither closer nor faster.  Against long double, rel L2 of a 256^3 forward
// transform 3.4e-16 (8 x 8 x 4: 3.2e-16), of 32 heat steps 9.4e-15 (7.5e-15); one
// field at P = 2 forward 293 us (291), inverse 302 (281), heat step 629 (611), and
// Laplacian + forward 391 (325), as 16 values per thread leave no registers for
// the fused 3D Laplacian.
zm::LinePassSize nat_size(const Geo& g, bool fp64) {
    return zm::LinePassSize{g.ln, false, fp64 && g.ln == 8 && g.p <= 2};
}

// The pass `kind` along `axis`, or grid 0 where it is not built.
template <typename T>
zm_plan::NatPass nat_pass(const zm_plan* p, int cus, zm::LinePass kind, int axis) {
    const Geo& g = p->geo;
    const zm::NatMaps m(g);
    zm_plan::NatPass np{kind, nat_size(g, sizeof(T) == 8), 0, nullptr, {}};
    const int lines = g.ln * (g.dims - 1);  // log2 of the lines per field
    zm::LinePassInfo info = zm::line_pass_info<T>(kind, np.size);
    if (info.lines_log2 < 0) return np;
    // too few groups to fill the CUs: fewer lines per group
    if (((int64_t)p->batch << (lines - info.lines_log2)) < cus) {
        np.size.small = true;
        const zm::LinePassInfo si = zm::line_pass_info<T>(kind, np.size);
        if (si.lines_log2 >= 0) info = si;
        else np.size.small = false;
    }
    const int64_t groups = (int64_t)p->batch << (lines - info.lines_log2);
    if (groups > INT32_MAX) return np;
    int64_t grid = groups;
    if (info.loop) {
        const int64_t resident = (int64_t)zm::line_pass_occupancy<T>(kind, np.size) * cus;
        if (resident < groups) grid = resident;
    }
    if (grid <= 0) return np;
    np.grid = (int)grid;
    const bool rows = !(kind >= zm::LP_TILE_FWD && kind <= zm::LP_TILE_SPEC);
    np.tables = p->nat_tables[rows ? 0 : 1];
    zm::LinePassArgs& a = np.args;
    a.lgroups = lines - info.lines_log2;
    a.groups = (int)groups;
    // Consecutive groups on one XCD, where they share cache lines or rows:
    // * tile loads (shorter runs, DRAM pages): 512^3 FP32 y + z 0.83 -> 0.80
    //   ms, 2048^2 FP32 0.32 -> 0.25 ms; not stores (2048^2 FP64 0.223 -> 0.234
    //   ms) nor short lines (128^3 FP32 0.091 -> 0.107 ms);
    // * Laplacian rows in 2D (x pass + y pass, 2048^2 x8 FP32 0.277 -> 0.241
    //   ms) and in 3D while the fields stay in the last-level cache, whose
    //   planes the XCDs share otherwise (256^3 FP64 0.362 -> 0.318 ms; four of
    //   them 1.32 -> 1.49, 512^3 FP64 2.81 -> 3.21).
    const bool lap = kind == zm::LP_ROW_LAP2 || kind == zm::LP_ROW_LAP3;
    const double mib = (double)p->batch * (double)g.field * sizeof(zm::Cx<T>) / (1 << 20);
    a.xcd = (kind == zm::LP_TILE_FWD && g.ln >= 9) || (lap && (g.dims == 2 || mib <= 384.0));
    a.field = g.field;
    m.ends(kind, axis, p->tiled, &a);
    return np;
}

// At N >= 4096 the specialised pass (line_fast.hip) is as fast as a row pass or
// faster where it is built (forward + inverse: 4096^2 FP32 0.293 against 0.306
// ms, eight fields 2.43 against 2.32; 8192^2 FP32 line 0.20 against 0.22-0.23
// ms); elsewhere the generic one took 8192^2, P = 1, B = 32 4.54 against 1.46 ms.
bool row_passes_lose(const Geo& g, bool fast) { return g.ln >= 12 && fast; }

// The grids of the specialised line pass (line_fast.hip) in the directions that
// a plan runs it in: the MFMA variant and N >= 4096 both, else only the forward
// x pass beside the fused Laplacian.
template <typename T>
void choose_fast_passes(zm_plan* p, int cus, bool mfma) {
    const Geo& g = p->geo;
    if (!zm::fast_line_supported<T>(g.vec, g.m)) return;
    const bool plain = zm::fast_line_plain<T>(g.vec, g.m, mfma);
    const bool lapx = zm::fast_line_lapx<T>(g.vec, g.m, mfma, g.dims, g.b);
    if (!plain && !lapx) return;
    const int of = zm::fast_line_occupancy<T>(g.vec, g.m, true, mfma, false);
    const int oi = plain ? zm::fast_line_occupancy<T>(g.vec, g.m, false, mfma, false) : 0;
    const int ol = lapx ? zm::fast_line_occupancy<T>(g.vec, g.m, true, mfma, true) : 0;
    if (of <= 0 || (plain && oi <= 0)) return;
    p->fast_grid_fwd = of * cus;
    p->fast_grid_inv = oi * cus;
    p->fast_grid_lapx = ol * cus;
    if (g.dims == 3 && ol > 0) {
        // 3D: row tiles times plane chunks, about the resident workgroups, the
        // chunks at least two planes long
        const int ntile = g.n >> zm::fast_line_lapx_lines_log2(g.vec, g.m);
        int nzc = 1;
        while (2 * nzc * ntile <= ol * cus && 2 * nzc <= g.n / 2) nzc *= 2;
        p->fast_grid_lapx = ntile * nzc;
    }
}

// Allocates and fills the tables that the plan's passes read: one allocation and
// one launch, in the plan's precision.  A 1024^2 FP64 plan on a caller's scratch
// takes 19 us to create; with an allocation and a launch for each table, those of
// passes it does not run, and every pass's occupancy queried it took 31.
template <typename T>
hipError_t make_tables(zm_plan* p, bool mfma) {
    const Geo& g = p->geo;
    const bool nat = !p->two_stage && !mfma, fast = p->fast_grid_fwd > 0;
    const zm::LinePassSize size = nat_size(g, sizeof(T) == 8);
    const zm::LinePassInfo none{-1, false, {}};
    const zm::LinePassInfo row = nat ? zm::line_pass_info<T>(zm::LP_ROW_FWD, size) : none;
    const zm::LinePassInfo tile = nat ? zm::line_pass_info<T>(zm::LP_TILE_FWD, size) : none;
    const zm::LinePassInfo solve = nat ? zm::line_pass_info<T>(zm::LP_ROW_SPEC, size) : none;
    const bool rows = row.lines_log2 >= 0 && (!row_passes_lose(g, fast) || solve.lines_log2 >= 0);
    const bool tiles = tile.lines_log2 >= 0;
    zm::PlanTables<T> t{};
    t.n = g.n;
    t.line_entries = fast ? zm::line_table_entries(g.vec, g.m) : 0;
    t.line_s = g.vec > g.m ? g.vec : g.m;
    t.radices[0] = row.radices;
    t.radices[1] = tile.radices;
    size_t bytes = 0;
    auto place = [&](size_t need) {
        const size_t at = bytes;
        bytes += (need + 255) & ~(size_t)255;
        return at;
    };
    const size_t es = sizeof(zm::Cx<T>);
    const size_t tw = place(es * (size_t)g.n), line = place(es * (size_t)t.line_entries);
    const size_t nat0 = place(rows ? es * (size_t)row.radices.entries : 0);
    const size_t nat1 = place(tiles ? es * (size_t)tile.radices.entries : 0);
    const size_t half = place(rows || tiles ? sizeof(double) * (size_t)g.n : 0);
    const hipError_t e = hipMalloc(&p->tables, bytes);
    if (e != hipSuccess) return e;
    char* const base = (char*)p->tables;
    p->tw = t.tw = (zm::Cx<T>*)(base + tw);
    if (fast) p->ltab = t.line = (zm::Cx<T>*)(base + line);
    if (rows) p->nat_tables[0] = t.nat[0] = (zm::Cx<T>*)(base + nat0);
    if (tiles) p->nat_tables[1] = t.nat[1] = (zm::Cx<T>*)(base + nat1);
    if (rows || tiles) p->half_sin = t.half_sin = (double*)(base + half);
    return zm::launch_plan_tables<T>(t, nullptr);
}

// The natural-order line passes of a plan.
template <typename T>
void choose_nat_passes(zm_plan* p, int cus) {
    const int d = p->geo.dims;
    p->tiled = p->nat_tables[1] != nullptr;
    for (int axis = 1; axis < d && p->tiled; axis++) {
        p->nat_fwd[axis] = nat_pass<T>(p, cus, zm::LP_TILE_FWD, axis);
        p->nat_inv[axis] = nat_pass<T>(p, cus, zm::LP_TILE_INV, axis);
        if (!p->nat_fwd[axis].grid || !p->nat_inv[axis].grid) p->tiled = false;
    }
    const bool rows = p->nat_tables[0] && !row_passes_lose(p->geo, p->fast_grid_fwd > 0);
    for (int axis = 0; axis < d; axis++) {
        if (axis > 0 && p->tiled) break;
        p->nat_fwd[axis] = p->nat_inv[axis] = zm_plan::NatPass{};
        if (!rows) continue;
        // the forward x pass keeps the fused Laplacian's radix order where the
        // plan has that pass: zm_laplace_forward is bit for bit
        // zm_forward(zm_laplace)
        if (axis > 0 || !p->fast_grid_lapx) p->nat_fwd[axis] = nat_pass<T>(p, cus, zm::LP_ROW_FWD, axis);
        p->nat_inv[axis] = nat_pass<T>(p, cus, zm::LP_ROW_INV, axis);
    }
    // with the forward x pass as a row pass, its Laplacian form has the same
    // radix order
    if (p->nat_fwd[0].grid && p->tiled)
        p->nat_lap = nat_pass<T>(p, cus, d == 2 ? zm::LP_ROW_LAP2 : zm::LP_ROW_LAP3, 0);
    p->nat_spec = nat_pass<T>(p, cus, p->tiled ? zm::LP_TILE_SPEC : zm::LP_ROW_SPEC, d - 1);
}

// The passes of a plan and their tables.
template <typename T>
hipError_t choose_passes(zm_plan* p, bool mfma) {
    int cus = 0;
    hipError_t e = hipDeviceGetAttribute(&cus, hipDeviceAttributeMultiprocessorCount, p->device);
    if (e != hipSuccess) return e;
    if (!p->two_stage) choose_fast_passes<T>(p, cus, mfma);
    e = make_tables<T>(p, mfma);
    if (e != hipSuccess) return e;
    if (!p->two_stage && !mfma) choose_nat_passes<T>(p, cus);
    // the specialised (VEC, M) pairs, as long as every pass of the plan has a
    // compile-time kernel
    p->fast = !p->two_stage && zm::fast_line_supported<T>(p->geo.vec, p->geo.m);
    for (int axis = 0; axis < p->geo.dims; axis++)
        if (!(p->nat_fwd[axis].grid || p->fast_grid_fwd) || !(p->nat_inv[axis].grid || p->fast_grid_inv))
            p->fast = false;
    return hipSuccess;
}

}  // namespace

extern "C" {

zm_status zm_shape_check(const zm_shape* s, zm_dims* out) {
    if (!s) return ZM_ERR_INVALID_ARG;
    if ((s->dims != 2 && s->dims != 3) || s->n <= 0 || s->p <= 0 || s->b <= 0) return ZM_ERR_SHAPE;
    // zmodel/utils.h:47 (LOCAL_DIM = N/P), :60 (VEC = L/B), fft_host_plans.h:46-50 (VEC/P)
    if (s->n % s->p) return ZM_ERR_SHAPE;
    const int l = s->n / s->p;
    if (l % s->b) return ZM_ERR_SHAPE;
    const int vec = l / s->b;
    if (vec % s->p) return ZM_ERR_SHAPE;
    if (!is_pow2(s->n) || !is_pow2(s->p) || !is_pow2(s->b)) return ZM_ERR_UNSUPPORTED;
    const double field = std::pow((double)s->n, s->dims);
    if (field >= 2147483648.0) return ZM_ERR_UNSUPPORTED;  // 32-bit element index inside a field
    if (out) {
        out->l = l;
        out->vec = vec;
        out->vp = vec / s->p;
        out->m = s->b * s->p;
        out->nranks = ipow(s->p, s->dims);
        out->local = (int64_t)l * l * (s->dims == 3 ? l : 1);
        out->field = out->local * out->nranks;
    }
    return ZM_OK;
}

zm_status zm_plan_create(zm_plan** plan, const zm_shape* shape, zm_precision precision, int batch, unsigned flags) {
    if (!plan || !shape) return ZM_ERR_INVALID_ARG;
    *plan = nullptr;
    if (precision != ZM_FP64 && precision != ZM_FP32 && precision != ZM_FP32_MFMA) return ZM_ERR_INVALID_ARG;
    if (batch < 1 || batch > 65535) return ZM_ERR_INVALID_ARG;
    if (flags & ~(ZM_FLAG_TWO_STAGE | ZM_FLAG_CALLER_SCRATCH)) return ZM_ERR_INVALID_ARG;
    zm_dims d;
    ZM_TRY(zm_shape_check(shape, &d));
    const bool mfma = precision == ZM_FP32_MFMA;
    // the split-precision radix-16 passes live in the specialised fused line
    // pass only
    if (mfma && ((flags & ZM_FLAG_TWO_STAGE) || !zm::fast_line_supported<float>(d.vec, d.m)))
        return ZM_ERR_UNSUPPORTED;

    const int n = shape->n;
    const int64_t rows = (int64_t)d.local / d.l;  // L^(dims-1) local rows per rank
    const size_t es = elem_bytes(precision);

    // Fused line kernel when a whole line (N elements) fits LDS; otherwise
    // the two-stage path.
    bool two_stage = (flags & ZM_FLAG_TWO_STAGE) != 0;
    int lpb = 1;
    if (!two_stage) {
        if (es * zm::padded_elems(n) > kMaxLds || n / zm::EPT > 512) two_stage = true;
    }
    if (!two_stage) {
        while ((int64_t)lpb * 2 * n <= kLineTarget && lpb * 2 <= rows) lpb *= 2;
        if ((int64_t)lpb * n < zm::EPT) return ZM_ERR_UNSUPPORTED;
    }
    int rpb = 1;
    while ((int64_t)rpb * 2 * d.l <= kStageTarget && rpb * 2 <= rows) rpb *= 2;
    if (two_stage) {
        if ((int64_t)rpb * d.l < zm::EPT || es * zm::padded_elems(rpb * d.l) > kMaxLds || rpb * d.l / zm::EPT > 512)
            return ZM_ERR_UNSUPPORTED;
    }

    int device = 0;
    if (hipGetDevice(&device) != hipSuccess) return ZM_ERR_DEVICE;
    int count = 0;
    if (hipGetDeviceCount(&count) != hipSuccess || count < 1) return ZM_ERR_DEVICE;

    noalloc::resolve(device);

    zm_plan* p = new (std::nothrow) zm_plan();
    if (!p) return ZM_ERR_NOMEM;
    p->shape = *shape;
    p->dims = d;
    p->precision = precision;
    p->batch = batch;
    p->flags = flags;
    p->device = device;
    p->two_stage = two_stage;
    p->lpb = lpb;
    p->rpb = rpb;
    Geo& g = p->geo;
    g.dims = shape->dims;
    g.n = n;
    g.p = shape->p;
    g.b = shape->b;
    g.l = d.l;
    g.vec = d.vec;
    g.vp = d.vp;
    g.m = d.m;
    g.nranks = d.nranks;
    g.local = d.local;
    g.field = d.field;
    g.ln = ilog2(n);
    g.lp = ilog2(shape->p);
    g.lb = ilog2(shape->b);
    g.ll = ilog2(d.l);
    g.lvec = ilog2(d.vec);
    p->scratch_bytes = (size_t)batch * (size_t)d.field * es;

    // The plan's own scratch is allocated here, once, so that the plan is
    // immutable after creation; ZM_FLAG_CALLER_SCRATCH plans own none and
    // every transform call must bring one.
    if (!(flags & ZM_FLAG_CALLER_SCRATCH) && hipMalloc(&p->own_scratch, p->scratch_bytes) != hipSuccess) {
        delete p;
        return ZM_ERR_NOMEM;
    }
    hipError_t e = precision == ZM_FP64 ? choose_passes<double>(p, false) : choose_passes<float>(p, mfma);
    if (e == hipSuccess) e = hipDeviceSynchronize();
    if (e != hipSuccess || (mfma && !p->fast)) {
        if (p->tables) (void)hipFree(p->tables);
        if (p->own_scratch) (void)hipFree(p->own_scratch);
        delete p;
        return e == hipErrorOutOfMemory ? ZM_ERR_NOMEM : e != hipSuccess ? ZM_ERR_DEVICE : ZM_ERR_UNSUPPORTED;
    }
    *plan = p;
    return ZM_OK;
}

zm_status zm_plan_destroy(zm_plan* p) {
    if (!p) return ZM_ERR_INVALID_ARG;
    zm_status st = ZM_OK;
    if (p->tables && hipFree(p->tables) != hipSuccess) st = ZM_ERR_DEVICE;
    if (p->own_scratch && hipFree(p->own_scratch) != hipSuccess) st = ZM_ERR_DEVICE;
    drop_timing(p);
    delete p;
    return st;
}

zm_status zm_plan_dims(const zm_plan* p, zm_shape* shape, zm_dims* dims, zm_precision* precision, int* batch) {
    if (!p) return ZM_ERR_INVALID_ARG;
    if (shape) *shape = p->shape;
    if (dims) *dims = p->dims;
    if (precision) *precision = p->precision;
    if (batch) *batch = p->batch;
    return ZM_OK;
}

zm_status zm_plan_path(const zm_plan* p, unsigned* path) {
    if (!p || !path) return ZM_ERR_INVALID_ARG;
    *path = (p->two_stage ? ZM_PATH_TWO_STAGE : 0u) | (p->fast ? ZM_PATH_FAST_LINE : 0u) |
            (p->precision == ZM_FP32_MFMA ? ZM_PATH_MFMA : 0u) | (p->tiled ? ZM_PATH_TILES : 0u) |
            (p->fast_grid_lapx || p->nat_lap.grid ? ZM_PATH_LAPLACE : 0u) | (p->nat_spec.grid ? ZM_PATH_SOLVE : 0u);
    return ZM_OK;
}

size_t zm_scratch_bytes(const zm_plan* p) { return p ? p->scratch_bytes : 0; }

size_t zm_field_bytes(const zm_plan* p) {
    return p ? (size_t)p->batch * (size_t)p->dims.field * elem_bytes(p->precision) : 0;
}

}  // extern "C"

// ---------------------------------------------------------------------------
// transform sequences
// ---------------------------------------------------------------------------
namespace {

int axis_stride(const zm_plan* p, int axis) { return axis == 0 ? 1 : (axis == 1 ? p->shape.p : p->shape.p * p->shape.p); }

enum RepackKind { REPACK_2D = 0, REPACK_XY = 1, REPACK_YZ = 2 };

zm::RepackArgs repack_args(const zm_plan* p, RepackKind k) {
    const int64_t L = p->dims.l;
    zm::RepackArgs a{};
    a.tx = p->dims.vec < zm::REPACK_TX ? p->dims.vec : zm::REPACK_TX;
    a.ty = L < zm::REPACK_TY ? (int)L : zm::REPACK_TY;
    if (k == REPACK_2D) {
        a.ecount = 1;
        a.ei = a.eo = 0;
        a.sxi = L;
        a.syo = L;
    } else if (k == REPACK_XY) {
        a.ecount = (int)L;
        a.ei = a.eo = L * L;
        a.sxi = L;
        a.syo = L;
    } else {
        a.ecount = (int)L;
        a.ei = a.eo = L;
        a.sxi = L * L;
        a.syo = L * L;
    }
    return a;
}

template <typename T>
struct Exec {
    zm_plan* p;
    hipStream_t st;
    bool compute;
    const zm::Cx<T>* tw;
    bool record = true;  // per-launch timing events when the plan records them

    const zm::Cx<T>* line_tables() const {
        return (const zm::Cx<T>*)p->ltab;
    }
    // natural-order line pass of one axis; a tile pass holds a repack stage,
    // counted inside it
    zm_status nat(const zm_plan::NatPass& np, const void* in, void* out, double scale,
                  const zm::SpectralArgs& sp = zm::SpectralArgs{}) const {
        const hipError_t e = timed_launch(p, ZM_STAGE_LINE, st, [&] {
            return zm::launch_line_pass<T>(np.kind, np.size, (const zm::Cx<T>*)in, (zm::Cx<T>*)out,
                                           np.args, (const zm::Cx<T>*)np.tables, scale, sp, np.grid, st);
        }, record);
        if (e == hipSuccess && np.kind >= zm::LP_TILE_FWD && np.kind <= zm::LP_TILE_SPEC)
            timed_inside(p, ZM_STAGE_REPACK, record);
        if (e == hipSuccess && np.kind == zm::LP_TILE_SPEC) timed_inside(p, ZM_STAGE_REPACK, record);
        if (e == hipSuccess && (np.kind == zm::LP_TILE_SPEC || np.kind == zm::LP_ROW_SPEC))
            timed_inside(p, ZM_STAGE_SPECTRAL, record);
        return launch_status(e);
    }
    // whether the transforms run without repack launches
    bool tiled() const { return compute && p->tiled; }

    // lapx: the x pass of zm_laplace_forward (fast_grid_lapx != 0 only),
    // transforming `scale` times the input's Laplacian
    zm_status line(const void* in, void* out, int axis, bool fwd, double scale, bool lapx = false) const {
        const zm_plan::NatPass& np = fwd ? p->nat_fwd[axis] : p->nat_inv[axis];
        if (lapx && p->nat_lap.grid) {
            ZM_TRY(nat(p->nat_lap, in, out, scale));
            timed_inside(p, ZM_STAGE_LAPLACE, record);
            return ZM_OK;
        }
        if (compute && !lapx && np.grid) return nat(np, in, out, scale);
        zm::LineArgs a{axis_stride(p, axis), (int)(p->dims.local / p->dims.l), p->lpb};
        const int grid = lapx ? p->fast_grid_lapx : fwd ? p->fast_grid_fwd : p->fast_grid_inv;
        if (compute && grid) {
            return launch_status(timed_launch(p, lapx ? ZM_STAGE_LINE_LAPLACE : ZM_STAGE_LINE, st, [&] {
                return zm::launch_line_fast<T>((const zm::Cx<T>*)in, (zm::Cx<T>*)out, p->geo, a, line_tables(),
                                               p->batch, fwd, scale, grid, p->precision == ZM_FP32_MFMA, lapx, st);
            }, record));
        }
        if (lapx) return ZM_ERR_UNSUPPORTED;
        return launch_status(timed_launch(p, ZM_STAGE_LINE, st, [&] {
            return zm::launch_line<T>((const zm::Cx<T>*)in, (zm::Cx<T>*)out, p->geo, a, tw, p->batch, fwd, compute,
                                      scale, st);
        }, record));
    }
    zm::StageArgs sargs(int axis) const {
        return zm::StageArgs{axis_stride(p, axis), (int)(p->dims.local / p->dims.l), p->rpb,
                             p->shape.dims == 3 ? p->dims.l : 1};
    }
    zm_status stage_a(const void* in, void* out, int axis, bool fwd, double scale) const {
        return launch_status(timed_launch(p, ZM_STAGE_A, st, [&] {
            return zm::launch_stage_a<T>((const zm::Cx<T>*)in, (zm::Cx<T>*)out, p->geo, sargs(axis), tw, p->batch,
                                         fwd, compute, scale, st);
        }, record));
    }
    zm_status stage_b(const void* in, void* out, int axis, bool fwd) const {
        return launch_status(timed_launch(p, ZM_STAGE_B, st, [&] {
            return zm::launch_stage_b<T>((const zm::Cx<T>*)in, (zm::Cx<T>*)out, p->geo, sargs(axis), tw, p->batch,
                                         fwd, compute, st);
        }, record));
    }
    zm_status repack(const void* in, void* out, RepackKind k, bool fwd) const {
        return launch_status(timed_launch(p, ZM_STAGE_REPACK, st, [&] {
            return zm::launch_repack<T>((const zm::Cx<T>*)in, (zm::Cx<T>*)out, p->geo, repack_args(p, k), p->batch,
                                        fwd, st);
        }, record));
    }

    // forward_fft / forward_fft_3d (zmodel/transforms/fft.cu:199-339,
    // fft3d.cu:234-412) as x-pass, repack, y-pass [, repack-yz, z-pass]; with
    // the tiled passes the repacks are part of the passes after them.
    zm_status forward(const void* in, void* out, void* s, bool lapx = false, double lap_scale = 1.0) const {
        const bool d3 = p->shape.dims == 3;
        if (!p->two_stage && tiled()) {
            void* a = d3 ? out : s;
            ZM_TRY(line(in, a, 0, true, lap_scale, lapx));
            if (!d3) return line(s, out, 1, true, 1.0);
            ZM_TRY(line(out, s, 1, true, 1.0));
            return line(s, out, 2, true, 1.0);
        }
        if (!p->two_stage) {
            ZM_TRY(line(in, s, 0, true, lap_scale, lapx));
            ZM_TRY(repack(s, out, d3 ? REPACK_XY : REPACK_2D, true));
            ZM_TRY(line(out, out, 1, true, 1.0));
            if (d3) {
                ZM_TRY(repack(out, s, REPACK_YZ, true));
                ZM_TRY(line(s, out, 2, true, 1.0));
            }
            return ZM_OK;
        }
        if (!d3) {
            ZM_TRY(stage_a(in, out, 0, true, 1.0));
            ZM_TRY(stage_b(out, s, 0, true));
            ZM_TRY(repack(s, out, REPACK_2D, true));
            ZM_TRY(stage_a(out, s, 1, true, 1.0));
            ZM_TRY(stage_b(s, out, 1, true));
            return ZM_OK;
        }
        ZM_TRY(stage_a(in, s, 0, true, 1.0));
        ZM_TRY(stage_b(s, out, 0, true));
        ZM_TRY(repack(out, s, REPACK_XY, true));
        ZM_TRY(stage_a(s, out, 1, true, 1.0));
        ZM_TRY(stage_b(out, s, 1, true));
        ZM_TRY(repack(s, out, REPACK_YZ, true));
        ZM_TRY(stage_a(out, s, 2, true, 1.0));
        ZM_TRY(stage_b(s, out, 2, true));
        return ZM_OK;
    }

    // The reference's laplace followed by forward_fft (zmodel/main.cu:50-63).
    // With a fused pass (line_fast.hip, or the row pass's Laplacian form) the
    // Laplacian is formed inside the x pass, one sweep of the field less;
    // otherwise the stencil writes `out` and the
    // forward chain runs in place on it (its first pass reads `out` whole
    // before the repack writes it).  Either way the result is bit for bit
    // zm_forward(zm_laplace(in)).
    zm_status laplace_forward(const void* in, void* out, void* s, double lap_scale) const {
        if (p->two_stage) return ZM_ERR_UNSUPPORTED;
        if (p->fast_grid_lapx > 0 || p->nat_lap.grid) return forward(in, out, s, true, lap_scale);
        ZM_TRY(launch_status(timed_launch(p, ZM_STAGE_LAPLACE, st, [&] {
            return zm::launch_stencil<T>(in, out, p->geo, p->batch, zm::OP_LAPLACE, true, lap_scale, false, st);
        }, record)));
        return forward(out, out, s);
    }

    // inverse_fft / inverse_fft_3d (zmodel/transforms/fft.cu:409-514,
    // fft3d.cu:508-633): the reverse chain, scale applied once on the x-pass.
    zm_status inverse(const void* in, void* out, void* s, double scale) const {
        const bool d3 = p->shape.dims == 3;
        if (!p->two_stage && tiled()) {
            if (!d3) {
                ZM_TRY(line(in, s, 1, false, 1.0));
                return line(s, out, 0, false, scale);
            }
            ZM_TRY(line(in, s, 2, false, 1.0));
            ZM_TRY(line(s, out, 1, false, 1.0));
            return line(out, out, 0, false, scale);
        }
        if (!p->two_stage) {
            if (d3) {
                ZM_TRY(line(in, s, 2, false, 1.0));
                ZM_TRY(repack(s, out, REPACK_YZ, false));
                ZM_TRY(line(out, out, 1, false, 1.0));
                ZM_TRY(repack(out, s, REPACK_XY, false));
                ZM_TRY(line(s, out, 0, false, scale));
                return ZM_OK;
            }
            ZM_TRY(line(in, s, 1, false, 1.0));
            ZM_TRY(repack(s, out, REPACK_2D, false));
            ZM_TRY(line(out, out, 0, false, scale));
            return ZM_OK;
        }
        if (!d3) {
            ZM_TRY(stage_b(in, out, 1, false));
            ZM_TRY(stage_a(out, s, 1, false, 1.0));
            ZM_TRY(repack(s, out, REPACK_2D, false));
            ZM_TRY(stage_b(out, s, 0, false));
            ZM_TRY(stage_a(s, out, 0, false, scale));
            return ZM_OK;
        }
        ZM_TRY(stage_b(in, s, 2, false));
        ZM_TRY(stage_a(s, out, 2, false, 1.0));
        ZM_TRY(repack(out, s, REPACK_YZ, false));
        ZM_TRY(stage_b(s, out, 1, false));
        ZM_TRY(stage_a(out, s, 1, false, 1.0));
        ZM_TRY(repack(s, out, REPACK_XY, false));
        ZM_TRY(stage_b(out, s, 0, false));
        ZM_TRY(stage_a(s, out, 0, false, scale));
        return ZM_OK;
    }
    zm_status multiply(const void* in, void* out, const zm::SpectralArgs& sp) const {
        return launch_status(timed_launch(p, ZM_STAGE_SPECTRAL, st, [&] {
            return zm::launch_spectral<T>((const zm::Cx<T>*)in, (zm::Cx<T>*)out, p->geo, p->batch, sp.kind, sp.p0,
                                          sp.p1, sp.kscale, sp.conj != 0, sp.factor, st);
        }, record));
    }

    // inverse(scale) after the multiplier after forward.  The last axis's
    // forward pass, the multiplier and its inverse pass are one kernel, which
    // holds the spectrum of a line group in LDS: two to four sweeps of the
    // field less than the three calls.
    zm_status solve(const void* in, void* out, void* s, double scale, zm::SpectralArgs sp) const {
        const bool d3 = p->shape.dims == 3;
        if (p->two_stage) return ZM_ERR_UNSUPPORTED;
        if (!p->nat_spec.grid) {
            ZM_TRY(forward(in, out, s));
            ZM_TRY(multiply(out, out, sp));
            return inverse(out, out, s, scale);
        }
        const zm::NatMaps m(p->geo);
        sp.f0 = m.frequency0();
        sp.f1 = m.frequency1();
        sp.half_sin = p->half_sin;
        if (!p->tiled) {  // 2D
            ZM_TRY(line(in, s, 0, true, 1.0));
            ZM_TRY(repack(s, out, REPACK_2D, true));
            ZM_TRY(nat(p->nat_spec, out, out, 1.0, sp));
            ZM_TRY(repack(out, s, REPACK_2D, false));
            return line(s, out, 0, false, scale);
        }
        if (!d3) {
            ZM_TRY(line(in, s, 0, true, 1.0));
            ZM_TRY(nat(p->nat_spec, s, out, 1.0, sp));
            return line(out, out, 0, false, scale);
        }
        ZM_TRY(line(in, out, 0, true, 1.0));
        ZM_TRY(line(out, s, 1, true, 1.0));
        ZM_TRY(nat(p->nat_spec, s, out, 1.0, sp));
        ZM_TRY(line(out, s, 1, false, 1.0));
        return line(s, out, 0, false, scale);
    }
};

zm_status check_io(const zm_plan* p, const void* in, const void* out) {
    if (!p || !in || !out) return ZM_ERR_INVALID_ARG;
    if (in == out) return ZM_ERR_ALIAS;
    return ZM_OK;
}

// The caller's scratch, else the one the plan allocated at creation (none
// for ZM_FLAG_CALLER_SCRATCH plans: then NULL is an invalid argument).
zm_status scratch_for(const zm_plan* p, void* scratch, void** s) {
    *s = scratch ? scratch : p->own_scratch;
    return *s ? ZM_OK : ZM_ERR_INVALID_ARG;
}

zm_status run_transform(zm_plan* p, const void* in, void* out, void* scratch, void* stream, bool fwd, bool compute,
                        double scale, bool record = true) {
    ZM_TRY(check_io(p, in, out));
    void* s = nullptr;
    ZM_TRY(scratch_for(p, scratch, &s));
    if (s == in || s == out) return ZM_ERR_ALIAS;
    hipStream_t st = (hipStream_t)stream;
    if (p->precision == ZM_FP64) {
        Exec<double> ex{p, st, compute, (const double2*)p->tw, record};
        return fwd ? ex.forward(in, out, s) : ex.inverse(in, out, s, scale);
    }
    Exec<float> ex{p, st, compute, (const float2*)p->tw, record};
    return fwd ? ex.forward(in, out, s) : ex.inverse(in, out, s, scale);
}

}  // namespace

extern "C" {

zm_status zm_forward(zm_plan* p, const void* in, void* out, void* scratch, void* stream) {
    return run_transform(p, in, out, scratch, stream, true, true, 1.0);
}

zm_status zm_forward_noalloc(zm_plan* p, const void* in, void* out, void* stream) {
    if (!p) return ZM_ERR_INVALID_ARG;
    if (p->scratch_bytes > ZM_NOALLOC_SCRATCH_BYTES) return ZM_ERR_SCRATCH_LIMIT;
    void* s = noalloc::device_copy(p->device);
    if (!s) return ZM_ERR_DEVICE;
    // no timing events: creating them is an allocation
    return run_transform(p, in, out, s, stream, true, true, 1.0, false);
}

zm_status zm_laplace_forward(zm_plan* p, const void* in, void* out, double scale, void* scratch, void* stream) {
    ZM_TRY(check_io(p, in, out));
    if (!std::isfinite(scale)) return ZM_ERR_INVALID_ARG;
    void* s = nullptr;
    ZM_TRY(scratch_for(p, scratch, &s));
    if (s == in || s == out) return ZM_ERR_ALIAS;
    const hipStream_t st = (hipStream_t)stream;
    if (p->precision == ZM_FP64) {
        Exec<double> ex{p, st, true, (const double2*)p->tw};
        return ex.laplace_forward(in, out, s, scale);
    }
    Exec<float> ex{p, st, true, (const float2*)p->tw};
    return ex.laplace_forward(in, out, s, scale);
}

zm_status zm_inverse(zm_plan* p, const void* in, void* out, double scale, void* scratch, void* stream) {
    return run_transform(p, in, out, scratch, stream, false, true, scale);
}

zm_status zm_permute_forward(zm_plan* p, const void* in, void* out, void* scratch, void* stream) {
    return run_transform(p, in, out, scratch, stream, true, false, 1.0);
}

zm_status zm_permute_inverse(zm_plan* p, const void* in, void* out, void* scratch, void* stream) {
    return run_transform(p, in, out, scratch, stream, false, false, 1.0);
}

zm_status zm_forward_adjoint(zm_plan* p, const void* in, void* out, void* scratch, void* stream) {
    // forward = P_out * DFT * P_in stage by stage, so its adjoint is the
    // inverse chain (conjugate twiddles, inverse DFTs) with scale 1.
    return run_transform(p, in, out, scratch, stream, false, true, 1.0);
}

zm_status zm_inverse_adjoint(zm_plan* p, const void* in, void* out, double scale, void* scratch, void* stream) {
    // (s * inverse)^H = s * forward; the scale goes on a separate pass only
    // when it is not 1.
    zm_status st = run_transform(p, in, out, scratch, stream, true, true, 1.0);
    if (st != ZM_OK || scale == 1.0) return st;
    return zm_spectral_multiply(p, out, out, ZM_SPECTRAL_SCALE, scale, 0.0, 1.0, stream);
}

// ---------------------------------------------------------------------------
// stencils
// ---------------------------------------------------------------------------

static zm_status run_stencil(zm_plan* p, const void* in, void* out, zm::StencilOp op, double coef, bool negate,
                             zm_element element, void* stream) {
    ZM_TRY(check_io(p, in, out));
    if (element != ZM_COMPLEX && element != ZM_REAL) return ZM_ERR_INVALID_ARG;
    const bool cplx = element == ZM_COMPLEX;
    const hipStream_t st = (hipStream_t)stream;
    return launch_status(timed_launch(p, op == zm::OP_LAPLACE ? ZM_STAGE_LAPLACE : ZM_STAGE_DERIV, st, [&] {
        if (p->precision == ZM_FP64) return zm::launch_stencil<double>(in, out, p->geo, p->batch, op, cplx, coef, negate, st);
        return zm::launch_stencil<float>(in, out, p->geo, p->batch, op, cplx, coef, negate, st);
    }));
}

zm_status zm_laplace(zm_plan* p, const void* in, void* out, double scale, zm_element element, void* stream) {
    return run_stencil(p, in, out, zm::OP_LAPLACE, scale, false, element, stream);
}

zm_status zm_laplace_add(zm_plan* p, const void* in, void* inout, double scale, double alpha, void* stream) {
    ZM_TRY(check_io(p, in, inout));
    const hipStream_t st = (hipStream_t)stream;
    return launch_status(timed_launch(p, ZM_STAGE_LAPLACE, st, [&] {
        if (p->precision == ZM_FP64)
            return zm::launch_laplace_add<double>((const double2*)in, (double2*)inout, p->geo, p->batch, scale, alpha, st);
        return zm::launch_laplace_add<float>((const float2*)in, (float2*)inout, p->geo, p->batch, scale, alpha, st);
    }));
}

zm_status zm_residual_norm(zm_plan* p, void* inout, const void* g, double* partials, void* norm2, void* stream) {
    ZM_TRY(check_io(p, g, inout));
    if (!partials || !norm2) return ZM_ERR_INVALID_ARG;
    const hipStream_t st = (hipStream_t)stream;
    const int64_t n = (int64_t)p->batch * p->dims.field;
    return launch_status(timed_launch(p, ZM_STAGE_SPECTRAL, st, [&] {
        if (p->precision == ZM_FP64)
            return zm::launch_residual_norm<double>((double2*)inout, (const double2*)g, n, partials, (double*)norm2, st);
        return zm::launch_residual_norm<float>((float2*)inout, (const float2*)g, n, partials, (float*)norm2, st);
    }));
}

static zm_status deriv(zm_plan* p, const void* in, void* out, double delta, zm_element element, void* stream,
                       zm::StencilOp op, bool negate) {
    if (!p) return ZM_ERR_INVALID_ARG;
    if (p->shape.b < 2) return ZM_ERR_UNSUPPORTED;  // dx.cu:94-100, dy.cu:117-124 need B >= 2
    if (op == zm::OP_DZ4 && p->shape.dims != 3) return ZM_ERR_UNSUPPORTED;
    if (!(delta != 0.0) || !std::isfinite(delta)) return ZM_ERR_INVALID_ARG;
    return run_stencil(p, in, out, op, 12 * delta, negate, element, stream);
}

zm_status zm_dx4(zm_plan* p, const void* in, void* out, double delta, zm_element element, void* stream) {
    return deriv(p, in, out, delta, element, stream, zm::OP_DX4, false);
}
zm_status zm_dy4(zm_plan* p, const void* in, void* out, double delta, zm_element element, void* stream) {
    return deriv(p, in, out, delta, element, stream, zm::OP_DY4, false);
}
zm_status zm_dx4_adjoint(zm_plan* p, const void* in, void* out, double delta, zm_element element, void* stream) {
    return deriv(p, in, out, delta, element, stream, zm::OP_DX4, true);
}
zm_status zm_dy4_adjoint(zm_plan* p, const void* in, void* out, double delta, zm_element element, void* stream) {
    return deriv(p, in, out, delta, element, stream, zm::OP_DY4, true);
}
zm_status zm_dz4(zm_plan* p, const void* in, void* out, double delta, zm_element element, void* stream) {
    return deriv(p, in, out, delta, element, stream, zm::OP_DZ4, false);
}
zm_status zm_dz4_adjoint(zm_plan* p, const void* in, void* out, double delta, zm_element element, void* stream) {
    return deriv(p, in, out, delta, element, stream, zm::OP_DZ4, true);
}

// Checks a multiplier's parameters; fills all of its arguments but the line
// maps of the fused pass.
static zm_status spectral_args(const zm_plan* p, zm_spectral kind, double p0, double p1, double length, bool conj,
                               zm::SpectralArgs* sp) {
    if ((int)kind < (int)ZM_SPECTRAL_POISSON || (int)kind > (int)ZM_SPECTRAL_POISSON_STENCIL) return ZM_ERR_INVALID_ARG;
    if (!(length > 0.0)) return ZM_ERR_INVALID_ARG;
    // the dx4 symbol is defined on the 2D layout only, like zm_dx4
    if ((kind == ZM_SPECTRAL_STENCIL || kind == ZM_SPECTRAL_POISSON_STENCIL) && p1 != 0.0 && p->shape.dims != 2)
        return ZM_ERR_INVALID_ARG;
    *sp = zm::SpectralArgs{(int)kind, conj ? 1 : 0, p->shape.dims, p0, p1, 2.0 * M_PI / length, {}, {}, nullptr, nullptr};
    return ZM_OK;
}

static zm_status spectral(zm_plan* p, const void* in, void* out, zm_spectral kind, double p0, double p1,
                          double length, void* stream, bool conj) {
    if (!p || !in || !out) return ZM_ERR_INVALID_ARG;
    zm::SpectralArgs sp;
    ZM_TRY(spectral_args(p, kind, p0, p1, length, conj, &sp));
    const hipStream_t st = (hipStream_t)stream;
    if (p->precision == ZM_FP64) return Exec<double>{p, st, true, (const double2*)p->tw}.multiply(in, out, sp);
    return Exec<float>{p, st, true, (const float2*)p->tw}.multiply(in, out, sp);
}

static zm_status spectral_solve(zm_plan* p, const void* in, void* out, zm_spectral kind, double p0, double p1,
                                double length, double scale, const double* factor, void* scratch, void* stream,
                                bool conj) {
    ZM_TRY(check_io(p, in, out));
    zm::SpectralArgs sp;
    ZM_TRY(spectral_args(p, kind, p0, p1, length, conj, &sp));
    sp.factor = factor;
    void* s = nullptr;
    ZM_TRY(scratch_for(p, scratch, &s));
    if (s == in || s == out) return ZM_ERR_ALIAS;
    const hipStream_t st = (hipStream_t)stream;
    if (p->precision == ZM_FP64) return Exec<double>{p, st, true, (const double2*)p->tw}.solve(in, out, s, scale, sp);
    return Exec<float>{p, st, true, (const float2*)p->tw}.solve(in, out, s, scale, sp);
}

zm_status zm_spectral_multiply(zm_plan* p, const void* in, void* out, zm_spectral kind, double p0, double p1,
                               double length, void* stream) {
    return spectral(p, in, out, kind, p0, p1, length, stream, false);
}

zm_status zm_spectral_multiply_adjoint(zm_plan* p, const void* in, void* out, zm_spectral kind, double p0, double p1,
                                       double length, void* stream) {
    return spectral(p, in, out, kind, p0, p1, length, stream, true);
}

zm_status zm_spectral_solve(zm_plan* p, const void* in, void* out, zm_spectral kind, double p0, double p1,
                            double length, double scale, const double* factor, void* scratch, void* stream) {
    return spectral_solve(p, in, out, kind, p0, p1, length, scale, factor, scratch, stream, false);
}

zm_status zm_spectral_solve_adjoint(zm_plan* p, const void* in, void* out, zm_spectral kind, double p0, double p1,
                                    double length, double scale, const double* factor, void* scratch,
                                    void* stream) {
    return spectral_solve(p, in, out, kind, p0, p1, length, scale, factor, scratch, stream, true);
}

zm_status zm_real_index_table(zm_plan* p, int64_t* out, void* stream) {
    if (!p || !out) return ZM_ERR_INVALID_ARG;
    return launch_status(timed_launch(p, ZM_STAGE_CONVERT, (hipStream_t)stream,
                                      [&] { return zm::launch_index_table(out, p->geo, false, (hipStream_t)stream); }));
}

zm_status zm_reciprocal_index_table(zm_plan* p, int64_t* out, void* stream) {
    if (!p || !out) return ZM_ERR_INVALID_ARG;
    return launch_status(timed_launch(p, ZM_STAGE_CONVERT, (hipStream_t)stream,
                                      [&] { return zm::launch_index_table(out, p->geo, true, (hipStream_t)stream); }));
}

static zm_status natural_packed(zm_plan* p, const void* in, void* out, bool to_packed, void* stream) {
    ZM_TRY(check_io(p, in, out));
    const hipStream_t st = (hipStream_t)stream;
    return launch_status(timed_launch(p, ZM_STAGE_CONVERT, st, [&] {
        if (p->precision == ZM_FP64)
            return zm::launch_natural_packed<double>((const double2*)in, (double2*)out, p->geo, p->batch, to_packed, st);
        return zm::launch_natural_packed<float>((const float2*)in, (float2*)out, p->geo, p->batch, to_packed, st);
    }));
}

zm_status zm_natural_to_packed(zm_plan* p, const void* natural, void* packed, void* stream) {
    return natural_packed(p, natural, packed, true, stream);
}

zm_status zm_packed_to_natural(zm_plan* p, const void* packed, void* natural, void* stream) {
    return natural_packed(p, packed, natural, false, stream);
}

// ---------------------------------------------------------------------------
// host index maps (zmodel/utils.h:122-320)
// ---------------------------------------------------------------------------

int zm_packed_to_block_cyclic(const zm_shape* s, int c) { return zm::packed_to_block_cyclic(map_shape(s), c); }
int zm_block_cyclic_to_packed(const zm_shape* s, int c) { return zm::block_cyclic_to_packed(map_shape(s), c); }

void zm_real_to_global(const zm_shape* s, int rid, int cid, int lr, int lc, int* gr, int* gc) {
    const zm::MapShape m = map_shape(s);
    *gr = zm::local_row_to_global(m, rid, lr);
    *gc = zm::packed_col_to_global(m, cid, lc);
}

void zm_global_to_real(const zm_shape* s, int gr, int gc, int* rid, int* cid, int* lr, int* lc) {
    const zm::MapShape m = map_shape(s);
    zm::global_row_to_local(m, gr, rid, lr);
    zm::global_col_to_local(m, gc, cid, lc);
}

void zm_real_to_global_3d(const zm_shape* s, int rid, int cid, int did, int ld, int lr, int lc, int* gd, int* gr,
                          int* gc) {
    const zm::MapShape m = map_shape(s);
    *gd = zm::local_row_to_global(m, did, ld);
    *gr = zm::local_row_to_global(m, rid, lr);
    *gc = zm::packed_col_to_global(m, cid, lc);
}

void zm_global_to_real_3d(const zm_shape* s, int gd, int gr, int gc, int* rid, int* cid, int* did, int* ld, int* lr,
                          int* lc) {
    const zm::MapShape m = map_shape(s);
    zm::global_row_to_local(m, gd, did, ld);
    zm::global_row_to_local(m, gr, rid, lr);
    zm::global_col_to_local(m, gc, cid, lc);
}

int zm_lp(const zm_shape* s, int i) { return zm::lp(map_shape(s), i); }
int zm_ct(const zm_shape* s, int q) { return zm::ct(map_shape(s), q); }
int zm_lp_inv(const zm_shape* s, int j) { return zm::lp_inv(map_shape(s), j); }
int zm_ct_inv(const zm_shape* s, int k) { return zm::ct_inv(map_shape(s), k); }

void zm_reciprocal_to_global(const zm_shape* s, int rid, int cid, int lr, int lc, int* ky, int* kx) {
    const zm::MapShape m = map_shape(s);
    *kx = zm::recip_to_freq(m, cid, lr);
    *ky = zm::recip_to_freq(m, rid, lc);
}

void zm_global_to_reciprocal(const zm_shape* s, int ky, int kx, int* rid, int* cid, int* lr, int* lc) {
    const zm::MapShape m = map_shape(s);
    zm::freq_to_recip(m, kx, cid, lr);
    zm::freq_to_recip(m, ky, rid, lc);
}

void zm_reciprocal_to_global_3d(const zm_shape* s, int rid, int cid, int did, int ld, int lr, int lc, int* kd, int* kr,
                                int* kc) {
    const zm::MapShape m = map_shape(s);
    *kc = zm::recip_to_freq(m, cid, lr);
    *kr = zm::recip_to_freq(m, rid, ld);
    *kd = zm::recip_to_freq(m, did, lc);
}

void zm_global_to_reciprocal_3d(const zm_shape* s, int kd, int kr, int kc, int* rid, int* cid, int* did, int* ld,
                                int* lr, int* lc) {
    const zm::MapShape m = map_shape(s);
    zm::freq_to_recip(m, kc, cid, lr);
    zm::freq_to_recip(m, kr, rid, ld);
    zm::freq_to_recip(m, kd, did, lc);
}

zm_status zm_timing_enable(zm_plan* p, int enable) {
    if (!p) return ZM_ERR_INVALID_ARG;
    p->timing = enable != 0;
    p->last_stop = nullptr;  // a new timed sequence starts with its own start event
    return ZM_OK;
}

zm_status zm_timing_read(zm_plan* p, zm_stage stage, int* count, double* total_ms) {
    if (!p || !count || !total_ms || (int)stage < 0 || stage >= ZM_STAGE_COUNT) return ZM_ERR_INVALID_ARG;
    int c = 0;
    double tot = 0.0;
    for (auto& t : p->timed) {
        if (t.stage != (int)stage) continue;
        if (hipEventSynchronize(t.stop) != hipSuccess) return ZM_ERR_DEVICE;
        float ms = 0.f;
        if (t.own_stop && hipEventElapsedTime(&ms, t.start, t.stop) != hipSuccess) return ZM_ERR_DEVICE;
        tot += ms;
        c++;
    }
    *count = c;
    *total_ms = tot;
    return ZM_OK;
}

zm_status zm_timing_reset(zm_plan* p) {
    if (!p) return ZM_ERR_INVALID_ARG;
    drop_timing(p);
    return ZM_OK;
}

zm_status zm_init_host(const zm_shape* s, double* host_grid, int ncomp) {
    zm_dims d;
    if (!host_grid || (ncomp != 1 && ncomp != 2)) return ZM_ERR_INVALID_ARG;
    ZM_TRY(zm_shape_check(s, &d));
    const zm::MapShape m = map_shape(s);
    const int64_t L = d.l, N = s->n;
    // every packed position holds the global linear index of its point: the
    // block-cyclic fill of utils.cu:17-32 followed by vector_pack (utils.h:100-108)
    for (int id = 0; id < d.nranks; id++) {
        const int cid = id % s->p;
        const int rid = (id / s->p) % s->p;
        const int did = s->dims == 3 ? id / (s->p * s->p) : 0;
        const int64_t ndep = s->dims == 3 ? L : 1;
        for (int64_t ld = 0; ld < ndep; ld++)
            for (int64_t lr = 0; lr < L; lr++)
                for (int64_t lc = 0; lc < L; lc++) {
                    const int64_t gr = zm::local_row_to_global(m, rid, (int)lr);
                    const int64_t gc = zm::packed_col_to_global(m, cid, (int)lc);
                    const int64_t gd = s->dims == 3 ? zm::local_row_to_global(m, did, (int)ld) : 0;
                    const double v = (double)((gd * N + gr) * N + gc);
                    const int64_t at = (int64_t)id * d.local + (ld * L + lr) * L + lc;
                    host_grid[at * ncomp] = v;
                    if (ncomp == 2) host_grid[at * ncomp + 1] = 0.0;
                }
    }
    return ZM_OK;
}

const char* zm_strerror(zm_status s) {
    switch (s) {
        case ZM_OK: return "ok";
        case ZM_ERR_INVALID_ARG: return "invalid argument";
        case ZM_ERR_SHAPE: return "invalid shape: need P | N, B | N/P and P | N/(P*B)";
        case ZM_ERR_UNSUPPORTED: return "unsupported configuration";
        case ZM_ERR_DEVICE: return "HIP device or runtime error";
        case ZM_ERR_ALIAS: return "input and output buffers alias";
        case ZM_ERR_LAUNCH: return "kernel launch failed";
        case ZM_ERR_NOMEM: return "device allocation failed";
        case ZM_ERR_IO: return "file I/O failed";
        case ZM_ERR_SCRATCH_LIMIT: return "the plan needs more scratch than the static no-allocation buffer holds";
    }
    return "unknown status";
}

const char* zm_version(void) { return "stencilfft-amd 0.1.0 (gfx950)"; }

}  // extern "C"
