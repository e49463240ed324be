// spectral.hip -- the plans' tables, reciprocal-space multipliers, the
// device forms of the index maps and the natural <-> packed converters.
#include <type_traits>

#include "common.hpp"
#include "kernels.hpp"
#include "line_maps.hpp"
#include "maps.hpp"
#include "spectral_math.hpp"

namespace zm {

// exp(-2 pi i num / den), num / den dyadic: sincospi of the exact argument, in
// FP64; an FP32 table holds the correctly rounded value
template <typename T>
__device__ __forceinline__ Cx<T> root(double num, double den) {
    double s, c;
    sincospi(-2.0 * num / den, &s, &c);
    return Cx<T>{(T)c, (T)s};
}

// All tables of a plan in one launch (a kernel for each took plan creation from
// 19 to 25 us at 1024^2 FP64).  tw replaces the host std::exp loops of
// init_forward_twiddles (zmodel/transforms/fft.cu:37-54): the reference's L x L
// table holds W_N^(k l) for k = fr + id*VP, l = fc, and the kernels index this
// length-N table with (k l) mod N instead.
template <typename T>
__global__ void plan_tables_kernel(PlanTables<T> a) {
    int t = blockIdx.x * blockDim.x + threadIdx.x;
    if (t < a.n) {
        a.tw[t] = root<T>(t, a.n);
        return;
    }
    t -= a.n;
    if (a.line) {
        if (t < a.line_entries) {
            // [W_S^u | W_N^u, u < 64 | W_N^(64 u) | W_N^u]
            const int s = a.line_s, nb = a.n / 64 > 0 ? a.n / 64 : 1;
            a.line[t] = t < s             ? root<T>(t, s)
                        : t < s + 64      ? root<T>(t - s, a.n)
                        : t < s + 64 + nb ? root<T>(64.0 * (t - s - 64), a.n)
                                          : root<T>(t - s - 64 - nb, a.n);
            return;
        }
        t -= a.line_entries;
    }
    for (int i = 0; i < 2; i++) {
        if (!a.nat[i]) continue;
        const LineRadices& r = a.radices[i];
        if (t < r.entries) {
            int p = 1, lns = r.lr[0], e = t;  // radix pass p, 2^lns = NS, entry e of the pass
            while (e >= 1 << (lns + r.lr[p])) {
                e -= 1 << (lns + r.lr[p]);
                lns += r.lr[p++];
            }
            a.nat[i][t] = root<T>((e & ((1 << lns) - 1)) * (e >> lns), 1 << (lns + r.lr[p]));
            return;
        }
        t -= r.entries;
    }
    if (a.half_sin && t < a.n) a.half_sin[t] = sinpi((double)signed_wavenumber(t, a.n) * (1.0 / (double)a.n));
}

template <typename T>
hipError_t launch_plan_tables(const PlanTables<T>& a, hipStream_t stream) {
    int entries = a.n + (a.line ? a.line_entries : 0) + (a.half_sin ? a.n : 0);
    for (int i = 0; i < 2; i++)
        if (a.nat[i]) entries += a.radices[i].entries;
    const unsigned threads = 256;
    hipLaunchKernelGGL((plan_tables_kernel<T>), dim3((entries + threads - 1) / threads), dim3(threads), 0, stream, a);
    return hipGetLastError();
}

template hipError_t launch_plan_tables<float>(const PlanTables<float>&, hipStream_t);
template hipError_t launch_plan_tables<double>(const PlanTables<double>&, hipStream_t);

struct Coord {
    int did, rid, cid, ld, lr, lc;
};

__device__ __forceinline__ Coord decode_coord(const Geo& g, int64_t i) {
    Coord c;
    const int id = (int)(i / g.local);
    const int64_t rem = i - (int64_t)id * g.local;
    c.lc = (int)(rem & (g.l - 1));
    c.lr = (int)((rem >> g.ll) & (g.l - 1));
    c.ld = (g.dims == 3) ? (int)(rem >> (2 * g.ll)) : 0;
    c.cid = id & (g.p - 1);
    c.rid = (id >> g.lp) & (g.p - 1);
    c.did = (g.dims == 3) ? (id >> (2 * g.lp)) : 0;
    return c;
}

// Frequencies of element i of the reciprocal layout: 2D kx <- (cid, lr),
// ky <- (rid, lc) (zmodel/utils.h:265-268); 3D kc <- (cid, lr),
// kr <- (rid, ld), kd <- (did, lc) (utils.h:298-302).  Returns the linear
// index ky*N + kx / (kd*N + kr)*N + kc and the three signed wavenumbers.
__device__ __forceinline__ int64_t recip_freq(const Geo& g, const MapShape& ms, int64_t i, int* s0, int* s1,
                                              int* s2) {
    const Coord c = decode_coord(g, i);
    if (g.dims == 2) {
        const int kx = recip_to_freq(ms, c.cid, c.lr);
        const int ky = recip_to_freq(ms, c.rid, c.lc);
        *s0 = signed_wavenumber(kx, g.n);
        *s1 = signed_wavenumber(ky, g.n);
        *s2 = 0;
        return (int64_t)ky * g.n + kx;
    }
    const int kc = recip_to_freq(ms, c.cid, c.lr);
    const int kr = recip_to_freq(ms, c.rid, c.ld);
    const int kd = recip_to_freq(ms, c.did, c.lc);
    *s0 = signed_wavenumber(kc, g.n);
    *s1 = signed_wavenumber(kr, g.n);
    *s2 = signed_wavenumber(kd, g.n);
    return ((int64_t)kd * g.n + kr) * g.n + kc;
}

// Real-space linear index gr*N + gc / (gd*N + gr)*N + gc of element i of the
// packed layout (zmodel/utils.h:166-170, 192-197).
__device__ __forceinline__ int64_t real_linear(const Geo& g, const MapShape& ms, int64_t i) {
    const Coord c = decode_coord(g, i);
    const int gr = local_row_to_global(ms, c.rid, c.lr);
    const int gc = packed_col_to_global(ms, c.cid, c.lc);
    if (g.dims == 2) return (int64_t)gr * g.n + gc;
    const int gd = local_row_to_global(ms, c.did, c.ld);
    return ((int64_t)gd * g.n + gr) * g.n + gc;
}

// Symbol of the periodic 5-/7-point Laplacian (scaled by `lap`) plus, in 2D,
// the 4th-order x-derivative [1, -8, 0, 8, -1] / (12 delta) when delta != 0:
// for the mode exp(2 pi i k x / N), theta = 2 pi k / N,
//   Laplacian: lap * sum_d (2 cos theta_d - 2) = -4 lap sum_d sin^2(theta_d / 2)
//   dx4:       i (8 sin theta_x - sin 2 theta_x) / (6 delta)
// (the sin^2 form has no cancellation at small k).  kx is the packed-column
// (gc) wavenumber, the axis zm_dx4 differentiates.
__device__ __forceinline__ void stencil_symbol(const Geo& g, int s0, int s1, int s2, double lap, double delta,
                                               double* re, double* im) {
    const double inv_n = 1.0 / (double)g.n;
    double acc = 0.0;
    const int s[3] = {s0, s1, s2};
    for (int d = 0; d < g.dims; ++d) {
        const double h = sinpi((double)s[d] * inv_n);  // sin(theta_d / 2)
        acc += h * h;
    }
    *re = -4.0 * lap * acc;
    *im = 0.0;
    if (delta != 0.0) {
        const double t = 2.0 * (double)s0 * inv_n;  // theta_x / pi
        *im = (8.0 * sinpi(t) - sinpi(2.0 * t)) / (6.0 * delta);
    }
}

// kind: 0 Poisson -1/|k|^2 (k = 0 -> 0), 1 heat exp(-p0 |k|^2 p1), 2 constant
// p0, 3 stencil symbol (Laplacian scale p0, dx4 delta p1), 4 Poisson times the
// stencil symbol.  conj = 1 applies the complex conjugate multiplier (the
// adjoint); the multiplier is formed in FP64 for every storage precision.
template <typename T>
__global__ void __launch_bounds__(256) spectral_kernel(const Cx<T>* in, Cx<T>* out, Geo g, int kind, double p0,
                                                       double p1, double kscale, int conj, const double* factor) {
    const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= g.field) return;
    const MapShape ms = make_map_shape(g.n, g.p, g.b);
    int s0, s1, s2;
    recip_freq(g, ms, i, &s0, &s1, &s2);
    const double k2 = kscale * kscale * ((double)s0 * s0 + (double)s1 * s1 + (double)s2 * s2);
    const double poisson = (k2 == 0.0) ? 0.0 : -1.0 / k2;  // 1 / (-|k|^2), mean mode removed
    double mr, mi = 0.0;
    if (kind == 0) mr = poisson;
    else if (kind == 1) mr = exp(-p0 * k2 * p1);  // heat: exp(-nu |k|^2 dt)
    else if (kind == 2) mr = p0;
    else {
        stencil_symbol(g, s0, s1, s2, p0, p1, &mr, &mi);
        if (kind == 4) {
            mr *= poisson;
            mi *= poisson;
        }
    }
    if (conj) mi = -mi;
    if (factor) mr *= *factor, mi *= *factor;
    const int64_t at = (int64_t)blockIdx.y * g.field + i;
    const Cx<T> v = in[at];
    const double vx = (double)v.x, vy = (double)v.y;
    out[at] = Cx<T>{(T)(vx * mr - vy * mi), (T)(vx * mi + vy * mr)};
}

template <typename T>
hipError_t launch_spectral(const Cx<T>* in, Cx<T>* out, const Geo& g, int batch, int kind, double p0, double p1,
                           double kscale, bool conj, const double* factor, hipStream_t stream) {
    const unsigned threads = 256;
    const dim3 grid((unsigned)((g.field + threads - 1) / threads), (unsigned)batch);
    hipLaunchKernelGGL((spectral_kernel<T>), grid, dim3(threads), 0, stream, in, out, g, kind, p0, p1, kscale,
                       conj ? 1 : 0, factor);
    return hipGetLastError();
}

template hipError_t launch_spectral<float>(const float2*, float2*, const Geo&, int, int, double, double, double,
                                           bool, const double*, hipStream_t);
template hipError_t launch_spectral<double>(const double2*, double2*, const Geo&, int, int, double, double, double,
                                            bool, const double*, hipStream_t);

// r -= g and the FP64 partial sums of |r|^2, one per block in a fixed order
// (the sum does not depend on scheduling); norm_kernel adds them.  Memory-bound:
// two reads and a write of the field, where the difference, its square and the
// sum as separate passes read four times and write twice (8 x 4096^2 FP32: 1.16
// ms as three torch kernels).
template <typename T>
__global__ void __launch_bounds__(256) residual_kernel(Cx<T>* r, const Cx<T>* g, int64_t n, double* partials) {
    __shared__ double sums[256];
    const int64_t step = (int64_t)gridDim.x * 1024;
    double acc = 0.0;
    for (int64_t i0 = (int64_t)blockIdx.x * 1024 + threadIdx.x; i0 < n; i0 += step) {
        Cx<T> a[4], b[4];
#pragma unroll
        for (int k = 0; k < 4; k++) {
            const int64_t i = i0 + 256 * k < n ? i0 + 256 * k : i0;
            a[k] = ld_nt(r + i);
            b[k] = ld_nt(g + i);
        }
#pragma unroll
        for (int k = 0; k < 4; k++) {
            if (i0 + 256 * k >= n) break;
            const Cx<T> d = csub(a[k], b[k]);
            st_nt(r + i0 + 256 * k, d);
            acc += (double)d.x * (double)d.x + (double)d.y * (double)d.y;
        }
    }
    sums[threadIdx.x] = acc;
    __syncthreads();
    for (int w = 128; w > 0; w >>= 1) {
        if ((int)threadIdx.x < w) sums[threadIdx.x] += sums[threadIdx.x + w];
        __syncthreads();
    }
    if (threadIdx.x == 0) partials[blockIdx.x] = sums[0];
}

template <typename T>
__global__ void __launch_bounds__(256) norm_kernel(const double* partials, int n, T* norm2) {
    __shared__ double sums[256];
    double acc = 0.0;
    for (int i = threadIdx.x; i < n; i += 256) acc += partials[i];
    sums[threadIdx.x] = acc;
    __syncthreads();
    for (int w = 128; w > 0; w >>= 1) {
        if ((int)threadIdx.x < w) sums[threadIdx.x] += sums[threadIdx.x + w];
        __syncthreads();
    }
    if (threadIdx.x == 0) *norm2 = (T)sums[0];
}

template <typename T>
hipError_t launch_residual_norm(Cx<T>* r, const Cx<T>* g, int64_t n, double* partials, T* norm2, hipStream_t stream) {
    const int64_t want = (n + 1023) / 1024;
    const int blocks = (int)(want < kNormBlocks ? want : kNormBlocks);
    hipLaunchKernelGGL((residual_kernel<T>), dim3(blocks), dim3(256), 0, stream, r, g, n, partials);
    hipLaunchKernelGGL((norm_kernel<T>), dim3(1), dim3(256), 0, stream, partials, blocks, norm2);
    return hipGetLastError();
}

template hipError_t launch_residual_norm<float>(float2*, const float2*, int64_t, double*, float*, hipStream_t);
template hipError_t launch_residual_norm<double>(double2*, const double2*, int64_t, double*, double*, hipStream_t);

__global__ void __launch_bounds__(256) index_table_kernel(int64_t* out, Geo g, int reciprocal) {
    const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= g.field) return;
    const MapShape ms = make_map_shape(g.n, g.p, g.b);
    if (reciprocal) {
        int s0, s1, s2;
        out[i] = recip_freq(g, ms, i, &s0, &s1, &s2);
    } else {
        out[i] = real_linear(g, ms, i);
    }
}

hipError_t launch_index_table(int64_t* out, const Geo& g, bool reciprocal, hipStream_t stream) {
    const unsigned threads = 256;
    hipLaunchKernelGGL(index_table_kernel, dim3((unsigned)((g.field + threads - 1) / threads)), dim3(threads), 0,
                       stream, out, g, reciprocal ? 1 : 0);
    return hipGetLastError();
}

// natural (row-major N^d) <-> real-space packed layout: the composition of the
// block-cyclic distribution and vector_pack that init_host performs on the host
// (zmodel/utils.cu:9-36, utils.h:99-108).
//
// Of a row, column jj M + r (r = gm B + j) goes to packed column j VEC + jj of
// rank column gm: a VEC x M transpose.  A workgroup moves a tile of RC
// consecutive r by JC consecutive jj of one row, or of several rows where a row
// is smaller, through LDS, so that both sides move runs (of RC elements in
// natural order, of JC elements or more in the packed rows); one thread per
// element had read or written every VEC-th element per lane.  Both sides are
// permutations of the bits of one element index q, whose low `ltile` bits are
// the element of the tile: r, jj, rows.
// Memory-bound: tiles of 8 KB (two FP64 or four FP32 elements per thread; half of
// it in FP32 took 128 MB fields from 34 to 43 us, twice of it in FP64 512 MB from
// 175 to 185), in FP64 consecutive tiles on one XCD (768 MB 261 -> 250 us; not in
// FP32, 128 MB 43 -> 45), non-temporal stores (256 MB FP64 93 -> 62 us), but plain
// ones in FP64 for rank rows shorter than a cache line while the last-level cache
// holds input and output together: 128 MB of 16^3 with P = 4, B = 1, 50 -> 38 us
// (256 MB as fast either way; longer rows, 32 MB of 128^3 9.1 -> 11.0 us with plain
// stores, 128 MB within 5%).
// Loads: plain while the last-level cache can still hold the field (256 MB FP64
// 62 us, non-temporal 85), non-temporal beyond (512 MB FP64 181 -> 169, FP32 179
// -> 169, 384 MB FP32 135 -> 129).  Geometric means over the distributions, to /
// from packed, against one thread per element: FP32 128 MB 65 / 67 -> 34 / 35
// us, 1 GB 661 / 803 -> 344 / 333; FP64 128 MB 39 / 41 -> 32 / 32, 512 MB 224 /
// 262 -> 169 / 171 (6.3 TB/s), where the best of the former, whose runs were long
// enough, took 167.
// FULL: the field holds at least one tile (no guards).  NTL, NTS: non-temporal
// loads and stores.
template <typename T, int LE, bool FULL, bool NTL, bool NTS>
__global__ void __launch_bounds__(256) convert_kernel(const Cx<T>* __restrict__ in, Cx<T>* __restrict__ out,
                                                      ConvertArgs a, int to_packed) {
    using C = Cx<T>;
    constexpr int EPT = (1 << LE) / 256, NB = LE - 8;
    __shared__ C tile[(1 << LE) + (1 << (LE - 4)) + (1 << (LE - 8)) + 1];
    const int tid = threadIdx.x;
    auto pad = [](int i) { return i + (i >> 4) + (i >> 8); };  // distinct banks at every power-of-two stride
    const int64_t f = (int64_t)blockIdx.y << a.lfield;
    const int base = (int)(sizeof(T) == 8 ? xcd_block(blockIdx.x, gridDim.x) : blockIdx.x) << a.ltile;
    // every address is a part of this tile, of this thread and of register k,
    // the last the sum of its bits' offsets
    const int slot = bits(a.order, tid);
    const C* const nat_in = in + f + bits(a.nat, base) + bits(a.nat, tid);
    C* const nat_out = out + f + bits(a.nat, base) + bits(a.nat, tid);
    const C* const pk_in = in + f + bits(a.pk, base) + bits(a.pk, slot);
    C* const pk_out = out + f + bits(a.pk, base) + bits(a.pk, slot);
    int nat_bit[NB], pk_bit[NB], slot_bit[NB];
#pragma unroll
    for (int i = 0; i < NB; i++) {
        nat_bit[i] = bits(a.nat, 256 << i);
        slot_bit[i] = bits(a.order, 256 << i);
        pk_bit[i] = bits(a.pk, slot_bit[i]);
    }
    auto sum = [&](const int* bit, int k) {
        int o = 0;
#pragma unroll
        for (int i = 0; i < NB; i++) o += (k >> i) & 1 ? bit[i] : 0;
        return o;
    };
    auto ld = [](const C* p) -> C {
        if constexpr (NTL) return ld_nt(p);
        else return *p;
    };
    auto st = [](C* p, const C& v) {
        if constexpr (NTS) st_nt(p, v);
        else *p = v;
    };
    const int n = FULL ? EPT : tid >= (1 << a.ltile) ? 0 : a.ltile > 8 ? 1 << (a.ltile - 8) : 1;
    C v[EPT];
    if (to_packed) {
#pragma unroll
        for (int k = 0; k < EPT; k++) v[k] = k < n ? ld(nat_in + sum(nat_bit, k)) : C{0, 0};
#pragma unroll
        for (int k = 0; k < EPT; k++)
            if (k < n) tile[pad(tid + 256 * k)] = v[k];
        __syncthreads();
#pragma unroll
        for (int k = 0; k < EPT; k++)
            if (k < n) st(pk_out + sum(pk_bit, k), tile[pad(sum(slot_bit, k) + slot)]);
    } else {
#pragma unroll
        for (int k = 0; k < EPT; k++) v[k] = k < n ? ld(pk_in + sum(pk_bit, k)) : C{0, 0};
#pragma unroll
        for (int k = 0; k < EPT; k++)
            if (k < n) tile[pad(sum(slot_bit, k) + slot)] = v[k];
        __syncthreads();
#pragma unroll
        for (int k = 0; k < EPT; k++)
            if (k < n) st(nat_out + sum(nat_bit, k), tile[pad(tid + 256 * k)]);
    }
}

template <typename T>
hipError_t launch_natural_packed(const Cx<T>* in, Cx<T>* out, const Geo& g, int batch, bool to_packed,
                                 hipStream_t stream) {
    constexpr int LE = kConvertTile<T>;
    const ConvertArgs a = convert_args(g, LE);
    const dim3 grid((unsigned)(g.field >> a.ltile), (unsigned)batch);
    const int tp = to_packed ? 1 : 0;
    const int64_t bytes = (int64_t)batch * g.field * (int64_t)sizeof(Cx<T>);
    auto launch = [&](auto full, auto ntl, auto nts) {
        hipLaunchKernelGGL((convert_kernel<T, LE, full.value, ntl.value, nts.value>), grid, dim3(256), 0, stream, in,
                           out, a, tp);
    };
    constexpr std::true_type yes{};
    constexpr std::false_type no{};
    if (a.ltile < LE) launch(no, no, yes);
    else if (bytes > kLastLevelCache) launch(yes, yes, yes);
    else if (sizeof(T) == 4 || g.l >= 8 || 2 * bytes > kLastLevelCache) launch(yes, no, yes);
    else if constexpr (sizeof(T) == 8) launch(yes, no, no);
    return hipGetLastError();
}

template hipError_t launch_natural_packed<float>(const float2*, float2*, const Geo&, int, bool, hipStream_t);
template hipError_t launch_natural_packed<double>(const double2*, double2*, const Geo&, int, bool, hipStream_t);

}  // namespace zm
