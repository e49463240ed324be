// line_pass.hpp -- N-point line passes over natural-order lines, the kernels of
// line_pass_f32.hip / line_pass_f64.hip.
//
// One direction of the transform is an N-point DFT of every line.  The
// reference splits it as VEC-point transforms, a twiddle and M-point
// transforms (N = VEC * M, zmodel/transforms/fft.cu:207-264); here a line is
// transformed whole, by two to four radix passes of up to 16 points, and the
// block-cyclic layouts appear only as address maps of its two ends:
//   packed      real space, x = row of a rank slab: sample n = jj M + gm B + j
//               at packed column j VEC + jj of member rank gm (utils.h:122-128);
//   row         reciprocal: frequency k = k1 + VEC k2 at position
//               k1 % VP + k2 VP of member rank k1 / VP (fft.cu:162-181);
//   tile        the other axes before (forward) or after (inverse) the
//               repack-transpose (fft.cu:183-187, fft3d.cu:203-220): sample n
//               of line y is element y of local row jj B + j of member rank
//               gm.  A workgroup takes a tile of consecutive y, so that the
//               pass reads or writes runs of contiguous elements and the
//               repack's sweep of the field disappears.
// Every end is a permutation of index bits (N, P, B are powers of two), so an
// address is the sum of a per-thread part and a uniform part per register.
#pragma once

#include <type_traits>

#include "common.hpp"
#include "kernels.hpp"
#include "spectral_math.hpp"

namespace zm {
namespace lp {

// Ends of a pass.  PACKED goes through LDS (its runs in n are strided in
// memory); ROW and TILE are loaded and stored straight from the registers of
// the first and last radix pass, lanes along n (ROW) or along the lines (TILE).
// LAP2 / LAP3 (input): the 5- / 7-point Laplacian of a packed end.
enum End { PACKED = 0, ROW = 1, TILE = 2, LAP2 = 3, LAP3 = 4 };
enum Dir { FWD = 0, INV = 1, SPEC = 2 };
// How a workgroup runs over line groups: one group each (ONCE); a loop with the
// next group's loads in flight, for lines that leave a CU one workgroup (LOOP).
enum Mode { ONCE = 0, LOOP = 1 };

// The radix passes of a line of 2^LN points with 2^LEPT elements per thread: of
// at most 16 points, as even as possible, the larger ones first.
template <int LN, int LEPT>
struct Radices {
    static constexpr int LR = LEPT < 4 ? LEPT : 4;
    static constexpr int NP = (LN + LR - 1) / LR;
    static constexpr int lr(int p) { return LN / NP + (p < LN % NP ? 1 : 0); }
    static constexpr int lns(int p) { return p == 0 ? 0 : lns(p - 1) + lr(p - 1); }
    // twiddles of pass p >= 1: W_{NS R}^(jm r) at r NS + jm
    static constexpr int tw_off(int p) { return p <= 1 ? 0 : tw_off(p - 1) + (1 << (lns(p - 1) + lr(p - 1))); }
    static constexpr int TW = tw_off(NP);
    static constexpr LineRadices list() {
        LineRadices r{NP, TW, {}};
        for (int p = 0; p < NP; p++) r.lr[p] = lr(p);
        return r;
    }
};

// Lines of N = 2^LN points, LP = 2^LLP of them per workgroup, 2^LEPT elements
// per thread.
template <typename T, int LN, int LLP, int LEPT>
struct Line : Radices<LN, LEPT> {
    using C = Cx<T>;
    using Base = Radices<LN, LEPT>;
    using Base::lns, Base::lr, Base::NP, Base::TW, Base::tw_off;
    static constexpr int N = 1 << LN, LP = 1 << LLP, E = N * LP, EPT = 1 << LEPT, NT = E >> LEPT;
    static_assert(NP >= 2 && NT >= 64 && NT <= 1024, "split");

    // LDS index of element n of line l.  One padding element after every
    // 2^PS, 2^(2 PS), ..: the lanes of an LDS phase (16 of 8 bytes, 8 of 16)
    // then hit distinct banks at every power-of-two stride.  The line stride
    // spreads the lines of a tile over the banks the same way.
    static constexpr int SLOTS = sizeof(T) == 4 ? 16 : 8;
    static constexpr int PS = sizeof(T) == 4 || LN > 10 ? 4 : 3;
    static __host__ __device__ constexpr int pad(int i) {
        return i + (i >> PS) + (i >> (2 * PS)) + (PS * 3 < LN ? (i >> (3 * PS)) : 0);
    }
    static constexpr int line_stride() {
        const int want = SLOTS / LP > 1 ? SLOTS / LP : 1;
        int s = pad(N - 1) + 1;
        while (s % SLOTS != want % SLOTS) s++;
        return s;
    }
    static constexpr int LS = line_stride();
    static constexpr size_t lds_bytes() { return sizeof(C) * (size_t)(LP * LS); }

    // work item k of this thread in pass P: line l, butterfly j
    template <int P, bool TILED>
    static __device__ __forceinline__ void item(int tid, int k, int& l, int& j) {
        constexpr int LB = LN - lr(P);
        const int u = tid + k * NT;
        if constexpr (TILED) {
            l = u & (LP - 1);
            j = u >> LLP;
        } else {
            j = u & ((1 << LB) - 1);
            l = u >> LB;
        }
    }

    // Forward pass P (Stockham: Govindaraju et al., SC08; Van Loan 1992, sec.
    // 1.7): inputs j + r N/R, outputs (j - jm) R + jm + r NS, jm = j mod NS,
    // the twiddle before the butterfly.  The inverse runs the adjoint of each
    // pass in reverse order (inputs and outputs exchanged, the conjugate
    // twiddle after the butterfly), on the same tables.
    template <int P, bool F, bool TILED>
    static __device__ __forceinline__ void butterflies(C* v, const C* tw, int tid) {
        constexpr int R = 1 << lr(P), NS = 1 << lns(P);
        const C* t = tw + tw_off(P);
#pragma unroll
        for (int k = 0; k < EPT / R; k++) {
            int l, j;
            item<P, TILED>(tid, k, l, j);
            const int jm = j & (NS - 1);
            if constexpr (F && P > 0) {
#pragma unroll
                for (int r = 1; r < R; r++) v[k * R + r] = cmul(v[k * R + r], t[r * NS + jm]);
            }
            dft<R, F>(v + k * R);
            if constexpr (!F && P > 0) {
#pragma unroll
                for (int r = 1; r < R; r++) v[k * R + r] = cmulc(v[k * R + r], t[r * NS + jm]);
            }
        }
    }
    // the forward pass's inputs (IN) or outputs in LDS
    template <int P, bool IN, bool TILED>
    static __device__ __forceinline__ int lds_base(int tid, int k) {
        constexpr int R = 1 << lr(P), NS = 1 << lns(P);
        int l, j;
        item<P, TILED>(tid, k, l, j);
        if constexpr (IN) return l * LS + pad(j);
        const int jm = j & (NS - 1);
        return l * LS + pad((j - jm) * R + jm);
    }
    template <int P, bool IN, bool TILED>
    static __device__ __forceinline__ void read(const C* lds, C* v, int tid) {
        constexpr int R = 1 << lr(P), ST = IN ? N / R : 1 << lns(P);
#pragma unroll
        for (int k = 0; k < EPT / R; k++) {
            const C* b = lds + lds_base<P, IN, TILED>(tid, k);
#pragma unroll
            for (int r = 0; r < R; r++) v[k * R + r] = b[pad(r * ST)];
        }
    }
    template <int P, bool IN, bool TILED>
    static __device__ __forceinline__ void write(C* lds, const C* v, int tid) {
        constexpr int R = 1 << lr(P), ST = IN ? N / R : 1 << lns(P);
#pragma unroll
        for (int k = 0; k < EPT / R; k++) {
            C* b = lds + lds_base<P, IN, TILED>(tid, k);
#pragma unroll
            for (int r = 0; r < R; r++) b[pad(r * ST)] = v[k * R + r];
        }
    }
};

template <int I>
using IC = std::integral_constant<int, I>;

// One pass over every line group.  SPEC transforms forward, multiplies by a
// spectral multiplier along the line's axis (the last of the transform) and
// transforms back: both transforms and the multiplier in one sweep.
//
// `tables` holds the twiddles of passes 1, 2, .. one after the other
// (Line::tw_off), read from there: the caches keep them, and the lanes read
// consecutive entries.  A copy in LDS for looping workgroups lost: 2048^2 FP64, P =
// 1 .. 8, one field forward 60-64 against 55-59 us, eight 450-480 against 443-478.
template <typename T, int LN, int LLP, int LEPT, int IN, int OUT, int DIR, int MODE>
__global__ void __launch_bounds__(1 << (LN + LLP - LEPT), (LN + LLP - LEPT) <= 9 ? 2 : 1)
    line_pass_kernel(const Cx<T>* in, Cx<T>* out, LinePassArgs a, const Cx<T>* __restrict__ tables, T scale,
                     SpectralArgs sp) {
    using C = Cx<T>;
    using K = Line<T, LN, LLP, LEPT>;
    constexpr int EPT = K::EPT, NT = K::NT, NP = K::NP, N = K::N;
    constexpr bool F = DIR != INV;
    // the pass whose registers the input arrives in, and the one that stores
    constexpr int PIN = F ? 0 : NP - 1, POUT = DIR == FWD ? NP - 1 : 0;
    constexpr int RIN = 1 << K::lr(PIN), ROUT = 1 << K::lr(POUT);
    constexpr bool TIN = IN == TILE, TOUT = OUT == TILE, LAP = IN == LAP2 || IN == LAP3;
    constexpr bool PIN_LDS = IN == PACKED || LAP;  // the input is staged through LDS
    static_assert(!LAP || (DIR == FWD && MODE == ONCE), "the Laplacian runs ahead of forward passes");
    extern __shared__ unsigned char smem_raw[];
    C* const lds = reinterpret_cast<C*>(smem_raw);
    int tid = threadIdx.x;

    auto group_base = [&](const auto& m, int g) -> int64_t {
        const int f = g >> a.lgroups;
        return (int64_t)f * a.field + bits(m, (g & ((1 << a.lgroups) - 1)) << LLP);
    };
    // offset of memory-order element e of the group (PACKED ends): line e / N,
    // element e % N of its P rank rows
    auto packed_off = [&](const auto& ml, const BitMap<3>& mn, int e) -> int {
        return bits(ml, e >> LN) + bits(mn, e & (N - 1));
    };
    auto packed_lds = [&](int e) -> int { return (e >> LN) * K::LS + K::pad(bits(a.pk, e & (N - 1))); };

    // a multiplier pass writes where it reads; a Laplacian's lines are global
    // rows, in their order
    const auto& in_l = [&]() -> const auto& {
        if constexpr (LAP) return a.rows;
        else return a.in_l;
    }();
    const auto& out_l = [&]() -> const auto& {
        if constexpr (LAP) return a.rows;
        else if constexpr (DIR == SPEC) return a.in_l;
        else return a.out_l;
    }();
    const BitMap<3>& out_n = DIR == SPEC ? a.in_n : a.out_n;
    // An address is a per-thread part plus a uniform one per register, the sum
    // of the offsets of the register number's bits: radix index r (ROW, TILE)
    // or memory-order sweep k (PACKED).
    constexpr int NB = PIN_LDS || OUT == PACKED ? LEPT : K::LR;
    int in_bit[NB], out_bit[NB], lds_bit[NB];
#pragma unroll
    for (int i = 0; i < NB; i++) {
        in_bit[i] = PIN_LDS ? packed_off(in_l, a.in_n, NT << i) : bits(a.in_n, (N / RIN) << i);
        out_bit[i] = OUT == PACKED ? packed_off(out_l, out_n, NT << i) : bits(out_n, (N / ROUT) << i);
        lds_bit[i] = packed_lds(NT << i);
    }
    const int in_thread = packed_off(in_l, a.in_n, tid), out_thread = packed_off(out_l, out_n, tid),
              lds_thread = packed_lds(tid);  // PACKED
    auto uniform_off = [&](const int* bit, int r) -> int {
        int o = 0;
#pragma unroll
        for (int i = 0; i < NB; i++) o += (r >> i) & 1 ? bit[i] : 0;
        return o;
    };

    // the next group's input registers: slot k R + r is element j + r N / R of
    // line l (ROW, TILE), or memory-order element tid + k NT (PACKED)
    C pre[EPT];
    auto fetch = [&](int g, auto k0c, auto k1c) __attribute__((always_inline)) {
        constexpr int K0 = decltype(k0c)::value, K1 = decltype(k1c)::value;
        const C* gb = in + group_base(in_l, g);
        if constexpr (LAP) {
            // rows and planes that other groups read too: plain loads
#pragma unroll
            for (int k = K0; k < K1; k++) pre[k] = gb[uniform_off(in_bit, k) + in_thread];
        } else if constexpr (IN == PACKED) {
#pragma unroll
            for (int k = K0; k < K1; k++)
                pre[k] = ld_nt(gb + uniform_off(in_bit, k) + in_thread);
        } else {
#pragma unroll
            for (int k = K0; k < K1; k++) {
                int l, j;
                K::template item<PIN, TIN>(tid, k / RIN, l, j);
                const C* p = gb + uniform_off(in_bit, k % RIN);
                pre[k] = ld_nt(p + (bits(in_l, l) + bits(a.in_n, j)));
            }
        }
    };
    auto store = [&](int g, const C* v) __attribute__((always_inline)) {
        C* gb = out + group_base(out_l, g);
#pragma unroll
        for (int k = 0; k < EPT; k++) {
            C x = v[k];
            if constexpr (DIR != FWD) x = C{x.x * scale, x.y * scale};
            if constexpr (OUT == PACKED) {
                st_nt(gb + uniform_off(out_bit, k) + out_thread, x);
            } else {
                int l, j;
                K::template item<POUT, TOUT>(tid, k / ROUT, l, j);
                C* p = gb + uniform_off(out_bit, k % ROUT);
                st_nt(p + (bits(out_l, l) + bits(out_n, j)), x);
            }
        }
    };

    // LAP: pre[] becomes `scale` times its Laplacian.  The rows above and below
    // (and the planes before and after) are loaded beside it, mostly from the
    // caches: the groups run in global row order.  The x neighbours come from
    // the raw rows in LDS, where they are samples n -+ 1.  Operations and their
    // order are the stencil kernels' (stencil.hip, lap_combine): bit for bit
    // zm_laplace.  The field is read and written once instead of twice: forward
    // chain of three 2048^2 FP64 fields, P = 8, 255 -> 183 us, 256^3 FP64 P = 4
    // 400 -> 318, 1024^2 FP64 25 -> 22, 64^2 8.6 -> 7.6.
    auto laplacian = [&](int g) __attribute__((always_inline)) {
#pragma clang fp contract(off)
        const int lam0 = (g & ((1 << a.lgroups) - 1)) << LLP;
        const C* const fb = in + (int64_t)(g >> a.lgroups) * a.field;
        const int in_row = bits(a.in_n, tid & (N - 1));
        // memory-order element k of the line `rows` down and `planes` on
        auto neighbour = [&](int k, int rows, int planes) -> C {
            const int gl = lam0 + (tid >> LN) + ((k * NT) >> LN);  // uniform where NT <= N
            int to = (gl & ~(N - 1)) | ((gl + rows) & (N - 1));
            if constexpr (IN == LAP3) to = (to + planes * N) & (N * N - 1);
            return fb[bits(a.rows, to) + bits(a.in_n, (k * NT) & (N - 1)) + in_row];
        };
        C y0[EPT], y1[EPT];
#pragma unroll
        for (int k = 0; k < EPT; k++) {
            y0[k] = neighbour(k, -1, 0);
            y1[k] = neighbour(k, 1, 0);
        }
        C z0[IN == LAP3 ? EPT : 1], z1[IN == LAP3 ? EPT : 1];
        if constexpr (IN == LAP3) {
#pragma unroll
            for (int k = 0; k < EPT; k++) {
                z0[k] = neighbour(k, 0, -1);
                z1[k] = neighbour(k, 0, 1);
            }
        }
#pragma unroll
        for (int k = 0; k < EPT; k++) lds[uniform_off(lds_bit, k) + lds_thread] = pre[k];
        __syncthreads();
#pragma unroll
        for (int k = 0; k < EPT; k++) {
            const int e = tid + k * NT, n = bits(a.pk, e & (N - 1));
            const C* const row = lds + (e >> LN) * K::LS;
            const C l = row[K::pad((n - 1) & (N - 1))], r = row[K::pad((n + 1) & (N - 1))], c = pre[k];
            C s;
            if constexpr (sizeof(T) == 8) {
                s = cadd(C{0, 0}, y0[k]);
                s = cadd(cadd(cadd(s, y1[k]), l), r);
                constexpr T centre = IN == LAP3 ? 6 : 4;
                if constexpr (IN == LAP3) s = cadd(cadd(s, z0[k]), z1[k]);
                s = csub(s, C{c.x * centre, c.y * centre});
            } else {
                s = cadd(cadd(csub(y0[k], c), csub(y1[k], c)), cadd(csub(l, c), csub(r, c)));
                if constexpr (IN == LAP3) s = cadd(s, cadd(csub(z0[k], c), csub(z1[k], c)));
            }
            pre[k] = C{s.x * scale, s.y * scale};
        }
        __syncthreads();  // the raw rows are overwritten
    };

    int g = a.xcd ? (int)xcd_block(blockIdx.x, gridDim.x) : (int)blockIdx.x;
    if (g < a.groups) fetch(g, IC<0>{}, IC<EPT>{});
    // keeps the first loads' addresses apart from what follows: without it the
    // one-line Laplacian passes spill 4 to 8 scalar registers
    __syncthreads();
    // exchanges through LDS in one group, each a point to issue a slice of
    // the next group's loads at
    constexpr int HIN = PIN_LDS ? 1 : 0;
    constexpr int HOOKS = (DIR == SPEC ? 2 : 1) * (NP - 1) + HIN + (OUT == PACKED ? 1 : 0);
    // Addresses and a multiplier's frequencies are the same for every group,
    // and the compiler would keep them all live across the loop (spills at 256
    // VGPRs, or of scalar registers): an opaque tid, and opaque bit offsets for
    // the uniform parts, have them recomputed per group.
    constexpr bool OPAQUE = DIR == SPEC;
    while (g < a.groups) {
        if constexpr (OPAQUE) asm volatile("" : "+v"(tid));
        if constexpr (MODE != ONCE) {
#pragma unroll
            for (int i = 0; i < NB; i++) {
                asm volatile("" : "+s"(in_bit[i]), "+s"(out_bit[i]));
                if constexpr (PIN_LDS || OUT == PACKED) asm volatile("" : "+s"(lds_bit[i]));
            }
        }
        const int nxt = g + (int)gridDim.x;
        auto hook = [&](auto hc) __attribute__((always_inline)) {
            constexpr int h = decltype(hc)::value;
            constexpr int K0 = h * EPT / HOOKS, K1 = (h + 1) * EPT / HOOKS;
            if constexpr (K1 > K0 && MODE != ONCE) {
                if (nxt < a.groups) fetch(nxt, IC<K0>{}, IC<K1>{});
            }
        };
        C v[EPT];
        if constexpr (LAP) laplacian(g);
        if constexpr (PIN_LDS) {
#pragma unroll
            for (int k = 0; k < EPT; k++) lds[uniform_off(lds_bit, k) + lds_thread] = pre[k];
            hook(IC<0>{});
            __syncthreads();
            K::template read<0, true, false>(lds, v, tid);
        } else {
#pragma unroll
            for (int k = 0; k < EPT; k++) v[k] = pre[k];
        }
        if constexpr (F) {
            auto fwd = [&](auto self, auto pc) __attribute__((always_inline)) -> void {
                constexpr int P = decltype(pc)::value;
                constexpr bool TL = P == 0 && TIN;
                K::template butterflies<P, true, TL>(v, tables, tid);
                if constexpr (P + 1 < NP) {
                    // the previous reads of LDS: this group's, or those
                    // before the barrier that ended the last group
                    if constexpr (P > 0 || PIN_LDS) __syncthreads();
                    K::template write<P, false, TL>(lds, v, tid);
                    hook(IC<HIN + P>{});
                    __syncthreads();
                    K::template read<P + 1, true, false>(lds, v, tid);
                    self(self, IC<P + 1>{});
                }
            };
            fwd(fwd, IC<0>{});
        }
        if constexpr (DIR == SPEC) {
            // v holds frequencies j + r N / R of the last pass's items.  They
            // go through this thread's own LDS slots (those it read last, so
            // without a barrier) for a rolled loop: unrolled over registers,
            // the FP64 multipliers' temporaries and constants spill.
            constexpr int R = 1 << K::lr(NP - 1);
            const int lam0 = (g & ((1 << a.lgroups) - 1)) << LLP;
            K::template write<NP - 1, true, false>(lds, v, tid);
            const double factor = sp.factor ? *sp.factor : 1.0;
            auto multiply = [&](auto fc) __attribute__((always_inline)) {
                constexpr int FAMILY = decltype(fc)::value;
#pragma unroll 1
                for (int k = 0; k < EPT / R; k++) {
                    int l, j;
                    K::template item<NP - 1, false>(tid, k, l, j);
                    int lam = lam0 + l;
                    asm volatile("" : "+v"(lam));  // uniform for one-line groups: scalar registers are short
                    // packed ends: 2D, N >= 4096
                    const LineSymbol ls = line_symbol<FAMILY, IN == PACKED>(sp, bits(sp.f0, lam), bits(sp.f1, lam), N);
                    // In the rolled loop each of a stencil's sines is waited
                    // for by itself.  The one-line groups have the registers
                    // to load a butterfly's R ahead and unroll (the whole
                    // solve, Poisson times stencil: 4096^2 FP32, eight fields
                    // 2.21 -> 2.11 ms, FP64, two fields 1.13 -> 1.08, 8192^2
                    // FP32 1.12 -> 1.09; the kernel 763 -> 687 us for 2.15 GB
                    // at the first); the tiled forms do not (4 to 10
                    // spilled scalar registers from 4 sines on), and gained
                    // nothing (256^3 FP32, four fields 1.07 ms either way).
                    constexpr int AHEAD = FAMILY == SF_STENCIL && IN == PACKED ? R : 1;
                    double hs[AHEAD] = {};
                    if constexpr (AHEAD > 1) {
#pragma unroll
                        for (int i = 0; i < AHEAD; i++) hs[i] = sp.half_sin[j + i * (N / R)];
                    }
#pragma unroll 1
                    for (int r = 0; r < R; r += AHEAD) {
                        if constexpr (FAMILY == SF_STENCIL && AHEAD == 1) hs[0] = sp.half_sin[j + r * (N / R)];
#pragma unroll
                        for (int i = 0; i < AHEAD; i++) {
                            const int f = j + (r + i) * (N / R);
                            C* p = lds + l * K::LS + K::pad(f);
                            double mr, mi;
                            line_multiplier<FAMILY>(sp, ls, f, N, hs[i], &mr, &mi);
                            mr *= factor, mi *= factor;
                            const double vx = (double)p->x, vy = (double)p->y;
                            *p = C{(T)(vx * mr - vy * mi), (T)(vx * mi + vy * mr)};
                        }
                    }
                }
            };
            if (sp.kind == 1) multiply(IC<SF_HEAT>{});
            else if (sp.kind >= 3) multiply(IC<SF_STENCIL>{});
            else multiply(IC<SF_PLAIN>{});
            K::template read<NP - 1, true, false>(lds, v, tid);
        }
        if constexpr (DIR != FWD) {
            constexpr int HB = HIN + (DIR == SPEC ? NP - 1 : 0);
            auto inv = [&](auto self, auto pc) __attribute__((always_inline)) -> void {
                constexpr int P = decltype(pc)::value;
                constexpr bool TL = P == 0 && TOUT;
                K::template butterflies<P, false, TL>(v, tables, tid);
                if constexpr (P > 0) {
                    // SPEC: the last forward pass read exactly the elements
                    // this thread now writes
                    if constexpr (P < NP - 1) __syncthreads();
                    K::template write<P, true, false>(lds, v, tid);
                    hook(IC<HB + NP - 1 - P>{});
                    __syncthreads();
                    K::template read<P - 1, false, P - 1 == 0 && TOUT>(lds, v, tid);
                    self(self, IC<P - 1>{});
                }
            };
            inv(inv, IC<NP - 1>{});
        }
        if constexpr (OUT == PACKED) {
            __syncthreads();
            K::template write<0, true, false>(lds, v, tid);
            hook(IC<HOOKS - 1>{});
            __syncthreads();
#pragma unroll
            for (int k = 0; k < EPT; k++) v[k] = lds[uniform_off(lds_bit, k) + lds_thread];
        }
        store(g, v);
        if constexpr (MODE == ONCE) break;
        __syncthreads();  // the next group's writes overwrite LDS
        g = nxt;
    }
}

}  // namespace lp
}  // namespace zm
