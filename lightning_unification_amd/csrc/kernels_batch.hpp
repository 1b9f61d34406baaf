// Batched forward + adjoint for layered ansatz circuits of uneven size.
//
// Circuit family (the hot path's batched and surrogate workloads, and the
// plain 20-qubit workload): `depth` layers, each = for every wire w, the
// rotations of `pattern` (e.g. RY then RZ) with their own angles, followed by
// a CNOT entangler (ladder i->i+1 or ring i->(i+1) mod n).  Observable: a
// Pauli sum per circuit.  Output: E = <psi|H|psi> and dE/dtheta for every
// angle, the quantities AdjointJacobianLQubit.hpp:212-336 returns for K = 1.
//
// Every launch covers all circuits that still have work at that step; block
// b finds its circuit by bisection in a per-launch prefix table.  Rotations
// run on register tiles (reg_tile.hpp): a tile holds 2^T amplitudes spanning T
// bit positions (the 3 lowest bits -- one 128-byte line -- plus up to W-3
// target bits), so one HBM pass applies the rotations of up to W wires.  The
// entangler is one GF(2)-linear gather (out[y] = in[src(y)], src bits are
// parities of y).  The adjoint holds tiles of lambda and H_lambda.
#pragma once

#include <hip/hip_runtime.h>
#include <stdint.h>

#include <type_traits>

#include "kernels_reduce.hpp"
#include "reg_tile.hpp"

namespace plamd {

constexpr int kBatchMaxQubits = 30;
constexpr int kBatchMaxPattern = 4;
constexpr int kBatchMaxTile = 13; // widest LDS tile (bits)

struct BCirc {
    int n;           // qubits
    int depth;       // layers
    int nstage;      // rotation stages per layer
    int ngroups;     // x-masks of the observable
    uint64_t off;    // amplitude offset of buffer 0 (buffers k at off + k * 2^n)
    uint32_t par;    // offset of this circuit's angles / gradients
    uint32_t group;  // offset of its groups
    uint32_t fwd_rows[kBatchMaxQubits]; // entangler gather:  src bit b = parity(y & fwd_rows[b])
    uint32_t adj_rows[kBatchMaxQubits]; // inverse entangler gather
};

struct BLaunch {
    const int *circ;        // active circuits of this launch
    const uint64_t *prefix; // exclusive block prefix (count + 1 entries)
    int count;
};

// The circuit of block b and the block's place in it: each wavefront narrows
// the prefix table 64-fold a load (bisection's ten dependent loads took longer
// than a small tile's rotations).
__device__ __forceinline__ int find_circ(const BLaunch &L, uint64_t b, uint64_t &local) {
    const int lane = threadIdx.x & 63;
    int lo = 0, n = L.count; // the largest c with prefix[c] <= b lies in [lo, lo + n)
    while (n > 1) {
        const int step = (n + 63) / 64, at = lane * step;
        const uint64_t below = __ballot(at < n && L.prefix[lo + (at < n ? at : 0)] <= b);
        const int k = __popcll(below) - 1; // prefix[lo] <= b always
        lo += k * step;
        n = n - k * step < step ? n - k * step : step;
    }
    lo = __builtin_amdgcn_readfirstlane(lo);
    local = b - L.prefix[lo];
    return L.circ[lo];
}

// Tile geometry of rotation stage s with tile width W: stage 0 spans bits
// [0, min(n, W)) and rotates all of them; stage s > 0 (only when n > W)
// rotates the target bits [alo, ahi) = [W + (s-1)(W-3), +W-3) clipped to n,
// inside a full W-bit tile: bits {0,1,2} (one 128-byte line, for coalescing)
// plus W-3 consecutive high bits ending no later than n, so the last stage's
// tile also holds some bits of the stage before it, left untouched.  Returns
// T, fills bits[] (ascending) and [alo, ahi).
__device__ __forceinline__ int stage_bits(int n, int W, int s, int *bits, int &alo, int &ahi) {
    if (s == 0) {
        const int T = n < W ? n : W;
        for (int k = 0; k < T; k++) {
            bits[k] = k;
        }
        alo = 0;
        ahi = T;
        return T;
    }
    alo = W + (s - 1) * (W - 3);
    ahi = alo + (W - 3) < n ? alo + (W - 3) : n;
    const int hlo = alo < n - (W - 3) ? alo : n - (W - 3);
    int T = 0;
    for (int k = 0; k < 3; k++) {
        bits[T++] = k;
    }
    for (int b = hlo; b < hlo + (W - 3); b++) {
        bits[T++] = b;
    }
    return T;
}

// The 2x2 of one wire's rotations in one layer.
struct BMat {
    dcx<double> u[4];
};

// Per (circuit, layer, wire), once per replay: (cos, sin) of every half angle
// and the product of the pattern's rotations, U = R_{npat-1} .. R_0 with
// R = exp(-i theta/2 sigma_axis) (LM.hpp:541-615), so the stages do no
// transcendental math and one 2x2 product per wire.
__global__ __launch_bounds__(kBlock) void k_batch_mats(const double *__restrict__ params, uint64_t nwires, int npat,
                                                      int4 pat, double2 *__restrict__ cs, BMat *__restrict__ mats) {
    const uint64_t i = static_cast<uint64_t>(blockIdx.x) * kBlock + threadIdx.x;
    if (i >= nwires) {
        return;
    }
    const int axes[4] = {pat.x, pat.y, pat.z, pat.w};
    BMat m;
    m.u[0] = m.u[3] = {1, 0};
    m.u[1] = m.u[2] = {0, 0};
    for (int a = 0; a < npat; a++) {
        double s, c;
        sincos(0.5 * params[i * npat + a], &s, &c);
        cs[i * npat + a] = double2{c, s};
        dcx<double> r[4] = {{c, 0}, {0, 0}, {0, 0}, {c, 0}};
        if (axes[a] == 0) {
            r[1] = r[2] = {0, -s};
        } else if (axes[a] == 1) {
            r[1] = {-s, 0};
            r[2] = {s, 0};
        } else {
            r[0].i = -s;
            r[3].i = s;
        }
        BMat p;
        for (int j = 0; j < 2; j++) {
            for (int k = 0; k < 2; k++) {
                const dcx<double> x = r[2 * j], y = m.u[k], u = r[2 * j + 1], v = m.u[2 + k];
                p.u[2 * j + k] = {x.r * y.r - x.i * y.i + u.r * v.r - u.i * v.i,
                                  x.r * y.i + x.i * y.r + u.r * v.i + u.i * v.r};
            }
        }
        m = p;
    }
    mats[i] = m;
}

// local tile index e -> global amplitude index.  Every stage's tile is bits
// {0, 1, 2} plus one contiguous run starting at bits[3] (stage 0: the run
// 3..T-1), so bits 0..2 of e stay in place and the rest shift to the run.
__device__ __forceinline__ uint64_t tile_index(uint64_t base, uint32_t e, const int *bits, int T) {
    const int hlo = T > 3 ? bits[3] : 3;
    return base | (e & 7U) | (static_cast<uint64_t>(e >> 3) << hlo);
}

// the tile's base: the block's local index spread over the non-tile bits
__device__ __forceinline__ uint64_t tile_base(uint64_t q, const int *bits, int T) {
    uint64_t g = q;
    for (int k = 0; k < T; k++) { // bits[] ascending: insert zeros in order
        const int p = bits[k];
        const uint64_t lo = g & ((uint64_t{1} << p) - 1);
        g = ((g >> p) << (p + 1)) | lo;
    }
    return g;
}

// source index of y under an entangler map: bit b = parity(y & rows[b])
__device__ __forceinline__ uint64_t gather_src(uint64_t y, const uint32_t *rows, int n) {
    uint64_t x = 0;
    for (int b = 0; b < n; b++) {
        x |= static_cast<uint64_t>(__popc(static_cast<uint32_t>(y) & rows[b]) & 1) << b;
    }
    return x;
}

// Entangler as a gather: dst[y] = src[src_index(y)] for the buffers given.
// adj = 0 forward map, 1 its inverse.  Up to two states per launch.
template <class T>
__global__ __launch_bounds__(kBlock) void k_batch_ring(v2<T> *__restrict__ arena,
                                                       const BCirc *__restrict__ circs,
                                                       const BLaunch L, int adj, int from0,
                                                       int to0, int from1, int to1) {
    uint64_t q;
    const BCirc &c = circs[find_circ(L, blockIdx.x, q)];
    const uint64_t len = uint64_t{1} << c.n;
    const uint64_t y = q * kBlock + threadIdx.x;
    if (y >= len) {
        return;
    }
    const uint64_t x = gather_src(y, adj ? c.adj_rows : c.fwd_rows, c.n);
    v2<T> *base = arena + c.off;
    base[to0 * len + y] = base[from0 * len + x];
    if (from1 >= 0) {
        base[to1 * len + y] = base[from1 * len + x];
    }
}

// |0...0> in buffer 0 of every circuit
template <class T>
__global__ __launch_bounds__(kBlock) void k_batch_init(v2<T> *__restrict__ arena,
                                                       const BCirc *__restrict__ circs,
                                                       const BLaunch L) {
    uint64_t q;
    const BCirc &c = circs[find_circ(L, blockIdx.x, q)];
    const uint64_t len = uint64_t{1} << c.n;
    const uint64_t y = q * kBlock + threadIdx.x;
    if (y < len) {
        v2<T> z;
        z.x = y == 0 ? T(1) : T(0);
        z.y = 0;
        arena[c.off + y] = z;
    }
}

// A term's coefficient with its (-i)^ny, and its Z/Y bits.
struct BTerm {
    double cr, ci;
    uint32_t zy, pad;
};
// The terms of one circuit that share an x-mask: terms [first, last).
struct BGroup {
    uint32_t x, first, last;
};

// H psi into buffer 2 + f, E += Re<psi|H psi> and N += <psi|psi> (FP64
// atomics per block), where psi sits in buffer f = depth mod 2 when layers
// end with an entangler (each one flips the buffer) and f = 0 otherwise.
// The amplitudes of four groups are loaded together (one at a time, a 20-qubit
// Ising sum was twenty dependent loads a thread), and a group's signed
// coefficients are added before its one complex product: 512 circuits, 3.07 ->
// 2.33 ms a replay; what is left are the L1 and L2 reads.
template <class T>
__global__ __launch_bounds__(kBlock) void k_batch_obs(v2<T> *__restrict__ arena,
                                                      const BCirc *__restrict__ circs,
                                                      const BLaunch L, int ent,
                                                      const BTerm *__restrict__ terms,
                                                      const BGroup *__restrict__ groups,
                                                      double *__restrict__ energy,
                                                      double *__restrict__ norm2) {
    uint64_t q;
    const int ci = find_circ(L, blockIdx.x, q);
    const BCirc &c = circs[ci];
    const uint64_t len = uint64_t{1} << c.n;
    const int pbuf = ent ? (c.depth & 1) : 0;
    const int hbuf = 2 + pbuf;
    const uint64_t y = q * kBlock + threadIdx.x;
    double e = 0, pn = 0;
    if (y < len) {
        const v2<T> *psi = arena + c.off + pbuf * len;
        const uint32_t yb = static_cast<uint32_t>(y);
        double hr = 0, hi = 0;
        for (int g0 = 0; g0 < c.ngroups; g0 += 4) {
            v2<T> a[4];
#pragma unroll
            for (int j = 0; j < 4; j++) {
                if (g0 + j < c.ngroups) {
                    a[j] = psi[yb ^ groups[c.group + g0 + j].x];
                }
            }
#pragma unroll
            for (int j = 0; j < 4; j++) {
                if (g0 + j < c.ngroups) {
                    const BGroup &g = groups[c.group + g0 + j];
                    double cr = 0, ci2 = 0;
                    for (uint32_t t = g.first; t < g.last; t++) {
                        const BTerm &tm = terms[t];
                        const bool minus = __popc(yb & tm.zy) & 1;
                        cr += minus ? -tm.cr : tm.cr;
                        ci2 += minus ? -tm.ci : tm.ci;
                    }
                    hr += cr * double(a[j].x) - ci2 * double(a[j].y);
                    hi += cr * double(a[j].y) + ci2 * double(a[j].x);
                }
            }
        }
        v2<T> hv;
        hv.x = T(hr);
        hv.y = T(hi);
        arena[c.off + hbuf * len + y] = hv;
        const v2<T> p = psi[y];
        e = double(p.x) * hr + double(p.y) * hi;
        pn = double(p.x) * double(p.x) + double(p.y) * double(p.y);
    }
    const double2 s = block_sum2(double2{e, pn});
    if (threadIdx.x == 0) {
        atomicAdd(energy + ci, s.x);
        atomicAdd(norm2 + ci, s.y);
    }
}

// One rotation stage of a layer over every circuit that has it: a tile of
// lambda (ADJ: and of H lambda) in registers, windows of three target bits
// from the highest down, each bit's 2x2 applied in registers.
//
// ADJ undoes the rotations.  The gradients of a wire's letters are linear
// forms of M_ab = sum conj(h_a) lambda_b on the states before any of them is
// undone: with W = U G U^dagger, U the letters after the one whose generator
// is G, W = x X + y Y + z Z and Im <H|G lambda> = z Im(M00 - M11) +
// x Im(M01 + M10) - y Re(M01 - M10).  So the three sums are accumulated in
// FP64 per wire and the wire is undone by one 2x2, whatever the pattern's
// length (scale -1/2 and the -2 of the reference's update cancel:
// dE/dtheta = Im <H|G lambda>, AdjointJacobianLQubit.hpp:70-75).
//
// gl >= 0: the entangler between this layer and the neighbouring one is fused
// in: at the layer's first stage in execution order (forward stage 0, adjoint
// stage nstage - 1) lambda and H are gathered from buffers gl and gh through
// the entangler's index map (forward) or its inverse and written to lb and hb.
// The map is linear over GF(2), so a source index is the exclusive or of the
// tile's, the thread's and the register's parts.
//
// A trip through LDS and a barrier per wire, as before, left the stages at 2.6
// (adjoint) and 3.3 TB/s; windows take a third of the trips.  complex64 states
// are rotated in double: a stage rounds an amplitude once.
// 512 circuits of 8-20 qubits complex128: 63.4 -> 32.3 ms a replay, the widest
// adjoint launch 1.67 ms -> 0.81 (3.8 TB/s, a large copy 4.35); one circuit of
// 16 qubits 485 -> 390 us.
template <class T, int NW, bool ADJ>
__global__ __launch_bounds__(64 * NW, NW == 16 || ADJ ? 4 : 8) void k_batch_stage(
    v2<T> *__restrict__ arena, const BCirc *__restrict__ circs, const BLaunch L, int W, int stage, int layer, int lb,
    int hb, int gl, int gh, int npat, int4 pat, const BMat *__restrict__ mats, const double2 *__restrict__ cs,
    double *__restrict__ grads) {
    constexpr int RB = 3, R = 1 << RB, S = ADJ ? 2 : 1;
    constexpr int TB = 6 + (NW == 16 ? 4 : NW == 8 ? 3 : NW == 4 ? 2 : NW == 2 ? 1 : 0);
    auto window_at = [](int p) { return static_cast<uint32_t>(p | (p + 1) << 4 | (p + 2) << 8); };
    constexpr uint32_t HOME = TB | (TB + 1) << 4 | (TB + 2) << 8;
    extern __shared__ unsigned char smem_raw[];
    __shared__ double wpart[ADJ ? NW : 1][ADJ ? kBatchMaxTile : 1][4];
    double *buf = reinterpret_cast<double *>(smem_raw);
    uint64_t q;
    const BCirc &c = circs[find_circ(L, blockIdx.x, q)];
    int bits[16];
    int alo, ahi;
    const uint32_t tid = threadIdx.x;
    const BMat *lm = mats + c.par / npat + static_cast<uint64_t>(layer) * c.n;
    // the layer's matrices and the circuit's index rows into the caches at
    // once: the scalar loads of each wire and row would meet memory one after
    // another (half of a small circuit's stage)
    if (tid < static_cast<uint32_t>(c.n)) {
        asm volatile("" ::"v"(*reinterpret_cast<const int *>(lm + tid)),
                     "v"((ADJ ? c.adj_rows : c.fwd_rows)[tid]));
    }
    const int Tn = stage_bits(c.n, W, stage, bits, alo, ahi);
    const uint32_t size = 1U << Tn;
    const uint64_t len = uint64_t{1} << c.n;
    v2<T> *st[2] = {arena + c.off + lb * len, arena + c.off + (ADJ ? hb : lb) * len};
    const uint64_t base = tile_base(q, bits, Tn);
    const uint64_t thread_at = tile_index(0, tid, bits, Tn);
    auto reg_at = [&](int r) { return tile_index(0, static_cast<uint32_t>(r) << TB, bits, Tn); };
    double2 x[S][R];
    const bool gather = gl >= 0 && stage == (ADJ ? c.nstage - 1 : 0);
    const uint32_t *rows = ADJ ? c.adj_rows : c.fwd_rows;
    const uint64_t from = gather ? gather_src(base, rows, c.n) ^ gather_src(thread_at, rows, c.n) : base | thread_at;
    const v2<T> *src[2] = {gather ? arena + c.off + gl * len : st[0], gather && ADJ ? arena + c.off + gh * len : st[1]};
    uint64_t reg_from[RB];
#pragma unroll
    for (int j = 0; j < RB; j++) {
        reg_from[j] = gather ? gather_src(reg_at(1 << j), rows, c.n) : reg_at(1 << j);
    }
#pragma unroll
    for (int r = 0; r < R; r++) {
        const uint64_t a = from ^ ((r & 1) ? reg_from[0] : 0) ^ ((r & 2) ? reg_from[1] : 0) ^ ((r & 4) ? reg_from[2] : 0);
        const bool in = ((static_cast<uint32_t>(r) << TB) | tid) < size;
#pragma unroll
        for (int i = 0; i < S; i++) {
            x[i][r] = double2{0, 0};
            if (in) {
                const v2<T> v = src[i][a];
                x[i][r] = double2{v.x, v.y};
            }
        }
    }
    // local positions of the target bits: [ka, kb)
    const int shift = stage == 0 ? 0 : bits[3] - 3;
    const int ka = alo - shift, kb = ahi - shift;
    const int lane = tid & 63, wave = tid >> 6;
    uint32_t win = HOME;
    for (int top = kb; top > ka;) { // target bits at and above `top` are done
        const int p = top >= 3 ? top - 3 : 0;
        if (window_at(p) != win) {
            rt_window<TB, RB, S, !ADJ>(x, buf, tid, win, window_at(p));
            win = window_at(p);
        }
        auto bit = [&](auto jt) {
            constexpr int J = decltype(jt)::value;
            const int k = p + J;
            if (k < ka || k >= top) {
                return;
            }
            const int b = k + shift;
            const BMat &mt = lm[c.n - 1 - b];
            dcx<double> u[4];
            if constexpr (ADJ) {
                u[0] = {mt.u[0].r, -mt.u[0].i};
                u[1] = {mt.u[2].r, -mt.u[2].i};
                u[2] = {mt.u[1].r, -mt.u[1].i};
                u[3] = {mt.u[3].r, -mt.u[3].i};
                double s0 = 0, s1 = 0, s2 = 0;
#pragma unroll
                for (int pr = 0; pr < R / 2; pr++) {
                    const int i0 = ((pr >> J) << (J + 1)) | (pr & ((1 << J) - 1)), i1 = i0 | (1 << J);
                    const double ax = x[0][i0].x, ay = x[0][i0].y, bx = x[0][i1].x, by = x[0][i1].y;
                    const double cx = x[S - 1][i0].x, cy = x[S - 1][i0].y, dx = x[S - 1][i1].x, dy = x[S - 1][i1].y;
                    s0 = rt_fma(cx, ay, rt_fma(-cy, ax, rt_fma(-dx, by, rt_fma(dy, bx, s0))));
                    s1 = rt_fma(cx, by, rt_fma(-cy, bx, rt_fma(dx, ay, rt_fma(-dy, ax, s1))));
                    s2 = rt_fma(cx, bx, rt_fma(cy, by, rt_fma(-dx, ax, rt_fma(-dy, ay, s2))));
                }
                const double t = rt_sum4(s0, s1, s2, 0.0);
                if ((lane & 15) == 0) {
                    wpart[wave][b - alo][rt_row(lane >> 4)] = t;
                }
            } else {
#pragma unroll
                for (int j = 0; j < 4; j++) {
                    u[j] = mt.u[j];
                }
            }
#pragma unroll
            for (int pr = 0; pr < R / 2; pr++) {
                const int i0 = ((pr >> J) << (J + 1)) | (pr & ((1 << J) - 1)), i1 = i0 | (1 << J);
#pragma unroll
                for (int i = 0; i < S; i++) {
                    rt_apply2(~uint64_t{0}, u, x[i][i0], x[i][i1]);
                }
            }
        };
        bit(std::integral_constant<int, 2>{});
        bit(std::integral_constant<int, 1>{});
        bit(std::integral_constant<int, 0>{});
        top = p > ka ? p : ka;
    }
    if (win != HOME) {
        rt_window<TB, RB, S, !ADJ>(x, buf, tid, win, HOME);
    }
#pragma unroll
    for (int r = 0; r < R; r++) {
        if (((static_cast<uint32_t>(r) << TB) | tid) < size) {
            const uint64_t a = base | thread_at | reg_at(r);
#pragma unroll
            for (int i = 0; i < S; i++) {
                st[i][a] = v2<T>{static_cast<T>(x[i][r].x), static_cast<T>(x[i][r].y)};
            }
        }
    }
    if constexpr (ADJ) {
        __syncthreads();
        const int axes[4] = {pat.x, pat.y, pat.z, pat.w};
        for (int t = tid; t < (ahi - alo) * npat; t += 64 * NW) {
            const int sl = t / npat, a = t - sl * npat;
            double s[3] = {0, 0, 0};
            for (int v = 0; v < NW; v++) {
#pragma unroll
                for (int j = 0; j < 3; j++) {
                    s[j] += wpart[v][sl][j];
                }
            }
            const uint64_t pidx = c.par + (static_cast<uint64_t>(layer) * c.n + (c.n - 1 - (alo + sl))) * npat;
            // W: the generator's axis turned by the letters after it
            double w[3] = {axes[a] == 0 ? 1.0 : 0.0, axes[a] == 1 ? 1.0 : 0.0, axes[a] == 2 ? 1.0 : 0.0};
            for (int l = a + 1; l < npat; l++) {
                const double2 h = cs[pidx + l];
                const double co = h.x * h.x - h.y * h.y, si = 2 * h.x * h.y;
                // right-handed about axis l: (e1, e2) the two following axes
                const double x0 = w[0], y0 = w[1], z0 = w[2];
                if (axes[l] == 0) {
                    w[1] = y0 * co - z0 * si;
                    w[2] = y0 * si + z0 * co;
                } else if (axes[l] == 1) {
                    w[2] = z0 * co - x0 * si;
                    w[0] = z0 * si + x0 * co;
                } else {
                    w[0] = x0 * co - y0 * si;
                    w[1] = x0 * si + y0 * co;
                }
            }
            atomicAdd(grads + pidx + a, w[2] * s[0] + (w[0] * s[1] - w[1] * s[2]));
        }
    }
}

// zero n doubles (graph-safe replacement for a memset)
__global__ __launch_bounds__(kBlock) void k_zero(double *__restrict__ p, uint64_t n) {
    const uint64_t i = static_cast<uint64_t>(blockIdx.x) * kBlock + threadIdx.x;
    if (i < n) {
        p[i] = 0;
    }
}

} // namespace plamd
