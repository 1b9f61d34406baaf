// The backward sweep of the adjoint Jacobian (AdjointJacobianLQubit.hpp:282-329)
// and of the vector-Jacobian product (VectorJacobianProduct.hpp:77-155) in tile
// passes.
//
// Per operation, in reverse, the sweep needs <H_k|G lambda> of a trainable
// operation's generator G, then undoes the operation on lambda and every H_k.
// A launch per operation moves (1 + K) states for a few FMAs an amplitude:
// 60 us a step with 10 observables at 20 qubits, all of it cache and HBM
// traffic.  Here a workgroup of NW wavefronts holds a tile of lambda and of KH
// of the H_k (all combinations of the pass's bits) in registers and runs every
// step of the pass on it, so a pass moves each state once however many steps
// it has.  A thread's 2^RB amplitudes differ in the window bits; a step mixes
// one window bit, with compile-time register indexes, and a change of window
// goes through LDS, one state at a time through one buffer.  A step per trip
// through LDS instead (amplitudes kept there) was bound by LDS latency and
// address arithmetic: 5 us a step for six resident wavefronts.
// 20 qubits, 600 parameters, 20 observables: 8 passes of 0.64 ms, 5.1 ms for
// the Jacobian against 84 ms; bound by FP64 issue (about 2.5 ms of multiply-adds
// at full rate, window changes, wavefront reductions) and by the states'
// traffic (0.16 ms a pass).
//
// Steps (sweep.hpp) hold runs of operations with one geometry.  A run of 2x2
// operations is one step: every <H|G_j lambda_j> inside it is a linear form of
// the transition matrix M_ab = sum conj(h_a) lambda_b at the run's start, whose
// needed parts are accumulated, in FP64, while the run's product matrix is
// applied.
#pragma once

#include <hip/hip_runtime.h>
#include <stdint.h>

#include "kernels_reduce.hpp"
#include "reg_tile.hpp"
#include "sweep_launch.hpp"

namespace plamd {

// Workgroups are numbered (tile walker w, observable group grp), groups of one
// walker on one XCD where the grid allows it, since they read the same lambda
// tiles.  Group grp takes KH observables.  The group numbered `writer` writes
// lambda to lam_out (which may be lam_in when no other group reads it).
// partial[(((slot0 + slot) * NC + c) * pk + k - pk0) * W + w], W walkers.
template <class T, int NW, int KH, bool FULL>
__global__ __launch_bounds__(64 * NW, 4) void k_sweep(const SweepArgs<T> A, const SweepStep *__restrict__ prog) {
    constexpr int NC = FULL ? kSweepFull : kSweepReal;
    constexpr int RB = kSweepRegBits, R = 1 << RB;
    static_assert(RB == 3, "the steps' switches name three register bits");
    constexpr int TB = 6 + (NW == 4 ? 2 : NW == 2 ? 1 : 0); // thread bits
    constexpr int S = 1 + KH;                               // states: lambda, then the H_k
    constexpr uint32_t HOME = [] { // window at a tile's load and store: the highest local bits
        uint32_t v = 0;
        for (int j = 0; j < RB; j++) {
            v |= static_cast<uint32_t>(TB + j) << (4 * j);
        }
        return v;
    }();
    extern __shared__ unsigned char smem_raw[];
    double *tile = reinterpret_cast<double *>(smem_raw);
    constexpr uint32_t IM = 1U << (TB + RB);
    double *sums = reinterpret_cast<double *>(tile + 2 * IM); // [wave][slot][KH][NC]
    const uint32_t tid = threadIdx.x;
    const int lane = tid & 63, wave = tid >> 6;
    int w, grp;
    if (A.W & 7) {
        grp = static_cast<int>(blockIdx.x) % A.ngrp;
        w = static_cast<int>(blockIdx.x) / A.ngrp;
    } else {
        const int xcd = blockIdx.x & 7, y = blockIdx.x >> 3;
        grp = y % A.ngrp;
        w = (y / A.ngrp) * 8 + xcd;
    }
    grp += A.grp0;
    const int k0 = grp * KH, nk = A.K - k0 < KH ? A.K - k0 : KH;
    v2<T> *h[KH];
#pragma unroll
    for (int kk = 0; kk < KH; kk++) {
        h[kk] = A.hs[k0 + (kk < nk ? kk : 0)];
    }
    // the program into the caches at once: a step's scalar loads would each
    // meet memory otherwise, one after another
    for (uint32_t o = tid * 64; o < A.nsteps * sizeof(SweepStep); o += 64 * NW * 64) {
        asm volatile("" ::"v"(*reinterpret_cast<const int *>(reinterpret_cast<const char *>(prog) + o)));
    }
    const int nsum = A.nslots * KH * NC;
    double *mine = sums + wave * nsum;
    for (int i = lane; i < nsum; i += 64) {
        mine[i] = 0;
    }
    const SweepGeom &geo = A.geo;
    auto spread = [&](uint32_t e) { // local index -> bits of the state index
        uint64_t g = e & ((1U << geo.low) - 1);
        for (int b = geo.low; b < geo.bits; b++) {
            g |= static_cast<uint64_t>((e >> b) & 1U) << geo.hb[b - geo.low];
        }
        return g;
    };
    const uint32_t size = 1U << geo.bits; // a state smaller than the tile leaves the rest zero
    const uint64_t thread_at = spread(tid);
    double2 x[S][R];
    for (uint64_t q = w; q < A.ntiles; q += A.W) {
        uint64_t base = q << geo.low;
        for (int b = 0; b < geo.bits - geo.low; b++) {
            const int p = geo.hb[b];
            base = ((base >> p) << (p + 1)) | (base & ((uint64_t{1} << p) - 1));
        }
#pragma unroll
        for (int r = 0; r < R; r++) {
            const uint32_t e = (static_cast<uint32_t>(r) << TB) | tid;
            const uint64_t a = base | thread_at | spread(static_cast<uint32_t>(r) << TB);
#pragma unroll
            for (int i = 0; i < S; i++) {
                x[i][r] = double2{0, 0};
                if (e < size && (i == 0 || i - 1 < nk)) {
                    const v2<T> v = (i == 0 ? A.lam_in : h[i ? i - 1 : 0])[a];
                    x[i][r] = double2{v.x, v.y};
                }
            }
        }
        uint32_t win = HOME;
        auto window = [&](uint32_t to) {
            rt_window<TB, RB>(x, tile, tid, win, to);
            win = to;
        };
        for (int s = 0; s < A.nsteps; s++) {
            const SweepStep &st = prog[s];
            const int kind = st.kind;
            if (kind == kSweepWindow) {
                window(st.rp);
                continue;
            }
            if ((base & st.omask) != st.oval) {
                continue;
            }
            const int slot = st.slot;
            const bool on = (tid & st.lm) == st.lv;
            const uint64_t lanes = __ballot(on);
            const uint32_t rm = st.rm, rv = st.rv;
            const uint32_t rp = st.rp;
            const uint32_t tpar = (__popc(tid & st.lp) + __popcll(base & st.op)) & 1U; // kSweepDiag
            // the sums first, reading only, then the update: together, the
            // old and the new amplitudes would be live at once
            if (slot >= 0) {
                double acc[KH][NC];
#pragma unroll
                for (int kk = 0; kk < KH; kk++) {
#pragma unroll
                    for (int c = 0; c < NC; c++) {
                        acc[kk][c] = 0;
                    }
                }
                auto pairs = [&](auto jt) {
                    constexpr int J = decltype(jt)::value;
#pragma unroll
                    for (int p = 0; p < R / 2; p++) {
                        const int i0 = ((p >> J) << (J + 1)) | (p & ((1 << J) - 1)), i1 = i0 | (1 << J);
                        if ((static_cast<uint32_t>(i0) & rm) != rv) {
                            continue;
                        }
                        const double ax = x[0][i0].x, ay = x[0][i0].y, bx = x[0][i1].x, by = x[0][i1].y;
#pragma unroll
                        for (int kk = 0; kk < KH; kk++) {
                            const double cx = x[1 + kk][i0].x, cy = x[1 + kk][i0].y, dx = x[1 + kk][i1].x,
                                         dy = x[1 + kk][i1].y;
                            double *t = acc[kk];
                            t[0] = rt_fma(cx, ay, rt_fma(-cy, ax, t[0]));
                            t[1] = rt_fma(dx, by, rt_fma(-dy, bx, t[1]));
                            t[2] = rt_fma(cx, by, rt_fma(-cy, bx, rt_fma(dx, ay, rt_fma(-dy, ax, t[2]))));
                            t[3] = rt_fma(cx, bx, rt_fma(cy, by, rt_fma(-dx, ax, rt_fma(-dy, ay, t[3]))));
                            if constexpr (FULL) {
                                t[4] = rt_fma(cx, ax, rt_fma(cy, ay, t[4]));
                                t[5] = rt_fma(dx, bx, rt_fma(dy, by, t[5]));
                                t[6] = rt_fma(cx, bx, rt_fma(cy, by, rt_fma(dx, ax, rt_fma(dy, ay, t[6]))));
                                t[7] = rt_fma(cx, by, rt_fma(-cy, bx, rt_fma(-dx, ay, rt_fma(dy, ax, t[7]))));
                            }
                        }
                    }
                };
                if (kind == kSweepDiag) { // even register parity plus, and less, odd
#pragma unroll
                    for (int r = 0; r < R; r++) {
                        if ((static_cast<uint32_t>(r) & rm) != rv) {
                            continue;
                        }
                        const bool odd = __popc(static_cast<uint32_t>(r) & rp) & 1U; // uniform
                        const double ax = x[0][r].x, ay = x[0][r].y;
#pragma unroll
                        for (int kk = 0; kk < KH; kk++) {
                            const double cx = x[1 + kk][r].x, cy = x[1 + kk][r].y;
                            const double im = rt_fma(cx, ay, -cy * ax);
                            acc[kk][0] += im;
                            acc[kk][1] += odd ? -im : im;
                            if constexpr (FULL) {
                                const double re = rt_fma(cx, ax, cy * ay);
                                acc[kk][4] += re;
                                acc[kk][5] += odd ? -re : re;
                            }
                        }
                    }
#pragma unroll
                    for (int kk = 0; kk < KH; kk++) {
#pragma unroll
                        for (int c = 0; c < NC; c += 4) {
                            const double both = acc[kk][c], less = tpar ? -acc[kk][c + 1] : acc[kk][c + 1];
                            acc[kk][c] = 0.5 * (both + less);
                            acc[kk][c + 1] = 0.5 * (both - less);
                        }
                    }
                } else {
                    switch (st.j) {
                    case 0: pairs(std::integral_constant<int, 0>{}); break;
                    case 1: pairs(std::integral_constant<int, 1>{}); break;
                    default: pairs(std::integral_constant<int, 2>{}); break;
                    }
                }
#pragma unroll
                for (int kk = 0; kk < KH; kk++) {
#pragma unroll
                    for (int c = 0; c < NC; c += 4) {
                        const double t = rt_sum4(on ? acc[kk][c] : 0.0, on ? acc[kk][c + 1] : 0.0,
                                                    on ? acc[kk][c + 2] : 0.0, on ? acc[kk][c + 3] : 0.0);
                        if ((lane & 15) == 0) {
                            mine[(slot * KH + kk) * NC + c + rt_row(lane >> 4)] += t;
                        }
                    }
                }
            }
            if (kind == kSweepDense) {
                dcx<double> u[4];
#pragma unroll
                for (int i = 0; i < 4; i++) {
                    u[i] = st.u[i];
                }
                auto dense = [&](auto jt) {
                    constexpr int J = decltype(jt)::value;
#pragma unroll
                    for (int p = 0; p < R / 2; p++) {
                        const int i0 = ((p >> J) << (J + 1)) | (p & ((1 << J) - 1)), i1 = i0 | (1 << J);
                        if ((static_cast<uint32_t>(i0) & rm) == rv) {
#pragma unroll
                            for (int i = 0; i < S; i++) {
                                rt_apply2(lanes, u, x[i][i0], x[i][i1]);
                            }
                        }
                    }
                };
                switch (st.j) {
                case 0: dense(std::integral_constant<int, 0>{}); break;
                case 1: dense(std::integral_constant<int, 1>{}); break;
                default: dense(std::integral_constant<int, 2>{}); break;
                }
            } else if (kind == kSweepFlip) {
                auto flip = [&](auto jt) {
                    constexpr int J = decltype(jt)::value;
#pragma unroll
                    for (int p = 0; p < R / 2; p++) {
                        const int i0 = ((p >> J) << (J + 1)) | (p & ((1 << J) - 1)), i1 = i0 | (1 << J);
                        if ((static_cast<uint32_t>(i0) & rm) == rv) {
#pragma unroll
                            for (int i = 0; i < S; i++) {
                                rt_exchange(lanes, x[i][i0], x[i][i1]);
                            }
                        }
                    }
                };
                switch (st.j) {
                case 0: flip(std::integral_constant<int, 0>{}); break;
                case 1: flip(std::integral_constant<int, 1>{}); break;
                default: flip(std::integral_constant<int, 2>{}); break;
                }
            } else { // kSweepDiag
                const dcx<double> u0 = st.u[0], u1 = st.u[1];
                // this lane's phase at even and at odd parity of the register index
                const dcx<double> ue{tpar ? u1.r : u0.r, tpar ? u1.i : u0.i}, uo{tpar ? u0.r : u1.r, tpar ? u0.i : u1.i};
#pragma unroll
                for (int r = 0; r < R; r++) {
                    if ((static_cast<uint32_t>(r) & rm) == rv) {
                        const bool odd = __popc(static_cast<uint32_t>(r) & rp) & 1U; // uniform
                        const dcx<double> u{odd ? uo.r : ue.r, odd ? uo.i : ue.i};
#pragma unroll
                        for (int i = 0; i < S; i++) {
                            rt_into(lanes, x[i][r], u.r, -u.i * x[i][r].y, u.i * x[i][r].x);
                        }
                    }
                }
            }
        }
        if (win != HOME) {
            window(HOME);
        }
#pragma unroll
        for (int r = 0; r < R; r++) {
            const uint32_t e = (static_cast<uint32_t>(r) << TB) | tid;
            const uint64_t a = base | thread_at | spread(static_cast<uint32_t>(r) << TB);
            if (e < size) {
                if (grp == A.writer) {
                    A.lam_out[a] = v2<T>{static_cast<T>(x[0][r].x), static_cast<T>(x[0][r].y)};
                }
#pragma unroll
                for (int kk = 0; kk < KH; kk++) {
                    if (kk < nk) {
                        h[kk][a] = v2<T>{static_cast<T>(x[1 + kk][r].x), static_cast<T>(x[1 + kk][r].y)};
                    }
                }
            }
        }
    }
    __syncthreads();
    for (int i = tid; i < nsum; i += 64 * NW) {
        const int c = i % NC, kk = (i / NC) % KH, slot = i / (NC * KH);
        double t = sums[i];
        for (int v = 1; v < NW; v++) {
            t += sums[v * nsum + i];
        }
        if (kk < nk) {
            A.partial[((static_cast<uint64_t>(A.slot0 + slot) * NC + c) * A.pk + k0 - A.pk0 + kk) * A.W + w] = t;
        }
    }
}

// One step by itself (SweepStepArgs), as it touches a part of the amplitudes
// only and a pass would read and write them all, or where a launch costs less
// than a pass's program.  Four states' loads are in flight before the stores.
// OBS: states with room for their sums; four are an instance of their own, whose
// registers let more wavefronts run.
template <class T, int OBS, bool FULL, bool DENSE, bool TRAIN>
__global__ __launch_bounds__(kBlock, 4) void k_sweep_step(const SweepStepArgs<T> A) {
    constexpr int NC = FULL ? kSweepFull : kSweepReal;
    constexpr int CH = OBS < 4 ? OBS : 4;
    double acc[OBS][NC] = {};
    auto mul2 = [](const dcx<double> &p, const double2 &x, const dcx<double> &q, const double2 &y) {
        return v2<T>{static_cast<T>(rt_fma(p.r, x.x, rt_fma(-p.i, x.y, rt_fma(q.r, y.x, -q.i * y.y)))),
                     static_cast<T>(rt_fma(p.r, x.y, rt_fma(p.i, x.x, rt_fma(q.r, y.y, q.i * y.x))))};
    };
    auto mul1 = [](const dcx<double> &p, const double2 &x) {
        return v2<T>{static_cast<T>(rt_fma(p.r, x.x, -p.i * x.y)), static_cast<T>(rt_fma(p.r, x.y, p.i * x.x))};
    };
    const uint64_t stride = static_cast<uint64_t>(gridDim.x) * kBlock;
    for (uint64_t g = static_cast<uint64_t>(blockIdx.x) * kBlock + threadIdx.x; g < A.nwork; g += stride) {
        const uint64_t i0 = expand(g, A.geo), i1 = i0 ^ A.flip;
        const bool odd = !DENSE && (__popcll(i0 & A.par) & 1);
        const dcx<double> ph = odd ? A.u[3] : A.u[0];
        const v2<T> a0 = A.lam[i0], b0 = DENSE ? A.lam[i1] : v2<T>{0, 0};
        const double2 a{a0.x, a0.y}, b{b0.x, b0.y};
        if (A.write_lam) {
            if constexpr (DENSE) {
                A.lam[i0] = mul2(A.u[0], a, A.u[1], b);
                A.lam[i1] = mul2(A.u[2], a, A.u[3], b);
            } else {
                A.lam[i0] = mul1(ph, a);
            }
        }
#pragma unroll
        for (int k0 = 0; k0 < OBS; k0 += CH) {
            v2<T> c0[CH], d0[CH];
#pragma unroll
            for (int j = 0; j < CH; j++) {
                if (k0 + j < A.nk) {
                    c0[j] = A.h[k0 + j][i0];
                    if constexpr (DENSE) {
                        d0[j] = A.h[k0 + j][i1];
                    }
                }
            }
#pragma unroll
            for (int j = 0; j < CH; j++) {
                if (k0 + j >= A.nk) {
                    continue;
                }
                const double2 c{c0[j].x, c0[j].y};
                double *t = acc[k0 + j];
                if constexpr (DENSE) {
                    const double2 d{d0[j].x, d0[j].y};
                    if constexpr (TRAIN) {
                        t[0] = rt_fma(c.x, a.y, rt_fma(-c.y, a.x, t[0]));
                        t[1] = rt_fma(d.x, b.y, rt_fma(-d.y, b.x, t[1]));
                        t[2] = rt_fma(c.x, b.y, rt_fma(-c.y, b.x, rt_fma(d.x, a.y, rt_fma(-d.y, a.x, t[2]))));
                        t[3] = rt_fma(c.x, b.x, rt_fma(c.y, b.y, rt_fma(-d.x, a.x, rt_fma(-d.y, a.y, t[3]))));
                        if constexpr (FULL) {
                            t[4] = rt_fma(c.x, a.x, rt_fma(c.y, a.y, t[4]));
                            t[5] = rt_fma(d.x, b.x, rt_fma(d.y, b.y, t[5]));
                            t[6] = rt_fma(c.x, b.x, rt_fma(c.y, b.y, rt_fma(d.x, a.x, rt_fma(d.y, a.y, t[6]))));
                            t[7] = rt_fma(c.x, b.y, rt_fma(-c.y, b.x, rt_fma(-d.x, a.y, rt_fma(d.y, a.x, t[7]))));
                        }
                    }
                    A.h[k0 + j][i0] = mul2(A.u[0], c, A.u[1], d);
                    A.h[k0 + j][i1] = mul2(A.u[2], c, A.u[3], d);
                } else {
                    if constexpr (TRAIN) {
                        const double im = rt_fma(c.x, a.y, -c.y * a.x);
                        t[0] += odd ? 0.0 : im;
                        t[1] += odd ? im : 0.0;
                        if constexpr (FULL) {
                            const double re = rt_fma(c.x, a.x, c.y * a.y);
                            t[4] += odd ? 0.0 : re;
                            t[5] += odd ? re : 0.0;
                        }
                    }
                    A.h[k0 + j][i0] = mul1(ph, c);
                }
            }
        }
    }
    if constexpr (TRAIN) {
        __shared__ double wpart[kBlock / 64][OBS * NC];
        const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
#pragma unroll
        for (int k = 0; k < OBS; k++) {
            if (k < A.nk) { // uniform
#pragma unroll
                for (int c = 0; c < NC; c += 4) {
                    const double s = rt_sum4(acc[k][c], acc[k][c + 1], acc[k][c + 2], acc[k][c + 3]);
                    if ((lane & 15) == 0) {
                        wpart[wave][k * NC + c + rt_row(lane >> 4)] = s;
                    }
                }
            }
        }
        __syncthreads();
        for (int i = threadIdx.x; i < A.nk * NC; i += kBlock) {
            double s = wpart[0][i];
#pragma unroll
            for (int w = 1; w < kBlock / 64; w++) {
                s += wpart[w][i];
            }
            const int k = i / NC, c = i % NC;
            A.partial[((static_cast<uint64_t>(A.slot) * NC + c) * A.pk + A.k0 + k) * gridDim.x + blockIdx.x] = s;
        }
    }
}

// launch_sweep_sums: one wavefront per value, fixed order
static __global__ __launch_bounds__(64) void k_sweep_sums(const double *__restrict__ partial, int W, int pk, int pk0, int K,
                                                          double *__restrict__ out) {
    const int sc = static_cast<int>(blockIdx.x) / pk, k = pk0 + static_cast<int>(blockIdx.x) % pk;
    if (k >= K) {
        return;
    }
    const double *p = partial + static_cast<uint64_t>(blockIdx.x) * W;
    double s = 0;
    for (int i = threadIdx.x; i < W; i += 64) {
        s += p[i];
    }
    s = wave_sum(s);
    if (threadIdx.x == 0) {
        out[static_cast<uint64_t>(sc) * K + k] = s;
    }
}

} // namespace plamd
