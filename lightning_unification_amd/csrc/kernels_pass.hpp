// Forward passes on register tiles: a tape's steps (sweep.hpp) applied to one
// state, many per read and write of it.
//
// A gate per launch moves the whole state (or half) for a few multiply-adds an
// amplitude, and on a small state is a launch and nothing else.  A workgroup
// here holds a tile of 2^(6 + log2 NW + 4) amplitudes in registers, 16 a
// thread, and runs every step of the pass on it with the step forms and
// windows of the backward sweep (kernels_adjoint.hpp; reg_tile.hpp).  A window
// of four bits holds more steps than the sweep's three, and one state leaves
// the registers for it.  complex64 states are updated in double: a pass rounds
// each amplitude once.
// Bound: HBM for shallow passes (1.9 ms a pass of 4 GiB at the copy rate), FP64
// issue from about twenty steps a pass on.  28 qubits complex128: 19 gates 22.4 ->
// 3.5 ms against a launch each; 220 gates 28.2 -> 17.6 ms against the
// wavefront tiles of kernels_tile.hpp, whose 2^11 amplitudes take 16 passes
// where 2^13 take 7.  13 qubits complex64, 90 gates: 275 -> 65 us a call.
#pragma once

#include <hip/hip_runtime.h>
#include <stdint.h>

#include "reg_tile.hpp"
#include "sweep_launch.hpp"

namespace plamd {

template <class T, int NW>
__global__ __launch_bounds__(64 * NW, 4) void k_pass(v2<T> *__restrict__ sv, uint64_t ntiles, const SweepGeom geo,
                                                     const SweepStep *__restrict__ prog, int nsteps) {
    constexpr int RB = kPassRegBits, R = 1 << RB;
    static_assert(RB == 4, "rt_pairs4 names four register bits");
    constexpr int TB = 6 + (NW == 8 ? 3 : NW == 4 ? 2 : NW == 2 ? 1 : 0);
    constexpr uint32_t HOME = TB | (TB + 1) << 4 | (TB + 2) << 8 | (TB + 3) << 12;
    extern __shared__ unsigned char smem_raw[];
    double *buf = reinterpret_cast<double *>(smem_raw);
    const uint32_t tid = threadIdx.x;
    if (ntiles < 1024) { // few workgroups: the program into the caches at once, as in k_sweep
        for (uint32_t o = tid * 64; o < nsteps * sizeof(SweepStep); o += 64 * NW * 64) {
            asm volatile("" ::"v"(*reinterpret_cast<const int *>(reinterpret_cast<const char *>(prog) + o)));
        }
    }
    auto spread = [&](uint32_t e) { // local index -> bits of the state index
        uint64_t g = e & ((1U << geo.low) - 1);
        for (int b = geo.low; b < geo.bits; b++) {
            g |= static_cast<uint64_t>((e >> b) & 1U) << geo.hb[b - geo.low];
        }
        return g;
    };
    const uint32_t size = 1U << geo.bits; // a state smaller than the tile leaves the rest zero
    uint64_t q = blockIdx.x;
    if ((gridDim.x & 7) == 0) { // each XCD one contiguous eighth
        q = (q & 7) * (gridDim.x >> 3) + (q >> 3);
    }
    uint64_t base = q << geo.low;
    for (int b = 0; b < geo.bits - geo.low; b++) {
        const int p = geo.hb[b];
        base = ((base >> p) << (p + 1)) | (base & ((uint64_t{1} << p) - 1));
    }
    const uint64_t at = base | spread(tid);
    uint64_t reg_at[RB];
#pragma unroll
    for (int j = 0; j < RB; j++) {
        reg_at[j] = spread(1U << (TB + j));
    }
    auto part = [&](int r) {
        uint64_t e = 0;
#pragma unroll
        for (int j = 0; j < RB; j++) {
            e |= ((r >> j) & 1) ? reg_at[j] : 0;
        }
        return e;
    };
    double2 x[1][R];
#pragma unroll
    for (int r = 0; r < R; r++) {
        x[0][r] = double2{0, 0};
        if (((static_cast<uint32_t>(r) << TB) | tid) < size) {
            const v2<T> v = ld_nt<T>(sv + (at | part(r)));
            x[0][r] = double2{v.x, v.y};
        }
    }
    uint32_t win = HOME;
    for (int s = 0; s < nsteps; s++) {
        const SweepStep &st = prog[s];
        const int kind = st.kind;
        if (kind == kSweepWindow) {
            rt_window<TB, RB, 1, true>(x, buf, tid, win, st.rp);
            win = st.rp;
            continue;
        }
        if ((base & st.omask) != st.oval) {
            continue;
        }
        const bool on = (tid & st.lm) == st.lv;
        const uint64_t lanes = __ballot(on);
        const uint32_t rm = st.rm, rv = st.rv;
        if (kind == kSweepDense) {
            dcx<double> u[4];
#pragma unroll
            for (int i = 0; i < 4; i++) {
                u[i] = st.u[i];
            }
            auto each = [&](auto apply) {
                rt_pairs4(st.j, [&](auto jt, auto j2t) {
                    constexpr int J = decltype(jt)::value, J2 = decltype(j2t)::value;
#pragma unroll
                    for (int p = 0; p < R / 2; p++) {
                        const int i0 = rt_member<J>(p), i1 = rt_partner<J, J2>(i0);
                        if ((static_cast<uint32_t>(i0) & rm) == rv) {
                            apply(x[0][i0], x[0][i1]);
                        }
                    }
                });
            };
            if (st.form == kSweepReal2) {
                each([&](double2 &a, double2 &b) { rt_apply2_real(lanes, u, a, b); });
            } else if (st.form == kSweepCross2) {
                each([&](double2 &a, double2 &b) { rt_apply2_cross(lanes, u, a, b); });
            } else {
                each([&](double2 &a, double2 &b) { rt_apply2(lanes, u, a, b); });
            }
        } else if (kind == kSweepFlip) {
            rt_pairs4(st.j, [&](auto jt, auto j2t) {
                constexpr int J = decltype(jt)::value, J2 = decltype(j2t)::value;
#pragma unroll
                for (int p = 0; p < R / 2; p++) {
                    const int i0 = rt_member<J>(p), i1 = rt_partner<J, J2>(i0);
                    if ((static_cast<uint32_t>(i0) & rm) == rv) {
                        rt_exchange(lanes, x[0][i0], x[0][i1]);
                    }
                }
            });
        } else { // kSweepDiag
            const uint32_t rp = st.rp;
            const uint32_t tpar = (__popc(tid & st.lp) + __popcll(base & st.op)) & 1U;
            const dcx<double> u0 = st.u[0], u1 = st.u[1];
            const dcx<double> ue{tpar ? u1.r : u0.r, tpar ? u1.i : u0.i}, uo{tpar ? u0.r : u1.r, tpar ? u0.i : u1.i};
            if (rp == 0) { // one phase a lane
#pragma unroll
                for (int r = 0; r < R; r++) {
                    if ((static_cast<uint32_t>(r) & rm) == rv) {
                        rt_into(lanes, x[0][r], ue.r, -ue.i * x[0][r].y, ue.i * x[0][r].x);
                    }
                }
            } else {
#pragma unroll
                for (int r = 0; r < R; r++) {
                    if ((static_cast<uint32_t>(r) & rm) == rv) {
                        const bool odd = __popc(static_cast<uint32_t>(r) & rp) & 1U; // uniform
                        const dcx<double> u{odd ? uo.r : ue.r, odd ? uo.i : ue.i};
                        rt_into(lanes, x[0][r], u.r, -u.i * x[0][r].y, u.i * x[0][r].x);
                    }
                }
            }
        }
    }
    if (win != HOME) {
        rt_window<TB, RB, 1, true>(x, buf, tid, win, HOME);
    }
#pragma unroll
    for (int r = 0; r < R; r++) {
        if (((static_cast<uint32_t>(r) << TB) | tid) < size) {
            st_nt<T>(sv + (at | part(r)), v2<T>{static_cast<T>(x[0][r].x), static_cast<T>(x[0][r].y)});
        }
    }
}

} // namespace plamd
