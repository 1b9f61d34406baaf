// Register tiles: a workgroup holds 2^(TB + RB) amplitudes, 2^RB of them in
// each of its 2^TB threads.  A thread's amplitudes differ in the RB window
// bits of the local index (`win`, four bits a position, ascending); its thread
// index supplies the other bits.  Gates on window bits need no exchange; a
// change of window goes through an LDS buffer of real parts and imaginary
// parts (an element of both would tie the two registers of an amplitude into
// one tuple, which in-place updates would have to copy out of and back into).
// Used by the backward sweep (kernels_adjoint.hpp), forward passes
// (kernels_pass.hpp) and the batched circuits (kernels_batch.hpp).
#pragma once

#include <hip/hip_runtime.h>
#include <stdint.h>

#include <type_traits>

#include "kernels_gate.hpp"

namespace plamd {

// Sums of a and b over lanes l and l ^ 32: a's in the lower half, b's in the upper.
__device__ __forceinline__ double rt_fold32(double a, double b) {
    const auto ua = static_cast<unsigned long long>(__double_as_longlong(a));
    const auto ub = static_cast<unsigned long long>(__double_as_longlong(b));
    const auto lo = __builtin_amdgcn_permlane32_swap(static_cast<unsigned>(ua), static_cast<unsigned>(ub), false, false);
    const auto hi = __builtin_amdgcn_permlane32_swap(static_cast<unsigned>(ua >> 32), static_cast<unsigned>(ub >> 32),
                                                     false, false);
    const double x = __longlong_as_double(static_cast<long long>((static_cast<unsigned long long>(hi[0]) << 32) | lo[0]));
    const double y = __longlong_as_double(static_cast<long long>((static_cast<unsigned long long>(hi[1]) << 32) | lo[1]));
    return x + y;
}
// Sums of a and b over lanes l and l ^ 16: a's in even rows of 16 lanes, b's in odd ones.
__device__ __forceinline__ double rt_fold16(double a, double b) {
    const auto ua = static_cast<unsigned long long>(__double_as_longlong(a));
    const auto ub = static_cast<unsigned long long>(__double_as_longlong(b));
    const auto lo = __builtin_amdgcn_permlane16_swap(static_cast<unsigned>(ua), static_cast<unsigned>(ub), false, false);
    const auto hi = __builtin_amdgcn_permlane16_swap(static_cast<unsigned>(ua >> 32), static_cast<unsigned>(ub >> 32),
                                                     false, false);
    const double x = __longlong_as_double(static_cast<long long>((static_cast<unsigned long long>(hi[0]) << 32) | lo[0]));
    const double y = __longlong_as_double(static_cast<long long>((static_cast<unsigned long long>(hi[1]) << 32) | lo[1]));
    return x + y;
}
template <int CTRL> __device__ __forceinline__ double rt_dpp(double v) {
    const auto u = static_cast<unsigned long long>(__double_as_longlong(v));
    const unsigned lo = static_cast<unsigned>(__builtin_amdgcn_mov_dpp(static_cast<int>(static_cast<unsigned>(u)), CTRL, 0xf, 0xf, true));
    const unsigned hi = static_cast<unsigned>(__builtin_amdgcn_mov_dpp(static_cast<int>(static_cast<unsigned>(u >> 32)), CTRL, 0xf, 0xf, true));
    return __longlong_as_double(static_cast<long long>((static_cast<unsigned long long>(hi) << 32) | lo));
}
// Totals of four values over the wavefront: row r of 16 lanes (lane / 16 = r)
// ends with the total of v[rt_row(r)].
__device__ __forceinline__ double rt_sum4(double v0, double v1, double v2, double v3) {
    // rows 0..3 after the folds: v0, v2, v1, v3
    double s = rt_fold16(rt_fold32(v0, v1), rt_fold32(v2, v3));
    s += rt_dpp<0x128>(s); // rotations within a row by 8, 4, 2, 1
    s += rt_dpp<0x124>(s);
    s += rt_dpp<0x122>(s);
    s += rt_dpp<0x121>(s);
    return s;
}
__device__ __forceinline__ int rt_row(int r) { return ((r & 1) << 1) | (r >> 1); }

// Local index -> place in the LDS buffer, linear in its bits.  With window bits
// p .. p + RB - 1, consecutive lanes differ in the local bits around them; the
// map folds bits 4..8 into the low five so that for windows of three and four
// neighbouring bits the first four lane bits give 16 places that differ mod 16
// and the first five 32 mod 32 (all but one case): no two lanes of an access
// share a bank.  Found by trying every such map.  Measured, conflicts take up to 2 % of
// the LDS cycles in the sweep and the batched stages, but 21 % there on tiles
// of 2^10 amplitudes, and 25 % in a forward pass at 28 qubits, whose windows
// hold any four bits.
__device__ __forceinline__ uint32_t rt_place(uint32_t e) {
    return e ^ ((e >> 4) & 1U) ^ ((e >> 3) & 4U) ^ (((e >> 6) & 1U) * 10U) ^ (((e >> 7) & 1U) * 28U) ^ ((e >> 4) & 16U);
}

// thread bits spread over the local bits outside the window
template <int RB> __device__ __forceinline__ uint32_t rt_thread_part(uint32_t t, uint32_t win) {
#pragma unroll
    for (int j = 0; j < RB; j++) {
        const uint32_t m = (1U << ((win >> (4 * j)) & 15U)) - 1;
        t = ((t & ~m) << 1) | (t & m);
    }
    return t;
}
__device__ __forceinline__ double rt_fma(double a, double b, double c) { return __builtin_fma(a, b, c); }

// Updates of the register tile.  The last multiply-add of every amplitude
// writes the amplitude's own register, in the lanes of `m` only; the lane
// condition is an execution mask inside the block, so a step has no divergent
// branch.  Left to the compiler (branches on the condition, results in
// registers of their own), every step's results were copied back where the
// steps' branches join: 241 registers and two wavefronts a SIMD for KH = 2 in
// complex128, a third of the instructions moves.  All 64 lanes are active
// around every block.
__device__ __forceinline__ void rt_into(uint64_t m, double2 &a, double u, double tx, double ty) {
    asm("s_mov_b64 exec, %2\n\t"
        "v_fma_f64 %0, %3, %0, %4\n\t"
        "v_fma_f64 %1, %3, %1, %5\n\t"
        "s_mov_b64 exec, -1"
        : "+v"(a.x), "+v"(a.y)
        : "s"(m), "v"(u), "v"(tx), "v"(ty));
}
__device__ __forceinline__ void rt_into2(uint64_t m, double2 &a, double2 &b, double ua, double ub, double t0,
                                            double t1, double t2, double t3) {
    asm("s_mov_b64 exec, %4\n\t"
        "v_fma_f64 %0, %5, %0, %7\n\t"
        "v_fma_f64 %1, %5, %1, %8\n\t"
        "v_fma_f64 %2, %6, %2, %9\n\t"
        "v_fma_f64 %3, %6, %3, %10\n\t"
        "s_mov_b64 exec, -1"
        : "+v"(a.x), "+v"(a.y), "+v"(b.x), "+v"(b.y)
        : "s"(m), "s"(ua), "s"(ub), "v"(t0), "v"(t1), "v"(t2), "v"(t3));
}
// a <-> b in the lanes of m
__device__ __forceinline__ void rt_exchange(uint64_t m, double2 &a, double2 &b) {
    double t;
    asm("s_mov_b64 exec, %5\n\t"
        "v_mov_b64 %4, %0\n\t"
        "v_mov_b64 %0, %2\n\t"
        "v_mov_b64 %2, %4\n\t"
        "v_mov_b64 %4, %1\n\t"
        "v_mov_b64 %1, %3\n\t"
        "v_mov_b64 %3, %4\n\t"
        "s_mov_b64 exec, -1"
        : "+v"(a.x), "+v"(a.y), "+v"(b.x), "+v"(b.y), "=&v"(t)
        : "s"(m));
}

// Partner of register index i0 in the pairs that differ in bit J, or in J and J2.
template <int J, int J2> __device__ __forceinline__ constexpr int rt_partner(int i0) {
    return i0 ^ (1 << J) ^ (J2 >= 0 ? 1 << J2 : 0);
}
// The p-th register index with bit J clear.
template <int J> __device__ __forceinline__ constexpr int rt_member(int p) {
    return ((p >> J) << (J + 1)) | (p & ((1 << J) - 1));
}
// f(J, J2) for a step's j (SweepStep) with four register bits: a single one
// (J2 = -1) or two.
template <class F> __device__ __forceinline__ void rt_pairs4(int j, F &&f) {
    using std::integral_constant;
    integral_constant<int, -1> none;
    integral_constant<int, 0> b0;
    integral_constant<int, 1> b1;
    integral_constant<int, 2> b2;
    integral_constant<int, 3> b3;
    switch (j) {
    case 0: f(b0, none); break;
    case 1: f(b1, none); break;
    case 2: f(b2, none); break;
    case 3: f(b3, none); break;
    case 4: f(b0, b1); break;
    case 5: f(b0, b2); break;
    case 6: f(b0, b3); break;
    case 7: f(b1, b2); break;
    case 8: f(b1, b3); break;
    default: f(b2, b3); break;
    }
}

// (a, b) <- u (a, b) in the lanes of m, 16 multiply-adds
__device__ __forceinline__ void rt_apply2(uint64_t m, const dcx<double> *u, double2 &a, double2 &b) {
    const double t0 = rt_fma(-u[0].i, a.y, rt_fma(u[1].r, b.x, -u[1].i * b.y));
    const double t1 = rt_fma(u[0].i, a.x, rt_fma(u[1].r, b.y, u[1].i * b.x));
    const double t2 = rt_fma(-u[3].i, b.y, rt_fma(u[2].r, a.x, -u[2].i * a.y));
    const double t3 = rt_fma(u[3].i, b.x, rt_fma(u[2].r, a.y, u[2].i * a.x));
    rt_into2(m, a, b, u[0].r, u[3].r, t0, t1, t2, t3);
}

// the same for a real u, and for one with a real diagonal and imaginary others:
// 8 multiply-adds
__device__ __forceinline__ void rt_apply2_real(uint64_t m, const dcx<double> *u, double2 &a, double2 &b) {
    rt_into2(m, a, b, u[0].r, u[3].r, u[1].r * b.x, u[1].r * b.y, u[2].r * a.x, u[2].r * a.y);
}
__device__ __forceinline__ void rt_apply2_cross(uint64_t m, const dcx<double> *u, double2 &a, double2 &b) {
    rt_into2(m, a, b, u[0].r, u[3].r, -u[1].i * b.y, u[1].i * b.x, -u[2].i * a.y, u[2].i * a.x);
}

// The S states of a tile moved from window `from` to window `to` through
// `buf`, one state at a time: 2^(TB + RB) real parts, then as many imaginary
// parts; HALF: the parts take turns in a buffer of half that size, for two
// more barriers a state.  All threads of the workgroup call it.
template <int TB, int RB, int S, bool HALF = false>
__device__ __forceinline__ void rt_window(double2 (&x)[S][1 << RB], double *buf, uint32_t tid, uint32_t from,
                                          uint32_t to) {
    constexpr uint32_t IM = 1U << (TB + RB);
    const uint32_t tf = rt_place(rt_thread_part<RB>(tid, from));
    const uint32_t tt = rt_place(rt_thread_part<RB>(tid, to));
    // the register index's part, from its bits' parts (uniform): computed per
    // register instead, it costs more scalar instructions than the step's
    // multiply-adds
    uint32_t fb[RB], ob[RB];
#pragma unroll
    for (int j = 0; j < RB; j++) {
        fb[j] = rt_place(1U << ((from >> (4 * j)) & 15U));
        ob[j] = rt_place(1U << ((to >> (4 * j)) & 15U));
    }
    auto part = [](int r, const uint32_t (&v)[RB]) {
        uint32_t e = 0;
#pragma unroll
        for (int j = 0; j < RB; j++) {
            e ^= ((r >> j) & 1) ? v[j] : 0U;
        }
        return e;
    };
#pragma unroll
    for (int i = 0; i < S; i++) {
#pragma unroll
        for (int h = 0; h < (HALF ? 2 : 1); h++) {
            __syncthreads();
#pragma unroll
            for (int r = 0; r < (1 << RB); r++) {
                const uint32_t p = tf ^ part(r, fb);
                buf[p] = h ? x[i][r].y : x[i][r].x;
                if constexpr (!HALF) {
                    buf[p + IM] = x[i][r].y;
                }
            }
            __syncthreads();
#pragma unroll
            for (int r = 0; r < (1 << RB); r++) {
                const uint32_t p = tt ^ part(r, ob);
                (h ? x[i][r].y : x[i][r].x) = buf[p];
                if constexpr (!HALF) {
                    x[i][r].y = buf[p + IM];
                }
            }
        }
    }
}

} // namespace plamd
