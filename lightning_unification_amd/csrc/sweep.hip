// The pass kernels of the backward sweep and of forward tapes, one translation unit per precision
// (PL_SWEEP_DOUBLE), compiled like the tile passes with uniform regions left
// unstructured: a step's branches are all on scalars, and structuring them
// makes the compiler copy the register tile at every join.
#include "kernels_adjoint.hpp"
#include "kernels_pass.hpp"

namespace plamd {

template <class T> hipError_t launch_sweep(int waves, int kh, bool full, const SweepArgs<T> &a, hipStream_t s) {
    auto go = [&](auto nw, auto k, auto f) {
        constexpr int NW = decltype(nw)::value, KH = decltype(k)::value;
        constexpr bool FULL = decltype(f)::value != 0;
        constexpr size_t tile = sizeof(double2) << (6 + kSweepRegBits + (NW == 4 ? 2 : NW == 2 ? 1 : 0));
        const size_t lds = tile + size_t(a.nslots) * NW * KH * (FULL ? kSweepFull : kSweepReal) * sizeof(double);
        hipLaunchKernelGGL((k_sweep<T, NW, KH, FULL>), dim3(static_cast<unsigned>(a.W * a.ngrp)), dim3(64 * NW), lds,
                           s, a, a.prog);
        return hipGetLastError();
    };
    using I1 = std::integral_constant<int, 1>;
    using I2 = std::integral_constant<int, 2>;
    using I4 = std::integral_constant<int, 4>;
    using I0 = std::integral_constant<int, 0>;
    if (full) { // one state is swept with lambda
        return waves == 4 ? go(I4{}, I1{}, I1{}) : waves == 2 ? go(I2{}, I1{}, I1{}) : go(I1{}, I1{}, I1{});
    }
    if (kh == 2) {
        return waves == 4 ? go(I4{}, I2{}, I0{}) : waves == 2 ? go(I2{}, I2{}, I0{}) : go(I1{}, I2{}, I0{});
    }
    return waves == 4 ? go(I4{}, I1{}, I0{}) : waves == 2 ? go(I2{}, I1{}, I0{}) : go(I1{}, I1{}, I0{});
}

template <class T> hipError_t launch_sweep_step(int W, bool full, const SweepStepArgs<T> &a, hipStream_t s) {
    auto go = [&](auto obs, auto f, auto dense, auto train) {
        hipLaunchKernelGGL((k_sweep_step<T, decltype(obs)::value, decltype(f)::value, decltype(dense)::value,
                                         decltype(train)::value>),
                           dim3(W), dim3(kBlock), 0, s, a);
        return hipGetLastError();
    };
    using Yes = std::true_type;
    using No = std::false_type;
    std::integral_constant<int, 1> one;
    std::integral_constant<int, 4> four;
    std::integral_constant<int, kStepObs> all;
    const bool dense = a.flip != 0;
    if (!a.partial) {
        return dense ? go(all, No{}, Yes{}, No{}) : go(all, No{}, No{}, No{});
    }
    if (full) {
        return dense ? go(one, Yes{}, Yes{}, Yes{}) : go(one, Yes{}, No{}, Yes{});
    }
    if (a.nk <= 4) {
        return dense ? go(four, No{}, Yes{}, Yes{}) : go(four, No{}, No{}, Yes{});
    }
    return dense ? go(all, No{}, Yes{}, Yes{}) : go(all, No{}, No{}, Yes{});
}

template <class T>
hipError_t launch_pass(int waves, v2<T> *sv, uint64_t ntiles, const SweepGeom &geo, const SweepStep *prog, int nsteps,
                       hipStream_t s) {
    auto go = [&](auto nw) {
        constexpr int NW = decltype(nw)::value;
        constexpr size_t lds = sizeof(double) << (6 + kPassRegBits + (NW == 8 ? 3 : NW == 4 ? 2 : NW == 2 ? 1 : 0));
        hipLaunchKernelGGL((k_pass<T, NW>), dim3(static_cast<unsigned>(ntiles)), dim3(64 * NW), lds, s, sv, ntiles, geo,
                           prog, nsteps);
        return hipGetLastError();
    };
    switch (waves) {
    case 8: return go(std::integral_constant<int, 8>{});
    case 4: return go(std::integral_constant<int, 4>{});
    case 2: return go(std::integral_constant<int, 2>{});
    default: return go(std::integral_constant<int, 1>{});
    }
}

#if PL_SWEEP_DOUBLE
template hipError_t launch_pass<double>(int, v2<double> *, uint64_t, const SweepGeom &, const SweepStep *, int,
                                        hipStream_t);
template hipError_t launch_sweep_step<double>(int, bool, const SweepStepArgs<double> &, hipStream_t);
template hipError_t launch_sweep<double>(int, int, bool, const SweepArgs<double> &, hipStream_t);

hipError_t launch_sweep_sums(const double *partial, int W, unsigned count, int pk, int pk0, int K, double *out,
                             hipStream_t s) {
    hipLaunchKernelGGL(k_sweep_sums, dim3(count * static_cast<unsigned>(pk)), dim3(64), 0, s, partial, W, pk, pk0, K, out);
    return hipGetLastError();
}
#else
template hipError_t launch_pass<float>(int, v2<float> *, uint64_t, const SweepGeom &, const SweepStep *, int,
                                       hipStream_t);
template hipError_t launch_sweep_step<float>(int, bool, const SweepStepArgs<float> &, hipStream_t);
template hipError_t launch_sweep<float>(int, int, bool, const SweepArgs<float> &, hipStream_t);
#endif

} // namespace plamd
