// Data of the backward sweep's passes and the launch of one
// (kernels_adjoint.hpp; the kernel is compiled in its own translation units,
// sweep.hip).
#pragma once

#include <hip/hip_runtime.h>
#include <stdint.h>

#include "kernels_gate.hpp"

namespace plamd {

enum SweepKind : int {
    kSweepWindow = 0, // other local bits become register bits
    kSweepDense,      // a 2x2 on the pairs of j
    kSweepFlip,       // the pairs of j exchanged (CNOT, Toffoli, SWAP)
    kSweepDiag,       // phase u[0] or u[1] by the parity of masked bits
};

// Entries of a kSweepDense step's 2x2 that vanish: none; the imaginary parts (RY,
// Hadamard); the diagonal's imaginary and the others' real parts (RX, IsingXX).
enum SweepForm : int { kSweepFull2 = 0, kSweepReal2, kSweepCross2 };

// One step on a tile whose local index is split into register bits (the
// window) and thread bits (the others, ascending).  It acts where all tested
// bits have their values: (register index & rm) == rv, (thread & lm) == lv and
// (bits outside the tile & omask) == oval, of a pair at the member with the lower
// bit clear.  j: the pairs differ in register bit j (j < RB, the number of
// register bits), or in two: the j - RB-th of (0,1) (0,2) .. (1,2) ..  kSweepDiag: the phase is u[parity
// of register & rp, thread & lp and outside & op].  kSweepWindow: rp holds the
// new window's positions, four bits each.
struct SweepStep {
    int kind;
    int j;
    uint32_t rm, rv, lm, lv, rp, lp;
    int slot; // accumulation slot of the pass, -1: not trainable
    int form; // kSweepDense: SweepForm
    uint64_t omask, oval, op;
    dcx<double> u[4];
};

// Sums kept per slot and observable, of M_ab = sum conj(h_a) lambda_b over the
// step's pairs (kSweepDiag: a = b = the parity):
//   0 Im M00, 1 Im M11, 2 Im(M01 + M10), 3 Re(M01 - M10)
// and for the complex form also
//   4 Re M00, 5 Re M11, 6 Re(M01 + M10), 7 Im(M01 - M10).
constexpr int kSweepReal = 4, kSweepFull = 8;
constexpr int kSweepSlots = 64;    // trainable steps per pass
constexpr int kSweepMaxBits = 13;  // widest tile

constexpr int kSweepRegBits = 3;   // register bits of a sweep tile: 8 amplitudes a thread and state
constexpr int kPassRegBits = 4;    // of a forward pass's: 16 amplitudes a thread

struct SweepGeom {
    int bits;              // local bits of the state: min(n, the tile's)
    int low;               // the lowest `low` bit positions are local bits 0 .. low - 1
    int hb[kSweepMaxBits]; // positions of local bits low .., ascending
};

// States are held in T and swept in double: a pass of complex64 states rounds
// each amplitude once, where its steps would round it once each.
template <class T> struct SweepArgs {
    const v2<T> *lam_in;
    v2<T> *lam_out;
    v2<T> *const *hs;
    int K, grp0, ngrp, writer, W;
    uint64_t ntiles;
    SweepGeom geo;
    const SweepStep *prog;
    int nsteps, nslots, slot0;
    double *partial;
    int pk, pk0; // observables per slot of `partial`, the first one's number
};

// One step on lambda and up to kStepObs states, read and written in place
// where it acts.  Pairs of a dense step: i = expand(g, geo) and i ^ flip (geo
// pins the bit and the tested ones, so a bit2 no test is on stays free in g).  Phases (flip = 0): u[0] or u[3] by the parity of i & par.  partial, of a
// trainable one: as SweepArgs, one walker a workgroup, the first state's
// observable at k0 of pk.
constexpr int kStepObs = 8;
template <class T> struct SweepStepArgs {
    v2<T> *lam;
    v2<T> *h[kStepObs];
    int nk, write_lam;
    uint64_t nwork, flip, par;
    Geom geo;
    dcx<double> u[4];
    double *partial; // nullptr: not trainable
    int slot, pk, k0;
};

// One launch of args.ngrp observable groups (kh observables each) with `waves`
// (1, 2 or 4) wavefronts per tile; full: the complex sums too.
template <class T> hipError_t launch_sweep(int waves, int kh, bool full, const SweepArgs<T> &args, hipStream_t s);
// W workgroups
template <class T> hipError_t launch_sweep_step(int W, bool full, const SweepStepArgs<T> &args, hipStream_t s);
// One forward pass (kernels_pass.hpp) of `waves` (1, 2, 4 or 8) wavefronts a tile.
template <class T>
hipError_t launch_pass(int waves, v2<T> *sv, uint64_t ntiles, const SweepGeom &geo, const SweepStep *prog, int nsteps,
                       hipStream_t s);
// Sums over the W walkers of partial[sc][k][W], sc < count, k < pk:
// out[sc K + pk0 + k] where that is an observable
hipError_t launch_sweep_sums(const double *partial, int W, unsigned count, int pk, int pk0, int K, double *out,
                             hipStream_t s);

} // namespace plamd
