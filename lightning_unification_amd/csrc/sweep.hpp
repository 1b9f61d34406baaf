// Host side of the backward sweep (kernels_adjoint.hpp): a tape, last
// operation first, becomes steps; steps become passes; a pass becomes a
// program of register windows.
//
// Step: a 2x2 on pairs that differ in one bit or two, or phases by the parity
// of some bits, where other bits have given values.  Every gate of at most four
// members is one or two such steps (IsingXX: one on pairs that differ in both
// bits).  Pairs that differ in more bits (DoubleExcitation) are brought
// together in a pass by CNOTs from one of those bits to the others, undone
// after.  A step merges into the last one that touched any of its bits when that has the same geometry: nothing in between
// touches those bits, so it commutes back.  The merged step keeps the product
// U^dagger = U_m^dagger .. U_1^dagger (U_1 the tape's last) and, for the j-th
// operation's generator, W = A^dagger G A with A the product before it:
// <H_j|G lambda_j> = <H|W lambda> on the states at the step's start, a linear
// form of the step's transition matrix.  Products and W are formed in double.
//
// Pass: like a tile pass (tile.hpp), steps whose mixing bits lie in the
// pass's tile and which touch no bit of a step left out before them.  Bits a
// step only tests (controls, phases, parities) need not be tile bits.
#pragma once

#include <algorithm>
#include <complex>
#include <cstdint>
#include <deque>
#include <vector>

#include "lower.hpp"
#include "sweep_launch.hpp"

namespace plamd {

struct SweepTrain {
    int row;                     // index into tp[]
    double scale;                // generator scale, negated for an inverted operation
    double w00 = 0, w11 = 0;     // W, Hermitian
    std::complex<double> w01{0};
};

struct SweepOp { // one step before it is placed on a tile
    bool big = false;  // applied state by state: operation `tape` of the tape
    bool alone = false; // in no pass
    int tape = -1;
    uint64_t bit = 0;  // the bit a 2x2 mixes (the lower of two); 0: phases only
    uint64_t bit2 = 0; // a second bit its pairs differ in; tests are on the member with `bit` clear
    uint64_t more = 0; // further ones, each tested
    uint64_t par = 0;  // phases: u[0] or u[3] by the parity of these bits
    uint64_t test = 0, value = 0; // bits tested, and their values
    std::complex<double> u[4] = {1, 0, 0, 1};
    std::vector<SweepTrain> train;

    uint64_t touch() const { return bit | bit2 | more | par | test | extra; }
    uint64_t extra = 0; // big operations: all their bits
    uint64_t need() const { return bit | bit2 | more; }
    bool same_place(const SweepOp &o) const {
        return !big && !o.big && bit == o.bit && bit2 == o.bit2 && more == o.more && par == o.par && test == o.test && value == o.value;
    }
    bool diagonal() const { return u[1] == 0.0 && u[2] == 0.0; }
    bool identity() const { return diagonal() && u[0] == 1.0 && u[3] == 1.0; }
    bool flip() const { return u[0] == 0.0 && u[3] == 0.0 && u[1] == 1.0 && u[2] == 1.0; }
};

// W of the steps before: W <- a^dagger W a (a single phase cancels).
inline void sweep_move(SweepTrain &t, const SweepOp &a) {
    const std::complex<double> w[4] = {t.w00, t.w01, std::conj(t.w01), t.w11};
    std::complex<double> r[4];
    for (int i = 0; i < 2; i++) {
        for (int j = 0; j < 2; j++) {
            r[2 * i + j] = 0;
            for (int p = 0; p < 2; p++) {
                for (int q = 0; q < 2; q++) {
                    r[2 * i + j] += std::conj(a.u[2 * p + i]) * w[2 * p + q] * a.u[2 * q + j];
                }
            }
        }
    }
    t.w00 = r[0].real();
    t.w11 = r[3].real();
    t.w01 = r[1];
}

// The steps of one lowered operation ud (U^dagger) and, if it is trainable,
// its generator g; false if the operation has no such form.
inline bool sweep_expand_op(const GroupOp<double> &ud, const GroupOp<double> *g, const SweepTrain &tr,
                            std::vector<SweepOp> &out) {
    using C = std::complex<double>;
    out.clear();
    if (ud.kind == GroupOp<double>::Parity) {
        if (g && (g->kind != GroupOp<double>::Parity || g->parity_mask != ud.parity_mask)) {
            return false;
        }
        SweepOp s;
        s.par = ud.parity_mask;
        s.u[0] = C(ud.parity_phase[0]);
        s.u[3] = C(ud.parity_phase[1]);
        if (g) {
            SweepTrain t = tr;
            t.w00 = g->parity_phase[0].real();
            t.w11 = g->parity_phase[1].real();
            s.train.push_back(t);
        }
        out.push_back(s);
        return true;
    }
    const int M = ud.M;
    if (M != 1 && M != 2 && M != 4) {
        return false;
    }
    if (g) { // the generator lives on the operation's groups
        if (!g->same_geometry(ud)) {
            return false;
        }
    }
    uint64_t touch = 0, mem[4] = {}, vary = 0;
    for (int j = 0; j < ud.nb; j++) {
        touch |= uint64_t{1} << ud.pos[j];
    }
    for (int j = 0; j < M; j++) {
        mem[j] = ud.fixed | ud.off[j];
        vary |= mem[j] ^ mem[0];
    }
    SweepOp proto;
    proto.test = touch & ~vary;
    proto.value = mem[0] & proto.test;
    auto U = [&](int r, int c) { return C(ud.mat[r * M + c]); };
    auto G = [&](int r, int c) { return g ? g->mat[r * M + c] : C(0); };
    if (M == 1) {
        // the phase u[0] at "parity 0" of no bits
        proto.u[0] = U(0, 0);
        if (g) {
            SweepTrain t = tr;
            t.w00 = G(0, 0).real();
            proto.train.push_back(t);
        }
        if (__builtin_popcountll(proto.test) == 1) { // on one bit: a diagonal 2x2, which merges with others there
            const bool one = proto.value != 0;
            proto.bit = proto.test;
            proto.test = proto.value = 0;
            if (one) {
                std::swap(proto.u[0], proto.u[3]);
                for (auto &t : proto.train) {
                    std::swap(t.w00, t.w11);
                }
            }
        }
        out.push_back(proto);
        return true;
    }
    // the 2x2 of members p and q, which differ in t, t2 and `more`
    auto pair = [&](int p, int q, uint64_t t, uint64_t t2, uint64_t more) {
        if (mem[p] & t) {
            std::swap(p, q);
        }
        SweepOp s = proto;
        s.bit = t;
        s.bit2 = t2;
        s.more = more;
        s.test = touch & ~t;
        s.value = mem[p] & s.test;
        s.u[0] = U(p, p);
        s.u[1] = U(p, q);
        s.u[2] = U(q, p);
        s.u[3] = U(q, q);
        if (g) {
            SweepTrain w = tr;
            w.w00 = G(p, p).real();
            w.w11 = G(q, q).real();
            w.w01 = G(p, q);
            s.train.push_back(w);
        }
        return s;
    };
    if (M == 2) {
        const uint64_t t = vary & (~vary + 1), up = vary & ~t, t2 = up & (~up + 1);
        out.push_back(pair(0, 1, t, t2, up & ~t2));
        return true;
    }
    if (__builtin_popcountll(vary) != 2) {
        return false;
    }
    // four members over two bits: blocks of members that differ in `mix`
    uint64_t mix = 0;
    for (int r = 0; r < 4; r++) {
        for (int c = 0; c < 4; c++) {
            if (r != c && (U(r, c) != 0.0 || G(r, c) != 0.0)) {
                const uint64_t m = mem[r] ^ mem[c];
                if (mix && mix != m) {
                    return false;
                }
                mix = m;
            }
        }
    }
    auto at = [&](uint64_t v) { // the member with these varying bits
        int j = 0;
        while ((mem[j] & vary) != v) {
            j++;
        }
        return j;
    };
    const uint64_t lo = vary & (~vary + 1), hi = vary & ~lo;
    if (mix == 0) {
        const int m0 = at(0), m1 = at(lo), m2 = at(hi), m3 = at(vary);
        if (U(m0, m0) == U(m3, m3) && U(m1, m1) == U(m2, m2) && G(m0, m0) == G(m3, m3) && G(m1, m1) == G(m2, m2)) {
            SweepOp s = proto;
            s.par = vary;
            s.u[0] = U(m0, m0);
            s.u[3] = U(m1, m1);
            if (g) {
                SweepTrain t = tr;
                t.w00 = G(m0, m0).real();
                t.w11 = G(m1, m1).real();
                s.train.push_back(t);
            }
            out.push_back(s);
            return true;
        }
        mix = lo;
    }
    const uint64_t t = mix & (~mix + 1), t2 = mix & ~t;
    const int a = at(0), b = at(mix), c = at(t == mix ? vary & ~mix : hi), d = at(t == mix ? vary : lo);
    SweepOp s0 = pair(a, b, t, t2, 0), s1 = pair(c, d, t, t2, 0);
    auto same = [](const SweepOp &x, const SweepOp &y) {
        bool eq = std::equal(x.u, x.u + 4, y.u) && x.train.size() == y.train.size();
        for (size_t j = 0; eq && j < x.train.size(); j++) {
            eq = x.train[j].w00 == y.train[j].w00 && x.train[j].w11 == y.train[j].w11 && x.train[j].w01 == y.train[j].w01;
        }
        return eq;
    };
    if (same(s0, s1)) { // whatever the other bit is
        s0.test = proto.test;
        s0.value = proto.value;
        out.push_back(s0);
    } else {
        out.push_back(s0);
        out.push_back(s1);
    }
    return true;
}

// Steps in sweep order.  The builder keeps, per bit, the last step touching it.
class SweepSteps {
  public:
    std::vector<SweepOp> steps;
    SweepSteps() { std::fill(last_, last_ + 64, -1); }

    void add(const SweepOp &s) {
        const uint64_t touch = s.touch();
        int at = -2; // the one step last touching all of its bits
        for (uint64_t b = touch; b; b &= b - 1) {
            const int l = last_[__builtin_ctzll(b)];
            at = at == -2 || at == l ? l : -1;
        }
        if (at >= 0 && s.same_place(steps[at])) {
            SweepOp &d = steps[at];
            for (SweepTrain t : s.train) {
                sweep_move(t, d);
                d.train.push_back(t);
            }
            const std::complex<double> m[4] = {
                s.u[0] * d.u[0] + s.u[1] * d.u[2], s.u[0] * d.u[1] + s.u[1] * d.u[3],
                s.u[2] * d.u[0] + s.u[3] * d.u[2], s.u[2] * d.u[1] + s.u[3] * d.u[3]};
            std::copy(m, m + 4, d.u);
            return;
        }
        for (uint64_t b = touch; b; b &= b - 1) {
            last_[__builtin_ctzll(b)] = static_cast<int>(steps.size());
        }
        steps.push_back(s);
    }

    // All steps added: identities leave, diagonal 2x2s become phases (which
    // need no tile bit).
    void finish() {
        std::vector<SweepOp> kept;
        for (auto &s : steps) {
            if (!s.big && s.identity() && s.train.empty()) {
                continue;
            }
            bool diag = !s.big && s.bit && s.diagonal() && !(s.test & (s.bit2 | s.more));
            for (const auto &t : s.train) {
                diag = diag && t.w01 == 0.0;
            }
            if (diag) {
                s.par = s.bit;
                s.bit = s.bit2 = 0;
            }
            kept.push_back(std::move(s));
        }
        steps.swap(kept);
    }

  private:
    int last_[64];
};

// What a step by itself works on: members expand(g, pins) of the state, with
// `value` set, and for pairs their partners across `flip`.
struct SweepLone {
    uint64_t pins = 0, value = 0, flip = 0, par = 0;
};
inline SweepLone sweep_lone(const SweepOp &s) {
    SweepLone l;
    l.pins = s.test | s.bit;
    l.value = s.value;
    if (s.bit) {
        l.flip = s.need();
        l.value &= ~s.bit;
    } else {
        l.par = s.par;
        const bool one = s.train.empty() && __builtin_popcountll(s.par) == 1;
        if (one && s.u[0] == 1.0) { // the other half of them stays
            l.pins |= s.par;
            l.value |= s.par;
        } else if (one && s.u[3] == 1.0) {
            l.pins |= s.par;
        }
    }
    return l;
}

// The step as an operation of the per-gate kernels.
template <class T> GroupOp<T> sweep_group(const SweepOp &s) {
    const SweepLone l = sweep_lone(s);
    auto cast = [](const std::complex<double> &z) {
        return std::complex<T>(static_cast<T>(z.real()), static_cast<T>(z.imag()));
    };
    const std::complex<T> u[4] = {cast(s.u[0]), cast(s.u[1]), cast(s.u[2]), cast(s.u[3])}, none(0);
    std::vector<int> pos;
    auto pin = [&](uint64_t bits) {
        for (uint64_t b = bits; b; b &= b - 1) {
            pos.push_back(__builtin_ctzll(b));
        }
    };
    if (!s.bit) {
        const uint64_t par = s.par & ~l.pins;
        if (l.pins == 0) {
            GroupOp<T> g;
            g.kind = GroupOp<T>::Parity;
            g.parity_mask = par;
            g.parity_phase[0] = u[0];
            g.parity_phase[1] = u[3];
            return g;
        }
        const int np = __builtin_popcountll(par);
        pin(l.pins | par);
        if (np == 0) {
            return make_group<T>(pos, l.value, {0}, {(l.value & s.par) ? u[3] : u[0]}, true);
        }
        const uint64_t p0 = par & (~par + 1);
        if (np == 1) {
            return make_group<T>(pos, l.value, {0, p0}, {u[0], none, none, u[3]}, true);
        }
        if (np > 2) {
            throw std::logic_error("tested phases by the parity of more than two bits");
        }
        return make_group<T>(pos, l.value, {0, p0, par & ~p0, par},
                             {u[0], none, none, none, none, u[3], none, none, none, none, u[3], none, none, none, none,
                              u[0]},
                             true);
    }
    const uint64_t in = l.value & l.flip; // tested bits the pairs differ in
    if (s.bit2 && !(s.test & s.bit2)) {   // (bit, bit2): 00 with 11, 01 with 10
        pin(l.pins | s.bit2);
        return make_group<T>(pos, l.value & ~l.flip, {0, s.bit, s.bit2, s.bit | s.bit2},
                             {u[0], none, none, u[1], none, u[3], u[2], none, none, u[1], u[0], none, u[2], none, none,
                              u[3]},
                             s.diagonal());
    }
    pin(l.pins);
    return make_group<T>(pos, l.value & ~l.flip, {in, in ^ l.flip}, {u[0], u[1], u[2], u[3]}, s.diagonal());
}

struct SweepPass {
    bool big = false;     // one step that no pass holds
    std::vector<int> ops; // step indices, in order
    std::vector<int> hb;  // tile bits above the low ones, ascending
};

// Microseconds a pass's steps take one by one (`alone`) and as a pass
// (`together`), from which the cheaper is taken.  A pass reads and writes every
// amplitude of its states and uploads a program, whatever its steps touch; a
// step by itself is a launch and the traffic of its part of the state.  So a
// few steps on a small state, and operations on an eighth of a large one, go
// one by one.  `first`: no pass before it in the call, so nothing hides its
// upload.
struct SweepCost {
    double alone = 0, together = 0;
};

// Fraction of the state's 128-byte lines that a step by itself touches.
inline double sweep_lines(const SweepLone &l, bool c128) {
    const uint64_t high = ~uint64_t{0} << (c128 ? 3 : 4);
    return ((l.flip & l.pins & high) ? 2.0 : 1.0) /
           static_cast<double>(uint64_t{1} << __builtin_popcountll(l.pins & high));
}

// Forward passes (kernels_pass.hpp against the per-gate kernels, both sides measured):
//   14 qubits       4 RX 34 us one by one, 38 as a pass; 8 65, 43
//   28 qubits c128  4 RX 5480, 1550; 4 CZ 4500, 1510
//   28 qubits c64   8 RX 5510, 1660; 8 CSWAP 1970, 2880
// Of the whole state's time, half its lines take 0.55, a quarter 0.33, and a
// wire inside a line adds 0.3; the phases of a parity take 1.3 times the whole, a
// DoubleExcitation its lines' share times 1.3, or 0.9 in the last-level cache.
// In a pass a DoubleExcitation is a frame of some six steps (16 at 18 qubits 190
// us in passes, 120 one by one; 28 qubits complex64 11.2 and 3.0 ms).
inline SweepCost sweep_forward_us(const std::vector<SweepOp> &steps, const SweepPass &ps, int n, bool c128,
                                  bool first) {
    const double amps = std::ldexp(1.0, n), rw = 2 * amps * (c128 ? 16 : 8); // bytes
    double units = 0; // steps, with the flips and windows of a frame
    SweepCost c;
    for (int i : ps.ops) {
        const SweepLone l = sweep_lone(steps[i]);
        const double f = sweep_lines(l, c128);
        units += 1 + 2.4 * __builtin_popcountll(steps[i].more);
        if (steps[i].more) {
            c.alone += 4 + (rw > 5.4e8 ? 1.3 : 0.9) * rw * f / 6.0e6;
            continue;
        }
        const bool in_line = ((l.pins | l.flip) & (c128 ? 7 : 15)) && l.pins != l.flip;
        const double all = l.flip ? 1 : 1.3;
        c.alone += 4 + rw * ((f >= 1 ? all : f >= 0.5 ? 0.55 : 0.33) + (in_line ? 0.3 : 0)) / 6.0e6;
    }
    c.together = std::max((first ? 19 : 8) + 1.1 * units,
                          rw / (c128 ? 5.7e6 : 3.7e6) + units * amps * (c128 ? 6.3e-8 : 1.9e-7));
    return c;
}

// The backward sweep of lambda and K states (k_sweep against k_sweep_step), for
// 1, 2 and 4 of a gate:
//   6 qubits,       K = 1   CRX 53 54 79 us one by one, 59 64 63 as passes
//   20 qubits c128, K = 4   RX 112 143 207, 118 125 130; CRX 104 118 170, 119 125 136
//   24 qubits c64,  K = 4   RX 570 900 1490, 830 900 960; DoubleExcitation 400 460 990, 920 1070 1850
//   26 qubits c128, K = 1   RX 1850 2720 4290, 1820 1810 1830; DoubleExcitation 1150 1260 2450, 1840 1940 2360
// complex64 passes work in double: their arithmetic is not hidden behind half
// the traffic.
inline double sweep_whole_us(int n, bool c128, int K) { // a step by itself on every amplitude
    return 2 * std::ldexp(1.0, n) * (c128 ? 16 : 8) * (1 + K) / 4.3e6;
}
// DoubleExcitations go alone: a pass's bits hold two of them (16 at 20 qubits c128,
// K = 12: 980 us in passes, 530 alone).  With several launches each on a
// state that passes hold whole, they stay in (6 us each in the pass).
inline bool sweep_backward_alone(const SweepOp &s, int n, bool c128, int K) {
    return s.more && (K <= kStepObs || sweep_whole_us(n, c128, K) > 10);
}
inline SweepCost sweep_backward_us(const std::vector<SweepOp> &steps, const SweepPass &ps, int n, bool c128, int K,
                                   bool first) {
    const double whole = sweep_whole_us(n, c128, K);
    const int launches = (K + kStepObs - 1) / kStepObs;
    SweepCost c;
    double units = 0;
    for (int i : ps.ops) {
        c.alone += 5.0 * launches + whole * std::min(1.0, sweep_lines(sweep_lone(steps[i]), c128) + 0.05);
        units += 1 + 1.7 * __builtin_popcountll(steps[i].more);
    }
    c.together = (first ? 14 : 7) + units * (1.2 + (c128 ? 0.03 : 0.2) * whole) + (c128 ? 1.2 : 1.6) * whole;
    return c;
}

constexpr size_t kSweepLookahead = 1024; // steps scanned per pass
constexpr int kSweepSearchQubits = 18;   // states whose passes outlast a search over single bits on the host

class SweepScheduler {
  public:
    SweepScheduler(int n, int bits, int low, const std::vector<SweepOp> &steps)
        : n_(n), low_(low), budget_(bits - low), lowm_((uint64_t{1} << low) - 1), steps_(steps) {
        pending_.resize(steps.size());
        for (size_t i = 0; i < steps.size(); i++) {
            pending_[i] = static_cast<int>(i);
        }
    }

    bool next(SweepPass &p) {
        p = SweepPass{};
        if (pending_.empty()) {
            return false;
        }
        all_ = 0;
        for (size_t j = 0; j < pending_.size() && j < kSweepLookahead; j++) {
            all_ |= steps_[pending_[j]].touch();
        }
        // high bits claimed in sweep order, padded with the lowest unused
        uint64_t hmask = 0, blocked = 0;
        for (size_t j = 0; j < pending_.size() && j < kSweepLookahead && blocked != all_; j++) {
            const SweepOp &s = steps_[pending_[j]];
            const uint64_t hi = s.need() & ~lowm_;
            if (!s.big && !s.alone && !(s.touch() & blocked) && __builtin_popcountll(hmask | hi) <= budget_) {
                hmask |= hi;
            } else {
                blocked |= s.touch();
            }
        }
        for (int b = low_; b < n_ && __builtin_popcountll(hmask) < budget_; b++) {
            hmask |= uint64_t{1} << b;
        }
        // or runs of neighbouring bits.  A ladder of entanglers makes the
        // steps' front a staircase over the bits: bits claimed in order advance
        // one layer by the whole tile, a run centred on the staircase advances
        // half as many layers as it has bits by half its length (20 qubits, 10
        // ladder layers: 18 passes in claimed order, 8 with runs)
        int best = take(hmask, nullptr, nullptr);
        for (int a = low_; a + budget_ <= n_; a++) {
            const uint64_t m = ((uint64_t{1} << budget_) - 1) << a;
            const int c = take(m, nullptr, nullptr);
            if (c > best) {
                best = c;
                hmask = m;
            }
        }
        if (n_ >= kSweepSearchQubits) {
            exchange(hmask);
        }
        std::vector<int> rest;
        take(hmask, &p.ops, &rest);
        if (p.ops.empty()) { // the first one fits no tile
            p.big = true;
            p.ops.push_back(pending_[0]);
            rest.assign(pending_.begin() + 1, pending_.end());
        }
        for (int b = low_; b < n_; b++) {
            if ((hmask >> b) & 1U) {
                p.hb.push_back(b);
            }
        }
        pending_.swap(rest);
        return true;
    }

  private:
    int take(uint64_t hmask, std::vector<int> *ops, std::vector<int> *left) const {
        uint64_t blocked = 0;
        int taken = 0, slots = 0;
        size_t j = 0;
        for (; j < pending_.size() && j < kSweepLookahead; j++) {
            const SweepOp &s = steps_[pending_[j]];
            const int more = s.train.empty() ? 0 : 1;
            if (!s.big && !s.alone && !(s.touch() & blocked) && (s.need() & ~lowm_ & ~hmask) == 0 && slots + more <= kSweepSlots) {
                taken++;
                slots += more;
                if (ops) {
                    ops->push_back(pending_[j]);
                }
            } else {
                blocked |= s.touch();
                if (left) {
                    left->push_back(pending_[j]);
                }
                if ((blocked & all_) == all_) {
                    j++;
                    break;
                }
            }
        }
        if (left) {
            left->insert(left->end(), pending_.begin() + static_cast<long>(j), pending_.end());
        }
        return taken;
    }

    // The best exchange of one high bit for another while the pass takes more.
    void exchange(uint64_t &hmask) const {
        int best = take(hmask, nullptr, nullptr);
        for (int round = 0; round < 8 && best > 0; round++) {
            uint64_t to = hmask;
            for (int a = low_; a < n_; a++) {
                for (int b = low_; b < n_ && ((hmask >> a) & 1U); b++) {
                    if ((hmask >> b) & 1U) {
                        continue;
                    }
                    const uint64_t m = (hmask & ~(uint64_t{1} << a)) | (uint64_t{1} << b);
                    const int c = take(m, nullptr, nullptr);
                    if (c > best) {
                        best = c;
                        to = m;
                    }
                }
            }
            if (to == hmask) {
                return;
            }
            hmask = to;
        }
    }

    int n_, low_, budget_;
    uint64_t lowm_, all_ = 0;
    const std::vector<SweepOp> &steps_;
    std::vector<int> pending_;
};

// Steps of the longest program a pass of these can have: a step, its window,
// its flips (two on bit2 unless the kernel takes pairs in two bits; a frame
// of two per further bit, each with a window).
inline size_t sweep_longest(const std::vector<SweepOp> &steps, bool two) {
    size_t per = 0;
    for (const SweepOp &s : steps) {
        if (s.big || s.alone) {
            continue;
        }
        per = std::max(per, size_t{2} * (1 + 2 * __builtin_popcountll(s.more)) + (s.bit2 && !two ? 2 : 0));
    }
    return per * std::min(steps.size(), kSweepLookahead);
}

// A pass's program: windows of RB register bits claimed in step order, each
// followed by the steps it can hold (those whose mixing bit is in the window
// and which touch no bit of a step held back).  tb: thread bits of the tile;
// local bits are numbered from the lowest, the first window is the highest RB.
// two: the kernel takes pairs that differ in two register bits (k_pass); else
// such a step runs on its lower bit between CNOTs from it to the other
// (k_sweep, whose registers the further pair patterns would not fit).
inline void sweep_program(const std::vector<SweepOp> &steps, const SweepPass &ps, int low, int tb, int RB, bool two,
                          std::vector<SweepStep> &prog) {
    const int bits = tb + RB;
    uint64_t tile = (uint64_t{1} << low) - 1;
    for (int b : ps.hb) {
        tile |= uint64_t{1} << b;
    }
    auto local = [&](uint64_t v) {
        uint32_t r = static_cast<uint32_t>(v & ((uint64_t{1} << low) - 1));
        for (size_t j = 0; j < ps.hb.size(); j++) {
            r |= static_cast<uint32_t>((v >> ps.hb[j]) & 1U) << (low + j);
        }
        return r;
    };
    uint32_t win = ((1U << RB) - 1) << tb; // local bits of the window
    // of a local mask: the part on register bits, and on thread bits
    auto reg = [&](uint32_t v) {
        uint32_t r = 0;
        for (int b = 0, j = 0; b < bits; b++) {
            if ((win >> b) & 1U) {
                r |= ((v >> b) & 1U) << j++;
            }
        }
        return r;
    };
    auto thread = [&](uint32_t v) {
        uint32_t r = 0;
        for (int b = 0, j = 0; b < bits; b++) {
            if (!((win >> b) & 1U)) {
                r |= ((v >> b) & 1U) << j++;
            }
        }
        return r;
    };
    struct Item {
        const SweepOp *op;
        int slot;
        uint64_t need; // window bits
    };
    std::vector<Item> pending, left;
    std::deque<SweepOp> frames;
    int slots = 0;
    for (int i : ps.ops) {
        const SweepOp &s = steps[i];
        // CNOTs from the pairs' lowest bit bring `more` together; the member
        // with that bit clear, which the tests are on, stays
        const size_t f0 = frames.size();
        for (uint64_t b = s.more; b; b &= b - 1) {
            SweepOp c;
            c.bit = b & (~b + 1);
            c.test = c.value = s.bit;
            c.u[0] = c.u[3] = 0;
            c.u[1] = c.u[2] = 1;
            frames.push_back(c);
            pending.push_back({&frames.back(), -1, c.bit});
        }
        pending.push_back({&s, s.train.empty() ? -1 : slots++, s.bit | s.bit2});
        for (size_t f = f0; f < frames.size(); f++) {
            pending.push_back({&frames[f], -1, frames[f].bit});
        }
    }
    auto put = [&](const Item &it) {
        const SweepOp &s = *it.op;
        SweepStep d{};
        d.slot = it.slot;
        d.omask = s.test & ~tile;
        d.oval = s.value & ~tile;
        d.rm = reg(local(s.test));
        d.rv = reg(local(s.value));
        d.lm = thread(local(s.test));
        d.lv = thread(local(s.value));
        auto cast = [](const std::complex<double> &z) { return dcx<double>{z.real(), z.imag()}; };
        if (s.bit) {
            d.kind = s.flip() && s.train.empty() ? kSweepFlip : kSweepDense;
            const int j1 = __builtin_ctz(reg(local(s.bit)));
            d.j = j1;
            if (s.bit2 && two) { // the pairs (0,1) (0,2) .. (1,2) .. of register bits, after the single ones
                const int j2 = __builtin_ctz(reg(local(s.bit2)));
                d.j = RB + j1 * (2 * RB - j1 - 1) / 2 + (j2 - j1 - 1);
            }
            for (int j = 0; j < 4; j++) {
                d.u[j] = cast(s.u[j]);
            }
            const bool real = s.u[0].imag() == 0 && s.u[1].imag() == 0 && s.u[2].imag() == 0 && s.u[3].imag() == 0;
            const bool cross = s.u[0].imag() == 0 && s.u[1].real() == 0 && s.u[2].real() == 0 && s.u[3].imag() == 0;
            d.form = real ? kSweepReal2 : cross ? kSweepCross2 : kSweepFull2;
        } else {
            d.kind = kSweepDiag;
            d.op = s.par & ~tile;
            d.rp = reg(local(s.par & tile));
            d.lp = thread(local(s.par & tile));
            d.u[0] = cast(s.u[0]);
            d.u[1] = cast(s.u[3]);
        }
        SweepStep f{};
        if (s.bit2 && !two) {
            f.kind = kSweepFlip;
            f.slot = -1;
            f.j = __builtin_ctz(reg(local(s.bit2)));
            f.rm = f.rv = reg(local(s.bit));
            prog.push_back(f);
        }
        prog.push_back(d);
        if (s.bit2 && !two) {
            prog.push_back(f);
        }
    };
    while (!pending.empty()) {
        // steps the window w would take; claim: w grows to RB bits in step order
        auto fill = [&](uint32_t &w, bool claim) {
            uint64_t blocked = 0;
            int taken = 0;
            for (const Item &it : pending) {
                const SweepOp &s = *it.op;
                const uint32_t nd = local(it.need);
                if (!(s.touch() & blocked) && ((nd & ~w) == 0 || (claim && __builtin_popcount(w | nd) <= RB))) {
                    w |= nd;
                    taken++;
                } else {
                    blocked |= s.touch();
                }
            }
            return taken;
        };
        const uint32_t need0 = local(pending[0].need);
        if (need0 & ~win) {
            // the better of the bits claimed in step order and the runs of
            // RB neighbours that hold the first step's bit
            uint32_t m = 0;
            int best = fill(m, true);
            for (int b = bits - 1; b >= 0 && __builtin_popcount(m) < RB; b--) {
                m |= 1U << b;
            }
            const int at = __builtin_ctz(need0);
            for (int b = std::max(0, at - RB + 1); b <= at && b + RB <= bits; b++) {
                uint32_t run = ((1U << RB) - 1) << b;
                const int c = fill(run, false);
                if (c > best) {
                    best = c;
                    m = run;
                }
            }
            win = m;
            SweepStep d{};
            d.kind = kSweepWindow;
            d.slot = -1;
            for (int b = 0, j = 0; b < bits; b++) {
                if ((win >> b) & 1U) {
                    d.rp |= static_cast<uint32_t>(b) << (4 * j++);
                }
            }
            prog.push_back(d);
        }
        left.clear();
        uint64_t blocked = 0;
        for (const Item &it : pending) {
            const SweepOp &s = *it.op;
            if ((s.touch() & blocked) || (local(it.need) & ~win)) {
                blocked |= s.touch();
                left.push_back(it);
            } else {
                put(it);
            }
        }
        pending.swap(left);
    }
}

// <H|W lambda> of a train from its step's sums (kernels_adjoint.hpp); c(i) is sum i.
template <class C> std::complex<double> sweep_value(const SweepTrain &t, bool full, C &&c) {
    const double u = t.w01.real(), v = t.w01.imag();
    const double im = t.w00 * c(0) + t.w11 * c(1) + (u * c(2) + v * c(3));
    return {full ? t.w00 * c(4) + t.w11 * c(5) + (u * c(6) - v * c(7)) : 0.0, im};
}

} // namespace plamd
