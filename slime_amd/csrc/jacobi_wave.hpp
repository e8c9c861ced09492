// jacobi_wave.hpp — the rotation and the schedule of the Jacobi solve in fitness.hip: the cyclic row order of
// the rotations (0,1), (0,2), ..., (0,D-1), (1,2), ..., (D-2,D-1), (0,1), ... run as a wave
// front. Plain C++ with no HIP types, shared with tests/jacobi_wave_check.cpp.
//
// Rotations on disjoint index pairs commute, so only the order of rotations that share an
// index matters. Pair (p, q), p < q, of sweep s runs at step T = s D + p + q: every
// rotation before it in cyclic order that shares p or q then has a smaller T, across
// sweeps too ((p, D-1) of one sweep at s D + p + D - 1, (0, p) of the next at
// (s + 1) D + p). All pairs of one T are disjoint: with sig = T mod D they are the pairs
// with p + q = sig (of the sweep that began at T - sig) and p + q = sig + D (of the sweep
// before), so a sweep takes D steps instead of D (D - 1) / 2.
#pragma once

#if defined(__HIPCC__)
#define SLIME_JHD __host__ __device__ __forceinline__
#else
#define SLIME_JHD inline
#endif

namespace slime {
namespace jacobi_wave {

// What lane p (0 .. D-1) does at a step: the pair (p, q) when q > p (pair), nothing but
// keep index p when q == p (self), nothing when index p is the larger one of its pair.
// `prev`: the pair belongs to the sweep before the one that starts at T - sig.
struct Role {
    int q;
    bool pair, self, prev;
};
SLIME_JHD Role role(int sig, int p, int D) {
    Role r;
    r.prev = p > sig;
    r.q = (sig - p) & (D - 1);  // D is a power of two
    r.pair = r.q > p;
    r.self = r.q == p;
    return r;
}

// The step before, index q of lane p's pair was rotated with index p - 1, in lane p - 1;
// for p = 0 with index D - 1 of the sweep before, in lane q (as that pair's smaller index).
SLIME_JHD int q_partner_before(int p, int D) { return p > 0 ? p - 1 : D - 1; }

// The two indices of slot d (0 .. D/2 - 1) at a step: the pairs of that step, and for even
// sig slot 0 with the two indices that rest.
SLIME_JHD void slot(int sig, int d, int D, int* i, int* j) {
    const int odd = sig & 1, h = sig >> 1;
    *i = (h - d) & (D - 1);
    *j = (!odd && d == 0 ? h + D / 2 : h + d + odd) & (D - 1);
}

// Work items of a step, one per unordered pair of slots: item n covers slots d1 = n mod S
// and d2 = (d1 + o) mod S, o = n / S + 1, S = D / 2; of the offset o = S / 2 only the first half
// counts, and no larger offset does (valid = false). A macro, because the compiler orders the
// kernel's loop differently when these expressions come from an inlined function: the
// solve of 128 Grams then takes 36 us longer (750 us -> 786 us for the whole fitness).
#define SLIME_JACOBI_ITEM(n, S, d1, d2, valid)                             \
    const int d1 = n & (S - 1), o = n / S + 1, d2 = (d1 + o) & (S - 1);    \
    const bool valid = o <= S / 2 && (o < S / 2 || d1 < S / 2)

// The rotation of the cyclic Jacobi solve for the 2x2 block [[app, apq], [apq, aqq]],
// |apq| > 0, the one with |angle| <= pi / 4: with d = aqq - app and b = 2 apq,
// |cos 2 theta| = |d| / sqrt(d^2 + b^2), c = sqrt((1 + |cos 2 theta|) / 2) and
// s = sin 2 theta / (2 c) with the sign of d b (+ at d = 0). The same angle as
// t = sign(tau) / (|tau| + sqrt(1 + tau^2)), tau = d / b, c = 1 / sqrt(1 + t^2), s = t c (the
// oracle's form), with two square roots in a row instead of four operations. No difference of
// close numbers appears, so with u = 2^-53 the roundings in turn give, relative to the exact
// rotation of the rounded d: 1 / sqrt(d^2 + b^2) 3 u, c 2.3 u, 1 / c 3.3 u and s 8.3 u.
// fp64.hpp has the same steps with short square roots, bit for bit.
SLIME_JHD void rotation(double app, double aqq, double apq, double& c, double& s) {
    const double d = aqq - app, b = 2.0 * apq;
    const double r = 1.0 / __builtin_sqrt(__builtin_fma(d, d, b * b));
    c = __builtin_sqrt(__builtin_fma(0.5 * __builtin_fabs(d), r, 0.5));
    const double sb = d < 0.0 ? -apq : (d > 0.0 ? apq : __builtin_fabs(apq));
    s = sb * r * (1.0 / c);
}

// Element (i, j) of the symmetric matrix, kept once.
SLIME_JHD int upper(int i, int j, int D) { return i < j ? i * D + j : j * D + i; }

}  // namespace jacobi_wave
}  // namespace slime
