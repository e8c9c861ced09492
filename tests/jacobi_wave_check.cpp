// Host check of the wave-front Jacobi schedule (slime_amd/csrc/jacobi_wave.hpp): a plain
// emulation of fitness_finalize_kernel's lanes and work items, step by step, against the
// cyclic row order done one rotation at a time. Test infrastructure: built with g++ by
// tests/test_jacobi_wave.py.
//
// The rotations of both are the kernel's own (jacobi_wave::rotation). `rotation` compares
// that form with the exact angle: t = sign(tau) / (|tau| + sqrt(1 + tau^2)), tau = d / 2 apq,
// c = 1 / sqrt(1 + t^2), s = t c in 64-bit-significand long double, over blocks of every kind
// (both signs of d and apq, d = 0, |d| far above and far below |apq|, |apq| just over 1e-6).
//
// Usage: jacobi_wave_check D seed kind [plant]   kind: dense | lowrank | diag | rank1
//        jacobi_wave_check rotation n seed [plant]   plant "sign": the reference's sine negated
//          for d < 0; "half": its angle taken with tau = d / apq
//   plant "swap-order": the emulation visits each row's pairs one step late against the
//   other rows (a planted mistake).
// Prints "OK sweeps rotations err" or "FAIL ..." and exits 1.
#include <cmath>
#include <cstdio>
#include <cstdlib>
#include <cstring>
#include <random>
#include <set>
#include <string>
#include <utility>
#include <vector>

#include "../slime_amd/csrc/jacobi_wave.hpp"

using namespace slime::jacobi_wave;

namespace {

constexpr double kTol = 1e-6;
constexpr int kUpdateThreads = 512;  // kFinUpdate of fitness.hip

// One rotation at a time, in cyclic row order.
int serial(std::vector<double> A, int D, std::vector<double>& diag, long* nrot) {
    int sweeps = 0;
    for (int sw = 0; sw < 30; ++sw) {
        ++sweeps;
        double off = 0.0;
        long before = *nrot;
        for (int p = 0; p < D - 1; ++p)
            for (int q = p + 1; q < D; ++q) {
                const double apq = A[p * D + q];
                off += std::fabs(apq);
                if (std::fabs(apq) <= kTol) continue;
                ++*nrot;
                double c, s;
                const double app = A[p * D + p], aqq = A[q * D + q];
                rotation(app, aqq, apq, c, s);
                for (int i = 0; i < D; ++i) {
                    if (i == p || i == q) continue;
                    const double ip = A[i * D + p], iq = A[i * D + q];
                    A[i * D + p] = A[p * D + i] = c * ip - s * iq;
                    A[i * D + q] = A[q * D + i] = s * ip + c * iq;
                }
                A[p * D + p] = c * c * app + s * s * aqq - 2.0 * c * s * apq;
                A[q * D + q] = s * s * app + c * c * aqq + 2.0 * c * s * apq;
                A[p * D + q] = A[q * D + p] = 0.0;
            }
        if (off < kTol * D) break;
        if (*nrot == before) {
            sweeps = 30;
            break;
        }
    }
    for (int i = 0; i < D; ++i) diag[i] = A[i * D + i];
    return sweeps;
}

struct Lane {
    double c = 1, s = 0, app = 0, aqq = 0, off = 0, snap = 0, offs = 0;
    bool rot = false, rots = false;
};

int wave(const std::vector<double>& A0, int D, std::vector<double>& diag, bool plant) {
    const int S = D / 2;
    std::vector<double> A[2] = {A0, A0};
    std::vector<Lane> L(D);
    for (int p = 0; p < D; ++p) {
        L[p].app = A0[p * D + p];
        const Role r = role(0, p, D);
        if (r.pair) L[p].aqq = A0[r.q * D + r.q];
    }
    int cur = 0;
    bool any = false;  // a rotation at step T
    for (int T = 0;; ++T) {
        const int sig = T % D, sig1 = (T + 1) % D;
        // the update of step T, from A[cur] to A[1 - cur]; its rotations are in L
        if (any) {
            std::vector<double> cc(D), ss(D);
            std::set<int> covered;
            for (int p = 0; p < D; ++p) {
                const Role r = role(sig, p, D);
                if (r.pair) {
                    cc[p] = cc[r.q] = L[p].c, ss[p] = -L[p].s, ss[r.q] = L[p].s;
                    covered.insert(p), covered.insert(r.q);
                } else if (r.self) {
                    cc[p] = 1, ss[p] = 0;
                    covered.insert(p);
                }
            }
            if ((int)covered.size() != D) std::printf("FAIL indices without a rotation at T=%d\n", T), std::exit(1);
            std::set<int> written;
            auto put = [&](int i, int j, double v) {
                if (!written.insert(upper(i, j, D)).second) std::printf("FAIL element written twice\n"), std::exit(1);
                A[1 - cur][upper(i, j, D)] = v;
            };
            for (int n = 0; n < kUpdateThreads; ++n) {  // one item per thread of the kernel
                int i1, j1, i2, j2;
                SLIME_JACOBI_ITEM(n, S, d1, d2, valid);
                if (!valid) continue;
                slot(sig, d1, D, &i1, &j1);
                slot(sig, d2, D, &i2, &j2);
                const std::vector<double>& M = A[cur];
                const double a = M[upper(i1, i2, D)], b = M[upper(i1, j2, D)], c = M[upper(j1, i2, D)],
                             d = M[upper(j1, j2, D)];
                const double c1 = cc[i1], s1 = ss[i1], c2 = cc[i2], s2 = ss[i2];
                const double ar = c1 * a + s1 * c, br = c1 * b + s1 * d, cr = c1 * c - s1 * a, dr = c1 * d - s1 * b;
                put(i1, i2, c2 * ar + s2 * br);
                put(i1, j2, c2 * br - s2 * ar);
                put(j1, i2, c2 * cr + s2 * dr);
                put(j1, j2, c2 * dr - s2 * cr);
            }
            for (int d = 0; d < S; ++d) {
                int i, j;
                slot(sig, d, D, &i, &j);
                put(i, j, ss[i] != 0.0 ? 0.0 : A[cur][upper(i, j, D)]);
            }
            if ((int)written.size() != D * (D - 1) / 2) std::printf("FAIL %d elements written\n", (int)written.size()), std::exit(1);
        }
        // the rotations of step T + 1, from A[cur] (before step T) and step T's rotations
        std::vector<Lane> N = L;
        bool any1 = false;
        for (int p = 0; p < D; ++p) {
            const Role r = role(sig1, p, D);
            if (!r.pair && !r.self) continue;
            const Lane& me = L[p];
            const double cB = p ? L[p - 1].c : L[sig1].c, sB = p ? L[p - 1].s : -L[sig1].s;
            const double dB = p ? L[p - 1].aqq : L[sig1].app;
            Lane& o = N[p];
            if (r.self) {
                o.app = p ? dB : me.app;
                o.c = 1, o.s = 0, o.off = 0, o.rot = false;
                if (p == D - 1) o.snap = o.app, o.offs = 0, o.rots = false;
                continue;
            }
            const int m = q_partner_before(p, D), q = r.q;
            const std::vector<double>& M = A[cur];
            const double e1 = M[upper(p, m, D)], e2 = M[upper(p, q, D)];
            const double e3 = M[upper(q - 1, m, D)], e4 = M[upper(q - 1, q, D)];
            const double x = me.c * e1 - me.s * e3, y = me.c * e2 - me.s * e4;
            double apq = sB * x + cB * y;
            if (plant) apq = e2;
            const bool real = T + 1 - sig1 - (r.prev ? D : 0) >= 0;
            const bool rotate = real && std::fabs(apq) > kTol;
            if (real) o.off += std::fabs(apq);
            o.rot |= rotate;
            any1 |= rotate;
            o.c = 1, o.s = 0, o.aqq = dB;
            if (rotate) {
                double c, s;
                const double app = me.app, aqq = dB;
                rotation(app, aqq, apq, c, s);
                o.c = c, o.s = s;
                o.app = c * c * app + s * s * aqq - 2.0 * c * s * apq;
                o.aqq = s * s * app + c * c * aqq + 2.0 * c * s * apq;
            }
            if (q == D - 1) o.snap = o.app, o.offs = o.off, o.rots = o.rot;
        }
        if (any) cur = 1 - cur;
        L = N;
        any = any1;
        if (sig1 == D - 2 && T + 1 >= 2 * D - 2) {
            const int sweeps = (T + 1) / D;
            double off = 0;
            bool rots = false;
            for (int p = 0; p < D; ++p) off += L[p].offs, rots |= L[p].rots;
            if (off < kTol * D || !rots || sweeps == 30) {
                for (int p = 0; p < D; ++p) diag[p] = L[p].snap;
                return !(off < kTol * D) && !rots ? 30 : sweeps;
            }
        }
    }
}

// The roundings of jacobi_wave::rotation in turn (stated there) bound c by 2.3 u and s by 8.3 u
// relative, u = 2^-53, and so c^2 + s^2 - 1 by 2 (2.3 c^2 + 8.3 s^2) u, at most 10.6 u.
int rotation_check(long n, int seed, const std::string& plant) {
    std::mt19937_64 rng(seed);
    std::uniform_real_distribution<double> u01(0.0, 1.0);
    auto mag = [&](double lo, double hi) { return std::exp2(lo + (hi - lo) * u01(rng)); };
    const long double u = 0x1p-53L;
    long double ec = 0, es = 0, en = 0;
    for (long i = 0; i < n; ++i) {
        double app = mag(-24, 8), aqq = mag(-24, 8), apq = mag(-19, 8);
        switch (i % 6) {
            case 1: aqq = app; break;
            case 2: apq = 1e-6 * (1.0 + 1e-3 * u01(rng)); break;
            case 3: app = mag(40, 290), apq = mag(-19, 0); break;      // |d| >> |b|
            case 4: aqq = app * (1.0 + 0x1p-50 * (double)(i % 13)); apq = mag(0, 290); break;  // |b| >> |d|
            case 5: std::swap(app, aqq); aqq = mag(40, 290), apq = mag(-19, 290); break;
            default: break;
        }
        if (i & 8) apq = -apq;
        if (i & 16) std::swap(app, aqq);
        double c, s;
        rotation(app, aqq, apq, c, s);
        const double d = aqq - app;  // rounded, as in every form
        const long double tau = (long double)d / ((plant == "half" ? 1.0L : 2.0L) * apq);
        long double t = 1.0L / (std::fabs(tau) + std::sqrt(1.0L + tau * tau));
        if (tau < 0.0L) t = -t;
        const long double rc = 1.0L / std::sqrt(1.0L + t * t);
        long double rs = t * rc;
        if (plant == "sign" && d < 0.0) rs = -rs;
        ec = std::fmax(ec, std::fabs(c - rc) / rc / u);
        es = std::fmax(es, std::fabs(s - rs) / std::fabs(rs) / u);
        en = std::fmax(en, std::fabs((long double)c * c + (long double)s * s - 1.0L) / u);
    }
    const bool ok = ec <= 2.3L && es <= 8.3L && en <= 10.6L;
    std::printf("%s rotation c %.2Lf u, s %.2Lf u, norm %.2Lf u\n", ok ? "OK" : "FAIL", ec, es, en);
    return ok ? 0 : 1;
}

}  // namespace

int main(int argc, char** argv) {
    if (argc < 4) return 2;
    if (!std::strcmp(argv[1], "rotation"))
        return rotation_check(std::atol(argv[2]), std::atoi(argv[3]), argc > 4 ? argv[4] : "");
    const int D = std::atoi(argv[1]);
    const std::string kind = argv[3];
    std::mt19937_64 rng(std::atoi(argv[2]));
    std::uniform_real_distribution<double> u(0.0, 1.0);
    const int n = kind == "lowrank" ? D / 2 : kind == "rank1" ? 1 : 16 * D;
    std::vector<double> X((size_t)n * D), A((size_t)D * D, 0.0);
    for (double& v : X) v = (float)(kind == "rank1" ? u(rng) - 0.5 : u(rng));
    for (int i = 0; i < D; ++i)
        for (int j = 0; j < D; ++j)
            for (int k = 0; k < n; ++k)
                if (kind != "diag" || i == j) A[i * D + j] += X[k * D + i] * X[k * D + j] / n;
    std::vector<double> d0(D), d1(D);
    long nrot = 0;
    const int s0 = serial(A, D, d0, &nrot), s1 = wave(A, D, d1, argc > 4 && !std::strcmp(argv[4], "swap-order"));
    double big = 0, err = 0;
    for (int i = 0; i < D; ++i) big = std::fmax(big, std::fabs(d0[i])), err = std::fmax(err, std::fabs(d0[i] - d1[i]));
    const bool ok = s0 == s1 && err <= 1e-12 * big;
    std::printf("%s sweeps %d %d rotations %ld err %.2e\n", ok ? "OK" : "FAIL", s0, s1, nrot, err / big);
    return ok ? 0 : 1;
}
