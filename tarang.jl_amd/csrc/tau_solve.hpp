// tau_solve.hpp -- direct O(N) solves of the per-mode Chebyshev-tau systems of the channel
// solvers (2-D and 3-D), FP64 throughout.
//
// Per mode (horizontal wavenumber kh, implicit coefficient c, s = 2/Lz), with ux = i ux~ and
// the horizontal velocity rotated onto k_h (3-D), every system is real:
//   E2  : (1 + c kappa kh^2) b - c kappa D^2 b  + taus = R2              walls b(0), b(Lz)
//   perp: (1 + c nu kh^2) v  - c nu D^2 v       + taus = -sin R3x + cos R3y   (3-D), v = 0
//   E3x : (1 + c nu kh^2) u~ - c nu D^2 u~ + c kh p + taus = R3x          u~ = 0 on the walls
//   E1  : -c kh u~ + c D uz + c tau_u1z T_{N-1} (+ c tau_p at kh = 0) = R1
//   E3z : (1 + c nu kh^2) uz - c nu D^2 uz + c D p - c b + taus = R3z     uz = 0
// The lift of a tau_*2 is T_{N-1}, that of a tau_*1 is D T_{N-1}.  D^2 keeps the parity of the
// Chebyshev index, so every line (one field, one parity) is a problem of its own:
//   alpha u - beta D^2 u = r + D G  (unit-interval D, beta = c diff s^2),  sum_k u_k = w.
//
// Line solve.  Applying the second integral B ((B f)_k from f_{k-2}, f_k, f_{k+2}, k >= 2)
// turns a line into a tridiagonal recursion (m = alpha/beta)
//   u_k - m (B u)_k = -((B r)_k + (int G)_k)/beta,   (int G)_k = (G_{k-1} - G_{k+1})/(2k),
// whose matrix is an M-matrix (diagonally dominant, so no pivoting), eliminated from the top
// degree down.  With j counting the degrees of the parity and t_k = (k-1)/(k+1):
//   e_j = a_j t_j e_{j+1} - (a_j/alpha) (r_{j-1} - (1 + t) r_j + t r_{j+1} + 2(k-1)(G_{k-1} - G_{k+1}))
//   u_j = a_j u_{j-1} + e_j,  and u_0 from the wall sum (all weights of one sign).
// (k = 2 halves all but r_{j-1}: T_0 integrates with twice the weight.)  The lifts only touch the
// top rows ("A": the parity of N - 1, "B": the other), and only through their coefficients:
//   A: row N-1 is the tau_*2 row: r_{N-1} leaves the recursion and u_{N-1} follows from the second
//      integral alone (t = -1, a = m/(4 (N-1)(N-2))); row N-3 has no upper neighbour
//   B: D T_{N-1} has the coefficients 2(N-1) (half of it at 0), which B maps to zero below row
//      N-2, so only row N-2 changes (t = 0, G_{N-1} drops out)
// Where m is large (tau_psi_bound) the same recursion runs on psi = m u - r/beta instead, closed by
// sum psi = m w - sum r/beta: u = (beta psi + r)/alpha then keeps the digits that the second
// integral would lose.
//
// Pressure.  kh E3x + D E3z - (1 + ...) E1 leaves, exactly, with d = R1/c,
//   p = p' + nu d,   c kh^2 p' - c s^2 D^2 p' = kh R3x + d - s D (R3z + c b) + lift terms:
// a line with an unknown wall value lambda per parity.  p = p_0 + lambda p_1 (and u~, uz alike);
// lambda follows from E1 on the wall, s sum k^2 uz_k + tau_u1z - sum d = 0.  The responses u~_1,
// uz_1, p_1 depend on (kh, c) only and come from the set-up kernel.  kh = 0 decouples: uz is the
// integral of E1, p the integral of E3z.
// At small kh (tau_low_kh) uz is what little the pressure gradient leaves of R3z, so the digits that
// E3z loses there are those of uz.  E1 keeps them: from degree 1 on uz is the integral of f = d + kh u~
// (row N - 1: tau_u1z = f_{N-1}), its degree 0 the wall sum, and lambda makes the two agree: for an odd
// uz the integral's wall sum vanishes, for an even one its degree 0 is that of the E3z line.
//
// A solve reads the right-hand-side rows and 6 N doubles per |k_h| key and writes the solution (3-D 256 x 256 x 128:
// 0.34 GB in FP32, 0.65 GB in FP64; measured 0.38 and 0.70); the set-up is one small kernel.
#pragma once
#include <cmath>
#include <type_traits>

#include "common.hpp"

namespace tarang {

// From which |m| on the psi-form takes u_{N-1} (A) from the wall sum's remainder, which rounds with sum |u|, and
// not from the recursion, whose amplitudes pass through a_{N-1} = m/(4 N^2).  Over N = 9 .. 256 and m = 0.2 N^2 ..
// 1e5 N^2 the mean errors are those of a choice by running error sums, which take a scan per line.
__host__ __device__ inline double tau_rest_bound(int N) { return 64.0 * N * N; }
// Where the psi-form starts, as a bound on |m|.  FP64: at N^2/8, where the two are equally far from a
// long-double solve (N = 128: 2e-16 and 1e-16 of the line's 2-norm at m = N^2/20, 4e-16 and 1e-16 at
// 16 N^2, 1e-15 and 2e-16 at 1000 N^2; a dense LU 2e-16); with uz from E1 (below) the psi-form costs 256 x 256 x
// 128 188 -> 210 us and 320 x 97 7.4 -> 9.4 us, at m = 20 .. 45 N^2.  FP32 rounds the result at 6e-8, and the psi-form
// keeps r in registers beside the recursion: it starts where the u-form's u_{N-1}, which loses
// m/(4 N^2) eps |u_{N-3}|, would lose 4 eps (64 from 64 degrees on).
inline double tau_psi_bound(int N, bool fp64) { return (fp64 ? 0.125 : N < 64 ? 16.0 : 256.0) * N * N; }
// Up to which kh uz is the integral of E1, in units of s; -1: never.  Against long-double solves at N = 128
// and m = 30 N^2 / 1000 N^2, uz from E3z / from E1 / by a dense inverse is off by 5e-14 / 1e-15 / 1e-15 and
// 1e-13 / 4e-16 / 2e-15 at kh = 0.8 s, 2e-15 / 7e-16 / 1e-15 at 8 s, 1e-15 / 1e-15 / 1e-15 at 18 s and
// 5e-16 / 2e-15 / 1e-15 at 50 s: the integral carries kh eps |u~|.  Few degrees bring the line
// forward.  FP32 rounds at 6e-8 and takes the E3z line throughout.
inline double tau_low_kh(int N, double s, bool fp64) { return fp64 ? s * (N < 64 ? 0.25 * N : 16.0) : -1.0; }

__host__ __device__ inline int npar(int N, int g) { return (N + 1 - g) / 2; }  // #k in [0,N) with k%2 == g

// Lanes of a wave per mode (G) and degrees per lane and parity (E): lane l holds k = 2 E l .. 2 E l +
// 2 E - 1.  A table row stores degree k at (k % 2E) G + k / 2E, so that the lanes read it side by side.
struct TauShape {
    int G, E;
};
// Which recursion the solves run: kTauU and kTauPsi eliminate without pivoting, which the M-matrix of positive
// diffusivities allows; with a negative one (kTauAny) the lines of m <= 0 are solved by tau_bordered.
enum TauForm : int { kTauU = 0, kTauPsi = 1, kTauAny = 2 };
inline bool tau_any_sign(double kappa, double nu) { return kappa < 0.0 || nu < 0.0; }
__host__ __device__ inline int tau_row(const TauShape& h) { return 2 * h.E * h.G; }
__host__ __device__ inline int tau_slot(const TauShape& h, int k) { return (k % (2 * h.E)) * h.G + k / (2 * h.E); }
// 3-D: four modes per pair of waves up to N = 128 (scans stay within the 16-lane rows of the DPP shifts),
// two above; 2-D has few modes: as many lanes per mode as degrees allow
// (any sign: one shape for all N, one mode per pair of waves)
inline TauShape tau_shape(int N, bool three, bool any) {
    if (any) return three ? TauShape{64, 2} : TauShape{64, 4};
    if (three) return N <= 32 ? TauShape{16, 1} : N <= 64 ? TauShape{16, 2} : N <= 128 ? TauShape{16, 4} : TauShape{32, 4};
    return N <= 64 ? TauShape{32, 1} : N <= 128 ? TauShape{64, 1} : N <= 256 ? TauShape{64, 2} : TauShape{64, 4};
}

// doubles per key of the set-up table: rows a_j of b, u, p (1 at k = 0, 1), responses p_1, u~_1, uz_1,
// then scalars; after the last key the four coefficient rows of tau_coeffs
enum { kTabB = 0, kTabU = 1, kTabP = 2, kTabP1 = 3, kTabX1 = 4, kTabZ1 = 5 };
// scalars, [parity]: 1/sum of the homogeneous b, u, p lines; 1/q_1 (q: the condition on lambda), tau_u1z of uz_1,
// top psi of u~_1 (by p's parity) and alpha/beta, 1/alpha, beta, 1/beta of the b, u, p lines (kScLine + 4 op)
enum { kScB = 0, kScU = 2, kScP = 4, kScQ = 6, kScTz = 8, kScPsi = 10, kScLine = 12 };
constexpr int kTauScalars = 24;
__host__ __device__ inline size_t tau_table_stride(const TauShape& h) { return (size_t)6 * tau_row(h) + kTauScalars; }
inline size_t tau_table_doubles(const TauShape& h, size_t keys) { return keys * tau_table_stride(h) + 4 * tau_row(h); }

struct TauLine {
    double m, ial, beta, ibeta;  // alpha/beta, 1/alpha, beta, 1/beta
    bool psi;
};
__host__ __device__ inline TauLine tau_line(double alpha, double beta, double bound) {
    const double m = alpha / beta;
    return TauLine{m, 1.0 / alpha, beta, 1.0 / beta, fabs(m) > bound};
}
// the r_{k-2} entry of row k of the second integral, k >= 2
__host__ __device__ inline double tau_lo(int k) { return (k == 2 ? 2.0 : 1.0) / (4.0 * k * (k - 1.0)); }
// Row k of the second integral, relative to its r_{k-2} entry: t1 r_{k+2} - t2 r_k + g1 G_{k-1} - g2 G_{k+1},
// with the lifts' changes in the top rows (A: rows N-3 and N-1, B: row N-2)
struct TauCoeffs {
    double t1, t2, g1, g2;
};
__host__ __device__ inline TauCoeffs tau_coeffs(int N, int k) {
    if (k < 2 || k >= N) return TauCoeffs{0.0, 0.0, 0.0, 0.0};
    const double icc = k == 2 ? 0.5 : 1.0, g = icc * 2.0 * (k - 1.0);
    if (k == N - 1) return TauCoeffs{0.0, 0.0, g, 0.0};
    if (k == N - 2) return TauCoeffs{0.0, icc, g, 0.0};
    const double t = (k - 1.0) / (k + 1.0);
    return TauCoeffs{k == N - 3 ? 0.0 : icc * t, icc * (1.0 + t), g, g};
}

// a_j of one line (a[k], k = 2j + g >= 2); returns 1/W_0, W_0 = the wall sum of u_0 = 1, u_j = a_j u_{j-1}
__host__ __device__ inline double tau_factor_line(int N, int g, double m, double* a) {
    const bool A = g == ((N - 1) & 1);
    const int n = npar(N, g);
    double an = 0.0, W = 1.0;  // a_{j+1}, W_j
    int j = n - 2;
    if (A) {
        a[N - 1] = m / (4.0 * (N - 1) * (N - 2));
        W = 1.0 + a[N - 1];
    } else {
        const int k = N - 2;
        const double lo = tau_lo(k), cb = k == 2 ? 0.5 : 1.0;
        an = m * lo / (1.0 + m * lo * cb);
        a[k] = an;
        W = 1.0 + an;
    }
    for (; j >= 1; --j) {
        const int k = 2 * j + g;
        const double lo = tau_lo(k);
        const bool up = !(A && j == n - 2);
        const double den = 1.0 + m / (2.0 * ((double)k * k - 1.0)) - (up ? m / (4.0 * k * (k + 1)) * an : 0.0);
        an = m * lo / den;
        a[k] = an;
        W = 1.0 + an * W;
    }
    return 1.0 / W;
}

// One line by pivoted elimination, for m of any sign: the rows j = 1 .. n-1 of the recursion (in columns
// j-1, j, j+1) are upper triangular when row j pivots column j-1, and the wall sum is a last row of ones.  Each
// step eliminates with the larger of the band row and that last row, which stays constant beyond its two
// leading entries, so a line costs O(n).  S: five doubles per row, S[5 j + 4] the right-hand side of row j on
// entry and u_j on return; wt: the wall sum.  False: an exactly zero pivot (the line is singular).
// Against long-double solves: 2e-15 of the line's 2-norm up to m = -10 N^2; beyond, where the 1 of a row is
// small beside m/(4 k^2) and nothing resolves the solution, up to 1e-13 (m = -300 N^2).
__host__ __device__ inline bool tau_bordered(int N, int g, double m, double wt, double* S) {
    const int n = npar(N, g);
    double d0 = 1.0, d1 = 1.0, dt = 1.0, dr = wt;  // the last row: columns j, j + 1, beyond; right-hand side
    bool ok = true;
    for (int j = 0; j < n - 1; ++j) {
        const int k = 2 * (j + 1) + g;
        const TauCoeffs t = tau_coeffs(N, k);
        const double lo = m * tau_lo(k), b0 = -lo, b1 = 1.0 + lo * t.t2, b2 = -lo * t.t1, br = S[5 * (j + 1) + 4];
        double* U = S + 5 * j;
        if (fabs(b0) >= fabs(d0)) {
            const double l = d0 / b0;
            ok = ok && b0 != 0.0;
            U[0] = b0, U[1] = b1, U[2] = b2, U[3] = 0.0, U[4] = br;
            d0 = d1 - l * b1;
            d1 = dt - l * b2;
            dr -= l * br;
        } else {
            const double l = b0 / d0;
            U[0] = d0, U[1] = d1, U[2] = dt, U[3] = dt, U[4] = dr;
            d0 = b1 - l * d1;
            d1 = b2 - l * dt;
            dt = -l * dt;
            dr = br - l * dr;
        }
    }
    ok = ok && d0 != 0.0;
    double x1 = dr / d0, x2 = 0.0, tail = 0.0;  // u_{j+1}, u_{j+2}, sum beyond
    S[5 * (n - 1) + 4] = x1;
    for (int j = n - 2; j >= 0; --j) {
        double* U = S + 5 * j;
        const double x = (U[4] - U[1] * x1 - U[2] * x2 - U[3] * tail) / U[0];
        U[4] = x;
        tail += x2;
        x2 = x1;
        x1 = x;
    }
    return ok;
}

struct TauSums {
    double k2;   // sum k^2 u_k
    double psi;  // B: psi at degree N - 2 (the D T_{N-1} amplitude before the G term)
    bool ok = true;  // no zero pivot
};

// One line of parity g by one thread (set-up, and the reference of the wave-parallel solve): r(k), G(k)
// read the data, e is scratch (ANY: 5 npar doubles, else N), iW = tau_factor_line's result.
template <bool ANY, typename RF, typename GF>
__host__ __device__ inline TauSums tau_solve_line(int N, int g, const TauLine& L, const double* a, double iW, RF r, GF G,
                                                  double* e, double* u, double w) {
    const int n = npar(N, g);
    const bool A = g == ((N - 1) & 1), piv = ANY && !(L.m > 0.0);
    auto rr = [&](int k) { return k >= N - 1 + (A ? 0 : 1) ? 0.0 : r(k); };  // r_{N-1} is the tau_*2 row
    auto GG = [&](int k) { return k >= N ? 0.0 : G(k); };
    double en = 0.0;
    for (int j = n - 1; j >= 1; --j) {
        const int k = 2 * j + g;
        const TauCoeffs t = tau_coeffs(N, k);
        const double dg = t.g1 * GG(k - 1) - t.g2 * GG(k + 1);
        const double f = L.psi ? 2.0 * k * t.g1 * rr(k) + L.m * dg : rr(k - 2) + t.t1 * rr(k + 2) - t.t2 * rr(k) + dg;
        if (piv) {
            e[5 * j + 4] = -tau_lo(k) * L.ibeta * f;
        } else {
            en = a[k] * (t.t1 * en - L.ial * f);
            e[k] = en;
        }
    }
    double Q = 0.0, sum = 0.0, rs = rr(g);
    for (int j = 1; j < n; ++j) {
        const int k = 2 * j + g;
        if (!piv) {
            Q = a[k] * Q + e[k];
            sum += Q;
        }
        rs += rr(k);
    }
    const double wt = L.psi ? L.m * w - rs * L.ibeta : w;
    const bool rest = A && L.psi && fabs(L.m) > tau_rest_bound(N);
    double x = 0.0, su = 0.0;
    TauSums out{0.0, 0.0};
    if (piv) out.ok = tau_bordered(N, g, L.m, wt, e);
    else x = (wt - sum) * iW;
    for (int j = 0; j < n; ++j) {
        const int k = 2 * j + g;
        if (piv) x = e[5 * j + 4];
        else if (j > 0) x = a[k] * x + e[k];
        double v = L.psi ? (L.beta * x + rr(k)) * L.ial : x;
        if (rest && k == N - 1) v = w - su;
        su += v;
        u[k] = v;
        out.k2 += (double)k * k * v;
    }
    if (!A) out.psi = L.psi ? x : L.m * x - rr(N - 2) * L.ibeta;
    return out;
}

struct TauSys {
    int N;
    TauShape shape;
    int nkeys;
    double c, s, kappa, nu;  // implicit coefficient, 2/Lz, diffusivities
    const double* kh;        // |k_h| per key (null: kh = k0x * key)
    double k0x;
    double* table;           // tau_table_doubles
    double bound, low;       // tau_psi_bound, tau_low_kh
    int* info;               // any sign: per key, the systems that met a zero pivot (bit 0 b, 1 perp, 2 u-p)
};
__device__ inline double tau_kh(const TauSys& t, int key) { return t.kh ? t.kh[key] : t.k0x * key; }
// set-up LDS: 6 N doubles of table rows, and the scratch of the lines that run side by side
inline size_t tau_setup_lds(int N, bool any) {
    return (size_t)(6 * N + (any ? 2 * 5 * npar(N, 0) : 4 * N)) * sizeof(double);
}

// The set-up table of one key per workgroup (64 threads): six lanes run the factor recursions, then
// the lambda = 1 responses run as lines of their own.  LDS: tau_setup_lds.
template <bool ANY>
__global__ __launch_bounds__(64) void k_tau_setup(TauSys t) {
    extern __shared__ unsigned char smem_raw[];
    const int N = t.N, key = (int)blockIdx.x, tid = (int)threadIdx.x;
    double* tab = reinterpret_cast<double*>(smem_raw);  // [6][N]
    double* E = tab + 6 * N + (ANY ? (tid & 1) * 5 * npar(N, 0) : (tid & 3) * N);  // scratch row of a thread at work
    __shared__ double sc[kTauScalars];
    __shared__ int bad;
    const double kh = tau_kh(t, key), c = t.c, s = t.s;
    const int PL = (N - 1) & 1;
    for (int i = tid; i < 6 * N; i += 64) tab[i] = 0.0;
    if (tid < kTauScalars) sc[tid] = 0.0;
    if (tid == 0) bad = 0;
    __syncthreads();
    const TauLine lb = tau_line(1.0 + c * t.kappa * kh * kh, c * t.kappa * s * s, t.bound);
    const TauLine lu = tau_line(1.0 + c * t.nu * kh * kh, c * t.nu * s * s, t.bound);
    const TauLine lp = tau_line(c * kh * kh, c * s * s, t.bound);  // kh = 0: no line is solved with it (1/alpha is inf)
    const auto none = [](int) { return 0.0; };
    if (tid < 3) {
        const TauLine L = tid == 0 ? lb : (tid == 1 ? lu : lp);
        double* o = sc + kScLine + 4 * tid;
        o[0] = L.m, o[1] = kh > 0.0 || tid < 2 ? L.ial : 0.0, o[2] = L.beta, o[3] = L.ibeta;
    }
    if (ANY)  // the pivots of the b and u lines, each in place of its factors
        for (int op = 0; op < 2; ++op) {
            const TauLine L = op == 0 ? lb : lu;
            if (tid < 2 && !(L.m > 0.0) && !tau_bordered(N, tid, L.m, 0.0, E)) atomicOr(&bad, op == 0 ? 1 : 2);
        }
    if (tid < 6) {
        const int op = tid >> 1, g = tid & 1;
        const double m = op == 0 ? lb.m : (op == 1 ? lu.m : lp.m);
        if (!ANY || m > 0.0) sc[2 * op + g] = tau_factor_line(N, g, m, tab + op * N);
    }
    __syncthreads();
    if (kh > 0.0) {
        double *p1 = tab + kTabP1 * N, *x1 = tab + kTabX1 * N, *z1 = tab + kTabZ1 * N;
        if (tid < 2) tau_solve_line<ANY>(N, tid, lp, tab + kTabP * N, sc[kScP + tid], none, none, E, p1, 1.0);
        __syncthreads();
        double q1 = 1.0;
        if (tid < 2) {
            const TauSums q = tau_solve_line<ANY>(N, tid, lu, tab + kTabU * N, sc[kScU + tid],
                                                  [&](int k) { return -c * kh * p1[k]; }, none, E, x1, 0.0);
            sc[kScPsi + tid] = q.psi;
        }
        if (ANY) __syncthreads();  // two scratch rows
        if (tid >= 2 && tid < 4) {
            const int h = tid - 2, g = h ^ 1;
            const TauSums q = tau_solve_line<ANY>(N, h, lu, tab + kTabU * N, sc[kScU + h], none,
                                                  [&](int k) { return -c * s * p1[k]; }, E, z1, 0.0);
            const double tz = g == PL ? q.psi * s / (2.0 * (N - 1)) + p1[N - 1] * c * s * s * lu.ibeta : 0.0;
            q1 = s * q.k2 + tz;
            sc[kScTz + g] = tz;
        }
        __syncthreads();
        if (kh <= t.low && tid >= 2 && tid < 4) {  // uz_1 as the integral of kh u~_1
            const int h = tid - 2, g = h ^ 1;
            double sum = 0.0;
            for (int k = N - 1 - ((N - 1 - h) & 1); k >= 1; k -= 2) {
                const double z = kh * ((k == 1 ? 2.0 : 1.0) * x1[k - 1] - (k + 1 <= N - 2 ? x1[k + 1] : 0.0)) / (2.0 * k * s);
                z1[k] = z;
                sum += z;
            }
            q1 = sum;
            if (h == 0) {
                q1 += z1[0];
                z1[0] = -sum;
            }
            sc[kScTz + g] = g == PL ? kh * x1[N - 1] : 0.0;
        }
        if (tid >= 2 && tid < 4) {
            sc[kScQ + ((tid - 2) ^ 1)] = 1.0 / q1;
            if (ANY && q1 == 0.0) atomicOr(&bad, 4);
        }
        __syncthreads();
    }
    if (ANY && tid == 0) t.info[key] = bad;
    const int S = tau_row(t.shape);
    double* out = t.table + (size_t)key * tau_table_stride(t.shape);
    for (int i = tid; i < 6 * S; i += 64) {
        const int row = i / S, k = i - row * S;
        out[row * S + tau_slot(t.shape, k)] = (row < 3 && k < 2) ? 1.0 : (k < N ? tab[row * N + k] : 0.0);
    }
    if (tid < kTauScalars) out[6 * S + tid] = sc[tid];
    if (key == 0) {
        double* co = t.table + (size_t)t.nkeys * tau_table_stride(t.shape);
        for (int k = tid; k < S; k += 64) {
            const TauCoeffs q = tau_coeffs(N, k);
            const int o = tau_slot(t.shape, k);
            co[o] = q.t1;
            co[S + o] = q.t2;
            co[2 * S + o] = q.g1;
            co[3 * S + o] = q.g2;
        }
    }
}

// ---------------------------------------------------------------------------
// Wave-parallel lines: G lanes per mode (16, 32 or 64), E degrees per lane and parity.  Scans run in the
// 16-lane rows by DPP and then carry over the rows through scalar registers; shifts give 0 beyond the
// ends of a group.  Contraction is off and the fused multiply-adds are written out: every launch
// variant then gives the same bits.
// ---------------------------------------------------------------------------
template <int CTRL>
__device__ inline double dpp_f64(double x) {
    const int lo = __builtin_amdgcn_update_dpp(0, __double2loint(x), CTRL, 0xf, 0xf, true);
    const int hi = __builtin_amdgcn_update_dpp(0, __double2hiint(x), CTRL, 0xf, 0xf, true);
    return __hiloint2double(hi, lo);
}
__device__ inline double lane_f64(double x, int lane) {  // wave-uniform lane
    const int lo = __builtin_amdgcn_readlane(__double2loint(x), lane), hi = __builtin_amdgcn_readlane(__double2hiint(x), lane);
    return __hiloint2double(hi, lo);
}
template <int G>
__device__ inline double lane_below(double x, int l) {  // the value of lane l - 1
    if constexpr (G == 16) return dpp_f64<0x111>(x);
    const double y = dpp_f64<0x138>(x);  // wave shift
    return G == 64 || l > 0 ? y : 0.0;
}
template <int G>
__device__ inline double lane_above(double x, int l) {  // the value of lane l + 1
    if constexpr (G == 16) return dpp_f64<0x101>(x);
    const double y = dpp_f64<0x130>(x);
    return G == 64 || l < G - 1 ? y : 0.0;
}
template <int G>
__device__ inline double lanes_sum(double x) {  // over the group, in every lane
    x += dpp_f64<0x128>(x);                     // rotations of the 16-lane row
    x += dpp_f64<0x124>(x);
    x += dpp_f64<0x122>(x);
    x += dpp_f64<0x121>(x);
    if constexpr (G == 64) return (lane_f64(x, 0) + lane_f64(x, 16)) + (lane_f64(x, 32) + lane_f64(x, 48));
    if constexpr (G == 32) {
        const double a = lane_f64(x, 0) + lane_f64(x, 16), b = lane_f64(x, 32) + lane_f64(x, 48);
        return (threadIdx.x & 32) ? b : a;
    }
    return x;
}

// e_i = e_i + h_i e_{i+1} over the group's degrees, downwards, for NV values with the same h
template <int G, int E, int NV>
__device__ inline void tau_scan_down(const double (&h)[E], double (&e)[NV][E], int l) {
#pragma clang fp contract(off)
    double H = h[0], B[NV];
#pragma unroll
    for (int i = 1; i < E; ++i) H *= h[i];
#pragma unroll
    for (int v = 0; v < NV; ++v) {
        B[v] = e[v][E - 1];
#pragma unroll
        for (int i = E - 2; i >= 0; --i) B[v] = fma(h[i], B[v], e[v][i]);
    }
    const int rl = (int)threadIdx.x & 15;
    auto level = [&](auto DC) {
        constexpr int d = decltype(DC)::value;
#pragma unroll
        for (int v = 0; v < NV; ++v) B[v] = fma(H, dpp_f64<0x100 + d>(B[v]), B[v]);
        const double s = dpp_f64<0x100 + d>(H);
        H *= (G == 16 || rl + d < 16) ? s : 1.0;  // past a group's end nothing follows: 0 will do
    };
    level(std::integral_constant<int, 1>{});
    level(std::integral_constant<int, 2>{});
    level(std::integral_constant<int, 4>{});
    level(std::integral_constant<int, 8>{});
    if constexpr (G > 16) {  // rows above: their first lanes hold whole-row results
        const int rowi = ((int)threadIdx.x & 63) >> 4;
        const double H16 = lane_f64(H, 16), H32 = lane_f64(H, 32);
#pragma unroll
        for (int v = 0; v < NV; ++v) {
            const double c2 = lane_f64(B[v], 48), b32 = lane_f64(B[v], 32), b16 = lane_f64(B[v], 16);
            double carry;
            if constexpr (G == 64) {
                const double c1 = fma(H32, c2, b32), c0 = fma(H16, c1, b16);
                carry = rowi == 0 ? c0 : (rowi == 1 ? c1 : (rowi == 2 ? c2 : 0.0));
            } else {
                carry = rowi == 0 ? b16 : (rowi == 2 ? c2 : 0.0);
            }
            B[v] = fma(H, carry, B[v]);
        }
    }
#pragma unroll
    for (int v = 0; v < NV; ++v) {
        double x = lane_above<G>(B[v], l);
#pragma unroll
        for (int i = E - 1; i >= 0; --i) e[v][i] = x = fma(h[i], x, e[v][i]);
    }
}
// x_i = e_i + a_i x_{i-1} upwards (x = 0 below the first), in place; pr = the running products of a
template <int G, int E, int NV>
__device__ inline void tau_scan_up(const double (&a)[E], double (&e)[NV][E], double (&pr)[E], int l) {
#pragma clang fp contract(off)
    double A = a[0], B[NV];
#pragma unroll
    for (int i = 1; i < E; ++i) A *= a[i];
#pragma unroll
    for (int v = 0; v < NV; ++v) {
        B[v] = e[v][0];
#pragma unroll
        for (int i = 1; i < E; ++i) B[v] = fma(a[i], B[v], e[v][i]);
    }
    const int rl = (int)threadIdx.x & 15;
    auto level = [&](auto DC) {
        constexpr int d = decltype(DC)::value;
#pragma unroll
        for (int v = 0; v < NV; ++v) B[v] = fma(A, dpp_f64<0x110 + d>(B[v]), B[v]);
        const double s = dpp_f64<0x110 + d>(A);
        A *= rl >= d ? s : 1.0;
    };
    level(std::integral_constant<int, 1>{});
    level(std::integral_constant<int, 2>{});
    level(std::integral_constant<int, 4>{});
    level(std::integral_constant<int, 8>{});
    if constexpr (G > 16) {  // rows below: their last lanes hold whole-row results
        const int rowi = ((int)threadIdx.x & 63) >> 4;
        const double A15 = lane_f64(A, 15), A31 = lane_f64(A, 31), A47 = lane_f64(A, 47);
#pragma unroll
        for (int v = 0; v < NV; ++v) {
            const double b15 = lane_f64(B[v], 15), b31 = lane_f64(B[v], 31), b47 = lane_f64(B[v], 47);
            double carry;
            if constexpr (G == 64) {
                const double c2 = fma(A31, b15, b31), c3 = fma(A47, c2, b47);
                carry = rowi == 0 ? 0.0 : (rowi == 1 ? b15 : (rowi == 2 ? c2 : c3));
            } else {
                carry = rowi == 1 ? b15 : (rowi == 3 ? b47 : 0.0);
            }
            B[v] = fma(A, carry, B[v]);
        }
        if constexpr (G == 64) {
            const double p2 = A31 * A15, p3 = A47 * p2;
            A *= rowi == 0 ? 1.0 : (rowi == 1 ? A15 : (rowi == 2 ? p2 : p3));
        } else {
            A *= rowi == 1 ? A15 : (rowi == 3 ? A47 : 1.0);
        }
    }
    const double pin = lane_below<G>(A, l);
    pr[0] = a[0] * (l > 0 ? pin : 1.0);
#pragma unroll
    for (int i = 1; i < E; ++i) pr[i] = pr[i - 1] * a[i];
#pragma unroll
    for (int v = 0; v < NV; ++v) {
        double x = lane_below<G>(B[v], l);
#pragma unroll
        for (int i = 0; i < E; ++i) e[v][i] = x = fma(a[i], x, e[v][i]);
    }
}

template <typename T>
struct TauArgs {
    TauSys t;
    int nmodes;
    const double2* bcv;   // [2 mode + w]: b on wall w (0: z = 0, 1: z = Lz) at the mode
    const int2* modes;    // 3-D: (mode, key), sorted by key
    const double* rot;    // 3-D: (cos, sin) of the k_h direction per mode
    int form;             // TauForm
    const cplx<T>*R1, *R2, *R3x, *R3y, *R3z;  // right-hand-side rows, mode-major (R1 null: zero)
    cplx<T>*P, *B, *UX, *UY, *UZ, *taus;
};

// LDS of one pair of waves: two row buffers in turn, and the scalars that the parities exchange
template <int G, int E>
constexpr size_t tau_pair_buf() {
    return (size_t)(64 / G) * (2 * E + 1) * G * sizeof(double2);
}
template <int G, int E>
constexpr size_t tau_pair_bytes() {
    return 2 * tau_pair_buf<G, E>() + (64 / G) * 16 * sizeof(double);
}
template <int G, int E>
constexpr size_t tau_park_bytes() {  // 3-D: the perp row of both waves
    return (size_t)128 * E * sizeof(double2);
}
template <int E, int FORM>
constexpr size_t tau_any_bytes() {  // any sign: tau_bordered's rows of both waves, two parts each
    return FORM == kTauAny ? (size_t)4 * 64 * E * 5 * sizeof(double) : 0;
}
template <int G, int E, bool THREE, int FORM>
constexpr size_t tau_lds_bytes() {  // of one pair of waves
    return tau_pair_bytes<G, E>() + (THREE ? tau_park_bytes<G, E>() : 0) + tau_any_bytes<E, FORM>();
}

// One pair of waves: 64 / G modes, `slot0` the first; wave g holds the degrees of parity g, all rows in
// registers ([degree][part]).  LDS turns the rows between the memory order (neighbouring lanes,
// neighbouring degrees) and a lane's run, and passes G of the other parity.  Every workgroup meets the
// same barriers: a pair beyond the last mode runs along without storing.
// Bound: 3-D, latency: at 256 registers two waves share a SIMD, and each waits for memory or LDS half of its
// cycles and issues vector instructions a fifth of them (256 x 256 x 128: 151 us at 2.5 TB/s in FP32, 210 us at
// 3.3 TB/s in FP64, of 5.1 that a copy reaches; dense inverses on the matrix cores read 3.2 / 5.1 GB in 787 /
// 1262 us; 96 x 80 x 49 FP64 18 against 89 us).  2-D: the latency of one wave's instructions, whose fetch is part
// of it, as the code runs once; a wave per parity halves it against one wave for both (1024 x 256 FP32: 13.7
// against 24.4 us, and 200 us with dense inverses; 320 x 97 FP64: 9.4 us, 19.4 with dense inverses).
template <typename T, bool THREE, int G, int E, int FORM, bool HASD, bool MEAN>
__device__ __attribute__((always_inline)) inline void tau_solve_pair_t(const TauArgs<T>& s, int slot0, int g, unsigned char* lds) {
#pragma clang fp contract(off)
    using V = cplx<T>;
    constexpr bool ANY = FORM == kTauAny, PSI = FORM != kTauU, LOW = sizeof(T) == 8;
    constexpr int NM = 64 / G, K = 2 * E, LS = (K + 1) * G;  // LDS: K + 1 values per lane, so lanes differ in bank
    const int lane = (int)threadIdx.x & 63, l = lane & (G - 1), grp = lane / G;
    const int N = s.t.N, S = K * G, k0 = K * l + g;  // own degrees: k0 + 2 i
    const bool live = slot0 + grp < s.nmodes;
    const int slot = live ? slot0 + grp : s.nmodes - 1;
    int mode = slot, key = slot;
    if constexpr (THREE) {
        const int2 mk = s.modes[slot];
        mode = mk.x;
        key = mk.y;
    }
    const double c = s.t.c, sz = s.t.s, nu = s.t.nu, kh = tau_kh(s.t, key);
    const int PL = (N - 1) & 1;
    const bool A = g == PL;
    const int kt = A ? N - 1 : N - 2, lt = kt / K;  // own top degree and its lane
    const size_t base = (size_t)mode * N;
    int flip = 0;  // the buffer of the row before is read until the barrier of this row
    auto next = [&] {
        flip ^= 1;
        return lds + flip * tau_pair_buf<G, E>();
    };
    double* xs = reinterpret_cast<double*>(lds + 2 * tau_pair_buf<G, E>()) + 16 * grp;
    auto fetch = [&](const V* src, V (&v)[E]) __attribute__((always_inline)) {
#pragma unroll
        for (int i = 0; i < E; ++i) {
            const int k = l + G * (2 * i + g);
            v[i] = k < N ? src[base + k] : V{T(0), T(0)};
        }
    };
    using Row = double[E][2];
    auto turn = [&](const V (&v)[E], Row& o) __attribute__((always_inline)) {
        V* buf = reinterpret_cast<V*>(next()) + grp * LS;
#pragma unroll
        for (int i = 0; i < E; ++i) {
            const int k = l + G * (2 * i + g);
            buf[k + k / K] = v[i];
        }
        __syncthreads();
#pragma unroll
        for (int i = 0; i < E; ++i) {
            const V x = buf[k0 + l + 2 * i];
            o[i][0] = (double)x.x;
            o[i][1] = (double)x.y;
        }
    };
    auto put = [&](V* dst, auto value) __attribute__((always_inline)) {  // value(i): degree k0 + 2 i
        V* buf = reinterpret_cast<V*>(next()) + grp * LS;
#pragma unroll
        for (int i = 0; i < E; ++i) buf[k0 + l + 2 * i] = value(i);
        __syncthreads();
#pragma unroll
        for (int i = 0; i < E; ++i) {
            const int k = l + G * (2 * i + g);
            const V x = buf[k + k / K];
            if (live && k < N) dst[base + k] = x;
        }
    };
    // the other parity's neighbours: o[i] at degree k - 1, o[i + 1] at degree k + 1 of own degree k = k0 + 2 i
    using Nbr = double[E + 1][2];
    auto swap = [&](const Row& v, Nbr& o) __attribute__((always_inline)) {
        double2* buf = reinterpret_cast<double2*>(next()) + grp * LS;
#pragma unroll
        for (int i = 0; i < E; ++i) buf[k0 + l + 2 * i] = double2{v[i][0], v[i][1]};
        __syncthreads();
#pragma unroll
        for (int i = 0; i <= E; ++i) {
            const int k = k0 + 2 * i - 1;
            const double2 x = k >= 0 && k < S ? buf[k + k / K] : double2{0.0, 0.0};
            o[i][0] = x.x;
            o[i][1] = x.y;
        }
    };
    const double* tab = s.t.table + (size_t)key * tau_table_stride(s.t.shape) + g * G + l;
    const double* sc = s.t.table + (size_t)key * tau_table_stride(s.t.shape) + 6 * S;
    const double* co = s.t.table + (size_t)s.t.nkeys * tau_table_stride(s.t.shape) + g * G + l;  // coefficient rows
    // 2-D, and short rows: few waves with registers to spare, so every table is asked for at once here (at
    // 64 x 64 x 18 each round trip saved shows); 3-D: each row is loaded where it is used, other waves fill the wait
    constexpr bool AHEAD = !THREE || E <= 2;
    double ahead[AHEAD ? 6 : 1][E], cof[AHEAD ? 4 : 1][E];
    double2 wall0, wall1;
    if constexpr (AHEAD) {
#pragma unroll
        for (int r = 0; r < 6; ++r)
#pragma unroll
            for (int i = 0; i < E; ++i) ahead[r][i] = tab[r * S + 2 * i * G];
#pragma unroll
        for (int r = 0; r < 4; ++r)
#pragma unroll
            for (int i = 0; i < E; ++i) cof[r][i] = co[r * S + 2 * i * G];
        wall0 = s.bcv[2 * (size_t)mode];
        wall1 = s.bcv[2 * (size_t)mode + 1];
    }
    auto table = [&](int r, double (&a)[E]) __attribute__((always_inline)) {
        if constexpr (!AHEAD) asm volatile("" ::: "memory");
#pragma unroll
        for (int i = 0; i < E; ++i) a[i] = AHEAD ? ahead[AHEAD ? r : 0][i] : tab[r * S + 2 * i * G];
    };
    auto coeff = [&](int r, int i) { return AHEAD ? cof[AHEAD ? r : 0][i] : co[r * S + 2 * i * G]; };
    auto line_of = [&](int op) {
        const double* q = sc + kScLine + 4 * op;
        return TauLine{q[0], q[1], q[2], q[3], fabs(q[0]) > s.t.bound};
    };
    // ---- right-hand sides ----
    Row b, x, z;
    double y[THREE ? E : 1][2];  // perp (3-D)
    double d[HASD ? E : 1][2];   // R1 / c
    {
        V v0[E], v1[E], v2[E], v3[THREE ? E : 1], v4[HASD ? E : 1];
        fetch(s.R2, v0);
        fetch(s.R3x, v1);
        fetch(s.R3z, v2);
        if constexpr (THREE) fetch(s.R3y, v3);
        if constexpr (HASD) fetch(s.R1, v4);
        turn(v0, b);
        turn(v1, x);
        turn(v2, z);
        if constexpr (THREE) turn(v3, y);
        if constexpr (HASD) turn(v4, d);
    }
    double cr = 1.0, sr = 0.0;
    if constexpr (THREE) {
        cr = s.rot[2 * (size_t)mode];
        sr = s.rot[2 * (size_t)mode + 1];
    }
    const double ic = 1.0 / c;
#pragma unroll
    for (int i = 0; i < E; ++i) {
        const double xr = x[i][1], xi = -x[i][0];  // rows -i E3x (and -i E3y)
        if constexpr (THREE) {
            const double yr = y[i][1], yi = -y[i][0];
            x[i][0] = cr * xr + sr * yr;
            x[i][1] = cr * xi + sr * yi;
            y[i][0] = -sr * xr + cr * yr;
            y[i][1] = -sr * xi + cr * yi;
        } else {
            x[i][0] = xr;
            x[i][1] = xi;
        }
        if constexpr (HASD) {
            d[i][0] *= ic;
            d[i][1] *= ic;
        }
    }
    double* const bordered = reinterpret_cast<double*>(lds + tau_pair_bytes<G, E>() + (THREE ? tau_park_bytes<G, E>() : 0)) +
                             2 * 64 * E * 5 * g;  // any sign only
    // One line (real and imaginary part) of an operator: r at the own degrees, G = gs Go of the other parity;
    // the result over r.  w = wall sums; tops receives r at N - 1 (A) or psi at N - 2 (B).
    auto line = [&](auto hasg, const TauLine& L, const double (&a)[E], double iW, Row& r, const Nbr& Go, double gs,
                    const double (&w)[2], double (&tops)[2]) __attribute__((always_inline)) {
        if constexpr (!AHEAD) __builtin_amdgcn_sched_barrier(0);  // one line at a time: interleaved, their registers would spill
        constexpr bool HASG = decltype(hasg)::value;
        const bool piv = ANY && !(L.m > 0.0);  // the same in the whole workgroup, which has one mode
        const bool rest = PSI && L.psi && fabs(L.m) > tau_rest_bound(N);
        double e[2][E], h[E], pr[E];
        {
            double t1[E], t2[E], g1[HASG || PSI ? E : 1], g2[HASG ? E : 1];
#pragma unroll
            for (int i = 0; i < E; ++i) {
                t1[i] = coeff(0, i);
                t2[i] = coeff(1, i);
                if (HASG || PSI) g1[HASG || PSI ? i : 0] = coeff(2, i);
                if (HASG) g2[HASG ? i : 0] = coeff(3, i);
                h[i] = a[i] * t1[i];
            }
#pragma unroll
            for (int p = 0; p < 2; ++p) {
                const double rup = lane_above<G>(r[0][p], l), rlo = lane_below<G>(r[E - 1][p], l);
#pragma unroll
                for (int i = 0; i < E; ++i) {
                    const double rl = i > 0 ? r[i > 0 ? i - 1 : 0][p] : rlo, ru = i < E - 1 ? r[i < E - 1 ? i + 1 : 0][p] : rup;
                    double dg = 0.0;
                    if (HASG) dg = fma(g1[HASG ? i : 0], Go[i][p], -(g2[HASG ? i : 0] * Go[i + 1][p]));
                    double v = fma(t1[i], ru, fma(-t2[i], r[i][p], rl));
                    if (HASG) v = fma(gs, dg, v);
                    if (PSI) {
                        const int k = k0 + 2 * i;
                        const double rk = k == N - 1 ? 0.0 : r[i][p];
                        const double vp = fma(2.0 * k * g1[PSI ? i : 0], rk, L.m * (gs * dg));
                        v = L.psi ? vp : v;
                    }
                    e[p][i] = -(a[i] * L.ial) * v;
                    if constexpr (ANY) {
                        const int k = k0 + 2 * i;
                        if (piv) e[p][i] = k >= 2 && k < N ? -(tau_lo(k) * L.ibeta) * v : 0.0;
                    }
                }
            }
        }
        if (!piv) {
            tau_scan_down<G, E, 2>(h, e, l);
            if (l == 0) e[0][0] = e[1][0] = 0.0;
        }
        if (!piv) tau_scan_up<G, E, 2>(a, e, pr, l);
        double wts[2];
#pragma unroll
        for (int p = 0; p < 2; ++p) {
            double rs = 0.0;
            wts[p] = w[p];
            if (PSI) {
#pragma unroll
                for (int i = 0; i < E; ++i)
                    if (k0 + 2 * i != N - 1) rs += r[i][p];
                rs = lanes_sum<G>(rs);
                if (L.psi) wts[p] = L.m * wts[p] - rs * L.ibeta;
            }
        }
        if (ANY && piv) {  // lane p solves part p, row by row
            double* S[2] = {bordered, bordered + 64 * E * 5};
#pragma unroll
            for (int p = 0; p < 2; ++p)
#pragma unroll
                for (int i = 0; i < E; ++i) S[p][5 * (E * l + i) + 4] = e[p][i];
            __syncthreads();
            if (l < 2) tau_bordered(N, g, L.m, l == 0 ? wts[0] : wts[1], l == 0 ? S[0] : S[1]);
            __syncthreads();
#pragma unroll
            for (int p = 0; p < 2; ++p)
#pragma unroll
                for (int i = 0; i < E; ++i) e[p][i] = k0 + 2 * i < N ? S[p][5 * (E * l + i) + 4] : 0.0;
        }
#pragma unroll
        for (int p = 0; p < 2; ++p) {
            double x0 = 0.0;
            if (!piv) {
                double sum = 0.0;
#pragma unroll
                for (int i = 0; i < E; ++i) sum += e[p][i];
                x0 = (wts[p] - lanes_sum<G>(sum)) * iW;
            }
            double uu[E], rt = 0.0, vt = 0.0;
#pragma unroll
            for (int i = 0; i < E; ++i) {
                const double v = piv ? e[p][i] : fma(pr[i], x0, e[p][i]);
                rt = k0 + 2 * i == kt ? r[i][p] : rt;
                vt = k0 + 2 * i == kt ? v : vt;
                e[p][i] = v;
                uu[i] = v;
                if (PSI) {
                    const double rk = k0 + 2 * i == N - 1 ? 0.0 : r[i][p];
                    uu[i] = L.psi ? fma(L.beta, v, rk) * L.ial : v;
                }
            }
            // the owner of the top degree: r_{N-1} (A) or psi_{N-2} (B); zero elsewhere
            tops[p] = l == lt ? (A ? rt : ((PSI && L.psi) ? vt : fma(L.m, vt, -(rt * L.ibeta)))) : 0.0;
            if (PSI && A && __any(rest)) {  // u_{N-1}: the wall sum's remainder
                double su = 0.0;
#pragma unroll
                for (int i = 0; i < E; ++i) su += k0 + 2 * i < N - 1 ? uu[i] : 0.0;
                su = lanes_sum<G>(su);
#pragma unroll
                for (int i = 0; i < E; ++i) uu[i] = rest && k0 + 2 * i == N - 1 ? w[p] - su : uu[i];
            }
#pragma unroll
            for (int i = 0; i < E; ++i) r[i][p] = uu[i];  // beyond N - 1 a, e and r are zero
        }
    };
    using no_g = std::integral_constant<bool, false>;
    using with_g = std::integral_constant<bool, true>;
    constexpr int TS = THREE ? 9 : 8;
    V* tm = s.taus + (size_t)mode * TS;
    auto part = [&](int slot_, int p, double v) { reinterpret_cast<T*>(tm + slot_)[p] = T(v); };
    auto horizontal = [&](int slot_, int p, double v) {  // u = i u~: the real part of u~ is the imaginary part of u
        reinterpret_cast<T*>(tm + slot_)[p ^ 1] = T(p ? -v : v);
    };
    const double tscale = sz / (2.0 * (N - 1));  // psi at degree N - 2 -> amplitude of a D T_{N-1} lift
    auto at_top = [&](const Row& v, int p) __attribute__((always_inline)) {
        double o = 0.0;
#pragma unroll
        for (int i = 0; i < E; ++i) o = k0 + 2 * i == kt ? v[i][p] : o;
        return o;
    };
    auto at_top_d = [&](int p) __attribute__((always_inline)) {
        double o = 0.0;
        if constexpr (HASD)
#pragma unroll
            for (int i = 0; i < E; ++i) o = k0 + 2 * i == kt ? d[i][p] : o;
        return o;
    };
    const double zero2[2] = {0.0, 0.0};
    const Nbr none{};
    double2* const park = reinterpret_cast<double2*>(lds + tau_pair_bytes<G, E>()) + 64 * E * g + lane;  // 3-D only
    // ---- perp ----
    const double au = 1.0 + c * nu * kh * kh, ckh = c * kh;
    const TauLine lu = line_of(1);
    double topy[2] = {0.0, 0.0};
    if constexpr (THREE) {
        double a[E];
        table(kTabU, a);
        line(no_g{}, lu, a, sc[kScU + g], y, none, 0.0, zero2, topy);
#pragma unroll
        for (int p = 0; p < 2; ++p)  // the lift tau's share of degree N - 1 needs y itself
            topy[p] = A ? (topy[p] - au * at_top(y, p)) * ic : topy[p] * tscale;
#pragma unroll
        for (int i = 0; i < E; ++i) park[64 * i] = double2{y[i][0], y[i][1]};  // until the rotation back: its registers are needed
    }
    // ---- b: wall values as half-sum (even part) / half-difference (odd part) ----
    {
        const double al = 1.0 + c * s.t.kappa * kh * kh;
        const TauLine L = line_of(0);
        double a[E];
        table(kTabB, a);
        if constexpr (!AHEAD) {
            wall0 = s.bcv[2 * (size_t)mode];
            wall1 = s.bcv[2 * (size_t)mode + 1];
        }
        const double w[2] = {g == 0 ? 0.5 * (wall1.x + wall0.x) : 0.5 * (wall1.x - wall0.x),
                             g == 0 ? 0.5 * (wall1.y + wall0.y) : 0.5 * (wall1.y - wall0.y)};
        double tops[2];
        line(no_g{}, L, a, sc[kScB + g], b, none, 0.0, w, tops);
        if (live && l == lt)
#pragma unroll
            for (int p = 0; p < 2; ++p) part(A ? 2 : 1, p, A ? (tops[p] - al * at_top(b, p)) * ic : tops[p] * tscale);
        put(s.B, [&](int i) { return V{T(b[i][0]), T(b[i][1])}; });
    }
#pragma unroll
    for (int i = 0; i < E; ++i)
#pragma unroll
        for (int p = 0; p < 2; ++p) z[i][p] = fma(c, b[i][p], z[i][p]);
    // ---- kh = 0 (one mode, in the first workgroup): uz is the integral of E1, p that of E3z ----
    double pm[MEAN ? E : 1][2], zm[MEAN ? E : 1][2];
    double tau1[2] = {0.0, 0.0}, tau2[2] = {0.0, 0.0}, taup[2] = {0.0, 0.0}, first[2] = {0.0, 0.0};
    if constexpr (MEAN) {
        Row dw, f;
        Nbr n;
        double tz[2];
#pragma unroll
        for (int p = 0; p < 2; ++p) {
            double t = 0.0, d0 = 0.0, w2 = 0.0;
#pragma unroll
            for (int i = 0; i < E; ++i) {
                const int k = k0 + 2 * i;
                const double dk = HASD ? d[HASD ? i : 0][p] : 0.0;
                if (k == N - 1) t = dk;  // row N - 1 of E1: D uz has no such degree
                if (k == 0) d0 = dk;
                dw[i][p] = k >= N - 1 ? 0.0 : dk / sz;
                if (k == 2) w2 = dw[i][p];
            }
            tz[p] = tau1[p] = lanes_sum<G>(t);
            taup[p] = d0 - 0.5 * sz * lanes_sum<G>(w2);  // and -sz uz_1, below
        }
        swap(dw, n);
#pragma unroll
        for (int p = 0; p < 2; ++p) {
            double sum = 0.0;
#pragma unroll
            for (int i = 0; i < E; ++i) {
                const int k = k0 + 2 * i;
                zm[i][p] = k >= 2 && k < N ? (n[i][p] - n[i + 1][p]) / (2.0 * k) : 0.0;
                sum += zm[i][p];
            }
            first[p] = -lanes_sum<G>(sum);  // uz at degree g: zero walls
            if (l == 0) zm[0][p] = first[p];
#pragma unroll
            for (int i = 0; i < E; ++i) {
                const int k = k0 + 2 * i;
                f[i][p] = k >= N - 1 ? 0.0 : z[i][p] - zm[i][p];
                if (k == N - 1) tau2[p] = (z[i][p] - zm[i][p]) * ic;  // z momentum lift T_{N-1}
            }
        }
        swap(f, n);
        const double ics = 1.0 / (c * sz), beta = c * nu * sz * sz;
#pragma unroll
        for (int p = 0; p < 2; ++p) {
            double integ = 0.0;
#pragma unroll
            for (int i = 0; i < E; ++i) {
                const int k = k0 + 2 * i;
                double v = 0.0;
                if (k >= 1 && k < N)
                    v = (((k == 1 ? 2.0 : 1.0) * n[i][p] - n[i + 1][p]) / (2.0 * k) + beta * dw[i][p] +
                         (k == N - 1 ? c * nu * sz * tz[p] : 0.0)) * ics;
                pm[i][p] = v;
                if (g == 0 && k >= 2) integ += v / ((double)k * k - 1.0);
            }
            integ = lanes_sum<G>(integ);  // integ(p) = 0: sum 2/(1 - k^2) p_k over even k
            if (k0 == 0) pm[0][p] = integ;
        }
    }
    const bool mean = MEAN && kh == 0.0;
    const bool low = LOW && kh <= s.t.low;  // uz from E1
    // ---- pressure, zero wall value of p - nu d ----
    Row q;
    double wd[2] = {0.0, 0.0};
    {
        const TauLine L = line_of(2);  // the mean mode's p is pm
        double a[E];
        table(kTabP, a);
        Nbr n;
        swap(z, n);
#pragma unroll
        for (int i = 0; i < E; ++i)
#pragma unroll
            for (int p = 0; p < 2; ++p) {
                q[i][p] = fma(kh, x[i][p], HASD ? d[HASD ? i : 0][p] : 0.0);
                if (HASD) wd[p] += d[HASD ? i : 0][p];
            }
        if (HASD)
#pragma unroll
            for (int p = 0; p < 2; ++p) wd[p] = lanes_sum<G>(wd[p]);
        const double w[2] = {-nu * wd[0], -nu * wd[1]};
        double tops[2];
        line(with_g{}, L, a, sc[kScP + g], q, n, -sz, w, tops);
#pragma unroll
        for (int i = 0; i < E; ++i)
#pragma unroll
            for (int p = 0; p < 2; ++p) {
                if (HASD) q[i][p] = fma(nu, d[HASD ? i : 0][p], q[i][p]);
                if constexpr (MEAN) q[i][p] = mean ? pm[i][p] : q[i][p];
            }
    }
    // ---- u~, uz ----
    double topx[2], topz[2], k2[2] = {0.0, 0.0}, zi[2] = {0.0, 0.0};
    {
        double a[E];
        table(kTabU, a);
        Nbr n;
        swap(q, n);
#pragma unroll
        for (int i = 0; i < E; ++i)
#pragma unroll
            for (int p = 0; p < 2; ++p) x[i][p] = fma(-ckh, q[i][p], x[i][p]);
        line(no_g{}, lu, a, sc[kScU + g], x, none, 0.0, zero2, topx);
        if constexpr (!AHEAD)
#pragma unroll
            for (int i = 0; i < E; ++i) asm volatile("" : "+v"(a[i]));  // u~'s running products are not kept for uz: registers
        line(with_g{}, lu, a, sc[kScU + g], z, n, -c * sz, zero2, topz);
#pragma unroll
        for (int p = 0; p < 2; ++p)
#pragma unroll
            for (int i = 0; i < E; ++i) {
                const double k = k0 + 2 * i;
                k2[p] = fma(k * k, z[i][p], k2[p]);
                if constexpr (MEAN && !LOW) z[i][p] = mean ? zm[i][p] : z[i][p];
            }
        if constexpr (LOW) {
            Row f;
#pragma unroll
            for (int i = 0; i < E; ++i)
#pragma unroll
                for (int p = 0; p < 2; ++p)
                    f[i][p] = k0 + 2 * i >= N - 1 ? 0.0 : fma(kh, x[i][p], HASD ? d[HASD ? i : 0][p] : 0.0);
            swap(f, n);
            double iz[E];
#pragma unroll
            for (int i = 0; i < E; ++i) iz[i] = 0.5 / (sz * (k0 + 2 * i > 0 ? k0 + 2 * i : 1));
#pragma unroll
            for (int p = 0; p < 2; ++p) {
                double v[E], sum = 0.0;
#pragma unroll
                for (int i = 0; i < E; ++i) {
                    const int k = k0 + 2 * i;
                    v[i] = k >= 1 && k < N ? ((k == 1 ? 2.0 : 1.0) * n[i][p] - n[i + 1][p]) * iz[i] : 0.0;
                    sum += v[i];
                }
                sum = lanes_sum<G>(sum);
                zi[p] = sum + lanes_sum<G>(k0 == 0 ? z[0][p] : 0.0);  // even: against the degree 0 of the line
                if (k0 == 0) v[0] = -sum;
#pragma unroll
                for (int i = 0; i < E; ++i) {
                    z[i][p] = low ? v[i] : z[i][p];
                    if constexpr (MEAN) z[i][p] = mean ? zm[i][p] : z[i][p];
                }
            }
        }
    }
    // ---- lambda per parity of p: E1 on the wall; uz has the other parity ----
    double lam[2], lamz[2], tz[2];  // lam: own parity; lamz: the other; tz: tau_u1z before the response
    {
#pragma unroll
        for (int p = 0; p < 2; ++p) {
            const double t = lanes_sum<G>(l == lt ? (A ? at_top(q, p) * (c * sz * sz * lu.ibeta) : topz[p] * tscale) : 0.0);
            k2[p] = lanes_sum<G>(k2[p]);
            if (l == 0) {
                xs[8 * g + p] = LOW && low ? zi[p] : k2[p];
                xs[8 * g + 2 + p] = wd[p];
                xs[8 * g + 4 + p] = t;
                if constexpr (MEAN) xs[8 * g + 6 + p] = first[p];
            }
        }
        __syncthreads();
        const double iq = sc[kScQ + g], iqz = sc[kScQ + (g ^ 1)];
#pragma unroll
        for (int p = 0; p < 2; ++p) {
            tz[p] = xs[4 + p] + xs[12 + p];
            double own = sz * xs[8 * (g ^ 1) + p] + (A ? tz[p] : 0.0) - xs[8 * g + 2 + p];
            double oth = sz * xs[8 * g + p] + (A ? 0.0 : tz[p]) - xs[8 * (g ^ 1) + 2 + p];
            if (LOW) {
                own = low ? xs[8 * (g ^ 1) + p] : own;
                oth = low ? xs[8 * g + p] : oth;
                if (A) {  // row N - 1 of E1
                    const double t = fma(kh, at_top(x, p), HASD ? at_top_d(p) : 0.0);
                    tz[p] = low ? t : tz[p];
                }
            }
            lam[p] = mean ? 0.0 : -own * iq;
            lamz[p] = mean ? 0.0 : -oth * iqz;
            if constexpr (MEAN) taup[p] -= sz * xs[8 + 6 + p];
        }
    }
    // ---- lift taus, by the lanes that hold degrees N - 1 (T_{N-1} lifts, u2) and N - 2 (D T_{N-1}, u1) ----
    double rp[E], rz[E], rx[E];
    table(kTabP1, rp);
    table(kTabZ1, rz);
    table(kTabX1, rx);
    if (live && l == lt) {
        double p1t = 0.0, x1t = 0.0, z1t = 0.0;
#pragma unroll
        for (int i = 0; i < E; ++i) {
            p1t = k0 + 2 * i == kt ? rp[i] : p1t;
            x1t = k0 + 2 * i == kt ? rx[i] : x1t;
            z1t = k0 + 2 * i == kt ? rz[i] : z1t;
        }
#pragma unroll
        for (int p = 0; p < 2; ++p) {
            double tx;
            if (A) {
                tx = (topx[p] - au * at_top(x, p) - lam[p] * (au * x1t + ckh * p1t)) * ic;
                const double tu2z = (topz[p] - au * (at_top(z, p) + lamz[p] * z1t)) * ic;
                part(THREE ? 8 : 6, p, mean ? tau2[p] : tu2z);
                part(THREE ? 5 : 4, p, mean ? tau1[p] : tz[p] + lam[p] * sc[kScTz + g]);
            } else {
                tx = (topx[p] + lam[p] * sc[kScPsi + g]) * tscale;
            }
            const int h = THREE ? (A ? 6 : 3) : (A ? 5 : 3);
            horizontal(h, p, THREE ? cr * tx - sr * topy[p] : tx);
            if constexpr (THREE) horizontal(h + 1, p, sr * tx + cr * topy[p]);
        }
    }
    if (live && g == 0 && l == 0)
#pragma unroll
        for (int p = 0; p < 2; ++p) part(0, p, mean ? taup[p] : 0.0);
    // ---- add the lambda responses, rotate back, store ----
    put(s.P, [&](int i) { return V{T(fma(lam[0], rp[i], q[i][0])), T(fma(lam[1], rp[i], q[i][1]))}; });
    put(s.UZ, [&](int i) { return V{T(fma(lamz[0], rz[i], z[i][0])), T(fma(lamz[1], rz[i], z[i][1]))}; });
#pragma unroll
    for (int i = 0; i < E; ++i) {
        x[i][0] = fma(lam[0], rx[i], x[i][0]);
        x[i][1] = fma(lam[1], rx[i], x[i][1]);
    }
    if constexpr (THREE)
#pragma unroll
        for (int i = 0; i < E; ++i) {
            const double2 v = park[64 * i];
            y[i][0] = v.x;
            y[i][1] = v.y;
        }
    put(s.UX, [&](int i) {  // u~x = cos par - sin perp, u = i u~
        if constexpr (THREE) return V{T(-(cr * x[i][1] - sr * y[i][1])), T(cr * x[i][0] - sr * y[i][0])};
        else return V{T(-x[i][1]), T(x[i][0])};
    });
    if constexpr (THREE)
        put(s.UY, [&](int i) {  // u~y = sin par + cos perp
            return V{T(-(sr * x[i][1] + cr * y[i][1])), T(sr * x[i][0] + cr * y[i][0])};
        });
}

// the workgroup with the kh = 0 mode (key 0 sorts first) has a body of its own
template <typename T, bool THREE, int G, int E, int FORM, bool HASD>
__device__ __attribute__((always_inline)) inline void tau_solve_pair(const TauArgs<T>& s, int slot0, bool first, int g,
                                                                      unsigned char* lds) {
    if (first) tau_solve_pair_t<T, THREE, G, E, FORM, HASD, true>(s, slot0, g, lds);
    else tau_solve_pair_t<T, THREE, G, E, FORM, HASD, false>(s, slot0, g, lds);
}

// 3-D: the pairs of a workgroup have modes of their own; one or two of them give the same bits.
// Dynamic LDS: tau_lds_bytes per pair.
template <typename T, int G, int E, int FORM, bool HASD>
__global__ __launch_bounds__(256, 2) void k3_tau_solve(TauArgs<T> s) {
    extern __shared__ unsigned char smem_raw[];
    const int w = __builtin_amdgcn_readfirstlane((int)threadIdx.x >> 6), pair = w >> 1;
    const int slot = ((int)blockIdx.x * ((int)blockDim.x >> 7) + pair) * (64 / G);
    tau_solve_pair<T, true, G, E, FORM, HASD>(s, slot, blockIdx.x == 0, w & 1,
                                              smem_raw + pair * tau_lds_bytes<G, E, true, FORM>());
}

// 2-D: one pair per workgroup
template <typename T, int G, int E, int FORM, bool HASD>
__global__ __launch_bounds__(128) void k_ch_tau_solve(TauArgs<T> s) {
    __shared__ double2 lds[tau_lds_bytes<G, E, false, FORM>() / sizeof(double2)];
    const int g = __builtin_amdgcn_readfirstlane((int)threadIdx.x >> 6);
    tau_solve_pair<T, false, G, E, FORM, HASD>(s, (int)blockIdx.x * (64 / G), blockIdx.x == 0, g,
                                              reinterpret_cast<unsigned char*>(lds));
}

// One problem of a group solve and its first workgroup; the modes of several problems (uneven nx and
// nz, their own dt and diffusivities) run in one launch: workgroup w belongs to the last item with
// wg0 <= w (items sorted by wg0).
template <typename T>
struct TauItem {
    TauArgs<T> s;
    int wg0;
};
template <typename T, int FORM, bool HASD>
__global__ __launch_bounds__(128) void k_ch_tau_solve_group(const TauItem<T>* __restrict__ items, int nitems) {
    __shared__ double2 lds[tau_pair_bytes<64, 4>() / sizeof(double2)];  // the largest shape's
    const int w = (int)blockIdx.x;
    int lo = 0, hi = nitems - 1;
    while (lo < hi) {  // workgroup-uniform binary search
        const int mid = (lo + hi + 1) >> 1;
        if (items[mid].wg0 <= w) lo = mid;
        else hi = mid - 1;
    }
    const TauArgs<T>& s = items[lo].s;
    const int wg = w - items[lo].wg0, g = __builtin_amdgcn_readfirstlane((int)threadIdx.x >> 6);
    unsigned char* const mem = reinterpret_cast<unsigned char*>(lds);
    switch (tau_row(s.t.shape)) {  // the 2-D shapes of tau_shape
        case 64: tau_solve_pair<T, false, 32, 1, FORM, HASD>(s, 2 * wg, wg == 0, g, mem); break;
        case 128: tau_solve_pair<T, false, 64, 1, FORM, HASD>(s, wg, wg == 0, g, mem); break;
        case 256: tau_solve_pair<T, false, 64, 2, FORM, HASD>(s, wg, wg == 0, g, mem); break;
        default: tau_solve_pair<T, false, 64, 4, FORM, HASD>(s, wg, wg == 0, g, mem); break;
    }
}

// f(form, has R1) with both as compile-time constants; f's any-sign kernels are launched by the caller
template <typename F>
inline void tau_flags(int form, bool hasd, F&& f) {
    using yes = std::true_type;
    using no = std::false_type;
    using psi = std::integral_constant<int, kTauPsi>;
    using u = std::integral_constant<int, kTauU>;
    if (form == kTauPsi && hasd) f(psi{}, yes{});
    else if (form == kTauPsi) f(psi{}, no{});
    else if (hasd) f(u{}, yes{});
    else f(u{}, no{});
}

// the recursion of the keys up to kh_max: kTauPsi when any line among them takes the psi-form
inline int tau_form(const TauSys& t, double kh_max) {
    if (tau_any_sign(t.kappa, t.nu)) return kTauAny;
    const double k2 = kh_max * kh_max / (t.s * t.s);  // m of the pressure lines, below those of b and u
    const double mb = 1.0 / (t.c * t.kappa * t.s * t.s) + k2, mu = 1.0 / (t.c * t.nu * t.s * t.s) + k2;
    return mb > t.bound || mu > t.bound ? kTauPsi : kTauU;
}

// whether the equation of a diffusivity has lost it (the D T_{N-1} lift is left without a coefficient): zero, or
// too small for FP64
inline bool tau_no_diffusion(double c, double s, double diff) { return std::isinf(1.0 / (c * diff * s * s)); }

}  // namespace tarang
