// channel3d_kernels.hpp -- kernels of the RealFourier(x) x RealFourier(y) x
// ChebyshevT(z) channel solver (3-D Rayleigh-Benard, Chebyshev tau).
//
// Layouts (mode = m + (Nx/2+1) n, m the kx index, n the ky index in FFT order,
// exactly the reference's column-major (Nx/2+1, Ny) flattening):
//   state / right-hand side rows : mode-major, f[mode*N + k]
//   z-grid planes                : P[z*nmodes + mode]          (N x Ny x (Nx/2+1), kx fastest)
//   y-padded planes              : Q[(z*MY + j)*nxh + m]        (N x MY x (Nx/2+1))
//
// The dealiased products follow the 2-D padded product of each z level
// (nonlinear_padding.jl:359-437; the Chebyshev axis is not padded):
//   y: Nyquist split onto +-Ny/2 of the MY grid, inverse FFT; the kx = 0 and
//      kx = Nx/2 lines keep the real part (the state's grid round trip)
//   x: Hermitian extension to MX (kx = Nx/2 halved), inverse FFT, products,
//      forward FFT, truncation to Nx/2+1
//   y: forward FFT, truncation with the y Nyquist fold, x Nyquist fold
//      F(Nx/2, ky) += conj F(Nx/2, -ky); scale 1/(Nx Ny MX MY).
#pragma once
#include "channel_kernels.hpp"

namespace tarang {

// operand planes of the 3-D right-hand side, f in (b, ux, uy, uz)
//   z-grid: f value, 4+f dz f;   y-padded: 0 ux, 1 uy, 2 uz, 3+f dy f, 7+f dz f, 11 b
// dy f is formed where the values enter the y transform, dx f where they enter the x transform: 8
// and 12 planes pass through memory for the products' 15 operands.
// Against 15 planes of both kinds, 256 x 256 x 128, FP32 / FP64 us: k3_zbwd 233 / 428 -> 196 / 337,
// k3_ybwd 365 / 622 -> 312 / 550, k3_xpass 341 / 740 -> 335 / 725.
constexpr int kCh3ZPlanes = 8;
constexpr int kCh3Planes = 12;

template <typename T, int NT, int QT = ZbwdTile<T>::QT>
__global__ __launch_bounds__(NT, 768 / NT) void k3_zbwd(const cplx<T>* __restrict__ b, const cplx<T>* __restrict__ ux,
                                                 const cplx<T>* __restrict__ uy, const cplx<T>* __restrict__ uz,
                                                 Ch3Geom geo, const T* __restrict__ BT, const T* __restrict__ BDT,
                                                 cplx<T>* __restrict__ G) {
    zbwd_mfma<T, NT, false, QT>(b, ux, uy, uz, geo, BT, BDT, G);
}

// ---------------------------------------------------------------------------
// k3_ybwd: padded inverse y transform of TK kx-lines of one z level and plane.
// grid (ceil(nxh/TK), N, planes), remapped so that the tiles of one row of kx (which
// share cache lines: rows of nxh values are not line-aligned) run on one XCD, with the
// value and dy tiles of a row one after the other: the second reads the row from L2.
// On the kx = 0 and kx = Nx/2 lines dy vanishes at the y Nyquist.
// ---------------------------------------------------------------------------
template <typename T, int NY, int MY, int TK, int NT>
__global__ __launch_bounds__(NT) void k3_ybwd(const cplx<T>* __restrict__ G, Ch3Geom geo, cplx<T>* __restrict__ Q,
                                              const cplx<T>* __restrict__ tw) {
    using V = cplx<T>;
    constexpr int LS = line_stride_lf<T, TK>(MY);  // the tile's TK lines side by side in every access
    constexpr bool TW_LDS = (size_t)(TK * LS + MY) * sizeof(V) <= 160 * 1024;
    __shared__ V buf[TK * LS];
    __shared__ V twl_lds[TW_LDS ? MY : 1];
    const V* twl = TW_LDS ? twl_lds : tw;
    if constexpr (TW_LDS) load_twiddles<T, MY, NT>(twl_lds, tw);
    const unsigned gxy = gridDim.x * gridDim.y;
    const unsigned lin = xcd_remap(blockIdx.x + gridDim.x * (blockIdx.y + gridDim.y * blockIdx.z), gxy * gridDim.z);
    const int nxh = geo.nxh, m0 = (int)(lin % gridDim.x) * TK;
    const bool both = lin < 8 * gxy;  // value and dy of a field in turn, then the dz planes
    const unsigned row = lin / gridDim.x;
    const int z = (int)((both ? row >> 1 : row) % gridDim.y);
    const bool dy = both && (row & 1);
    const int f = (int)(both ? lin / (2 * gxy) : lin / gxy - 8);
    const int pl = both ? (dy ? 3 + f : (f == 0 ? 11 : f - 1)) : 7 + f;
    const size_t plane = (size_t)geo.N * geo.nmodes;
    const V* in = G + (size_t)(both ? f : 4 + f) * plane + (size_t)z * geo.nmodes;
    const bool xeven = (geo.nx % 2) == 0;
    cplx<T>* out = Q + (size_t)pl * geo.N * MY * nxh + (size_t)z * MY * nxh;
    // padded position j: ky = j below NY/2, the Nyquist row halved at j = NY/2 and
    // j = MY - NY/2, the negative ky above, zero in between
    auto load = [&](int c, int j) -> V {
        const int m = m0 + c;
        int n;
        bool half = false;
        if (j < NY / 2) n = j;
        else if (j == NY / 2 || j == MY - NY / 2) { n = NY / 2; half = true; }
        else if (j > MY - NY / 2) n = NY - MY + j;
        else return V{T(0), T(0)};
        if (m >= nxh) return V{T(0), T(0)};
        V v = in[(size_t)n * nxh + m];
        if (dy) {  // workgroup-uniform
            const T ky = half && (m == 0 || (xeven && m == geo.nx / 2)) ? T(0) : T(ch3_ky(geo, n));
            v = V{-ky * v.y, ky * v.x};
        }
        return half ? V{v.x * T(0.5), v.y * T(0.5)} : v;
    };
    auto store = [&](int c, int j, V v) {
        const int m = m0 + c;
        if (m >= nxh) return;
        if (m == 0 || (xeven && m == geo.nx / 2)) v.y = T(0);  // real lines of the grid round trip
        out[(size_t)j * nxh + m] = v;
    };
    fft_regs_io<T, MY, TK, NT, true, true, false, true, LS>(buf, twl, load, store);  // radix 8/4/2/3: fewer registers
}

// ---------------------------------------------------------------------------
// k3_xpass: one padded row (z, j) per workgroup: 15 operand rows, dx f = i kx f formed from the
// value rows, packed two per complex line (8 lines), inverse x FFT, the four advection
// products, two forward x FFTs.  Output: four rows of nxh values (scaled by `scale`).
//   F_b  = -(ux dx b  + uy dy b  + uz dz b)   (and likewise F_ux, F_uy, F_uz)
// ---------------------------------------------------------------------------
template <typename T, int NX, int MX, int NT>
__global__ __launch_bounds__(NT) void k3_xpass(const cplx<T>* __restrict__ Q, int N, int MY, double k0x, T scale,
                                               cplx<T>* __restrict__ H, const cplx<T>* __restrict__ tw) {
    using V = cplx<T>;
    constexpr int NXH = NX / 2 + 1;
    constexpr int NL = 8;
    constexpr int LS = line_stride(MX);
    constexpr bool TW_LDS = (size_t)(NL * LS + MX) * sizeof(V) <= 160 * 1024;
    __shared__ V buf[NL * LS];
    __shared__ V twl_lds[TW_LDS ? MX : 1];
    const V* twl = TW_LDS ? twl_lds : tw;
    if constexpr (TW_LDS) load_twiddles<T, MX, NT>(twl_lds, tw);
    const size_t row = (size_t)blockIdx.y * MY + blockIdx.x;  // (z, j)
    const size_t plane = (size_t)N * MY * NXH;
    // element i of packed line l: a + i b at k = i < NXH (real parts only at k = 0), conj(a) + i conj(b) at the
    // mirror i = MX - k, zero in between.  Lines 0..5 hold planes (2l, 2l+1), 6 and 7 the x derivatives of
    // (b, ux) and (uy, uz): i kx (a + i b) with the mirror's kx negative, zero on the kx = Nx/2 line
    auto load = [&](int line, int i) -> V {
        const bool mirror = i > MX - NXH;
        if (i >= NXH && !mirror) return V{T(0), T(0)};
        const int k = mirror ? MX - i : i;
        const size_t off = row * NXH + k;
        const bool dx = line >= 6;
        const V a = Q[(size_t)(dx ? 71 - 10 * line : 2 * line) * plane + off];
        V bb = Q[(size_t)(dx ? 2 * line - 12 : 2 * line + 1) * plane + off];
        if (line == 5) bb = V{T(0), T(0)};
        const V p = k == 0 ? V{a.x, bb.x} : (mirror ? V{a.x + bb.y, bb.x - a.y} : V{a.x - bb.y, a.y + bb.x});
        const T kx = 2 * k == NX ? T(0) : T(k0x * (mirror ? -k : k));
        return V{dx ? -kx * p.y : p.x, dx ? kx * p.x : p.y};  // selects: a thread's loads stay in flight together
    };
    fft_regs_io<T, MX, NL, NT, true, false, true, false>(buf, twl, load, [](int, int, V) {});  // lines are rows
    // l0 = (ux, uy), l1 = (uz, dy b), l2 = (dy ux, dy uy), l3 = (dy uz, dz b), l4 = (dz ux, dz uy),
    // l5 = (dz uz, 0), l6 = (dx b, dx ux), l7 = (dx uy, dx uz)
    for (int x = threadIdx.x; x < MX; x += NT) {
        const V l0 = buf[0 * LS + pidx(x)], l1 = buf[1 * LS + pidx(x)], l2 = buf[2 * LS + pidx(x)];
        const V l3 = buf[3 * LS + pidx(x)], l4 = buf[4 * LS + pidx(x)], l5 = buf[5 * LS + pidx(x)];
        const V l6 = buf[6 * LS + pidx(x)], l7 = buf[7 * LS + pidx(x)];
        const T vx = l0.x, vy = l0.y, vz = l1.x;
        const T fb = -(vx * l6.x + vy * l1.y + vz * l3.y) * scale;
        const T fux = -(vx * l6.y + vy * l2.x + vz * l4.x) * scale;
        const T fuy = -(vx * l7.x + vy * l2.y + vz * l4.y) * scale;
        const T fuz = -(vx * l7.y + vy * l3.x + vz * l5.x) * scale;
        // each thread reads and rewrites only its own x positions: no barrier needed here
        buf[0 * LS + pidx(x)] = V{fb, fux};
        buf[1 * LS + pidx(x)] = V{fuy, fuz};
    }
    __syncthreads();
    fft_lds<T, MX, 2, NT, false>(buf, twl);
    const size_t hplane = (size_t)N * MY * NXH;
    for (int k = threadIdx.x; k < NXH; k += NT) {
        const size_t o = row * NXH + k;
#pragma unroll
        for (int l = 0; l < 2; ++l) {
            const V zk = buf[l * LS + pidx(k)], zm = buf[l * LS + pidx((MX - k) % MX)];
            H[(size_t)(2 * l) * hplane + o] = V{(zk.x + zm.x) * T(0.5), (zk.y - zm.y) * T(0.5)};
            H[(size_t)(2 * l + 1) * hplane + o] = V{(zk.y + zm.y) * T(0.5), (zm.x - zk.x) * T(0.5)};
        }
    }
}

// ---------------------------------------------------------------------------
// k3_yfwd: forward y transform of TK padded kx-lines, truncation with the y
// Nyquist fold, the x Nyquist fold on the kx = Nx/2 line.  Output z-grid planes.
// grid (ceil(nxh/TK), N, 4), XCD-remapped like k3_ybwd.
// ---------------------------------------------------------------------------
template <typename T, int NY, int MY, int TK, int NT>
__global__ __launch_bounds__(NT) void k3_yfwd(const cplx<T>* __restrict__ H, Ch3Geom geo, cplx<T>* __restrict__ F,
                                              const cplx<T>* __restrict__ tw) {
    using V = cplx<T>;
    constexpr int LS = line_stride_lf<T, TK>(MY);  // the tile's TK lines side by side in every access
    constexpr bool TW_LDS = (size_t)(TK * LS + MY) * sizeof(V) <= 160 * 1024;
    __shared__ V buf[TK * LS];
    __shared__ V twl_lds[TW_LDS ? MY : 1];
    const V* twl = TW_LDS ? twl_lds : tw;
    if constexpr (TW_LDS) load_twiddles<T, MY, NT>(twl_lds, tw);
    const unsigned gxy = gridDim.x * gridDim.y;
    const unsigned lin = xcd_remap(blockIdx.x + gridDim.x * (blockIdx.y + gridDim.y * blockIdx.z), gxy * gridDim.z);
    const int nxh = geo.nxh, z = (int)((lin / gridDim.x) % gridDim.y), o = (int)(lin / gxy);
    const int m0 = (int)(lin % gridDim.x) * TK;
    const V* in = H + (size_t)o * geo.N * MY * nxh + (size_t)z * MY * nxh;
    auto load = [&](int c, int j) -> V {
        const int m = m0 + c;
        return m < nxh ? in[(size_t)j * nxh + m] : V{T(0), T(0)};
    };
    fft_regs_io<T, MY, TK, NT, false, false, true, true, LS>(buf, twl, load, [](int, int, V) {});
    // truncation (in place: entries n < NY/2 stay, n > NY/2 come from MY - NY + n, Nyquist folded)
    constexpr int NTR = TK * NY, PT = (NTR + NT - 1) / NT;
    V tr[PT];
#pragma unroll
    for (int e = 0; e < PT; ++e) {
        const int idx = threadIdx.x + e * NT;
        if (NTR % NT != 0 && idx >= NTR) break;
        const int c = idx % TK, n = idx / TK;
        const V* L = buf + c * LS;
        V v;
        if (n < NY / 2) v = L[pidx(n)];
        else if (n == NY / 2) {
            const V a = L[pidx(NY / 2)], bb = L[pidx(MY - NY / 2)];
            v = V{a.x + bb.x, a.y + bb.y};
        } else v = L[pidx(MY - NY + n)];
        tr[e] = v;
    }
    __syncthreads();
#pragma unroll
    for (int e = 0; e < PT; ++e) {
        const int idx = threadIdx.x + e * NT;
        if (NTR % NT != 0 && idx >= NTR) break;
        const int c = idx % TK, n = idx / TK;
        buf[c * LS + pidx(n)] = tr[e];
    }
    __syncthreads();
    const bool xeven = (geo.nx % 2) == 0;
    V* out = F + (size_t)o * geo.N * geo.nmodes + (size_t)z * geo.nmodes;
    for (int idx = threadIdx.x; idx < TK * NY; idx += NT) {
        const int c = idx % TK, n = idx / TK;
        const int m = m0 + c;
        if (m >= nxh) continue;
        V v = buf[c * LS + pidx(n)];
        if (xeven && m == geo.nx / 2) {  // F(Nx/2, ky) += conj F(Nx/2, -ky)
            const V p = buf[c * LS + pidx((NY - n) % NY)];
            v = V{v.x + p.x, v.y - p.y};
        }
        out[(size_t)n * nxh + m] = v;
    }
}

// 3-D tau slots: 0 tau_p, 1 tau_b1, 2 tau_b2, 3 tau_u1x, 4 tau_u1y, 5 tau_u1z, 6 tau_u2x, 7 tau_u2y, 8 tau_u2z
constexpr int kCh3TauStride = 9;

// Multistep right-hand side with the grid round trip of the state (Hermitian part
// of the kx = 0 and kx = Nx/2 lines), scaled by 1/a0; histories replaced in place.
template <typename T>
struct Ch3SbdfArgs {
    const cplx<T>* X[4];   // b, ux, uy, uz
    const cplx<T>* F[4];   // F_n rows E2, E3x, E3y, E3z
    cplx<T>* Fm1[4];
    cplx<T>* MXm1[4];
    cplx<T>* R[4];         // E2, E3x, E3y, E3z (E1: zero)
    T c1, c2, a1, a2, inv_a0;
    Ch3Geom geo;
};

template <typename T>
__global__ void k3_sbdf(Ch3SbdfArgs<T> a, size_t n) {
    const int N = a.geo.N, nxh = a.geo.nxh, ny = a.geo.ny;
    for (size_t i = blockIdx.x * (size_t)blockDim.x + threadIdx.x; i < n; i += (size_t)gridDim.x * blockDim.x) {
        const int mode = (int)(i / N), k = (int)(i - (size_t)mode * N);
        const int m = mode % nxh, nn = mode / nxh;
        const bool xline = m == 0 || ((a.geo.nx % 2) == 0 && m == a.geo.nx / 2);
        const size_t partner = ((size_t)(m + nxh * ((ny - nn) % ny))) * N + k;
#pragma unroll
        for (int r = 0; r < 4; ++r) {
            cplx<T> x = a.X[r][i];
            if (xline) {
                const cplx<T> q = a.X[r][partner];
                x = cplx<T>{(x.x + q.x) * T(0.5), (x.y - q.y) * T(0.5)};
            }
            const cplx<T> f = a.F[r][i], fo = a.Fm1[r][i], mo = a.MXm1[r][i];
            const T vx = a.c1 * f.x + a.c2 * fo.x - a.a1 * x.x - a.a2 * mo.x;
            const T vy = a.c1 * f.y + a.c2 * fo.y - a.a1 * x.y - a.a2 * mo.y;
            a.R[r][i] = cplx<T>{vx * a.inv_a0, vy * a.inv_a0};
            a.Fm1[r][i] = f;
            a.MXm1[r][i] = x;
        }
    }
}

// L P(x) per mode (one workgroup per mode) for the RK stage loop; P is the grid round
// trip (Hermitian part of the kx = 0 and kx = Nx/2 lines, through the partner mode
// (m, -n)); tau_p has no basis and is not projected.  Dz and Dzz = Dz(Dz .) by
// cheb_dz_wave, one wavefront per (field, real / imaginary part).
//   E1  = i kx ux + i ky uy + Dz uz + [N-1] tau_u1z + [k=0, mode 0] tau_p
//   E2  = kappa (kh^2 b - Dzz b) - kappa Dz[:,N-1] tau_b1 + [N-1] tau_b2
//   E3a = nu (kh^2 ua - Dzz ua) - nu Dz[:,N-1] tau_u1a + i ka p + [N-1] tau_u2a   (a = x, y)
//   E3z = nu (kh^2 uz - Dzz uz) - nu Dz[:,N-1] tau_u1z + Dz p - b + [N-1] tau_u2z
template <typename T, int NT>
__global__ __launch_bounds__(NT) void k3_lx(const cplx<T>* __restrict__ p, const cplx<T>* __restrict__ b,
                                            const cplx<T>* __restrict__ ux, const cplx<T>* __restrict__ uy,
                                            const cplx<T>* __restrict__ uz, const cplx<T>* __restrict__ taus,
                                            Ch3Geom geo, double sz, double kappa, double nu, cplx<T>* E1,
                                            cplx<T>* E2, cplx<T>* E3x, cplx<T>* E3y, cplx<T>* E3z) {
    extern __shared__ unsigned char smem_raw[];
    const int N = geo.N, nxh = geo.nxh;
    static_assert(NT % 64 == 0, "whole wavefronts");
    double2* v = reinterpret_cast<double2*>(smem_raw);  // [5][N]: p, b, ux, uy, uz
    double2* d1 = v + 5 * N;                             // Dz of each
    double2* d2 = d1 + 5 * N;                            // Dzz of b, ux, uy, uz
    const int mode = blockIdx.x, m = mode % nxh, n = mode / nxh;
    const bool xline = m == 0 || ((geo.nx % 2) == 0 && m == geo.nx / 2);
    const int partner = m + nxh * ((geo.ny - n) % geo.ny);
    const cplx<T>* src[5] = {p, b, ux, uy, uz};
    for (int idx = threadIdx.x; idx < 5 * N; idx += NT) {
        const int f = idx / N, k = idx - f * N;
        const cplx<T> x = src[f][(size_t)mode * N + k];
        double2 w{(double)x.x, (double)x.y};
        if (xline) {
            const cplx<T> q = src[f][(size_t)partner * N + k];
            w = double2{0.5 * (w.x + (double)q.x), 0.5 * (w.y - (double)q.y)};
        }
        v[idx] = w;
    }
    __syncthreads();
    // z derivatives by wavefront suffix scans, one wavefront per (field, real / imaginary part)
    for (int q = threadIdx.x >> 6; q < 10; q += NT / 64)
        cheb_dz_wave(reinterpret_cast<const double*>(v + (q >> 1) * N) + (q & 1),
                     reinterpret_cast<double*>(d1 + (q >> 1) * N) + (q & 1), 2, N, sz);
    __syncthreads();
    for (int q = threadIdx.x >> 6; q < 8; q += NT / 64)
        cheb_dz_wave(reinterpret_cast<const double*>(d1 + (1 + (q >> 1)) * N) + (q & 1),
                     reinterpret_cast<double*>(d2 + (q >> 1) * N) + (q & 1), 2, N, sz);
    __syncthreads();
    double2 tau[kCh3TauStride];
    for (int t = 0; t < kCh3TauStride; ++t) {
        const cplx<T> x = taus[(size_t)mode * kCh3TauStride + t];
        double2 w{(double)x.x, (double)x.y};
        if (xline && t > 0) {
            const cplx<T> q = taus[(size_t)partner * kCh3TauStride + t];
            w = double2{0.5 * (w.x + (double)q.x), 0.5 * (w.y - (double)q.y)};
        }
        tau[t] = w;
    }
    const double kx = geo.k0x * m, ky = ch3_ky(geo, n), kh2 = kx * kx + ky * ky;
    for (int k = threadIdx.x; k < N; k += NT) {
        const double2 dzz[4] = {d2[k], d2[N + k], d2[2 * N + k], d2[3 * N + k]};  // Dzz of b, ux, uy, uz
        const double dN = cheb_dz(k, N - 1, sz);
        const double2 P = v[k], Bv = v[N + k], Ux = v[2 * N + k], Uy = v[3 * N + k], Uz = v[4 * N + k];
        const double2 DP = d1[k], DUz = d1[4 * N + k];
        const bool last = k == N - 1;
        double2 e1{-kx * Ux.y - ky * Uy.y + DUz.x, kx * Ux.x + ky * Uy.x + DUz.y};
        if (last) { e1.x += tau[5].x; e1.y += tau[5].y; }
        if (k == 0 && mode == 0) { e1.x += tau[0].x; e1.y += tau[0].y; }
        double2 e2{kappa * (kh2 * Bv.x - dzz[0].x) - kappa * dN * tau[1].x,
                   kappa * (kh2 * Bv.y - dzz[0].y) - kappa * dN * tau[1].y};
        double2 ex{nu * (kh2 * Ux.x - dzz[1].x) - nu * dN * tau[3].x - kx * P.y,
                   nu * (kh2 * Ux.y - dzz[1].y) - nu * dN * tau[3].y + kx * P.x};
        double2 ey{nu * (kh2 * Uy.x - dzz[2].x) - nu * dN * tau[4].x - ky * P.y,
                   nu * (kh2 * Uy.y - dzz[2].y) - nu * dN * tau[4].y + ky * P.x};
        double2 ez{nu * (kh2 * Uz.x - dzz[3].x) - nu * dN * tau[5].x + DP.x - Bv.x,
                   nu * (kh2 * Uz.y - dzz[3].y) - nu * dN * tau[5].y + DP.y - Bv.y};
        if (last) {
            e2.x += tau[2].x; e2.y += tau[2].y;
            ex.x += tau[6].x; ex.y += tau[6].y;
            ey.x += tau[7].x; ey.y += tau[7].y;
            ez.x += tau[8].x; ez.y += tau[8].y;
        }
        const size_t o = (size_t)mode * N + k;
        E1[o] = cplx<T>{T(e1.x), T(e1.y)};
        E2[o] = cplx<T>{T(e2.x), T(e2.y)};
        E3x[o] = cplx<T>{T(ex.x), T(ex.y)};
        E3y[o] = cplx<T>{T(ey.x), T(ey.y)};
        E3z[o] = cplx<T>{T(ez.x), T(ez.y)};
    }
}

// IMEX RK stage right-hand side on the five row blocks (E1, E2, E3x, E3y, E3z):
//   rhs = M X0 + dt sum_j (AE_j F_j - AI_j LX_j);  final update writes b, ux, uy, uz
template <typename T>
struct Ch3StageArgs {
    const cplx<T>* X0[4];      // b, ux, uy, uz at the start of the step
    const cplx<T>* F[4][4];    // F_j rows E2, E3x, E3y, E3z
    const cplx<T>* LX[4][5];   // LX_j rows E1..E3z (null: no weight in this stage)
    T ae[4], ai[4];
    int nterms;
    T dt;
    cplx<T>* out[5];
    int final_update;
};

template <typename T>
__global__ void k3_stage(Ch3StageArgs<T> a, size_t n) {
    for (size_t i = blockIdx.x * (size_t)blockDim.x + threadIdx.x; i < n; i += (size_t)gridDim.x * blockDim.x) {
        for (int r = 0; r < 5; ++r) {
            if (a.final_update && r == 0) continue;
            cplx<T> v = r == 0 ? cplx<T>{T(0), T(0)} : a.X0[r - 1][i];
            for (int j = 0; j < a.nterms; ++j) {
                if (r > 0) {
                    const cplx<T> f = a.F[j][r - 1][i];
                    v.x += a.dt * a.ae[j] * f.x;
                    v.y += a.dt * a.ae[j] * f.y;
                }
                if (a.LX[j][r]) {
                    const cplx<T> l = a.LX[j][r][i];
                    v.x -= a.dt * a.ai[j] * l.x;
                    v.y -= a.dt * a.ai[j] * l.y;
                }
            }
            a.out[a.final_update ? r - 1 : r][i] = v;
        }
    }
}

}  // namespace tarang
