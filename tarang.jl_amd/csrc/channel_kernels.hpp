// channel_kernels.hpp -- kernels of the RealFourier(x) x ChebyshevT(z) channel
// solver (2-D Rayleigh-Benard with the Chebyshev-tau method).
//
// Internal layout is mode-major: a field's coefficients are stored per Fourier
// mode m (kx = 2 pi m/Lx, m = 0..Nx/2) with the Chebyshev degree k contiguous:
// index m*N + k.  The reference layout (kx fastest) is used only at the ABI.
//
// Per-mode operators (T basis, z in [0, Lz]):
//   (Dz c)_k  = (2/c_k) sum_{j>k, j-k odd} j c_j * (2/Lz),             c_0 = 2, c_k = 1
//   (Dzz c)_k = (1/c_k) sum_{j>=k+2, j-k even} j (j^2 - k^2) c_j * (2/Lz)^2
// (src/core/basis/basis_operators.jl:826-852; the second is Dz applied twice).
#pragma once
#include <cmath>
#include <vector>

#include "fft_lds.hpp"
#include "fourier_kernels.hpp"
#include "mfma.hpp"
#include "tau_solve.hpp"

namespace tarang {

__host__ __device__ inline double cheb_dz(int k, int j, double s) {  // s = 2/Lz
    if (j <= k || ((j - k) & 1) == 0) return 0.0;
    return (k == 0 ? 1.0 : 2.0) * j * s;
}
__host__ __device__ inline double cheb_dzz(int k, int j, double s) {
    if (j < k + 2 || ((j - k) & 1)) return 0.0;
    return (k == 0 ? 0.5 : 1.0) * (double)j * ((double)j * j - (double)k * k) * s * s;
}

// Chebyshev matrices on the Gauss-Lobatto grid z_j = (1 - cos(pi j/(N-1))) Lz/2:
//   Bm[z][k] = T_k at point z = (-1)^k cos(pi k z/(N-1))             (backward)
//   Fm[k][z] = (-1)^k w_k/(N-1) * (DCT-I kernel)                       (forward, its inverse)
//   BD = Bm * Dz                                                        (backward of the z derivative)
inline void chebyshev_tables(int N, double Lz, std::vector<double>& BT, std::vector<double>& BDT, std::vector<double>& FT) {
    const long period = 2L * (N - 1);
    auto cospi = [&](long num) {
        const long r = ((num % period) + period) % period;
        return (double)cosl(3.14159265358979323846264338327950288L * (long double)r / (long double)(N - 1));
    };
    std::vector<double> Bm((size_t)N * N), Fm((size_t)N * N);
    for (int z = 0; z < N; ++z)
        for (int k = 0; k < N; ++k) Bm[(size_t)z * N + k] = ((k & 1) ? -1.0 : 1.0) * cospi((long)k * z);
    for (int k = 0; k < N; ++k)
        for (int z = 0; z < N; ++z) {
            const double sgn = (k & 1) ? -1.0 : 1.0;
            const double wk = (k == 0 || k == N - 1) ? 0.5 : 1.0;
            double e;
            if (z == 0) e = 1.0;
            else if (z == N - 1) e = sgn;
            else e = 2.0 * cospi((long)z * k);
            Fm[(size_t)k * N + z] = sgn * wk / (N - 1) * e;
        }
    const double s = 2.0 / Lz;
    BT.assign((size_t)N * N, 0.0);
    BDT.assign((size_t)N * N, 0.0);
    FT.assign((size_t)N * N, 0.0);
    for (int z = 0; z < N; ++z)
        for (int k = 0; k < N; ++k) {
            BT[(size_t)k * N + z] = Bm[(size_t)z * N + k];
            FT[(size_t)z * N + k] = Fm[(size_t)k * N + z];
            long double acc = 0;  // (Bm Dz)[z][k] = sum_{q<k} Bm[z][q] Dz[q][k]
            for (int q = 0; q < k; ++q) acc += (long double)Bm[(size_t)z * N + q] * cheb_dz(q, k, s);
            BDT[(size_t)k * N + z] = (double)acc;
        }
}

// ---------------------------------------------------------------------------
struct Ch3Geom {
    int nx, ny, nxh, N, nmodes;
    double k0x, k0y;
};

__host__ __device__ inline double ch3_ky(const Ch3Geom& g, int n) {
    const int kk = n < (g.ny + 1) / 2 ? n : n - g.ny;  // FFT order
    return g.k0y * kk;
}

// ---------------------------------------------------------------------------
// zbwd_mfma: z-backward transform of the operands on the matrix cores (k3_zbwd in 3-D,
// k_ch_zbwd in 2-D).  Workgroup = (tile of QT modes, field f in (b, ux, uy, uz), or
// (b, ux, uz) in 2-D; with gridDim.z > 1 a share of the z tiles); the field's
// coefficients of the tile are the columns of an LDS block C[k][col], in groups of 16
// modes: column 32 g + j is Re, 32 g + 16 + j is Im of mode q0 + 16 g + j.
// Parity split: the Gauss-Lobatto grid is symmetric (point N-1-z mirrors z) and
// T_k(-x) = (-1)^k T_k(x), T_k'(-x) = (-1)^(k+1) T_k'(x), so with the even- and odd-k sums
//   E = sum_{k even} BT[k][z] C[k],  O = sum_{k odd} BT[k][z] C[k]  (and E', O' with BDT)
// over the first half of the points (z < ceil(N/2)):
//   value[z] = E + O,  value[N-1-z] = E - O,  dz[z] = E' + O',  dz[N-1-z] = O' - E'
// half the products of evaluating every point.  Wave w takes first-half z tile w (then
// the next pass) with every column tile, both products and both parities, its loads one
// batch ahead of its products.  A lane then holds Re and Im of one mode and writes whole
// complex values straight to the z-major planes (16 consecutive modes per row).
// The kx = Nx/2 line is halved.  3-D: eight planes, value (b, ux, uy, uz) and dz; the y
// and x passes form dy and dx from the values.  2-D: eight planes, dx f = i kx value among
// them (zero on the kx = 0 and kx = Nx/2 lines, where the projected state's x derivative
// vanishes), and those lines keep only their real part (the grid round trip of the state).
// ---------------------------------------------------------------------------
// modes per workgroup (QT, a multiple of 16), threads per workgroup (NT) and k steps per load batch
// of a tile of qt modes: eight for the FP32 tiles of 16 that the few modes of a 2-D problem take, a round
// trip to L2 per batch (1024 x 256: 19.9 us, four steps 22.3); FP64 loses registers by four (3-D 281 us, two 263)
template <typename T> struct ZbwdTile {
    static constexpr int QT = 32, NT = 256;
    static constexpr int steps(int qt) { return qt == 16 ? 8 : 4; }
};
template <> struct ZbwdTile<double> {
    static constexpr int QT = 16, NT = 256;
    static constexpr int steps(int) { return 2; }
};

__host__ __device__ inline int zbwd_lds_stride(int qt) { return 2 * qt + 1; }
// first-half z tiles of the parity-split evaluation
__host__ __device__ inline int zbwd_half_tiles(int N) { return ((N + 1) / 2 + 15) / 16; }

template <typename T, int NT, bool TWO_D, int QT = ZbwdTile<T>::QT>
__device__ inline void zbwd_mfma(const cplx<T>* __restrict__ b, const cplx<T>* __restrict__ ux,
                                 const cplx<T>* __restrict__ uy, const cplx<T>* __restrict__ uz, const Ch3Geom& geo,
                                 const T* __restrict__ BT, const T* __restrict__ BDT, cplx<T>* __restrict__ G) {
    static_assert(NT == ZbwdTile<T>::NT && QT % 16 == 0, "workgroup size of the tile plan, 16-mode groups");
    using Op = MfmaOp<T>;
    using acc4 = typename Op::acc4;
    using V = cplx<T>;
    constexpr int NG = QT / 16, CT = 2 * NG, S = 2 * QT + 1;
    constexpr int U = ZbwdTile<T>::steps(QT), NWV = NT / 64;
    extern __shared__ unsigned char smem_raw[];
    T* C = reinterpret_cast<T*>(smem_raw);  // [KP][S]
    const int N = geo.N, nmodes = geo.nmodes;
    const int KP = (N + 15) & ~15, NH = (N + 1) / 2, nzh = zbwd_half_tiles(N);
    const int f = blockIdx.y, q0 = blockIdx.x * QT;
    const V* in = f == 0 ? b : (f == 1 ? ux : (f == 2 && !TWO_D ? uy : uz));
    // eight loads in flight per thread: one at a time, each turn waited for memory (3-D 256 x 256 x 128: 196 / 337 us
    // in FP32 / FP64 against 152 / 263; 2-D 1024 x 256 FP32 24.6 against 22.3, 320 x 97 FP64 14.0 against 12.4)
    constexpr int FB = 8;
    for (int i0 = threadIdx.x; i0 < QT * KP; i0 += FB * NT) {
        T re[FB], im[FB];
#pragma unroll
        for (int u = 0; u < FB; ++u) {
            const int idx = i0 + u * NT, q = idx / KP, k = idx - q * KP;
            const bool ok = q < QT && q0 + q < nmodes && k < N;
            const V v = in[ok ? (size_t)(q0 + q) * N + k : 0];
            re[u] = ok ? v.x : T(0);
            im[u] = ok ? v.y : T(0);
        }
#pragma unroll
        for (int u = 0; u < FB; ++u) {
            const int idx = i0 + u * NT, q = idx / KP, k = idx - q * KP;
            const int col = 32 * (q >> 4) + (q & 15);
            if (q < QT) {
                C[k * S + col] = re[u];
                C[k * S + col + 16] = im[u];
            }
        }
    }
    __syncthreads();
    const int lane = threadIdx.x & 63, r16 = lane & 15, q4 = lane >> 4;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const size_t plane = (size_t)N * nmodes;
    const bool xeven = (geo.nx % 2) == 0;
    // per mode group: this lane's mode and its factors
    T kxv[NG], wv[NG];
    bool xline[NG], live[NG];
    int qq[NG];
#pragma unroll
    for (int g = 0; g < NG; ++g) {
        const int q = q0 + 16 * g + r16;
        qq[g] = q;
        live[g] = q < nmodes;
        const int m = q % geo.nxh;
        const bool xny = xeven && m == geo.nx / 2;
        kxv[g] = T(geo.k0x * m);
        wv[g] = xny ? T(0.5) : T(1);
        xline[g] = m == 0 || xny;
    }
    // first-half z tiles of this workgroup: all, or a share when the grid splits z (blockIdx.z)
    const int zper = (nzh + (int)gridDim.z - 1) / (int)gridDim.z;
    const int zbeg = zper * (int)blockIdx.z, zend = min(nzh, zbeg + zper);
    for (int zt = zbeg + wave; zt < zend; zt += NWV) {
        const int z = 16 * zt + r16;  // this lane's row of the A operand
        acc4 acc[2][2][CT];           // [parity][value, dz][column tile]
#pragma unroll
        for (int par = 0; par < 2; ++par)
#pragma unroll
            for (int p = 0; p < 2; ++p)
#pragma unroll
                for (int ct = 0; ct < CT; ++ct) acc[par][p][ct] = acc4{T(0), T(0), T(0), T(0)};
        // k steps of both parities in one sequence: step s < s0 is even-k step s, then odd;
        // k = 2 (4 s' + q4) + parity
        const int s0 = (NH + 3) >> 2, s1 = (N / 2 + 3) >> 2, nsteps = s0 + s1;
        // two batches in turn: one batch's loads are in flight while the other's products run
        T amA[U][2], bvA[U][CT], amB[U][2], bvB[U][CT];
        auto load = [&](int sb, T (&am)[U][2], T (&bv)[U][CT]) {
#pragma unroll
            for (int u = 0; u < U; ++u) {
                const int st = sb + u, par = st < s0 ? 0 : 1, sp = par ? st - s0 : st;
                const int k = 2 * (4 * sp + q4) + par;
                const bool ok = st < nsteps && k < N && z < N;
                const int o = ok ? k * N + z : 0;
                am[u][0] = BT[o];
                am[u][1] = BDT[o];
                am[u][0] = ok ? am[u][0] : T(0);
                am[u][1] = ok ? am[u][1] : T(0);
                const int kr = k < KP ? k : KP - 1;  // rows N .. KP - 1 are zero; beyond, a is zero
#pragma unroll
                for (int ct = 0; ct < CT; ++ct) bv[u][ct] = C[kr * S + 16 * ct + r16];
            }
        };
        auto multiply = [&](int sb, const T (&am)[U][2], const T (&bv)[U][CT]) {
#pragma unroll
            for (int u = 0; u < U; ++u) {
                if (sb + u >= nsteps) break;  // wave-uniform
#pragma unroll
                for (int ct = 0; ct < CT; ++ct) {
                    if (sb + u < s0) {  // even k
                        acc[0][0][ct] = Op::mma(am[u][0], bv[u][ct], acc[0][0][ct]);
                        acc[0][1][ct] = Op::mma(am[u][1], bv[u][ct], acc[0][1][ct]);
                    } else {
                        acc[1][0][ct] = Op::mma(am[u][0], bv[u][ct], acc[1][0][ct]);
                        acc[1][1][ct] = Op::mma(am[u][1], bv[u][ct], acc[1][1][ct]);
                    }
                }
            }
        };
        load(0, amA, bvA);
        for (int sb = 0; sb < nsteps; sb += 2 * U) {
            if (sb + U < nsteps) load(sb + U, amB, bvB);
            multiply(sb, amA, bvA);
            if (sb + U >= nsteps) break;
            if (sb + 2 * U < nsteps) load(sb + 2 * U, amA, bvA);
            multiply(sb + U, amB, bvB);
        }
        auto put = [&](int zz, int g, V val, V dzv) {
            const size_t o = (size_t)zz * nmodes + qq[g];
            if constexpr (TWO_D) {
                const V dx = xline[g] ? V{T(0), T(0)} : V{-kxv[g] * val.y, kxv[g] * val.x};  // i kx v
                // no y transform follows: the kx = 0 and kx = Nx/2 lines keep their real part here
                if (xline[g]) val.y = dzv.y = T(0);
                // planes 0 ux, 1 uz, 2 dx b, 3 dz b, 4 dx ux, 5 dz ux, 6 dx uz, 7 dz uz
                if (f > 0) G[(size_t)(f - 1) * plane + o] = val;
                G[(size_t)(2 + 2 * f) * plane + o] = dx;
                G[(size_t)(3 + 2 * f) * plane + o] = dzv;
            } else {
                G[(size_t)f * plane + o] = val;
                G[(size_t)(4 + f) * plane + o] = dzv;
            }
        };
#pragma unroll
        for (int g = 0; g < NG; ++g)
#pragma unroll
            for (int v = 0; v < 4; ++v) {
                const int zr = 16 * zt + Op::row(v, q4);
                if (zr >= NH || !live[g]) continue;
                const T w = wv[g];
                const T er = acc[0][0][2 * g][v], ei = acc[0][0][2 * g + 1][v];
                const T orr = acc[1][0][2 * g][v], oi = acc[1][0][2 * g + 1][v];
                const T dr = acc[0][1][2 * g][v], di = acc[0][1][2 * g + 1][v];
                const T pr = acc[1][1][2 * g][v], pi = acc[1][1][2 * g + 1][v];
                put(zr, g, V{(er + orr) * w, (ei + oi) * w}, V{(dr + pr) * w, (di + pi) * w});
                const int zm = N - 1 - zr;
                if (zm != zr) put(zm, g, V{(er - orr) * w, (ei - oi) * w}, V{(pr - dr) * w, (pi - di) * w});
            }
    }
}

// k_ch_zbwd: the 2-D z-backward transform, zbwd_mfma with planes 0 ux, 1 uz, 2 dx b,
// 3 dz b, 4 dx ux, 5 dz ux, 6 dx uz, 7 dz uz (kx fastest, one N x nxh plane each).
// grid (ceil(nxh / QT), 3 fields, z shares).
template <typename T, int NT, int QT = ZbwdTile<T>::QT>
__global__ __launch_bounds__(NT, 768 / NT) void k_ch_zbwd(const cplx<T>* __restrict__ b, const cplx<T>* __restrict__ ux,
                                                   const cplx<T>* __restrict__ uz, Ch3Geom geo,
                                                   const T* __restrict__ BT, const T* __restrict__ BDT,
                                                   cplx<T>* __restrict__ G) {
    zbwd_mfma<T, NT, true, QT>(b, ux, nullptr, uz, geo, BT, BDT, G);
}

// ---------------------------------------------------------------------------
// k_ch_xpass: one z level per workgroup.  The eight operand rows are packed
// two per complex line (a + i b, Hermitian extension to MX), inverse FFT, then
//   F_b  = -(ux dx b  + uz dz b),  F_ux = -(ux dx ux + uz dz ux),
//   F_uz = -(ux dx uz + uz dz uz)
// and the three real products go through two forward FFTs (F_b + i F_ux, F_uz).
// Output: three N x nxh planes (kx fastest), scaled by 1/(Nx MX).
// ---------------------------------------------------------------------------
template <typename T, int NX, int MX, int NT>
__global__ __launch_bounds__(NT) void k_ch_xpass(const cplx<T>* __restrict__ G, int N, T scale,
                                                 cplx<T>* __restrict__ H, const cplx<T>* __restrict__ tw) {
    using V = cplx<T>;
    constexpr int NXH = NX / 2 + 1;
    constexpr int NL = 4;
    constexpr int LS = line_stride(MX);
    constexpr bool TW_LDS = (size_t)(NL * LS + MX) * sizeof(V) <= 160 * 1024;
    __shared__ V buf[NL * LS];
    __shared__ V twl_lds[TW_LDS ? MX : 1];
    const V* twl = TW_LDS ? twl_lds : tw;
    const int z = blockIdx.x;
    const size_t plane = (size_t)N * NXH;
    if constexpr (TW_LDS) load_twiddles<T, MX, NT>(twl_lds, tw);
    constexpr int NSRC = NL * NXH;
    constexpr int PS = (NSRC + NT - 1) / NT;
    V va[PS], vb[PS];
#pragma unroll
    for (int e = 0; e < PS; ++e) {
        const int idx = threadIdx.x + e * NT;
        if (NSRC % NT == 0 || idx < NSRC) {
            const int line = idx / NXH, k = idx - line * NXH;
            const size_t off = (size_t)z * NXH + k;
            va[e] = G[(size_t)(2 * line) * plane + off];
            vb[e] = G[(size_t)(2 * line + 1) * plane + off];
        }
    }
    constexpr int GAPN = MX - 2 * NXH + 1;
    for (int idx = threadIdx.x; idx < NL * GAPN; idx += NT) {
        const int line = idx / GAPN, k = NXH + (idx - line * GAPN);
        buf[line * LS + pidx(k)] = V{T(0), T(0)};
    }
#pragma unroll
    for (int e = 0; e < PS; ++e) {
        const int idx = threadIdx.x + e * NT;
        if (NSRC % NT == 0 || idx < NSRC) {
            const int line = idx / NXH, k = idx - line * NXH;
            const V a = va[e], bb = vb[e];
            V* L = buf + line * LS;
            if (k == 0) {
                L[pidx(0)] = V{a.x, bb.x};
            } else {
                L[pidx(k)] = V{a.x - bb.y, a.y + bb.x};
                L[pidx(MX - k)] = V{a.x + bb.y, bb.x - a.y};
            }
        }
    }
    __syncthreads();
    fft_lds<T, MX, NL, NT, true>(buf, twl);
    for (int x = threadIdx.x; x < MX; x += NT) {
        const V l0 = buf[0 * LS + pidx(x)];  // ux + i uz
        const V l1 = buf[1 * LS + pidx(x)];  // dx b + i dz b
        const V l2 = buf[2 * LS + pidx(x)];  // dx ux + i dz ux
        const V l3 = buf[3 * LS + pidx(x)];  // dx uz + i dz uz
        const T fb = -(l0.x * l1.x + l0.y * l1.y) * scale;
        const T fux = -(l0.x * l2.x + l0.y * l2.y) * scale;
        const T fuz = -(l0.x * l3.x + l0.y * l3.y) * scale;
        buf[0 * LS + pidx(x)] = V{fb, fux};
        buf[1 * LS + pidx(x)] = V{fuz, T(0)};
    }
    __syncthreads();
    fft_lds<T, MX, 2, NT, false>(buf, twl);
    for (int k = threadIdx.x; k < NXH; k += NT) {
        const V zk = buf[pidx(k)], zm = buf[pidx((MX - k) % MX)];
        const size_t o = (size_t)z * NXH + k;
        H[0 * plane + o] = V{(zk.x + zm.x) * T(0.5), (zk.y - zm.y) * T(0.5)};
        H[1 * plane + o] = V{(zk.y + zm.y) * T(0.5), (zm.x - zk.x) * T(0.5)};
        H[2 * plane + o] = buf[LS + pidx(k)];
    }
}

// ---------------------------------------------------------------------------
// k_ch_zfwd: z-forward Chebyshev transform of the product planes on the matrix cores
// (grid (ceil(nmodes/QT), planes, k splits), XCD-remapped) into mode-major F arrays:
//   F[m][k] = sum_z Fm[k][z] H[z][m],   FT[z*N + k] = Fm[k][z]
// Parity split: Fm[k][N-1-z] = (-1)^k Fm[k][z] on the symmetric Gauss-Lobatto grid, so
//   F[m][k even] = sum_{z < N/2} Fm[k][z] (H[z] + H[N-1-z]) (+ Fm[k][mid] H[mid], N odd)
//   F[m][k odd]  = sum_{z < N/2} Fm[k][z] (H[z] - H[N-1-z])
// half the products.  The sums HS and the differences HA of the plane tile sit in LDS as
// columns in groups of 16 modes (Re block, Im block), first-half rows only.  Output tiles
// hold 16 k of one parity (k = 2 (16 t + r) + parity; even tiles first, then odd); split s
// of the workgroup takes tiles [s*kps, (s+1)*kps), wave w tiles KPW w .. KPW w + KPW - 1 of
// it, then the next pass.  A lane holds Re and Im of one mode for four k and stores them
// directly.  The kx = Nx/2 column takes the x Nyquist fold 2 Re(H) (nx odd switches the
// fold off: the 3-D path folds in its y pass).
// ---------------------------------------------------------------------------
// z steps per load batch (U), threads per workgroup (NT) and k tiles per wavefront and
// pass (KPW), per arithmetic type (modes per workgroup QT: 16 or 32)
template <typename T> struct ZfwdTile { static constexpr int U = 2, NT = 512, KPW = 1; };
template <> struct ZfwdTile<double> { static constexpr int U = 4, NT = 256, KPW = 2; };

// LDS elements of k_ch_zfwd: the sum and difference blocks of the first-half rows
__host__ __device__ inline size_t ch_zfwd_lds_elems(int N, int qt) {
    return (size_t)2 * (((N + 1) / 2 + 15) & ~15) * (2 * qt + 1);
}
// output k tiles of k_ch_zfwd: even-k tiles, then odd-k tiles
__host__ __device__ inline int zfwd_k_tiles(int N) { return ((N + 1) / 2 + 15) / 16 + (N / 2 + 15) / 16; }

template <typename T, int QT, int NT>
__global__ __launch_bounds__(NT, 768 / NT) void k_ch_zfwd(const cplx<T>* __restrict__ H, int nmodes, int nx, int N,
                                                   const T* __restrict__ FT, cplx<T>* __restrict__ F0,
                                                   cplx<T>* __restrict__ F1, cplx<T>* __restrict__ F2,
                                                   cplx<T>* __restrict__ F3 = nullptr) {
    static_assert(NT == ZfwdTile<T>::NT && QT % 16 == 0, "workgroup size of the tile plan, 16-mode groups");
    using V = cplx<T>;
    using Op = MfmaOp<T>;
    using acc4 = typename Op::acc4;
    constexpr int NG = QT / 16, CT = 2 * NG, S = 2 * QT + 1;
    constexpr int KPW = ZfwdTile<T>::KPW, NWV = NT / 64;
    extern __shared__ unsigned char smem_raw[];
    const int NH = (N + 1) / 2, NHP = (NH + 15) & ~15, zsteps = (NH + 3) >> 2;
    T* CS = reinterpret_cast<T*>(smem_raw);  // [NHP][S] sums (even k)
    T* CA = CS + (size_t)NHP * S;            // [NHP][S] differences (odd k)
    const int nke = (NH + 15) / 16, nkt = zfwd_k_tiles(N);  // even tiles, all tiles
    const unsigned gxy = gridDim.x * gridDim.y;
    const unsigned lin = xcd_remap(blockIdx.x + gridDim.x * (blockIdx.y + gridDim.y * blockIdx.z), gxy * gridDim.z);
    const int f = (int)((lin / gridDim.x) % gridDim.y), q0 = (int)(lin % gridDim.x) * QT;
    const int kps = (nkt + (int)gridDim.z - 1) / (int)gridDim.z, kb = (int)(lin / gxy) * kps;
    const int ke = kb + kps < nkt ? kb + kps : nkt;
    const V* in = H + (size_t)f * N * nmodes;
    const bool xeven = (nx % 2) == 0;
    // four rows in flight per thread: one at a time, each turn waited for memory (3-D 256 x 256 x 128: 114 / 180 us
    // in FP32 / FP64 against 109 / 165)
    constexpr int FB = 4;
    for (int i0 = threadIdx.x; i0 < QT * NHP; i0 += FB * NT) {
        T zr[FB], zi[FB], mr[FB], mi[FB];
#pragma unroll
        for (int u = 0; u < FB; ++u) {
            const int idx = i0 + u * NT, zz = idx / QT, m = q0 + idx - zz * QT, zm = N - 1 - zz;
            const bool ok = zz < NH && m < nmodes, two = ok && zm != zz;
            const V hz = in[ok ? (size_t)zz * nmodes + m : 0], hm = in[two ? (size_t)zm * nmodes + m : 0];
            zr[u] = ok ? hz.x : T(0);
            zi[u] = ok ? hz.y : T(0);
            mr[u] = two ? hm.x : T(0);
            mi[u] = two ? hm.y : T(0);
        }
#pragma unroll
        for (int u = 0; u < FB; ++u) {
            const int idx = i0 + u * NT, zz = idx / QT, q = idx - zz * QT;
            if (zz >= NHP) continue;
            V hz{zr[u], zi[u]}, hm{mr[u], mi[u]};
            if (xeven && q0 + q == nx / 2) {
                hz = V{T(2) * hz.x, T(0)};
                hm = V{T(2) * hm.x, T(0)};
            }
            const int col = 32 * (q >> 4) + (q & 15);
            const bool mid = N - 1 - zz == zz;  // the middle point (N odd) counts once, in the even sums
            CS[zz * S + col] = hz.x + hm.x;
            CS[zz * S + col + 16] = hz.y + hm.y;
            CA[zz * S + col] = mid ? T(0) : hz.x - hm.x;
            CA[zz * S + col + 16] = mid ? T(0) : hz.y - hm.y;
        }
    }
    __syncthreads();
    const int lane = threadIdx.x & 63, r16 = lane & 15, q4 = lane >> 4;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    V* out = f == 0 ? F0 : (f == 1 ? F1 : (f == 2 ? F2 : F3));
    for (int kt0 = kb + KPW * wave; kt0 < ke; kt0 += KPW * NWV) {
        int par[KPW], kk[KPW];  // parity of each tile and this lane's k as the A operand's row
#pragma unroll
        for (int a = 0; a < KPW; ++a) {
            const int t = kt0 + a;
            par[a] = t < nke ? 0 : 1;
            kk[a] = 2 * (16 * (par[a] ? t - nke : t) + r16) + par[a];
        }
        acc4 acc[KPW][CT];  // [k tile][column tile]
#pragma unroll
        for (int a = 0; a < KPW; ++a)
#pragma unroll
            for (int ct = 0; ct < CT; ++ct) acc[a][ct] = acc4{T(0), T(0), T(0), T(0)};
        constexpr int U = ZfwdTile<T>::U;
        for (int zs = 0; zs < zsteps; zs += U) {
            T am[U][KPW], bs[U][CT], ba[U][CT];
#pragma unroll
            for (int u = 0; u < U; ++u) {
                const int zz = 4 * (zs + u) + q4;
#pragma unroll
                for (int a = 0; a < KPW; ++a) {
                    const bool ok = zz < NH && kk[a] < N && kt0 + a < ke;
                    am[u][a] = FT[ok ? zz * N + kk[a] : 0];
                    am[u][a] = ok ? am[u][a] : T(0);
                }
                const int zr = zz < NHP ? zz : NHP - 1;  // rows NH .. NHP - 1 are zero; beyond, a is zero
#pragma unroll
                for (int ct = 0; ct < CT; ++ct) {
                    bs[u][ct] = CS[zr * S + 16 * ct + r16];
                    ba[u][ct] = CA[zr * S + 16 * ct + r16];
                }
            }
#pragma unroll
            for (int u = 0; u < U; ++u)
#pragma unroll
                for (int a = 0; a < KPW; ++a)
#pragma unroll
                    for (int ct = 0; ct < CT; ++ct)
                        acc[a][ct] = Op::mma(am[u][a], par[a] ? ba[u][ct] : bs[u][ct], acc[a][ct]);
        }
#pragma unroll
        for (int g = 0; g < NG; ++g) {
            const int m = q0 + 16 * g + r16;
            if (m >= nmodes) continue;
#pragma unroll
            for (int a = 0; a < KPW; ++a) {
                if (kt0 + a >= ke) continue;
                const int t = kt0 + a, base = 16 * (par[a] ? t - nke : t);
#pragma unroll
                for (int v = 0; v < 4; ++v) {
                    const int k = 2 * (base + Op::row(v, q4)) + par[a];
                    if (k < N) out[(size_t)m * N + k] = V{acc[a][2 * g][v], acc[a][2 * g + 1][v]};
                }
            }
        }
    }
}

// ---------------------------------------------------------------------------
// Stage pieces.  Equation rows per mode: E1 (divergence), E2 (b), E3x, E3z,
// each N long; BC rows are overridden inside the solve.
// ---------------------------------------------------------------------------
template <typename T>
struct ChStageArgs {
    const cplx<T>* X0[3];      // b, ux, uz at the start of the step (M x0)
    const cplx<T>* F[4][3];    // F_j rows E2, E3x, E3z
    const cplx<T>* LX[4][4];   // LX_j rows E1, E2, E3x, E3z
    T ae[4], ai[4];
    int nterms;
    T dt;
    cplx<T>* out[4];           // rhs rows E1, E2, E3x, E3z  (or, final: b, ux, uz)
    int final_update;
    cplx<T>* clr;              // final: p (n values) and the taus (ntau) cleared in the same pass
    cplx<T>* taus;
    size_t ntau;
};

// rhs = M x0 + dt sum_j (AE_j F_j - AI_j LX_j) on the four row blocks; the final
// update applies M^+ (evolved rows only) and clears p and the taus.
template <typename T>
__global__ void k_ch_stage(ChStageArgs<T> a, size_t n) {
    const size_t i0 = blockIdx.x * (size_t)blockDim.x + threadIdx.x, step = (size_t)gridDim.x * blockDim.x;
    if (a.taus)
        for (size_t i = i0; i < a.ntau; i += step) a.taus[i] = cplx<T>{T(0), T(0)};
    for (size_t i = i0; i < n; i += step) {
        if (a.clr) a.clr[i] = cplx<T>{T(0), T(0)};
        for (int r = 0; r < 4; ++r) {
            if (a.final_update && r == 0) continue;
            cplx<T> v = r == 0 ? cplx<T>{T(0), T(0)} : a.X0[r - 1][i];
            for (int j = 0; j < a.nterms; ++j) {
                if (r > 0 && a.F[j][r - 1]) {
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

// Per-mode multistep right-hand side (step_subproblem_multistep.jl:197-420), scaled by
// 1/a0 so that the solve uses M + (1/a0) L:
//   R = (c1 F_n + c2 F_{n-1} - a1 M P(x_n) - a2 M P(x_{n-1})) / a0;   E1 rows 0, not stored
// M P(x) is the evolved part (b, ux, uz) of the grid-round-tripped state.  The
// histories F_{n-1}, M P(x_{n-1}) are replaced by the current values in the same pass.
template <typename T>
struct ChSbdfArgs {
    const cplx<T>* X[3];   // state b, ux, uz
    const cplx<T>* F[3];   // F_n rows E2, E3x, E3z
    cplx<T>* Fm1[3];
    cplx<T>* MXm1[3];
    cplx<T>* R[3];         // rhs rows E2, E3x, E3z (E1: zero)
    T c1, c2, a1, a2, inv_a0;
    int N, nx;
};

template <typename T>
__global__ void k_ch_sbdf(ChSbdfArgs<T> a, size_t n) {
    for (size_t i = blockIdx.x * (size_t)blockDim.x + threadIdx.x; i < n; i += (size_t)gridDim.x * blockDim.x) {
        const int m = (int)(i / a.N);
        const bool proj = m == 0 || ((a.nx % 2) == 0 && m == a.nx / 2);
#pragma unroll
        for (int r = 0; r < 3; ++r) {
            cplx<T> x = a.X[r][i];
            if (proj) x.y = T(0);
            const cplx<T> f = a.F[r][i], fo = a.Fm1[r][i], mo = a.MXm1[r][i];
            const T vx = a.c1 * f.x + a.c2 * fo.x - a.a1 * x.x - a.a2 * mo.x;
            const T vy = a.c1 * f.y + a.c2 * fo.y - a.a1 * x.y - a.a2 * mo.y;
            a.R[r][i] = cplx<T>{vx * a.inv_a0, vy * a.inv_a0};
            a.Fm1[r][i] = f;
            a.MXm1[r][i] = x;
        }
    }
}

// d_r = s_r (n values); with clr / taus given, also clears clr (n values) and taus (ntau)
template <typename T>
__global__ void k_ch_copy(const cplx<T>* __restrict__ s0, const cplx<T>* __restrict__ s1,
                          const cplx<T>* __restrict__ s2, cplx<T>* d0, cplx<T>* d1, cplx<T>* d2, size_t n,
                          cplx<T>* __restrict__ clr = nullptr, cplx<T>* __restrict__ taus = nullptr, size_t ntau = 0) {
    const size_t i0 = blockIdx.x * (size_t)blockDim.x + threadIdx.x, step = (size_t)gridDim.x * blockDim.x;
    for (size_t i = i0; i < n; i += step) {
        d0[i] = s0[i];
        d1[i] = s1[i];
        d2[i] = s2[i];
        if (clr) clr[i] = cplx<T>{T(0), T(0)};
    }
    if (taus)
        for (size_t i = i0; i < ntau; i += step) taus[i] = cplx<T>{T(0), T(0)};
}

template <typename T>
__global__ void k_ch_zero(cplx<T>* a, size_t n) {
    for (size_t i = blockIdx.x * (size_t)blockDim.x + threadIdx.x; i < n; i += (size_t)gridDim.x * blockDim.x)
        a[i] = cplx<T>{T(0), T(0)};
}

// (Dz f)_k = sum_{j > k, j - k odd} 2 j sz f_j, halved at k = 0 (the closed form of the
// descending Chebyshev recurrence u_k = u_{k+2} + 2 (k+1) sz f_{k+1}), for one real sequence
// f_j = in[j st], j < N, into out[k st], by one whole wavefront: each lane sums a run of
// ceil(N/64) consecutive j by parity, a shuffle scan gives every lane the sums past its run,
// and the lane then walks its run downwards.
__device__ inline void cheb_dz_wave(const double* in, double* out, int st, int N, double sz) {
    const int lane = threadIdx.x & 63, PL = (N + 63) / 64, j0 = lane * PL;
    double se = 0.0, so = 0.0;  // this lane's sums of 2 j sz f_j over even / odd j
    for (int i = 0; i < PL; ++i) {
        const int j = j0 + i;
        if (j < N) {
            const double w = 2.0 * j * sz * in[(size_t)j * st];
            if (j & 1) so += w;
            else se += w;
        }
    }
    double te = se, to = so;  // inclusive suffix sums over lanes >= lane
    for (int d = 1; d < 64; d <<= 1) {
        const double ne = __shfl_down(te, d), no = __shfl_down(to, d);
        if (lane + d < 64) {
            te += ne;
            to += no;
        }
    }
    double ae = te - se, ao = to - so;  // sums over j past this lane's run
    for (int i = PL - 1; i >= 0; --i) {
        const int k = j0 + i;
        if (k < N) {
            const double u = (k & 1) ? ae : ao;  // j > k of the other parity
            out[(size_t)k * st] = k == 0 ? 0.5 * u : u;
            const double w = 2.0 * k * sz * in[(size_t)k * st];
            if (k & 1) ao += w;
            else ae += w;
        }
    }
}

// L * P(x) per mode (one workgroup per mode), P = real part at kx = 0, Nx/2.
// taus[m*8 + t]: 0 tau_p, 1 tau_b1, 2 tau_b2, 3 tau_u1x, 4 tau_u1z, 5 tau_u2x, 6 tau_u2z
// The z derivatives come from cheb_dz_wave; Dzz = Dz(Dz .).
template <typename T, int NT>
__global__ __launch_bounds__(NT) void k_ch_lx(const cplx<T>* __restrict__ p, const cplx<T>* __restrict__ b,
                                              const cplx<T>* __restrict__ ux, const cplx<T>* __restrict__ uz,
                                              const cplx<T>* __restrict__ taus, int nxh, int nx, int N, double k0x,
                                              double sz, double kappa, double nu, cplx<T>* E1, cplx<T>* E2,
                                              cplx<T>* E3x, cplx<T>* E3z) {
    static_assert(NT % 64 == 0, "whole wavefronts");
    extern __shared__ unsigned char smem_raw[];
    double* v = reinterpret_cast<double*>(smem_raw);  // [4][N][2]: p, b, ux, uz
    double* d1 = v + 8 * N;                             // Dz of each
    double* d2 = d1 + 8 * N;                            // Dzz of b, ux, uz
    const int m = blockIdx.x;
    const bool proj = (m == 0) || ((nx % 2) == 0 && m == nx / 2);
    const cplx<T>* src[4] = {p, b, ux, uz};
    for (int idx = threadIdx.x; idx < 4 * N; idx += NT) {
        const int f = idx / N, k = idx - f * N;
        const cplx<T> s = src[f][(size_t)m * N + k];
        v[2 * idx] = (double)s.x;
        v[2 * idx + 1] = proj ? 0.0 : (double)s.y;
    }
    __syncthreads();
    // out[(f - f0) N + k] = (Dz in[f])_k for nf fields starting at f0 (real and imaginary parts
    // interleaved): one wavefront per (field, part)
    auto dz = [&](const double* in, double* out, int f0, int nf) {
        for (int q = threadIdx.x >> 6; q < 2 * nf; q += NT / 64) {
            const int f = f0 + (q >> 1), c = q & 1;
            cheb_dz_wave(in + 2 * (size_t)f * N + c, out + 2 * (size_t)(f - f0) * N + c, 2, N, sz);
        }
    };
    dz(v, d1, 0, 4);
    __syncthreads();
    dz(d1, d2, 1, 3);
    __syncthreads();
    double2 tau[7];
    for (int t = 0; t < 7; ++t) {  // tau_p has no x basis: it does not go through the x transform
        const cplx<T> s = taus[(size_t)m * 8 + t];
        tau[t] = double2{(double)s.x, (proj && t > 0) ? 0.0 : (double)s.y};
    }
    const double kx = k0x * m;
    auto at = [&](const double* a, int f, int k) { return double2{a[2 * (f * N + k)], a[2 * (f * N + k) + 1]}; };
    for (int k = threadIdx.x; k < N; k += NT) {
        const double2 dzz[3] = {at(d2, 0, k), at(d2, 1, k), at(d2, 2, k)};  // Dzz of b, ux, uz
        const double dN = cheb_dz(k, N - 1, sz);  // Dz[:, N-1], the derivative of the lift
        const double2 P = at(v, 0, k), Bv = at(v, 1, k), Ux = at(v, 2, k), Uz = at(v, 3, k);
        const double2 DP = at(d1, 0, k), DUz = at(d1, 3, k);
        double2 e1{-kx * Ux.y + DUz.x, kx * Ux.x + DUz.y};
        if (k == N - 1) { e1.x += tau[4].x; e1.y += tau[4].y; }
        if (k == 0 && m == 0) { e1.x += tau[0].x; e1.y += tau[0].y; }
        double2 e2{-kappa * (dzz[0].x - kx * kx * Bv.x) - kappa * dN * tau[1].x,
                   -kappa * (dzz[0].y - kx * kx * Bv.y) - kappa * dN * tau[1].y};
        double2 e3x{-nu * (dzz[1].x - kx * kx * Ux.x) - nu * dN * tau[3].x - kx * P.y,
                    -nu * (dzz[1].y - kx * kx * Ux.y) - nu * dN * tau[3].y + kx * P.x};
        double2 e3z{-nu * (dzz[2].x - kx * kx * Uz.x) - nu * dN * tau[4].x + DP.x - Bv.x,
                    -nu * (dzz[2].y - kx * kx * Uz.y) - nu * dN * tau[4].y + DP.y - Bv.y};
        if (k == N - 1) {
            e2.x += tau[2].x; e2.y += tau[2].y;
            e3x.x += tau[5].x; e3x.y += tau[5].y;
            e3z.x += tau[6].x; e3z.y += tau[6].y;
        }
        const size_t o = (size_t)m * N + k;
        E1[o] = cplx<T>{T(e1.x), T(e1.y)};
        E2[o] = cplx<T>{T(e2.x), T(e2.y)};
        E3x[o] = cplx<T>{T(e3x.x), T(e3x.y)};
        E3z[o] = cplx<T>{T(e3z.x), T(e3z.y)};
    }
}

// ---------------------------------------------------------------------------
// Wall values of b -> per-mode boundary values: the unnormalised rfft along x (and FFT
// along y) of each wall's grid array, in FP64, as the reference projects an array BC
// onto a Fourier mode.  Stage 1: h[w][y][kx] = sum_x v_w[x + nx y] e^{-2 pi i kx x/nx};
// stage 2: out[2 (kx + nxh ky) + w] = sum_y h[w][y][kx] e^{-2 pi i ky y/ny}.
template <typename S>
__global__ void k_wall_dft_x(const S* __restrict__ v0, const S* __restrict__ v1, int nx, int ny, int nxh,
                             const double2* __restrict__ tw, double2* __restrict__ h) {
    const int idx = blockIdx.x * blockDim.x + threadIdx.x;
    if (idx >= 2 * nxh * ny) return;
    const int w = idx / (nxh * ny), r = idx - w * nxh * ny, kx = r % nxh, y = r / nxh;
    const S* v = (w ? v1 : v0) + (size_t)y * nx;
    double re = 0.0, im = 0.0;
    for (int x = 0; x < nx; ++x) {
        const double2 t = tw[(kx * x) % nx];
        const double a = (double)v[x];
        re += a * t.x;
        im += a * t.y;
    }
    h[idx] = double2{re, im};
}

static __global__ void k_wall_dft_y(const double2* __restrict__ h, int ny, int nxh, const double2* __restrict__ tw,
                             double2* __restrict__ out) {
    const int idx = blockIdx.x * blockDim.x + threadIdx.x;
    if (idx >= 2 * nxh * ny) return;
    const int w = idx / (nxh * ny), r = idx - w * nxh * ny, kx = r % nxh, ky = r / nxh;
    const double2* hw = h + (size_t)w * nxh * ny;
    double re = 0.0, im = 0.0;
    for (int y = 0; y < ny; ++y) {
        const double2 t = tw[(ky * y) % ny], a = hw[(size_t)y * nxh + kx];
        re += a.x * t.x - a.y * t.y;
        im += a.x * t.y + a.y * t.x;
    }
    out[2 * (size_t)(kx + nxh * ky) + w] = double2{re, im};
}

// Per-mode boundary values of constant walls: nx ny b_w at mode 0, zero elsewhere.
inline std::vector<double2> constant_wall_values(size_t nmodes, double scale, double b0, double b1) {
    std::vector<double2> v(2 * nmodes, double2{0.0, 0.0});
    v[0] = double2{scale * b0, 0.0};
    v[1] = double2{scale * b1, 0.0};
    return v;
}

// reference layout (kx fastest, (nxh, N)) <-> mode-major (N contiguous per mode)
template <typename T>
__global__ void k_ch_transpose(const cplx<T>* __restrict__ in, cplx<T>* __restrict__ out, int rows, int cols) {
    // in: rows x cols, element (r, c) at r*cols + c; out: (c, r) at c*rows + r
    __shared__ cplx<T> tile[32][33];
    const int c0 = blockIdx.x * 32, r0 = blockIdx.y * 32;
    for (int j = threadIdx.y; j < 32; j += blockDim.y) {
        const int r = r0 + j, c = c0 + threadIdx.x;
        if (r < rows && c < cols) tile[j][threadIdx.x] = in[(size_t)r * cols + c];
    }
    __syncthreads();
    for (int j = threadIdx.y; j < 32; j += blockDim.y) {
        const int c = c0 + j, r = r0 + threadIdx.x;
        if (r < rows && c < cols) out[(size_t)c * rows + r] = tile[threadIdx.x][j];
    }
}

}  // namespace tarang
