// channel3d_solver.hip -- 3-D Rayleigh-Benard channel, per-mode multistep on the GPU.
//
// Step (src/core/timesteppers/step_subproblem_multistep.jl:197-420, _sbdf2_coefs :544-552):
//   F_n = F(P(x_n)) (z-backward, padded y and x passes, z-forward), M P(x_n)
//   rhs = (c1 F_n + c2 F_{n-1} - a1 M P(x_n) - a2 M P(x_{n-1})) / a0, BC rows c ALG
//   x_{n+1} = (M + L/a0)^-1 rhs  per mode: direct FP64 line solves (tau_solve.hpp)
// SBDF1 on the first step after create / set_field, SBDF2 (w = dt/dt_prev) after.
#include <algorithm>
#include <array>
#include <cmath>
#include <mutex>
#include <cstdlib>
#include <type_traits>
#include <cstring>
#include <map>
#include <string>
#include <vector>

#include "channel3d_kernels.hpp"
#include "channel3d_solver.hpp"
#include "diagnostics.hpp"
#include "flow_tools.hpp"
#include "dispatch.hpp"

namespace tarang {

namespace {
bool size_ok(int n) {
    bool ok = false;
    dispatch_size(n, [&](auto) { ok = true; }, Sizes2D{});
    return ok;
}
}  // namespace

void Channel3Solver::validate(const Channel3Desc& d) {
    TG_REQUIRE(d.dtype == kF32 || d.dtype == kF64, kErrInvalid, "3-D channel solver: dtype must be f32 or f64");
    TG_REQUIRE(d.stepper == kSBDF2 || d.stepper == kSBDF1 || d.stepper == kRK222 || d.stepper == kRK443, kErrInvalid,
               "3-D channel solver: timestepper must be SBDF2, SBDF1, RK222 or RK443");
    const int xmax = d.dtype == kF64 ? 512 : 1024;
    TG_REQUIRE(size_ok(d.nx) && d.nx <= xmax && size_ok(d.ny) && d.ny <= 1024, kErrInvalid,
               "3-D channel solver: RealFourier sizes " + std::to_string(d.nx) + "x" + std::to_string(d.ny) +
                   " unsupported (2^k 8..2048, 3 2^k 48..768, 5 2^k 80..640; x up to " + std::to_string(xmax) +
                   ", y up to 1024)");
    TG_REQUIRE(d.nz >= 4 && d.nz <= 256, kErrInvalid,
               "3-D channel solver: ChebyshevT size " + std::to_string(d.nz) + " unsupported (4..256)");
    TG_REQUIRE(d.refine_sweeps >= 0 && d.refine_sweeps <= 2, kErrInvalid,
               "3-D channel solver: refine_sweeps must be 0, 1 or 2");
    TG_REQUIRE(d.refine_sweeps == 0 || d.nz <= 208, kErrInvalid,
               "3-D channel solver: refinement sweeps need nz <= 208");
    TG_REQUIRE(d.split_inverse == 0 || (d.split_inverse == 1 && d.dtype == kF32), kErrInvalid,
               "3-D channel solver: split_inverse is 0, or 1 with an FP32 state");
    TG_REQUIRE(d.Lx > 0 && d.Ly > 0 && d.Lz > 0 && d.dt > 0, kErrInvalid,
               "3-D channel solver: lengths and dt must be positive");
}

Channel3Solver::Channel3Solver(Context* ctx, const Channel3Desc& d) : ctx_(ctx), d_(d) {
    validate(d);
    nxh_ = d.nx / 2 + 1;
    nmodes_ = nxh_ * d.ny;
    mx_ = padded_len(d.nx);
    my_ = padded_len(d.ny);
    dt_prev_ = d.dt;
    ctx_->activate();
    hipStream_t s = ctx_->stream;
    const size_t fb = field_bytes(), vb = 2 * dtype_size((DType)d.dtype);
    auto zeroed = [&](DevBuf& b, size_t bytes) {
        b = DevBuf(ctx_, bytes);
        TG_HIP(hipMemsetAsync(b.ptr, 0, bytes, s));
    };
    zeroed(P_, fb);
    zeroed(B_, fb);
    zeroed(UX_, fb);
    zeroed(UY_, fb);
    zeroed(UZ_, fb);
    zeroed(TAU_, (size_t)nmodes_ * kCh3TauStride * vb);
    for (int r = 0; r < 4; ++r) {
        zeroed(F_[r], fb);
        zeroed(Fm1_[r], fb);
        zeroed(MXm1_[r], fb);
    }
    for (int r = multistep() ? 1 : 0; r < 5; ++r) zeroed(R_[r], fb);  // the multistep E1 rows are zero
    tab_ = make_tableau(d.stepper);
    if (!multistep()) {
        for (int r = 0; r < 4; ++r) zeroed(X0_[r], fb);
        for (int st = 0; st < tab_.stages; ++st) {
            for (int r = 0; r < 4; ++r) zeroed(Frk_[st][r], fb);
            for (int r = 0; r < 5 && uses_lx(tab_, st); ++r) zeroed(LX_[st][r], fb);
        }
    }
    const size_t prow = (size_t)d.nz * my_ * nxh_ * vb;  // one y-padded plane
    G_ = DevBuf(ctx_, (size_t)kCh3ZPlanes * fb);
    Q_ = DevBuf(ctx_, (size_t)kCh3Planes * prow);
    H_ = DevBuf(ctx_, (size_t)4 * prow);
    // Chebyshev tables
    std::vector<double> BT, BDT, FT;
    chebyshev_tables(d.nz, d.Lz, BT, BDT, FT);
    const size_t nn = (size_t)d.nz * d.nz;
    auto upload = [&](DevBuf& b, const std::vector<double>& h) {
        if (d.dtype == kF64) {
            b = DevBuf(ctx_, nn * sizeof(double));
            TG_HIP(hipMemcpyAsync(b.ptr, h.data(), nn * sizeof(double), hipMemcpyHostToDevice, s));
            TG_HIP(hipStreamSynchronize(s));
        } else {
            std::vector<float> f(h.begin(), h.end());
            b = DevBuf(ctx_, nn * sizeof(float));
            TG_HIP(hipMemcpyAsync(b.ptr, f.data(), nn * sizeof(float), hipMemcpyHostToDevice, s));
            TG_HIP(hipStreamSynchronize(s));
        }
    };
    upload(BT_, BT);
    upload(BDT_, BDT);
    upload(FT_, FT);
    // |k_h|^2 keys: integer m^2 + kk^2 when Lx == Ly, the pair (m^2, kk^2) otherwise; key 0 = kx = ky = 0
    const double k0x = 2.0 * M_PI / d.Lx, k0y = 2.0 * M_PI / d.Ly;
    std::map<std::pair<long, long>, int> keymap;
    std::vector<int> key(nmodes_);
    std::vector<double> khv, rot(2 * (size_t)nmodes_);
    const bool iso = d.Lx == d.Ly;
    keymap[{0, 0}] = 0;
    khv.push_back(0.0);
    for (int q = 0; q < nmodes_; ++q) {
        const int m = q % nxh_, n = q / nxh_;
        const long kk = n < (d.ny + 1) / 2 ? n : n - d.ny;
        const std::pair<long, long> kp = iso ? std::make_pair((long)m * m + kk * kk, 0L) : std::make_pair((long)m * m, kk * kk);
        auto it = keymap.find(kp);
        if (it == keymap.end()) {
            const double kx = k0x * m, ky = k0y * kk;
            it = keymap.emplace(kp, (int)khv.size()).first;
            khv.push_back(std::sqrt(kx * kx + ky * ky));
        }
        key[q] = it->second;
        const double kx = k0x * m, ky = k0y * kk, kh = std::sqrt(kx * kx + ky * ky);
        rot[2 * q] = kh > 0 ? kx / kh : 1.0;
        rot[2 * q + 1] = kh > 0 ? ky / kh : 0.0;
    }
    // the only mode with key 0 is kx = ky = 0 (integer keys), so the tau_p system is key 0
    nkeys_ = (int)khv.size();
    // modes sorted by key: neighbouring waves of the solve read the same key's table
    std::vector<int2> modes(nmodes_);
    for (int q = 0; q < nmodes_; ++q) modes[q] = int2{q, key[q]};
    std::stable_sort(modes.begin(), modes.end(), [](const int2& a, const int2& b) { return a.y < b.y; });
    kh_max_ = *std::max_element(khv.begin(), khv.end());
    auto up = [&](DevBuf& b, const void* h, size_t bytes) {
        b = DevBuf(ctx_, bytes);
        TG_HIP(hipMemcpyAsync(b.ptr, h, bytes, hipMemcpyHostToDevice, s));
        TG_HIP(hipStreamSynchronize(s));
    };
    up(kh_, khv.data(), khv.size() * sizeof(double));
    up(modes_, modes.data(), modes.size() * sizeof(int2));
    up(rot_, rot.data(), rot.size() * sizeof(double));
    tab_tau_ = DevBuf(ctx_, tau_table_doubles(tau_shape(d.nz, true, any_sign()), nkeys_) * sizeof(double));
    if (any_sign()) info_ = DevBuf(ctx_, nkeys_ * sizeof(int));
    {
        const auto bcv = constant_wall_values((size_t)nmodes_, (double)d.nx * d.ny, d.b_bottom, d.b_top);
        bcv_ = DevBuf(ctx_, bcv.size() * sizeof(double2));
        bch_ = DevBuf(ctx_, bcv.size() * sizeof(double2));
        TG_HIP(hipMemcpyAsync(bcv_.ptr, bcv.data(), bcv.size() * sizeof(double2), hipMemcpyHostToDevice, s));
    }
    ctx_->twiddle(mx_, (DType)d.dtype);
    ctx_->twiddle(my_, (DType)d.dtype);
    TG_HIP(hipStreamSynchronize(s));
    factor(implicit_c(first_step()));
    autotune();
}

void Channel3Solver::set_tuning(const Chan3Tuning& t) {
    TG_REQUIRE(t.solve == 0 || t.solve == 1, kErrInvalid, "3-D channel solver: solve variant is 0 or 1");
    TG_REQUIRE(t.zbwd == 0 || (t.zbwd == 1 && d_.dtype == kF32), kErrInvalid,
               "3-D channel solver: z-backward variant is 0, or 1 with an FP32 state");
    tune_ = t;
    invalidate_graph();
}

// Times the variants of k3_tau_solve and k3_zbwd on this solver's own buffers (HIP events,
// medians of 7 launches alternating with the default's) at creation.  A variant replaces the
// default only when it is at least 3 % faster, so timing noise does not flip the choice.  The
// choices are cached per (nx, ny, nz, dtype, solve form, |k_h|^2 keys) for the life of the process;
// TARANG_AUTOTUNE=0 keeps the defaults.
void Channel3Solver::autotune() {
    const char* env = std::getenv("TARANG_AUTOTUNE");
    if (env && std::string(env) == "0") return;
    const std::array<int, 7> key{d_.nx, d_.ny, d_.nz, d_.dtype, d_.refine_sweeps, d_.split_inverse, nkeys_};
    static std::mutex mu;
    static std::map<std::array<int, 7>, Chan3Tuning> cache;
    {
        std::lock_guard<std::mutex> lk(mu);
        auto it = cache.find(key);
        if (it != cache.end()) {
            tune_ = it->second;
            return;
        }
    }
    ctx_->activate();
    hipStream_t s = ctx_->stream;
    hipEvent_t a, b;
    TG_HIP(hipEventCreate(&a));
    TG_HIP(hipEventCreate(&b));
    // the two variants' launches alternate (a warm-up pair, then 7 timed pairs), so that
    // clock and temperature drift during the measurement falls on both; medians compared
    auto pick = [&](int& field, auto&& launch) {
        std::vector<float> v[2];
        for (int r = 0; r < 8; ++r)
            for (int var = 0; var < 2; ++var) {
                field = var;
                TG_HIP(hipEventRecord(a, s));
                launch();
                TG_HIP(hipEventRecord(b, s));
                TG_HIP(hipEventSynchronize(b));
                float ms = 0;
                TG_HIP(hipEventElapsedTime(&ms, a, b));
                if (r > 0) v[var].push_back(ms);
            }
        for (auto& x : v) std::sort(x.begin(), x.end());
        return v[1][v[1].size() / 2] < 0.97f * v[0][v[0].size() / 2] ? 1 : 0;
    };
    Chan3Tuning chosen;
    auto go = [&](auto tag) {
        using T = decltype(tag);
        chosen.solve = pick(tune_.solve, [&] { solve_t<T>(); });
        if (sizeof(T) == 4)
            chosen.zbwd = pick(tune_.zbwd, [&] { rhs_t<T>(F_[0].ptr, F_[1].ptr, F_[2].ptr, F_[3].ptr); });
    };
    if (d_.dtype == kF32) go(float{});
    else go(double{});
    (void)hipEventDestroy(a);
    (void)hipEventDestroy(b);
    tune_ = chosen;
    // the timed launches wrote the state and the products: back to the zero state of a new solver
    for (DevBuf* x : {&P_, &B_, &UX_, &UY_, &UZ_, &TAU_, &F_[0], &F_[1], &F_[2], &F_[3]})
        TG_HIP(hipMemsetAsync(x->ptr, 0, x->bytes, s));
    TG_HIP(hipStreamSynchronize(s));
    std::lock_guard<std::mutex> lk(mu);
    cache[key] = tune_;
}

Channel3Solver::~Channel3Solver() {
    if (graph_) (void)hipGraphExecDestroy(graph_);
}

void* Channel3Solver::field_ptr(int var) const {
    switch (var) {
        case kC3P: return P_.ptr;
        case kC3B: return B_.ptr;
        case kC3UX: return UX_.ptr;
        case kC3UY: return UY_.ptr;
        case kC3UZ: return UZ_.ptr;
        default: break;
    }
    TG_REQUIRE(false, kErrInvalid, "3-D channel solver: variable must be 0 (p), 1 (b), 2 (ux), 3 (uy) or 4 (uz)");
    return nullptr;
}

template <typename T>
void Channel3Solver::transpose_t(const void* in, void* out, int rows, int cols) {
    dim3 grid((unsigned)((cols + 31) / 32), (unsigned)((rows + 31) / 32));
    hipLaunchKernelGGL((k_ch_transpose<T>), grid, dim3(32, 8), 0, ctx_->stream, static_cast<const cplx<T>*>(in),
                       static_cast<cplx<T>*>(out), rows, cols);
    TG_HIP(hipGetLastError());
}

// reference layout (mode fastest, nz rows of nmodes) <-> mode-major (nmodes rows of nz)
void Channel3Solver::set_field(int var, const void* dev, bool restart) {
    ctx_->activate();
    void* dst = field_ptr(var);
    if (d_.dtype == kF32) transpose_t<float>(dev, dst, d_.nz, nmodes_);
    else transpose_t<double>(dev, dst, d_.nz, nmodes_);
    if (restart) {  // a new initial condition restarts the clock and the multistep history
        t_ = 0;
        iter_ = 0;
    }
}

void Channel3Solver::set_bc(const void* b_bottom, const void* b_top) {
    TG_REQUIRE(b_bottom && b_top, kErrInvalid, "channel solver: set_bc needs both wall arrays");
    ctx_->activate();
    const int nx = d_.nx, ny = d_.ny, nmodes = nxh_ * ny;
    const unsigned nb = (unsigned)((2 * nmodes + 255) / 256);
    const double2* twx = static_cast<const double2*>(ctx_->twiddle(nx, kF64));
    const double2* twy = static_cast<const double2*>(ctx_->twiddle(ny, kF64));
    if (d_.dtype == kF32)
        hipLaunchKernelGGL((k_wall_dft_x<float>), dim3(nb), dim3(256), 0, ctx_->stream,
                           static_cast<const float*>(b_bottom), static_cast<const float*>(b_top), nx, ny, nxh_, twx,
                           bch_.as<double2>());
    else
        hipLaunchKernelGGL((k_wall_dft_x<double>), dim3(nb), dim3(256), 0, ctx_->stream,
                           static_cast<const double*>(b_bottom), static_cast<const double*>(b_top), nx, ny, nxh_, twx,
                           bch_.as<double2>());
    hipLaunchKernelGGL(k_wall_dft_y, dim3(nb), dim3(256), 0, ctx_->stream, bch_.as<const double2>(), ny, nxh_, twy,
                       bcv_.as<double2>());
    TG_HIP(hipGetLastError());
}

void Channel3Solver::get_field(int var, void* dev) {
    ctx_->activate();
    const void* src = field_ptr(var);
    if (d_.dtype == kF32) transpose_t<float>(src, dev, nmodes_, d_.nz);
    else transpose_t<double>(src, dev, nmodes_, d_.nz);
}

void Channel3Solver::get_tau(int t, void* dev) {
    TG_REQUIRE(t >= 0 && t < kCh3TauStride, kErrInvalid, "3-D channel solver: tau index must be 0..8");
    ctx_->activate();
    const size_t vb = 2 * dtype_size((DType)d_.dtype);
    TG_HIP(hipMemcpy2DAsync(dev, vb, static_cast<const char*>(TAU_.ptr) + t * vb, kCh3TauStride * vb, vb, nmodes_,
                            hipMemcpyDeviceToDevice, ctx_->stream));
}

void Channel3Solver::set_dt(double dt) {
    TG_REQUIRE(dt > 0, kErrInvalid, "3-D channel solver: dt must be positive");
    d_.dt = dt;
}

double Channel3Solver::implicit_c(bool first) const {
    if (!multistep()) return d_.dt * tab_.AI[1][1];
    if (first) return d_.dt;
    const double w = d_.dt / dt_prev_;
    return (1.0 + w) * d_.dt / (1.0 + 2.0 * w);
}

TauSys Channel3Solver::tau_sys(double c) const {
    const bool fp64 = d_.dtype == kF64;
    const double sz = 2.0 / d_.Lz;
    return TauSys{d_.nz, tau_shape(d_.nz, true, any_sign()), nkeys_, c, sz, d_.kappa, d_.nu, kh_.as<const double>(), 0.0,
                  tab_tau_.as<double>(), tau_psi_bound(d_.nz, fp64), tau_low_kh(d_.nz, sz, fp64), info_.as<int>()};
}

bool Channel3Solver::any_sign() const { return tau_any_sign(d_.kappa, d_.nu); }

void Channel3Solver::factor(double c) {
    if (c == factored_c_) return;
    const TauSys t = tau_sys(c);
    std::string bad;
    const std::string par = ", parity " + std::to_string(d_.nz & 1) + ")";  // the parity of N - 2
    for (int k = 0; k < nkeys_ && bad.size() < 200; ++k) {
        const std::string key = "(|k_h| key " + std::to_string(k) + par;
        if (tau_no_diffusion(c, t.s, d_.kappa)) bad += " b-system" + key;
        if (tau_no_diffusion(c, t.s, d_.nu)) bad += " perp-system" + key + " u-p-system" + key;
    }
    TG_REQUIRE(bad.empty(), kErrSingular, "3-D channel solver: singular per-mode system:" + bad);
    invalidate_graph();
    factored_c_ = -1;  // until the set-up is in the stream: a failed launch is not taken for done by the next step
    const size_t lds = tau_setup_lds(d_.nz, any_sign());
    if (any_sign()) {
        hipLaunchKernelGGL((k_tau_setup<true>), dim3(nkeys_), dim3(64), lds, ctx_->stream, t);
        TG_HIP(hipGetLastError());
        std::vector<int> info(nkeys_);
        TG_HIP(hipMemcpyAsync(info.data(), info_.ptr, info.size() * sizeof(int), hipMemcpyDeviceToHost, ctx_->stream));
        TG_HIP(hipStreamSynchronize(ctx_->stream));
        for (int k = 0; k < nkeys_ && bad.size() < 200; ++k) {
            const std::string key = "(|k_h| key " + std::to_string(k) + ")";
            if (info[k] & 1) bad += " b-system" + key;
            if (info[k] & 2) bad += " perp-system" + key;
            if (info[k] & 6) bad += " u-p-system" + key;
        }
        TG_REQUIRE(bad.empty(), kErrSingular, "3-D channel solver: singular per-mode system:" + bad);
    } else {
        hipLaunchKernelGGL((k_tau_setup<false>), dim3(nkeys_), dim3(64), lds, ctx_->stream, t);
        TG_HIP(hipGetLastError());
    }
    factored_c_ = c;
}

template <typename T>
void Channel3Solver::rhs_t(void* F0, void* F1, void* F2, void* F3) {
    using V = cplx<T>;
    const int N = d_.nz;
    hipStream_t s = ctx_->stream;
    const DType dt = std::is_same<T, float>::value ? kF32 : kF64;
    Ch3Geom geo{d_.nx, d_.ny, nxh_, N, nmodes_, 2.0 * M_PI / d_.Lx, 2.0 * M_PI / d_.Ly};
    V* G = G_.as<V>();
    V* Q = Q_.as<V>();
    V* H = H_.as<V>();
    {
        constexpr int NTZ = ZbwdTile<T>::NT;
        auto zb = [&](auto QTC) {
            constexpr int QT = decltype(QTC)::value;
            const size_t blds = (size_t)((N + 15) & ~15) * zbwd_lds_stride(QT) * sizeof(T);
            timed(0, [&] {
                hipLaunchKernelGGL((k3_zbwd<T, NTZ, QT>), dim3((unsigned)((nmodes_ + QT - 1) / QT), 4), dim3(NTZ),
                                   blds, s, B_.as<const V>(), UX_.as<const V>(), UY_.as<const V>(), UZ_.as<const V>(),
                                   geo, BT_.as<const T>(), BDT_.as<const T>(), G);
            });
        };
        if (sizeof(T) == 4 && tune_.zbwd == 1) zb(std::integral_constant<int, 16>{});
        else zb(std::integral_constant<int, ZbwdTile<T>::QT>{});
    }
    TG_HIP(hipGetLastError());
    dispatch_size(d_.ny, [&](auto NC) {
        constexpr int NY = decltype(NC)::value;
        constexpr int MY = padded_len(NY);
        constexpr int TK = tile_cols<T, MY>();
        const V* tw = static_cast<const V*>(ctx_->twiddle(MY, dt));
        timed(1, [&] {
            hipLaunchKernelGGL((k3_ybwd<T, NY, MY, TK, 256>), dim3((nxh_ + TK - 1) / TK, N, kCh3Planes), dim3(256), 0,
                               s, G, geo, Q, tw);
        });
    }, Sizes2D{});
    TG_HIP(hipGetLastError());
    const T scale = T(1.0 / ((double)d_.nx * d_.ny * (double)mx_ * my_));
    dispatch_size(d_.nx, [&](auto NC) {
        constexpr int NX = decltype(NC)::value;
        constexpr int MX = padded_len(NX);
        if constexpr ((size_t)8 * line_stride(MX) * sizeof(V) <= 128 * 1024) {
            const V* tw = static_cast<const V*>(ctx_->twiddle(MX, dt));
            constexpr int NT = NX >= 512 ? 512 : 256;
            timed(2, [&] {
                hipLaunchKernelGGL((k3_xpass<T, NX, MX, NT>), dim3(my_, N), dim3(NT), 0, s, Q, N, my_, geo.k0x, scale,
                                   H, tw);
            });
        } else {
            TG_REQUIRE(false, kErrInvalid, "3-D channel solver: x size too large for this dtype");
        }
    }, Sizes2D{});
    TG_HIP(hipGetLastError());
    V* Fz = G;  // the operand planes are consumed: the four product planes reuse them
    dispatch_size(d_.ny, [&](auto NC) {
        constexpr int NY = decltype(NC)::value;
        constexpr int MY = padded_len(NY);
        constexpr int TK = tile_cols<T, MY>();
        const V* tw = static_cast<const V*>(ctx_->twiddle(MY, dt));
        timed(3, [&] {
            hipLaunchKernelGGL((k3_yfwd<T, NY, MY, TK, 256>), dim3((nxh_ + TK - 1) / TK, N, 4), dim3(256), 0, s, H,
                               geo, Fz, tw);
        });
    }, Sizes2D{});
    TG_HIP(hipGetLastError());
    {
        constexpr int QT = std::is_same<T, float>::value ? 32 : 16;  // 64 or 32 columns
        const size_t flds = ch_zfwd_lds_elems(N, QT) * sizeof(T);
        timed(4, [&] {
            hipLaunchKernelGGL((k_ch_zfwd<T, QT, ZfwdTile<T>::NT>), dim3((unsigned)((nmodes_ + QT - 1) / QT), 4),
                               dim3(ZfwdTile<T>::NT), flds, s,
                               Fz, nmodes_, 1, N, FT_.as<const T>(), static_cast<V*>(F0), static_cast<V*>(F1),
                               static_cast<V*>(F2), static_cast<V*>(F3));
        });
    }
    TG_HIP(hipGetLastError());
}

template <typename T>
void Channel3Solver::sbdf_t(bool first) {
    using V = cplx<T>;
    Ch3SbdfArgs<T> a;
    const double dt = d_.dt;
    double a0, a1, a2, c1, c2;
    if (first) {
        a0 = 1.0 / dt; a1 = -1.0 / dt; a2 = 0.0; c1 = 1.0; c2 = 0.0;
    } else {
        const double w = dt / dt_prev_;
        a0 = (1.0 + 2.0 * w) / ((1.0 + w) * dt);
        a1 = -(1.0 + w) / dt;
        a2 = w * w / ((1.0 + w) * dt);
        c1 = 1.0 + w;
        c2 = -w;
    }
    const DevBuf* X[4] = {&B_, &UX_, &UY_, &UZ_};
    for (int r = 0; r < 4; ++r) {
        a.X[r] = X[r]->as<const V>();
        a.F[r] = F_[r].as<const V>();
        a.Fm1[r] = Fm1_[r].as<V>();
        a.MXm1[r] = MXm1_[r].as<V>();
    }
    for (int r = 0; r < 4; ++r) a.R[r] = R_[r + 1].as<V>();
    a.c1 = T(c1); a.c2 = T(c2); a.a1 = T(a1); a.a2 = T(a2); a.inv_a0 = T(1.0 / a0);
    a.geo = Ch3Geom{d_.nx, d_.ny, nxh_, d_.nz, nmodes_, 2.0 * M_PI / d_.Lx, 2.0 * M_PI / d_.Ly};
    const size_t n = field_elems();
    const unsigned nblk = (unsigned)std::min<size_t>((n + 255) / 256, 8192);
    timed(5, [&] { hipLaunchKernelGGL((k3_sbdf<T>), dim3(nblk), dim3(256), 0, ctx_->stream, a, n); });
    TG_HIP(hipGetLastError());
}

template <typename T>
void Channel3Solver::solve_t() {
    using V = cplx<T>;
    TauArgs<T> a{};
    a.t = tau_sys(factored_c_);
    a.nmodes = nmodes_;
    a.bcv = bcv_.as<const double2>();
    a.modes = modes_.as<const int2>();
    a.rot = rot_.as<const double>();
    a.form = tau_form(a.t, kh_max_);
    a.R1 = multistep() ? nullptr : R_[0].as<const V>();  // the multistep E1 rows are zero
    a.R2 = R_[1].as<const V>();
    a.R3x = R_[2].as<const V>();
    a.R3y = R_[3].as<const V>();
    a.R3z = R_[4].as<const V>();
    a.P = P_.as<V>();
    a.B = B_.as<V>();
    a.UX = UX_.as<V>();
    a.UY = UY_.as<V>();
    a.UZ = UZ_.as<V>();
    a.taus = TAU_.as<V>();
    const TauShape h = a.t.shape;
    auto launch = [&](auto GC, auto EC) {
        constexpr int G = decltype(GC)::value, E = decltype(EC)::value;
        const unsigned np = tune_.solve == 1 ? 2 : 1, per = np * 64 / G;  // pairs of waves per workgroup
        const dim3 grid((nmodes_ + per - 1) / per), block(128 * np);
        auto go = [&](auto form, auto hasd) {
            constexpr int F = decltype(form)::value;
            const size_t lds = np * tau_lds_bytes<G, E, true, F>();
            hipLaunchKernelGGL((k3_tau_solve<T, G, E, F, decltype(hasd)::value>), grid, block, lds, ctx_->stream, a);
        };
        tau_flags(a.form, a.R1 != nullptr, go);
    };
    timed(6, [&] {
        if (a.form == kTauAny) {  // one mode per workgroup
            constexpr size_t lds = tau_lds_bytes<64, 2, true, kTauAny>();
            if (a.R1)
                hipLaunchKernelGGL((k3_tau_solve<T, 64, 2, kTauAny, true>), dim3(nmodes_), dim3(128), lds, ctx_->stream, a);
            else
                hipLaunchKernelGGL((k3_tau_solve<T, 64, 2, kTauAny, false>), dim3(nmodes_), dim3(128), lds, ctx_->stream, a);
        } else if (h.G == 32) launch(std::integral_constant<int, 32>{}, std::integral_constant<int, 4>{});
        else if (h.E == 4) launch(std::integral_constant<int, 16>{}, std::integral_constant<int, 4>{});
        else if (h.E == 2) launch(std::integral_constant<int, 16>{}, std::integral_constant<int, 2>{});
        else launch(std::integral_constant<int, 16>{}, std::integral_constant<int, 1>{});
    });
    TG_HIP(hipGetLastError());
}

template <typename T>
void Channel3Solver::lx_t(int st) {
    using V = cplx<T>;
    const int N = d_.nz;
    constexpr int NT = 256;
    Ch3Geom geo{d_.nx, d_.ny, nxh_, N, nmodes_, 2.0 * M_PI / d_.Lx, 2.0 * M_PI / d_.Ly};
    timed(7, [&] {
        hipLaunchKernelGGL((k3_lx<T, NT>), dim3(nmodes_), dim3(NT), (size_t)14 * N * sizeof(double2), ctx_->stream,
                           P_.as<const V>(), B_.as<const V>(), UX_.as<const V>(), UY_.as<const V>(), UZ_.as<const V>(),
                           TAU_.as<const V>(), geo, 2.0 / d_.Lz, d_.kappa, d_.nu, LX_[st][0].as<V>(),
                           LX_[st][1].as<V>(), LX_[st][2].as<V>(), LX_[st][3].as<V>(), LX_[st][4].as<V>());
    });
    TG_HIP(hipGetLastError());
}

template <typename T>
void Channel3Solver::stage_t(int st, bool final_update) {
    using V = cplx<T>;
    Ch3StageArgs<T> a;
    std::memset(&a, 0, sizeof(a));
    for (int r = 0; r < 4; ++r) a.X0[r] = X0_[r].as<const V>();
    const int nterms = final_update ? tab_.stages : st;
    for (int j = 0; j < nterms; ++j) {
        for (int r = 0; r < 4; ++r) a.F[j][r] = Frk_[j][r].as<const V>();
        const double ai = final_update ? tab_.bI[j] : tab_.AI[st][j];
        for (int r = 0; r < 5; ++r) a.LX[j][r] = ai != 0.0 ? LX_[j][r].as<const V>() : nullptr;
        a.ae[j] = T(final_update ? tab_.bE[j] : tab_.AE[st][j]);
        a.ai[j] = T(ai);
    }
    a.nterms = nterms;
    a.dt = T(d_.dt);
    a.final_update = final_update ? 1 : 0;
    if (final_update) {
        a.out[0] = B_.as<V>();
        a.out[1] = UX_.as<V>();
        a.out[2] = UY_.as<V>();
        a.out[3] = UZ_.as<V>();
    } else {
        for (int r = 0; r < 5; ++r) a.out[r] = R_[r].as<V>();
    }
    const size_t n = field_elems();
    const unsigned nblk = (unsigned)std::min<size_t>((n + 255) / 256, 8192);
    timed(5, [&] { hipLaunchKernelGGL((k3_stage<T>), dim3(nblk), dim3(256), 0, ctx_->stream, a, n); });
    TG_HIP(hipGetLastError());
}

template <typename T>
void Channel3Solver::zero_t(void* p, size_t n) {
    const unsigned nblk = (unsigned)std::min<size_t>((n + 255) / 256, 8192);
    timed(5, [&] {
        hipLaunchKernelGGL((k_ch_zero<T>), dim3(nblk), dim3(256), 0, ctx_->stream, static_cast<cplx<T>*>(p), n);
    });
    TG_HIP(hipGetLastError());
}

void Channel3Solver::launch_step_body() {
    if (!multistep()) {  // IMEX RK stage loop, as in the 2-D solver
        auto run = [&](auto tag) {
            using T = decltype(tag);
            using V = cplx<T>;
            const size_t n = field_elems();
            const unsigned nblk = (unsigned)std::min<size_t>((n + 255) / 256, 8192);
            const DevBuf* X[4] = {&B_, &UX_, &UY_, &UZ_};
            for (int r = 0; r < 4; r += 2)  // the second pass also clears p and the taus
                timed(5, [&] {
                    hipLaunchKernelGGL((k_ch_copy<T>), dim3(nblk), dim3(256), 0, ctx_->stream, X[r]->as<const V>(),
                                       X[r + 1]->as<const V>(), X[r + 1]->as<const V>(), X0_[r].as<V>(),
                                       X0_[r + 1].as<V>(), X0_[r + 1].as<V>(), n, r == 2 ? P_.as<V>() : nullptr,
                                       r == 2 ? TAU_.as<V>() : nullptr, r == 2 ? (size_t)nmodes_ * kCh3TauStride : 0);
                });
            rhs_t<T>(Frk_[0][0].ptr, Frk_[0][1].ptr, Frk_[0][2].ptr, Frk_[0][3].ptr);
            if (uses_lx(tab_, 0)) lx_t<T>(0);
            for (int st = 1; st < tab_.stages; ++st) {
                stage_t<T>(st, false);
                solve_t<T>();
                rhs_t<T>(Frk_[st][0].ptr, Frk_[st][1].ptr, Frk_[st][2].ptr, Frk_[st][3].ptr);
                if (uses_lx(tab_, st)) lx_t<T>(st);
            }
            stage_t<T>(0, true);
            zero_t<T>(P_.ptr, n);
            zero_t<T>(TAU_.ptr, (size_t)nmodes_ * kCh3TauStride);
        };
        if (d_.dtype == kF32) run(float{}); else run(double{});
        return;
    }
    const bool first = first_step();
    if (d_.dtype == kF32) {
        rhs_t<float>(F_[0].ptr, F_[1].ptr, F_[2].ptr, F_[3].ptr);
        sbdf_t<float>(first);
        solve_t<float>();
    } else {
        rhs_t<double>(F_[0].ptr, F_[1].ptr, F_[2].ptr, F_[3].ptr);
        sbdf_t<double>(first);
        solve_t<double>();
    }
}

void Channel3Solver::step_once(bool allow_graph) {
    const bool first = first_step();
    factor(implicit_c(first));
    if (!(allow_graph && graph_on_)) {
        launch_step_body();
    } else {
        if (graph_ && (graph_dt_ != d_.dt || graph_first_ != first || (multistep() && graph_dtp_ != dt_prev_)))
            invalidate_graph();
        if (!graph_) {
            hipGraph_t g = nullptr;
            TG_HIP(hipStreamBeginCapture(ctx_->stream, hipStreamCaptureModeThreadLocal));
            try {
                launch_step_body();
            } catch (...) {
                (void)hipStreamEndCapture(ctx_->stream, &g);
                if (g) (void)hipGraphDestroy(g);
                throw;
            }
            TG_HIP(hipStreamEndCapture(ctx_->stream, &g));
            TG_HIP(hipGraphInstantiate(&graph_, g, nullptr, nullptr, 0));
            TG_HIP(hipGraphDestroy(g));
            graph_dt_ = d_.dt;
            graph_dtp_ = dt_prev_;
            graph_first_ = first;
        }
        TG_HIP(hipGraphLaunch(graph_, ctx_->stream));
    }
    dt_prev_ = d_.dt;
    t_ += d_.dt;
    ++iter_;
}

void Channel3Solver::step(int nsteps) {
    TG_REQUIRE(nsteps >= 0, kErrInvalid, "3-D channel solver: nsteps must be >= 0");
    ctx_->activate();
    for (int i = 0; i < nsteps; ++i) step_once(true);
}

void Channel3Solver::rhs(void* Fb, void* Fux, void* Fuy, void* Fuz) {
    ctx_->activate();
    void* outs[4] = {Fb, Fux, Fuy, Fuz};
    if (d_.dtype == kF32) rhs_t<float>(F_[0].ptr, F_[1].ptr, F_[2].ptr, F_[3].ptr);
    else rhs_t<double>(F_[0].ptr, F_[1].ptr, F_[2].ptr, F_[3].ptr);
    for (int r = 0; r < 4; ++r) {
        if (!outs[r]) continue;
        if (d_.dtype == kF32) transpose_t<float>(F_[r].ptr, outs[r], nmodes_, d_.nz);
        else transpose_t<double>(F_[r].ptr, outs[r], nmodes_, d_.nz);
    }
}

template <typename F>
void Channel3Solver::timed(int kind, F&& launch) {
    if (!profiling_) {
        launch();
        return;
    }
    Mark m{kind, nullptr, nullptr};
    TG_HIP(hipEventCreate(&m.a));
    TG_HIP(hipEventCreate(&m.b));
    TG_HIP(hipEventRecord(m.a, ctx_->stream));
    launch();
    TG_HIP(hipEventRecord(m.b, ctx_->stream));
    marks_.push_back(m);
}

void Channel3Solver::profile(int nsteps, double* avg_ms, long* counts) {
    ctx_->activate();
    marks_.clear();
    profiling_ = true;
    try {
        for (int i = 0; i < nsteps; ++i) step_once(false);
    } catch (...) {
        profiling_ = false;
        throw;
    }
    profiling_ = false;
    TG_HIP(hipStreamSynchronize(ctx_->stream));
    double sum[kKinds] = {};
    long cnt[kKinds] = {};
    for (auto& m : marks_) {
        float ms = 0.f;
        TG_HIP(hipEventElapsedTime(&ms, m.a, m.b));
        sum[m.kind] += ms;
        cnt[m.kind] += 1;
        (void)hipEventDestroy(m.a);
        (void)hipEventDestroy(m.b);
    }
    marks_.clear();
    for (int k = 0; k < kKinds; ++k) {
        if (avg_ms) avg_ms[k] = cnt[k] ? sum[k] / cnt[k] : 0.0;
        if (counts) counts[k] = cnt[k];
    }
}

void Channel3Solver::kernel_bytes(double* out) const {
    const double vb = 2.0 * dtype_size((DType)d_.dtype), rb = dtype_size((DType)d_.dtype);
    const double nc = (double)nmodes_ * d_.nz, N = d_.nz;
    const double pad = (double)d_.nz * my_ * nxh_;
    out[0] = (4 * nc + kCh3ZPlanes * nc) * vb + 2 * N * N * rb;  // read 4 fields, write 8 planes
    out[1] = (kCh3ZPlanes * nc + kCh3Planes * pad) * vb;        // read 8 planes, write 12 y-padded planes
    out[2] = (kCh3Planes * pad + 4 * pad) * vb;                 // read 12 padded planes, write 4
    out[3] = (4 * pad + 4 * nc) * vb;                           // read 4 padded planes, write 4
    out[4] = (8 * nc) * vb + N * N * rb;                        // read 4 planes, write 4 rows
    out[5] = (4 * 4 + 3 * 4) * nc * vb;                         // read state, F, histories; write histories, rhs
    // solve: rhs rows and the per-key tables in, five fields out
    out[6] = (multistep() ? 9 : 10) * nc * vb +
             (double)nkeys_ * tau_table_stride(tau_shape(d_.nz, true, any_sign())) * sizeof(double);
    out[7] = 10 * nc * vb;  // L x: read p, b, u (and partners on two lines), write five rows
}

double Channel3Solver::nusselt() {
    ctx_->activate();
    return channel_nusselt(ctx_, B_.ptr, UZ_.ptr, (DType)d_.dtype, d_.nx, d_.ny, d_.nz, d_.Lz, d_.kappa,
                           d_.b_bottom - d_.b_top);
}

size_t footprint(const Channel3Desc& d) {
    // every buffer the constructor allocates, in 2 MiB pages
    const size_t nxh = d.nx / 2 + 1, nmodes = nxh * d.ny, N = d.nz, vb = 2 * dtype_size((DType)d.dtype);
    const size_t fb = nmodes * N * vb, prow = N * (size_t)padded_len(d.ny) * nxh * vb, ib = dtype_size((DType)d.dtype);
    const bool ms = d.stepper == kSBDF2 || d.stepper == kSBDF1;
    size_t nfields = 5 + 12 + (ms ? 4 : 5 + 4);  // state, history, rhs rows, RK initial state
    if (!ms) {
        const Tableau tab = make_tableau(d.stepper);
        for (int st = 0; st < tab.stages; ++st) nfields += 4 + (uses_lx(tab, st) ? 5 : 0);  // RK stage rows
    }
    // distinct |k_h|^2 keys: at most one per mode (about nmodes / 5.6 at 256 x 256 when Lx == Ly)
    const size_t keys = d.Lx == d.Ly ? nmodes / 3 + 64 : nmodes;
    size_t b = nfields * alloc_granule(fb) + alloc_granule(kCh3ZPlanes * fb) + alloc_granule(kCh3Planes * prow) +
               alloc_granule(4 * prow);                                                           // G, Q, H
    b += alloc_granule(nmodes * kCh3TauStride * vb) + 3 * alloc_granule(N * N * ib);           // taus, tables
    const bool any = tau_any_sign(d.kappa, d.nu);
    b += alloc_granule(tau_table_doubles(tau_shape(d.nz, true, any), keys) * sizeof(double));  // tau-solve tables
    if (any) b += alloc_granule(keys * sizeof(int));
    b += 8 * alloc_granule(nmodes * 32);                                 // keys, rotations, modes, walls
    return b;
}

void Channel3Solver::flag_nonfinite(int* dflag) const {
    for (const DevBuf* b : {&P_, &B_, &UX_, &UY_, &UZ_})
        tarang::flag_nonfinite(ctx_, b->ptr, 2 * field_elems(), (DType)d_.dtype, dflag);
}

}  // namespace tarang
