// pic_ua.hip -- the uniformly accurate (UA) PIC step of src/ua_steps.jl on
// the device: preparation!, update_particles_e! (the tau-fold M6 gather of
// interpolation_m6.jl:3-123), compute_f!, both ua_step! forms,
// update_particles_x! (the reconstruction and M6 deposit of
// compute_rho_m6.jl:29-179) and compute_v!, and the loop of test/bupdate.jl.
//
// A particle is worked by ntau consecutive lanes of one wave, lane m holding
// the tau-sample m of its (ntau, 2) arrays; the reference's (ntau, 2, n)
// layout is then read and written coalesced.  The tau-FFTs are radix-2
// transforms across those lanes (FFTW's signs; the inverse scales by 1/ntau
// as Julia's ifft does): decimation in frequency forward, in time backward, so
// that a spectrum stays in the bit-reversed order it comes out in, lane m
// holding the frequency of bitrev(m), and no permutation is needed between the
// two.  What a transform would only undo or what is known in closed form is
// not transformed (see ua_prep and k_ua_predict).
//
// The kernels are bound by FP64 VALU issue: 16 samples of a particle at ntau
// 16 are 16 lanes, so every instruction counts per sample.  Transforms with
// general lane shuffles, selects and a bit-reversal each, 18 of them in the
// prediction and 20 in the correction, and twiddles, cosines and FP64
// divisions formed anew for every particle took 304 and 458 us (204,800
// particles, 128 x 64 cells, ntau 16, deposit not counted) against 190 and 215
// now: 1,213 and 1,705 VALU instructions per wave, 59 % and 73 % of the issue
// rate, the rest waiting for the gather's nodes.  Three waves per SIMD at every
// ntau: at four the correction spills.  Measured at two, three and four waves,
// 3,276,800 samples each, correction: ntau 2 359, 358 and 358 us, 8 205, 204 and
// 260, 16 183, 184 and 229, 64 200, 200 and 298; prediction at 16 145, 146 and 144.
//
// The fused loop keeps between the prediction and the correction only the
// positions at the step's start and the tau-spectra of fx, fy; everything else
// is recomputed from them.
#include <algorithm>
#include <cmath>
#include <vector>

#include "pic_fftlanes.h"
#include "pic_internal.h"

namespace pic {

namespace {

constexpr int UB = 256;  // threads per block
constexpr int UA_WAVES = 3;

struct cd {
    double re, im;
};
__device__ __forceinline__ cd mk(double r, double i = 0.0) { return {r, i}; }
__device__ __forceinline__ cd operator+(cd a, cd b) { return {a.re + b.re, a.im + b.im}; }
__device__ __forceinline__ cd operator-(cd a, cd b) { return {a.re - b.re, a.im - b.im}; }
__device__ __forceinline__ cd operator*(cd a, cd b) {
    return {a.re * b.re - a.im * b.im, a.re * b.im + a.im * b.re};
}
__device__ __forceinline__ cd operator*(double s, cd a) { return {s * a.re, s * a.im}; }
__device__ __forceinline__ cd operator/(cd a, double s) { return {a.re / s, a.im / s}; }
__device__ __forceinline__ cd operator+(double s, cd a) { return {s + a.re, a.im}; }

// Keeps the computation of x where it is written.
__device__ __forceinline__ void pin(double &x) { asm volatile("" : "+v"(x)); }
__device__ __forceinline__ cd shfl(cd z, int src) { return {__shfl(z.re, src), __shfl(z.im, src)}; }

template <int NT>
__device__ __forceinline__ int bitrev(int m) {
    int r = 0;
#pragma unroll
    for (int b = 1; b < NT; b <<= 1) r = (r << 1) | ((m & b) ? 1 : 0);
    return r;
}

constexpr int ilog2(int n) { return n <= 1 ? 0 : 1 + ilog2(n / 2); }

struct Div : picd::Div {
    using picd::Div::Div;
    using picd::Div::of;
    __device__ __forceinline__ cd of(cd a) const { return {of(a.re), of(a.im)}; }
};

// Tables of ntau entries, made once for an ntau (k_ua_tables): cos and sin of
// tau[k] = k dtau and 1/ltau[k], 1/ltau[k]^2 (ua_type.jl:18-24; 1 at k = 0),
// cos and sin of 2 pi k / ntau.
struct UaTable {
    double c, s, rl, rl2, wc, ws;
};
__global__ void k_ua_tables(int nt, UaTable *t) {
    const int k = threadIdx.x;
    if (k >= nt) return;
    const double l = k == 0 ? 1.0 : k < nt / 2 ? (double)k : (double)(k - nt);
    sincos((double)k * (2 * M_PI / nt), &t[k].s, &t[k].c);
    sincospi((double)(2 * k) / nt, &t[k].ws, &t[k].wc);
    t[k].rl = 1.0 / l;
    t[k].rl2 = 1.0 / (l * l);
}

// This lane's constants of UA(ntau, eps): cos(tau[m]), sin(tau[m]); ltau of
// the frequency bitrev(m) it holds of a spectrum, and its square, as divisors
// (1 at frequency 0); the lane that holds the opposite frequency; and of every
// transform stage h the sign of its own value, -1 in the upper half of a pair,
// and its twiddle exp(-pi i (m mod h) / h) there (1 in the lower half).
template <int NT>
struct UaLane {
    static constexpr int LOG = ilog2(NT);
    int m, base, mirror;
    double l, c, s;
    Div dl, dl2;
    double sg[LOG], wr[LOG], wi[LOG];
    __device__ UaLane(const UaTable *__restrict__ t, int m_, int base_) : m(m_), base(base_) {
        const int k = bitrev<NT>(m);
        l = k < NT / 2 ? (double)k : (double)(k - NT);
        mirror = base + bitrev<NT>((NT - k) & (NT - 1));
        c = t[m].c;
        s = t[m].s;
        dl = Div(k == 0 ? 1.0 : l, t[k].rl);
        dl2 = Div(k == 0 ? 1.0 : l * l, t[k].rl2);
#pragma unroll
        for (int q = 0; q < LOG; ++q) {
            const int h = 1 << q;
            const bool up = (m & h) != 0;
            const int j = up ? (m & (h - 1)) * (NT / (2 * h)) : 0;
            sg[q] = up ? -1.0 : 1.0;
            wr[q] = t[j].wc;
            wi[q] = -t[j].ws;
        }
    }
};

template <int H>
__device__ __forceinline__ cd xor_cd(cd z) {
    return {xor_lane<H>(z.re), xor_lane<H>(z.im)};
}

// One stage of distance H = 2^Q: the lower lane of a pair takes a + b, the
// upper (a - b) w forward, a + b w backward (conj w).
template <int NT, int Q, bool INV>
__device__ __forceinline__ cd fft_pair(cd z, const UaLane<NT> &L) {
    const double wi = INV ? -L.wi[Q] : L.wi[Q];
    if (INV && Q > 0)
        z = {__builtin_fma(z.re, L.wr[Q], -(z.im * wi)), __builtin_fma(z.re, wi, z.im * L.wr[Q])};
    const cd p = xor_cd<(1 << Q)>(z);
    z = {__builtin_fma(L.sg[Q], z.re, p.re), __builtin_fma(L.sg[Q], z.im, p.im)};
    if (!INV && Q > 0)
        z = {__builtin_fma(z.re, L.wr[Q], -(z.im * wi)), __builtin_fma(z.re, wi, z.im * L.wr[Q])};
    return z;
}

// Forward: lane m's sample in, frequency bitrev(m) out.
template <int NT>
__device__ __forceinline__ cd fft_fwd(cd z, const UaLane<NT> &L) {
    if constexpr (NT >= 64) z = fft_pair<NT, 5, false>(z, L);
    if constexpr (NT >= 32) z = fft_pair<NT, 4, false>(z, L);
    if constexpr (NT >= 16) z = fft_pair<NT, 3, false>(z, L);
    if constexpr (NT >= 8) z = fft_pair<NT, 2, false>(z, L);
    if constexpr (NT >= 4) z = fft_pair<NT, 1, false>(z, L);
    return fft_pair<NT, 0, false>(z, L);
}

// Backward, scaled by 1/NT: frequency bitrev(m) in, sample m out.
template <int NT>
__device__ __forceinline__ cd fft_inv(cd z, const UaLane<NT> &L) {
    z = fft_pair<NT, 0, true>(z, L);
    if constexpr (NT >= 4) z = fft_pair<NT, 1, true>(z, L);
    if constexpr (NT >= 8) z = fft_pair<NT, 2, true>(z, L);
    if constexpr (NT >= 16) z = fft_pair<NT, 3, true>(z, L);
    if constexpr (NT >= 32) z = fft_pair<NT, 4, true>(z, L);
    if constexpr (NT >= 64) z = fft_pair<NT, 5, true>(z, L);
    return mk(z.re * (1.0 / NT), z.im * (1.0 / NT));
}

// Sum over the NT lanes of a group (every lane receives it).
template <int NT>
__device__ __forceinline__ double lane_sum(double z) {
    z += xor_lane<1>(z);
    if constexpr (NT >= 4) z += xor_lane<2>(z);
    if constexpr (NT >= 8) z += xor_lane<4>(z);
    if constexpr (NT >= 16) z += xor_lane<8>(z);
    if constexpr (NT >= 32) z += xor_lane<16>(z);
    if constexpr (NT >= 64) z += xor_lane<32>(z);
    return z;
}
template <int NT>
__device__ __forceinline__ cd lane_sum(cd z) {
    return {lane_sum<NT>(z.re), lane_sum<NT>(z.im)};
}

// exp(-1im l t / eps) as Julia evaluates it: cis(((-l) t) / eps).
__device__ __forceinline__ cd ua_cis(double l, double t, Div eps) {
    const double th = eps.of(-l * t);
    double s, c;
    sincos(th, &s, &c);
    return mk(c, s);
}

// pl, ql of preparation! (ua_steps.jl:26-33) at this lane's frequency; elt =
// exp(-1im l t / eps).
template <int NT>
__device__ __forceinline__ void ua_plql(const UaLane<NT> &L, double t, double eps, cd elt, cd &pl,
                                        cd &ql) {
    if (L.m == 0) {
        pl = mk(t);
        ql = mk(t * t / 2);
        return;
    }
    pl = L.dl.of(mk(0.0, eps) * (elt - mk(1.0)));                          // eps*1im*(elt-1)/l
    ql = L.dl2.of(eps * (eps * (mk(1.0) - elt) - mk(0.0 * t, L.l * t)));  // eps*(eps*(1-elt)-1im*l*t)/l^2
}

// preparation! for one particle (ua_steps.jl:3-83): b, t, xt (real) at this
// lane's tau, and the spectrum Z of r~ = r[0] + 1im r[1] (both real).
struct UaPrep {
    double b, t, interv, vxb, vyb, xt[2];
    Div db;
    cd Z;
};
template <int NT>
__device__ __forceinline__ void ua_prep(const UaLane<NT> &L, double x1, double x2, double vx,
                                        double vy, double ex, double ey, double dt, double eps,
                                        Div deps, UaPrep &p) {
    // sin(x1) on the even lanes, sin(x2) on the odd ones, exchanged
    const double sq = sin((L.m & 1) ? x2 : x1), so = xor_lane<1>(sq);
    p.b = 1 + 0.5 * ((L.m & 1) ? so : sq) * ((L.m & 1) ? sq : so);
    p.t = dt * p.b;
    p.db = Div(p.b);
    p.vxb = p.db.of(vx);
    p.vyb = p.db.of(vy);
    const double c = L.c, s = L.s;
    const double h1 = eps * (s * p.vxb - c * p.vyb);
    const double h2 = eps * (s * p.vyb + c * p.vxb);
    p.xt[0] = x1 + h1 + eps * p.vyb;
    p.xt[1] = x2 + h2 - eps * p.vxb;
    p.interv = deps.of(1 + 0.5 * sin(p.xt[0]) * sin(p.xt[1]) - p.b);
    const double exb = p.db.of((c * vy - s * vx) * p.interv + ex);
    const double eyb = p.db.of((-c * vx - s * vy) * p.interv + ey);
    p.Z = fft_fwd<NT>(mk(c * exb - s * eyb, s * exb + c * eyb), L);
}

// -1im R / l, the spectrum of the tau-antiderivative of preparation!
// (ua_steps.jl:60-74); frequency 0 stays.
template <int NT>
__device__ __forceinline__ cd ua_integrate(const UaLane<NT> &L, cd R) {
    if (L.m == 0) return R;
    return L.dl.of(mk(R.im, -R.re));
}

// yt of preparation! (ua_steps.jl:76-82) at this lane's tau.  The integral is
// linear, so both components go through one inverse transform as the real and
// imaginary part of r~'s; but for the middle frequency -NT/2, whose -1im/l
// makes the term of a real sequence imaginary: it is left out there and added
// to each component by itself.
template <int NT>
__device__ __forceinline__ void ua_yt(const UaLane<NT> &L, const UaPrep &p, double vx, double vy,
                                      double eps, cd yt[2]) {
    // lane 1 holds frequency -NT/2: Z there is R0 + 1im R1, both real
    const cd mid = shfl(p.Z, L.base + 1);
    const cd w = fft_inv<NT>(L.m == 1 ? mk(0.0) : ua_integrate<NT>(L, p.Z), L);
    const cd w0 = shfl(w, L.base);
    // -1im R / (-NT/2) (-1)^m / NT, less its value at m = 0
    const double n = (L.m & 1) ? -4.0 / ((double)NT * NT) : 0.0;
    yt[0] = mk(vx + eps * (w.re - w0.re), eps * (n * mid.re));
    yt[1] = mk(vy + eps * (w.im - w0.im), eps * (n * mid.im));
}

// The spectra of xt and yt at this lane's frequency, without transforms: xt is
// a constant and the first harmonic, and fft(r) is the spectrum r came from.
template <int NT>
__device__ __forceinline__ void ua_xs(const UaLane<NT> &L, const UaPrep &p, double x1, double x2,
                                      double eps, cd xs[2]) {
    xs[0] = xs[1] = mk(0.0);
    if (L.m == 0) {
        xs[0] = mk(NT * (x1 + eps * p.vyb));
        xs[1] = mk(NT * (x2 - eps * p.vxb));
    } else if (NT == 2) {  // tau = 0, pi: cos = 1, -1, sin = 0
        xs[0] = mk(-2.0 * (eps * p.vyb));
        xs[1] = mk(2.0 * (eps * p.vxb));
    } else if (L.l == 1.0 || L.l == -1.0) {
        const double q = -0.5 * NT * L.l;  // sin: -1im NT/2 at l = 1
        xs[0] = mk(-0.5 * NT * (eps * p.vyb), q * (eps * p.vxb));
        xs[1] = mk(0.5 * NT * (eps * p.vxb), q * (eps * p.vyb));
    }
}
template <int NT>
__device__ __forceinline__ void ua_ys(const UaLane<NT> &L, const UaPrep &p, double vx, double vy,
                                      double eps, cd ys[2]) {
    const cd zm = shfl(p.Z, L.mirror);
    const cd r[2] = {ua_integrate<NT>(L, mk(0.5 * (p.Z.re + zm.re), 0.5 * (p.Z.im - zm.im))),
                     ua_integrate<NT>(L, mk(0.5 * (p.Z.im + zm.im), -0.5 * (p.Z.re - zm.re)))};
    const double v[2] = {vx, vy};
#pragma unroll
    for (int q = 0; q < 2; ++q) {
        const cd r0 = lane_sum<NT>(r[q]);  // NT r at tau = 0
        ys[q] = eps * r[q];
        if (L.m == 0) ys[q] = ys[q] + mk(NT * v[q]) - eps * r0;
    }
}

// (1 + sin(x1) sin(x2)/2 - b)/eps at the lane's position (ua_steps.jl:55, :130).
__device__ __forceinline__ double ua_interv(const double xt[2], double b, Div deps) {
    return deps.of(1 + 0.5 * sin(xt[0]) * sin(xt[1]) - b);
}

// compute_f! at this lane's tau (ua_steps.jl:117-145), before its FFTs;
// interv from ua_interv at xt.
template <int NT>
__device__ __forceinline__ void ua_f(const UaLane<NT> &L, Div db, double interv, const cd yt[2],
                                     const double et[2], cd fx[2], cd fy[2]) {
    const double c = L.c, s = L.s;
    fx[0] = db.of(c * yt[0] + s * yt[1]);
    fx[1] = db.of(-s * yt[0] + c * yt[1]);
    const cd tmp1 = et[0] + interv * (c * yt[1] - s * yt[0]);
    const cd tmp2 = et[1] + interv * (-c * yt[0] - s * yt[1]);
    fy[0] = db.of(c * tmp1 - s * tmp2);
    fy[1] = db.of(s * tmp1 + c * tmp2);
}

struct UaGrid {
    int nx, ny;
    double xmin, ymin, dimx, dimy, dx, dy;
    Div ddx, ddy;
    const double2 *e;       // node fields (ex, ey), nx x ny
    double *rho_acc;        // raw charge, nx x ny, or null: no deposit here
    double w;               // particle weight
};

// The gather of update_particles_e! at real(xt) (interpolation_m6.jl:22-120):
// nodes i-2..i+3 and j-2..j+3, wrapped, (ex, ey) of a node in one 16-byte load
// at a 32-bit offset.  Sums with FMAs, y inner.
__device__ __forceinline__ void ua_gather(const double xt[2], const UaGrid &g, double et[2]) {
    const double px = g.ddx.of(picd::jl_mod_pos(xt[0] - g.xmin, g.dimx));
    const double py = g.ddy.of(picd::jl_mod_pos(xt[1] - g.ymin, g.dimy));
    // (clamped: NaN and what rounding leaves on the far edge stay in the mesh)
    const int i = min(max((int)px, 0), g.nx), j = min(max((int)py, 0), g.ny);
    double wx[6], wy[6];
    picd::m6_weights_d(px - (double)i, wx);
    picd::m6_weights_d(py - (double)j, wy);
    unsigned row[6];
#pragma unroll
    for (int b = 0; b < 6; ++b) {
        int q = j - 2 + b;
        q = q < 0 ? q + g.ny : q;
        q = q >= g.ny ? q - g.ny : q;
        row[b] = (unsigned)(q * g.nx);
    }
    et[0] = 0.0;
    et[1] = 0.0;
#pragma unroll
    for (int a = 0; a < 6; ++a) {
        int q = i - 2 + a;
        q = q < 0 ? q + g.nx : q;
        q = q >= g.nx ? q - g.nx : q;
        double t1 = 0.0, t2 = 0.0;
#pragma unroll
        for (int b = 0; b < 6; ++b) {
            const double2 e = g.e[row[b] + (unsigned)q];
            t1 = __builtin_fma(wy[b], e.x, t1);
            t2 = __builtin_fma(wy[b], e.y, t2);
        }
        et[0] = __builtin_fma(wx[a], t1, et[0]);
        et[1] = __builtin_fma(wx[a], t2, et[1]);
    }
    // the sums are taken here: left to itself the compiler moves them past the
    // branches of the cosines that follow and spills the 36 loaded nodes
    pin(et[0]);
    pin(et[1]);
}

// update_particles_x! for one particle (compute_rho_m6.jl:37-164): x(t) from
// the spectrum of its tau-samples, into the domain, stored (as x - xmin where
// pic_deposit.hip's deposit follows); else the M6 deposit (nodes i-2..i+3,
// wrapped, as in :70-81) spread over the group's lanes.  eplus = exp(+1im l t / eps), the
// conjugate of elt (cos is even and sin odd in the device library, and the two
// angles differ only in sign).
template <int NT>
__device__ __forceinline__ void ua_reconstruct_deposit(const UaLane<NT> &L, cd eplus,
                                                       const cd xs[2], const UaGrid &g, bool live,
                                                       double *xo, double *yo) {
    double pos[2];
#pragma unroll
    for (int q = 0; q < 2; ++q)
        pos[q] = lane_sum<NT>(__builtin_fma(xs[q].re, eplus.re, -(xs[q].im * eplus.im))) *
                 (1.0 / NT);
    const double xt1 = picd::jl_mod_pos(pos[0] - g.xmin, g.dimx);
    const double xt2 = picd::jl_mod_pos(pos[1] - g.ymin, g.dimy);
    if (!live) return;
    const bool follows = !g.rho_acc;  // the deposit, in launches of its own, from the residues
    if (L.m == 0) {
        *xo = follows ? xt1 : xt1 + g.xmin;
        *yo = follows ? xt2 : xt2 + g.ymin;
    }
    if (follows) return;
    const double px = xt1 / g.dx, py = xt2 / g.dy;
    const int i = min(max((int)px, 0), g.nx), j = min(max((int)py, 0), g.ny);
    double wx[6], wy[6];
    picd::m6_weights_d(px - (double)i, wx);
    picd::m6_weights_d(py - (double)j, wy);
    for (int q = L.m; q < 36; q += NT) {
        const int a = q / 6, bb = q % 6;
        const int ii = picd::wrap2(i - 2 + a, g.nx), jj = picd::wrap2(j - 2 + bb, g.ny);
        unsafeAtomicAdd(&g.rho_acc[ii + (size_t)g.nx * jj], wx[a] * wy[bb] * g.w);
    }
}

// compute_v! for one particle (ua_steps.jl:206-224) from the tau-spectrum yt;
// cos and sin of t/eps are elt's at l = 1.
template <int NT>
__device__ __forceinline__ void ua_v(const UaLane<NT> &L, double t, Div deps, cd eplus,
                                     const cd yt[2], double &v1, double &v2) {
    double p[2];
#pragma unroll
    for (int q = 0; q < 2; ++q)
        p[q] = lane_sum<NT>(__builtin_fma(yt[q].re, eplus.re, -(yt[q].im * eplus.im))) * (1.0 / NT);
    cd e1;
    if (NT == 2) {  // frequencies 0 and -1 only
        const double th = deps.of(t);
        sincos(th, &e1.im, &e1.re);
    } else {
        e1 = shfl(eplus, L.base + NT / 2);
    }
    v1 = e1.re * p[0] + e1.im * p[1];
    v2 = e1.re * p[1] - e1.im * p[0];
}

// Lane, group and particle of this thread.
template <int NT>
struct Slot {
    int m, base;
    int64_t k;
    bool live;
    __device__ Slot(int64_t n) {
        const int lane = threadIdx.x & 63;
        m = lane & (NT - 1);
        base = lane & ~(NT - 1);
        const int64_t k0 = (int64_t)blockIdx.x * (UB / NT) + threadIdx.x / NT;
        live = k0 < n;
        k = live ? k0 : n - 1;  // idle groups shadow the last particle
    }
};

// (m, c, k) of a (ntau, 2, n) array.
__device__ __forceinline__ size_t ux(int m, int c, int64_t k, int nt) {
    return (size_t)m + (size_t)nt * ((size_t)c + 2 * (size_t)k);
}

// (m, q, k) of the (ntau, 4, n) spectra of fx (q = 0, 1) and fy (q = 2, 3), in
// the lanes' bit-reversed order.
__device__ __forceinline__ size_t uf(int m, int q, int64_t k, int nt) {
    return (size_t)m + (size_t)nt * ((size_t)q + 4 * (size_t)k);
}

struct UaArgs {
    int64_t n;
    double eps, dt;
    Div deps;
    const UaTable *tab;
    double *x, *y, *vx, *vy;  // Particles.x, .v (SoA)
    const double *epx, *epy;  // Particles.e
    double *b, *t;            // Particles.b, .t
    double *x0, *y0;          // positions at the step's start
    cd *fhat;                 // tau-spectra of fx, fy: (ntau, 4, n)
    UaGrid g;
};

// ---------------------------------------------------------------- the loop

// Prediction of test/bupdate.jl:64-84: preparation!, update_particles_e!,
// compute_f!, x~t = fft(xt), ua_step!, then update_particles_x!, which takes the
// spectrum that the reference's ifft! and fft! would give back.  (The
// predicted yt is formed by the correction.)  Keeps x at the step's start and
// the spectra of fx, fy.
template <int NT>
__global__ __launch_bounds__(UB, UA_WAVES) void k_ua_predict(UaArgs a) {
    const Slot<NT> S(a.n);
    const UaLane<NT> L(a.tab, S.m, S.base);
    const bool live = S.live;
    const int64_t k = S.k;
    const double x1 = a.x[k], x2 = a.y[k], vx = a.vx[k], vy = a.vy[k];
    UaPrep p;
    ua_prep<NT>(L, x1, x2, vx, vy, a.epx[k], a.epy[k], a.dt, a.eps, a.deps, p);
    cd yt[2], fx[2], fy[2], xs[2];
    ua_yt<NT>(L, p, vx, vy, a.eps, yt);
    double et[2];
    ua_gather(p.xt, a.g, et);
    ua_f<NT>(L, p.db, p.interv, yt, et, fx, fy);
    const cd elt = ua_cis(L.l, p.t, a.deps);
    cd pl, ql;
    ua_plql<NT>(L, p.t, a.eps, elt, pl, ql);
    ua_xs<NT>(L, p, x1, x2, a.eps, xs);
#pragma unroll
    for (int q = 0; q < 2; ++q) {
        fx[q] = fft_fwd<NT>(fx[q], L);
        fy[q] = fft_fwd<NT>(fy[q], L);
        xs[q] = elt * xs[q] + pl * fx[q];
    }
    if (live) {
        if (S.m == 0) {
            a.x0[k] = x1;
            a.y0[k] = x2;
            a.b[k] = p.b;
            a.t[k] = p.t;
        }
#pragma unroll
        for (int q = 0; q < 2; ++q) {
            a.fhat[uf(S.m, q, k, NT)] = fx[q];
            a.fhat[uf(S.m, 2 + q, k, NT)] = fy[q];
        }
    }
    ua_reconstruct_deposit<NT>(L, mk(elt.re, -elt.im), xs, a.g, live, &a.x[k], &a.y[k]);
}

// Correction of test/bupdate.jl:90-114: the predicted xt, yt rebuilt from the
// step's start, update_particles_e! on the new field, compute_f!, the
// corrected ua_step!s, update_particles_x! and compute_v!.
template <int NT>
__global__ __launch_bounds__(UB, UA_WAVES) void k_ua_correct(UaArgs a) {
    const Slot<NT> S(a.n);
    const UaLane<NT> L(a.tab, S.m, S.base);
    const bool live = S.live;
    const int64_t k = S.k;
    const double x1 = a.x0[k], x2 = a.y0[k], vx = a.vx[k], vy = a.vy[k];
    cd fx[2], fy[2];
#pragma unroll
    for (int q = 0; q < 2; ++q) {
        fx[q] = a.fhat[uf(S.m, q, k, NT)];
        fy[q] = a.fhat[uf(S.m, 2 + q, k, NT)];
    }
    UaPrep p;
    ua_prep<NT>(L, x1, x2, vx, vy, a.epx[k], a.epy[k], a.dt, a.eps, a.deps, p);
    const cd elt = ua_cis(L.l, p.t, a.deps);
    cd pl, ql;
    ua_plql<NT>(L, p.t, a.eps, elt, pl, ql);
    cd xs[2], ys[2], yp[2];
    ua_xs<NT>(L, p, x1, x2, a.eps, xs);
    ua_ys<NT>(L, p, vx, vy, a.eps, ys);
    double xr[2];
#pragma unroll
    for (int q = 0; q < 2; ++q) {
        xs[q] = elt * xs[q] + pl * fx[q];
        ys[q] = elt * ys[q] + pl * fy[q];
        xr[q] = fft_inv<NT>(xs[q], L).re;
        yp[q] = fft_inv<NT>(ys[q], L);
    }
    double et[2];
    ua_gather(xr, a.g, et);
    cd gx[2], gy[2];
    ua_f<NT>(L, p.db, ua_interv(xr, p.b, a.deps), yp, et, gx, gy);
    const Div dt(p.t);
#pragma unroll
    for (int q = 0; q < 2; ++q) {
        xs[q] = xs[q] + dt.of(ql * (fft_fwd<NT>(gx[q], L) - fx[q]));
        ys[q] = ys[q] + dt.of(ql * (fft_fwd<NT>(gy[q], L) - fy[q]));
    }
    const cd eplus = mk(elt.re, -elt.im);
    ua_reconstruct_deposit<NT>(L, eplus, xs, a.g, live, &a.x[k], &a.y[k]);
    double v1, v2;
    ua_v<NT>(L, p.t, a.deps, eplus, ys, v1, v2);
    if (live && S.m == 0) {
        a.vx[k] = v1;
        a.vy[k] = v2;
    }
}

// ------------------------------------------------------- per-call pieces
//
// Spectra enter and leave in the reference's order: lane m's element is that of
// frequency mr.
#define UA_CALL_PROLOGUE                  \
    const Slot<NT> S(a.n);                \
    const UaLane<NT> L(a.tab, S.m, S.base); \
    const bool live = S.live;             \
    const int64_t k = S.k;                \
    const int mr = bitrev<NT>(S.m);       \
    (void)mr

// preparation!: b, t, pl, ql, xt, yt (any output may be null).
template <int NT>
__global__ __launch_bounds__(UB) void k_ua_prep_call(UaArgs a, cd *pl, cd *ql, cd *xt, cd *yt) {
    UA_CALL_PROLOGUE;
    const double vx = a.vx[k], vy = a.vy[k];
    UaPrep pr;
    ua_prep<NT>(L, a.x[k], a.y[k], vx, vy, a.epx[k], a.epy[k], a.dt, a.eps, a.deps, pr);
    cd y[2], p, q;
    ua_yt<NT>(L, pr, vx, vy, a.eps, y);
    ua_plql<NT>(L, pr.t, a.eps, ua_cis(L.l, pr.t, a.deps), p, q);
    if (!live) return;
    if (S.m == 0) {
        a.b[k] = pr.b;
        a.t[k] = pr.t;
    }
    if (pl) pl[mr + (size_t)NT * k] = p;
    if (ql) ql[mr + (size_t)NT * k] = q;
    for (int c = 0; c < 2; ++c) {
        if (xt) xt[ux(S.m, c, k, NT)] = mk(pr.xt[c]);
        if (yt) yt[ux(S.m, c, k, NT)] = y[c];
    }
}

// update_particles_e!: et from real(xt).
template <int NT>
__global__ __launch_bounds__(UB) void k_ua_gather_call(UaArgs a, const cd *xt, double *et) {
    const Slot<NT> S(a.n);
    const bool live = S.live;
    const int64_t k = S.k;
    const double x[2] = {xt[ux(S.m, 0, k, NT)].re, xt[ux(S.m, 1, k, NT)].re};
    double e[2];
    ua_gather(x, a.g, e);
    if (!live) return;
    et[ux(S.m, 0, k, NT)] = e[0];
    et[ux(S.m, 1, k, NT)] = e[1];
}

// compute_f!, with its closing FFTs.
template <int NT>
__global__ __launch_bounds__(UB) void k_ua_f_call(UaArgs a, const cd *xt, const cd *yt,
                                                  const double *et, cd *fx, cd *fy) {
    UA_CALL_PROLOGUE;
    const double x[2] = {xt[ux(S.m, 0, k, NT)].re, xt[ux(S.m, 1, k, NT)].re};
    const cd y[2] = {yt[ux(S.m, 0, k, NT)], yt[ux(S.m, 1, k, NT)]};
    const double e[2] = {et[ux(S.m, 0, k, NT)], et[ux(S.m, 1, k, NT)]};
    const double b = a.b[k];
    cd f[2], h[2];
    ua_f<NT>(L, Div(b), ua_interv(x, b, a.deps), y, e, f, h);
    for (int c = 0; c < 2; ++c) {
        f[c] = fft_fwd<NT>(f[c], L);
        h[c] = fft_fwd<NT>(h[c], L);
    }
    if (!live) return;
    for (int c = 0; c < 2; ++c) {
        fx[ux(mr, c, k, NT)] = f[c];
        fy[ux(mr, c, k, NT)] = h[c];
    }
}

// ua_step! (gx null) or its corrected form.
template <int NT>
__global__ __launch_bounds__(UB) void k_ua_step_call(UaArgs a, const cd *xtil, const cd *fx,
                                                     const cd *gx, cd *xt) {
    UA_CALL_PROLOGUE;
    const double t = a.t[k];
    const cd elt = ua_cis(L.l, t, a.deps);
    cd pl, ql;
    ua_plql<NT>(L, t, a.eps, elt, pl, ql);
    if (!live) return;
    for (int c = 0; c < 2; ++c) {
        const size_t u = ux(mr, c, k, NT);
        const cd f = fx[u];
        cd z = elt * xtil[u] + pl * f;
        if (gx) z = z + (ql * (gx[u] - f)) / t;
        xt[u] = z;
    }
}

// update_particles_x!: reconstruction into Particles.x and the deposit.
template <int NT>
__global__ __launch_bounds__(UB) void k_ua_rho_call(UaArgs a, const cd *xt) {
    UA_CALL_PROLOGUE;
    cd x[2] = {xt[ux(S.m, 0, k, NT)], xt[ux(S.m, 1, k, NT)]};
    for (int c = 0; c < 2; ++c) x[c] = fft_fwd<NT>(x[c], L);
    const cd elt = ua_cis(L.l, a.t[k], a.deps);
    ua_reconstruct_deposit<NT>(L, mk(elt.re, -elt.im), x, a.g, live, &a.x[k], &a.y[k]);
}

// compute_v!.
template <int NT>
__global__ __launch_bounds__(UB) void k_ua_v_call(UaArgs a, const cd *yt) {
    UA_CALL_PROLOGUE;
    const cd y[2] = {yt[ux(mr, 0, k, NT)], yt[ux(mr, 1, k, NT)]};
    const double t = a.t[k];
    const cd elt = ua_cis(L.l, t, a.deps);
    double v1, v2;
    ua_v<NT>(L, t, a.deps, mk(elt.re, -elt.im), y, v1, v2);
    if (live && S.m == 0) {
        a.vx[k] = v1;
        a.vy[k] = v2;
    }
}

// ------------------------------------------------------------------ host

#define UA_NT_SWITCH(nt, ...)                          \
    switch (nt) {                                      \
        case 2: { constexpr int NT = 2; __VA_ARGS__; } break;   \
        case 4: { constexpr int NT = 4; __VA_ARGS__; } break;   \
        case 8: { constexpr int NT = 8; __VA_ARGS__; } break;   \
        case 16: { constexpr int NT = 16; __VA_ARGS__; } break; \
        case 32: { constexpr int NT = 32; __VA_ARGS__; } break; \
        case 64: { constexpr int NT = 64; __VA_ARGS__; } break; \
        default: return fail(PIC_ERR_ARG, "ntau %d", nt);       \
    }

int ua_alloc(double **p, size_t count) {
    if (*p) return PIC_OK;
    const hipError_t e = hipMalloc((void **)p, std::max<size_t>(count, 2) * 8);
    if (e != hipSuccess) return fail(PIC_ERR_NOMEM, "hipMalloc(%zu bytes): %s", count * 8, hipGetErrorString(e));
    return PIC_OK;
}

void ua_free(Ctx *c) {
    for (double **p : {&c->ua_b, &c->ua_t, &c->ua_x0, &c->ua_y0, &c->ua_fhat}) {
        if (*p) (void)hipFree(*p);
        *p = nullptr;
    }
    c->ua_cap = 0;
}

// The per-particle UA buffers for the context's particle count.
int ua_ensure(Ctx *c) {
    PIC_CHECK(c->ua_ntau > 0, PIC_ERR_STATE, "pic_ua_init has not been called");
    PIC_CHECK(c->state == PIC_STATE_F64, PIC_ERR_STATE, "the UA step runs in the FP64 state");
    PIC_CHECK(c->uniform_w, PIC_ERR_STATE, "the UA step needs one particle weight (Particles.w)");
    if (c->ua_cap < c->n) ua_free(c);
    if (!c->ua_b) {
        const size_t n = (size_t)std::max<int64_t>(c->n, 1);
        PIC_TRY(ua_alloc(&c->ua_b, n));
        PIC_TRY(ua_alloc(&c->ua_t, n));
        PIC_TRY(ua_alloc(&c->ua_x0, n));
        PIC_TRY(ua_alloc(&c->ua_y0, n));
        PIC_TRY(ua_alloc(&c->ua_fhat, n * (size_t)c->ua_ntau * 8));
        c->ua_cap = (int64_t)n;
    }
    PIC_TRY(ensure_pfields(c));
    PIC_TRY(ua_alloc(&c->ua_e, (size_t)2 * c->nx * c->ny));
    if (!c->ua_tab) {  // made for the ntau of pic_ua_init, which drops an older one
        PIC_HIP(hipMalloc(&c->ua_tab, (size_t)c->ua_ntau * sizeof(UaTable)));
        hipLaunchKernelGGL(k_ua_tables, dim3(1), dim3(64), 0, c->stream, c->ua_ntau,
                           static_cast<UaTable *>(c->ua_tab));
        PIC_HIP(hipGetLastError());
    }
    return PIC_OK;
}

UaArgs ua_args(Ctx *c, double dt) {
    UaArgs a;
    a.n = c->n;
    a.eps = c->ua_eps;
    a.deps = Div(c->ua_eps);
    a.tab = static_cast<const UaTable *>(c->ua_tab);
    a.dt = dt;
    a.x = c->x; a.y = c->y; a.vx = c->vx; a.vy = c->vy;
    a.epx = c->epx; a.epy = c->epy;
    a.b = c->ua_b; a.t = c->ua_t;
    a.x0 = c->ua_x0; a.y0 = c->ua_y0;
    a.fhat = reinterpret_cast<cd *>(c->ua_fhat);
    a.g.nx = c->nx; a.g.ny = c->ny;
    a.g.xmin = c->xmin; a.g.ymin = c->ymin;
    a.g.dimx = c->dimx; a.g.dimy = c->dimy;
    a.g.dx = c->dx; a.g.dy = c->dy;
    a.g.ddx = Div(c->dx); a.g.ddy = Div(c->dy);
    a.g.e = reinterpret_cast<const double2 *>(c->ua_e);
    a.g.rho_acc = c->rho_acc;
    a.g.w = c->w0;
    return a;
}

inline dim3 ua_grid(int64_t n, int nt) {
    return dim3((unsigned)((n + UB / nt - 1) / (UB / nt)));
}

// A (ntau, 2, n) complex host array (interleaved doubles) on the device.
struct DevC {
    cd *p = nullptr;
    ~DevC() {
        if (p) (void)hipFree(p);
    }
};

int to_dev(Ctx *c, DevC &d, const double *host, size_t count_c) {
    if (!host) return PIC_OK;
    PIC_HIP(hipMalloc((void **)&d.p, std::max<size_t>(count_c, 1) * 16));
    PIC_HIP(hipMemcpyAsync(d.p, host, count_c * 16, hipMemcpyHostToDevice, c->stream));
    return PIC_OK;
}

int alloc_dev(DevC &d, size_t count_c) {
    PIC_HIP(hipMalloc((void **)&d.p, std::max<size_t>(count_c, 1) * 16));
    return PIC_OK;
}

int from_dev(Ctx *c, double *host, const DevC &d, size_t count_c) {
    if (!host) return PIC_OK;
    PIC_HIP(hipMemcpyAsync(host, d.p, count_c * 16, hipMemcpyDeviceToHost, c->stream));
    return PIC_OK;
}

// Particles.b or .t from the host into the context (NULL: keep the ones of
// the last preparation).
int load_bt(Ctx *c, double *dst, const double *src) {
    if (src && c->n)
        PIC_HIP(hipMemcpyAsync(dst, src, (size_t)c->n * 8, hipMemcpyHostToDevice, c->stream));
    return PIC_OK;
}

int ua_begin(pic_ctx *ctx, Ctx *&c) {
    PIC_CHECK(ctx, PIC_ERR_ARG, "null context");
    c = ctx_of(ctx);
    PIC_HIP(hipSetDevice(c->device));
    return ua_ensure(c);
}

}  // namespace

}  // namespace pic

using namespace pic;

extern "C" {

int pic_ua_init(pic_ctx *ctx, int ntau, double eps) {
    PIC_CHECK(ctx, PIC_ERR_ARG, "null context");
    PIC_CHECK(ntau >= 2 && ntau <= 64 && (ntau & (ntau - 1)) == 0, PIC_ERR_ARG,
              "ntau must be a power of two from 2 to 64 (got %d)", ntau);
    PIC_CHECK(eps > 0.0, PIC_ERR_ARG, "eps must be positive");
    Ctx *c = ctx_of(ctx);
    PIC_HIP(hipSetDevice(c->device));
    if (c->ua_ntau != ntau) {
        ua_free(c);
        if (c->ua_tab) (void)hipFree(c->ua_tab);
        c->ua_tab = nullptr;
    }
    c->ua_ntau = ntau;
    c->ua_eps = eps;
    return PIC_OK;
}

int pic_ua_preparation(pic_ctx *ctx, double dt, double *b, double *t, double *pl, double *ql,
                       double *xt, double *yt) {
    Ctx *c = nullptr;
    PIC_TRY(ua_begin(ctx, c));
    const int nt = c->ua_ntau;
    const size_t n = (size_t)c->n, nc = (size_t)nt * 2 * n;
    DevC dpl, dql, dxt, dyt;
    if (pl) PIC_TRY(alloc_dev(dpl, (size_t)nt * n));
    if (ql) PIC_TRY(alloc_dev(dql, (size_t)nt * n));
    if (xt) PIC_TRY(alloc_dev(dxt, nc));
    if (yt) PIC_TRY(alloc_dev(dyt, nc));
    if (n) {
        const UaArgs a = ua_args(c, dt);
        UA_NT_SWITCH(nt, hipLaunchKernelGGL(k_ua_prep_call<NT>, ua_grid(c->n, NT), dim3(UB), 0,
                                            c->stream, a, dpl.p, dql.p, dxt.p, dyt.p));
        PIC_HIP(hipGetLastError());
    }
    if (b) PIC_HIP(hipMemcpyAsync(b, c->ua_b, n * 8, hipMemcpyDeviceToHost, c->stream));
    if (t) PIC_HIP(hipMemcpyAsync(t, c->ua_t, n * 8, hipMemcpyDeviceToHost, c->stream));
    PIC_TRY(from_dev(c, pl, dpl, (size_t)nt * n));
    PIC_TRY(from_dev(c, ql, dql, (size_t)nt * n));
    PIC_TRY(from_dev(c, xt, dxt, nc));
    PIC_TRY(from_dev(c, yt, dyt, nc));
    PIC_HIP(hipStreamSynchronize(c->stream));
    return PIC_OK;
}

int pic_ua_interpol(pic_ctx *ctx, const double *xt, double *et) {
    PIC_CHECK(xt && et, PIC_ERR_ARG, "null pointer");
    Ctx *c = nullptr;
    PIC_TRY(ua_begin(ctx, c));
    const int nt = c->ua_ntau;
    const size_t n = (size_t)c->n, nc = (size_t)nt * 2 * n;
    DevC dxt, det;
    PIC_TRY(to_dev(c, dxt, xt, nc));
    PIC_TRY(alloc_dev(det, (nc + 1) / 2));
    if (n) {
        PIC_TRY(interleave_fields(c, reinterpret_cast<double2 *>(c->ua_e)));
        const UaArgs a = ua_args(c, 0.0);
        UA_NT_SWITCH(nt, hipLaunchKernelGGL(k_ua_gather_call<NT>, ua_grid(c->n, NT), dim3(UB), 0,
                                            c->stream, a, dxt.p, (double *)det.p));
        PIC_HIP(hipGetLastError());
        PIC_HIP(hipMemcpyAsync(et, det.p, nc * 8, hipMemcpyDeviceToHost, c->stream));
    }
    PIC_HIP(hipStreamSynchronize(c->stream));
    return PIC_OK;
}

int pic_ua_compute_f(pic_ctx *ctx, const double *b, const double *xt, const double *yt,
                     const double *et, double *fx, double *fy) {
    PIC_CHECK(xt && yt && et && fx && fy, PIC_ERR_ARG, "null pointer");
    Ctx *c = nullptr;
    PIC_TRY(ua_begin(ctx, c));
    PIC_TRY(load_bt(c, c->ua_b, b));
    const int nt = c->ua_ntau;
    const size_t n = (size_t)c->n, nc = (size_t)nt * 2 * n;
    DevC dxt, dyt, det, dfx, dfy;
    PIC_TRY(to_dev(c, dxt, xt, nc));
    PIC_TRY(to_dev(c, dyt, yt, nc));
    PIC_TRY(alloc_dev(det, (nc + 1) / 2));
    if (n) PIC_HIP(hipMemcpyAsync(det.p, et, nc * 8, hipMemcpyHostToDevice, c->stream));
    PIC_TRY(alloc_dev(dfx, nc));
    PIC_TRY(alloc_dev(dfy, nc));
    if (n) {
        const UaArgs a = ua_args(c, 0.0);
        UA_NT_SWITCH(nt, hipLaunchKernelGGL(k_ua_f_call<NT>, ua_grid(c->n, NT), dim3(UB), 0,
                                            c->stream, a, dxt.p, dyt.p, (const double *)det.p,
                                            dfx.p, dfy.p));
        PIC_HIP(hipGetLastError());
    }
    PIC_TRY(from_dev(c, fx, dfx, nc));
    PIC_TRY(from_dev(c, fy, dfy, nc));
    PIC_HIP(hipStreamSynchronize(c->stream));
    return PIC_OK;
}

int pic_ua_step(pic_ctx *ctx, const double *t, const double *xtilde, const double *fx,
                const double *gx, double *xt) {
    PIC_CHECK(xtilde && fx && xt, PIC_ERR_ARG, "null pointer");
    Ctx *c = nullptr;
    PIC_TRY(ua_begin(ctx, c));
    PIC_TRY(load_bt(c, c->ua_t, t));
    const int nt = c->ua_ntau;
    const size_t n = (size_t)c->n, nc = (size_t)nt * 2 * n;
    DevC dxs, dfx, dgx, dxt;
    PIC_TRY(to_dev(c, dxs, xtilde, nc));
    PIC_TRY(to_dev(c, dfx, fx, nc));
    PIC_TRY(to_dev(c, dgx, gx, nc));
    PIC_TRY(alloc_dev(dxt, nc));
    if (n) {
        const UaArgs a = ua_args(c, 0.0);
        UA_NT_SWITCH(nt, hipLaunchKernelGGL(k_ua_step_call<NT>, ua_grid(c->n, NT), dim3(UB), 0,
                                            c->stream, a, dxs.p, dfx.p, dgx.p, dxt.p));
        PIC_HIP(hipGetLastError());
    }
    PIC_TRY(from_dev(c, xt, dxt, nc));
    PIC_HIP(hipStreamSynchronize(c->stream));
    return PIC_OK;
}

int pic_ua_compute_rho(pic_ctx *ctx, const double *t, const double *xt) {
    PIC_CHECK(xt, PIC_ERR_ARG, "null pointer");
    Ctx *c = nullptr;
    PIC_TRY(ua_begin(ctx, c));
    PIC_TRY(load_bt(c, c->ua_t, t));
    const int nt = c->ua_ntau;
    const size_t n = (size_t)c->n, nc = (size_t)nt * 2 * n;
    DevC dxt;
    PIC_TRY(to_dev(c, dxt, xt, nc));
    const bool lds = deposit_lds_ok(c);
    if (!lds) PIC_TRY(launch_fill(c, c->rho_acc, 0.0, (int64_t)c->nx * c->ny));
    if (n) {
        UaArgs a = ua_args(c, 0.0);
        if (lds) a.g.rho_acc = nullptr;
        UA_NT_SWITCH(nt, hipLaunchKernelGGL(k_ua_rho_call<NT>, ua_grid(c->n, NT), dim3(UB), 0,
                                            c->stream, a, dxt.p));
        PIC_HIP(hipGetLastError());
    }
    if (lds) PIC_TRY(deposit_rho_residues(c));
    else PIC_TRY(finalize_rho(c, PIC_M6));
    PIC_HIP(hipStreamSynchronize(c->stream));
    new_particles(c);
    return PIC_OK;
}

int pic_ua_compute_v(pic_ctx *ctx, const double *t, const double *yt) {
    PIC_CHECK(yt, PIC_ERR_ARG, "null pointer");
    Ctx *c = nullptr;
    PIC_TRY(ua_begin(ctx, c));
    PIC_TRY(load_bt(c, c->ua_t, t));
    const int nt = c->ua_ntau;
    const size_t n = (size_t)c->n, nc = (size_t)nt * 2 * n;
    DevC dyt;
    PIC_TRY(to_dev(c, dyt, yt, nc));
    if (n) {
        const UaArgs a = ua_args(c, 0.0);
        UA_NT_SWITCH(nt, hipLaunchKernelGGL(k_ua_v_call<NT>, ua_grid(c->n, NT), dim3(UB), 0,
                                            c->stream, a, dyt.p));
        PIC_HIP(hipGetLastError());
    }
    PIC_HIP(hipStreamSynchronize(c->stream));
    return PIC_OK;
}

int pic_ua_run(pic_ctx *ctx, double dt, int nsteps, double *energy) {
    PIC_CHECK(nsteps >= 0, PIC_ERR_ARG, "nsteps %d", nsteps);
    Ctx *c = nullptr;
    PIC_TRY(ua_begin(ctx, c));
    const int nt = c->ua_ntau;
    const int64_t m = (int64_t)c->nx * c->ny;
    hipEvent_t ev[2] = {nullptr, nullptr};
    if (c->timing) {
        PIC_HIP(hipEventCreate(&ev[0]));
        PIC_HIP(hipEventCreate(&ev[1]));
    }
    struct EvFree {
        hipEvent_t *e;
        ~EvFree() {
            for (int k = 0; k < 2; ++k)
                if (e[k]) (void)hipEventDestroy(e[k]);
        }
    } evfree{ev};
    // energies of every half step queued on the device (pairs of interior
    // sums, then the ghost-node terms) and read once after the loop
    const int64_t nh = 2 * (int64_t)nsteps;
    if (energy) PIC_TRY(ensure_energy(c, nh + (nh + 1) / 2));
    double *ghost = c->energy_hist + 2 * nh;
    const bool lds = deposit_lds_ok(c);
    // the gather reads (ex, ey) side by side: the loop's solves write them so
    double2 *const e2 = reinterpret_cast<double2 *>(c->ua_e);
    if (c->n && nsteps) PIC_TRY(interleave_fields(c, e2));
    for (int s = 0; s < nsteps; ++s) {
        for (int half = 0; half < 2; ++half) {
            if (!lds) PIC_TRY(launch_fill(c, c->rho_acc, 0.0, m));
            if (c->n) {
                UaArgs a = ua_args(c, dt);
                if (lds) a.g.rho_acc = nullptr;
                if (c->timing) PIC_HIP(hipEventRecord(ev[0], c->stream));
                if (half == 0) {
                    UA_NT_SWITCH(nt, hipLaunchKernelGGL(k_ua_predict<NT>,
                                                        ua_grid(c->n, NT),
                                                        dim3(UB), 0, c->stream, a));
                } else {
                    UA_NT_SWITCH(nt, hipLaunchKernelGGL(k_ua_correct<NT>,
                                                        ua_grid(c->n, NT),
                                                        dim3(UB), 0, c->stream, a));
                }
                PIC_HIP(hipGetLastError());
                if (c->timing) {
                    // timing waits for each kernel (the untimed loop does not wait)
                    PIC_HIP(hipEventRecord(ev[1], c->stream));
                    PIC_HIP(hipEventSynchronize(ev[1]));
                    float ms = 0.0f;
                    PIC_HIP(hipEventElapsedTime(&ms, ev[0], ev[1]));
                    c->t_ua_ms[half] += ms;
                    c->t_ua_n[half] += 1;
                }
            }
            if (lds) PIC_TRY(deposit_rho_residues(c));
            else PIC_TRY(finalize_rho(c, PIC_M6));
            // pic_solve_fields without its wait: E and the energy sums
            PIC_TRY(solve_fields_async(c, energy ? 2 * s + half : -1,
                                       energy ? ghost + 2 * s + half : nullptr, e2));
        }
    }
    if (energy && nh > 0) {
        std::vector<double> h(3 * (size_t)nh);
        PIC_HIP(hipMemcpyAsync(h.data(), c->energy_hist, h.size() * sizeof(double),
                               hipMemcpyDeviceToHost, c->stream));
        PIC_HIP(hipStreamSynchronize(c->stream));
        for (int64_t k = 0; k < nh; ++k)
            energy[k] = h[2 * k] + h[2 * k + 1] + h[2 * nh + k] * c->dx * c->dy;
    }
    PIC_HIP(hipStreamSynchronize(c->stream));
    new_particles(c);
    return PIC_OK;
}

int pic_get_ua_timing(pic_ctx *ctx, double *ms, int64_t *launches) {
    PIC_CHECK(ctx, PIC_ERR_ARG, "null context");
    Ctx *c = ctx_of(ctx);
    for (int k = 0; k < 2; ++k) {
        if (ms) ms[k] = c->t_ua_ms[k];
        if (launches) launches[k] = c->t_ua_n[k];
    }
    return PIC_OK;
}

}  // extern "C"
