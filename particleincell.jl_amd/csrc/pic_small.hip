// pic_small.hip -- pic_run's time loop with one launch per iteration on small
// grids (power-of-two nx, ny <= 64).
//
// On a 64 x 64 grid the loop of separate kernels (three transform kernels, the
// particle pass and its deferred-list kernel, a lane sort every few steps)
// is bound by launch latency: each kernel runs a few microseconds with most
// of the chip idle.  Here every block of one launch holds the whole grid in
// LDS and does:
//   1. the E solve of the previous deposit, redundantly on its own LDS copy
//      (the same operations on the same inputs, so every block holds the
//      same field): transforms along x and y of the raw charge, the spectral
//      multiplier of the E solve, the inverse transforms along y and x,
//      (ex, ey) = (Re, Im).  Block 0 writes the field energy, and at the last
//      iteration ex, ey and their FP32 copy;
//   2. the particles in any order (no sort): gather from the LDS field, kick,
//      drift, deposit into an LDS charge grid;
//   3. the charge grid added to the global accumulator with global atomics.
// The raw charge rotates through three buffers (the one read, the one summed
// into, the one cleared for the next launch), so no launch writes what
// another block of the same launch reads.
//
// Transforms (es_line): N/8 lanes of one wave hold a line's N <= 64 points,
// eight each (N = 4: one lane, four).  Two steps, N = 8 B: eight-point
// transforms over the points B apart, twiddles, the lanes' exchange through
// their line in LDS (no block barrier: a line's lanes are in one wave), then
// B-point transforms.  Four passes: along x of two real rows packed as one
// complex line, along y of the half spectrum's columns, back along y, back
// along x, with three block barriers between them and one within the third.
// Same transforms (unnormalised, exp(-+2 pi i jk/N)) and the spectral
// values as the three-kernel solve of pic_poisson.hip; results agree to rounding.
// Measured on MI355X, Landau CIC 64 x 64 with 204,800 particles, FP32 state, 100
// steps: 18.6 us per step of wall time against 23.1 (FP64 state 20.2 against
// 25.9) with a point per lane and
// radix-2 stages exchanged between lanes (and the self-conjugate columns'
// projection formed from both halves).  In a block's timestamps: loads 3.4 us,
// the passes 1.6, 2.0, 2.2 (0.8 of it the spectral values), 2.0 and barriers
// 1.6, particles 1.3, flush 1.9; the loads and the flush are latency of memory
// past the L2, the passes that of LDS and of dependent FP64 operations at two
// waves per SIMD.
//
// Charge: FP32 state: int32 fixed-point LDS grid (charge32_fixed) with one
// quantum for every block, flushed as int64 sums, so the raw charge is exact
// and the same on every run; FP64 state: FP64 LDS atomics and FP64 global
// atomics, as in the segment passes.
//
// Per-particle arithmetic is the segment passes' (pic_push32.h,
// pic_push64.h): the same operations on the same field values.
#include <algorithm>
#include <cmath>
#include <vector>

#include "pic_internal.h"
#include "pic_push32.h"
#include "pic_push64.h"

namespace pic {

constexpr int ES_T = 1024;                 // threads per block
constexpr int ES_WAVES = ES_T / 64;
constexpr int ES_MAX_SIDE = 64;
constexpr int ES_EPAD = 8;
// Particles per block.  Every block loads the whole charge and adds its own
// charge grid to the global one, so fewer, fuller blocks do less of both;
// measured on MI355X, Landau CIC 64 x 64 with 204,800 particles in the FP32
// state: 128 blocks (1.6 particles per thread) 18.4 us per step, 200 blocks
// 20.2, 86 blocks 18.5, 50 blocks 18.5.
constexpr int64_t ES_BLOCK_PARTICLES = 1600;

struct EsStep {
    int nx, ny, lognx, logny;
    int mode;     // 0: drift dt/2 + deposit; 1: kick + drift dt + deposit; 2: kick + drift dt/2
    int solve;    // E from rin first (modes 1, 2)
    int write_e;  // block 0 stores ex, ey, e32
    int slot;     // energy history entry (-1: none)
    int64_t n;
    SegF64 s64;   // FP64 state: arrays and the step's constants (kick64, drift64)
    int32_t *cell;  // FP32 state
    float4 *ov;
    float hdt, dtdx, dtdy, bz0;
    float wu;     // |w| in quanta
    int R, conserve;
    double unit;  // charge of one quantum
    const void *rin;  // raw charge read (FP64, or int64 quanta in the FP32 state)
    void *racc;       // summed into
    void *rclr;       // cleared
    const double *kxk2, *kyk2;
    double scale, dxdy;
    double *ex, *ey;
    float2 *e32;
    double *hist;
    const double2 *tw;  // twiddles: nx along x, then ny along y
    int nbp;            // particle blocks; block nbp (if launched) the field block
};

__device__ __forceinline__ double2 operator+(double2 a, double2 b) {
    return make_double2(a.x + b.x, a.y + b.y);
}
__device__ __forceinline__ double2 operator-(double2 a, double2 b) {
    return make_double2(a.x - b.x, a.y - b.y);
}
// a - 1i sg d and a + 1i sg d (sg = 1 forward, -1 backward)
__device__ __forceinline__ double2 es_sub_i(double2 a, double2 d, double sg) {
    return make_double2(__builtin_fma(sg, d.y, a.x), __builtin_fma(-sg, d.x, a.y));
}
__device__ __forceinline__ double2 es_add_i(double2 a, double2 d, double sg) {
    return make_double2(__builtin_fma(-sg, d.y, a.x), __builtin_fma(sg, d.x, a.y));
}

// In-register transforms X[k] = sum_j z[j] exp(-2 pi i sg jk / N), natural
// order in and out, of the points z[o], z[o + S], ..
template <int N, int S>
__device__ __forceinline__ void es_dft(double2 *z, double sg) {
    if constexpr (N == 2) {
        const double2 a = z[0], b = z[S];
        z[0] = a + b;
        z[S] = a - b;
    } else if constexpr (N == 4) {
        const double2 t0 = z[0] + z[2 * S], t1 = z[0] - z[2 * S], t2 = z[S] + z[3 * S],
                      t3 = z[S] - z[3 * S];
        z[0] = t0 + t2;
        z[S] = es_sub_i(t1, t3, sg);
        z[2 * S] = t0 - t2;
        z[3 * S] = es_add_i(t1, t3, sg);
    } else {
        static_assert(N == 8 && S == 1, "eight points side by side");
        constexpr double h = 0.70710678118654752440;
        double2 b[4], c[4];
#pragma unroll
        for (int k = 0; k < 4; ++k) {
            b[k] = z[k] + z[k + 4];
            c[k] = z[k] - z[k + 4];
        }
        // c[k] exp(-2 pi i sg k / 8)
        const double2 c1 = make_double2(h * __builtin_fma(sg, c[1].y, c[1].x),
                                        h * __builtin_fma(-sg, c[1].x, c[1].y));
        const double2 c2 = make_double2(sg * c[2].y, -sg * c[2].x);
        const double2 c3 = make_double2(h * __builtin_fma(sg, c[3].y, -c[3].x),
                                        -h * __builtin_fma(sg, c[3].x, c[3].y));
        c[1] = c1;
        c[2] = c2;
        c[3] = c3;
        es_dft<4, 1>(b, sg);
        es_dft<4, 1>(c, sg);
#pragma unroll
        for (int k = 0; k < 4; ++k) {
            z[2 * k] = b[k];
            z[2 * k + 1] = c[k];
        }
    }
}

// One line of N = 2^LOG points: this lane, t of the line's N/8, holds the
// points t + B n (n < 8) in z[n].  swap(t, c) is the LDS word of element t + c of
// the line, out(t, c, v) takes element t + c of the result (c, without bits in
// common with t, is a constant once the loops are unrolled, so that the words
// share their address arithmetic); tw[k] = exp(-2 pi i k / N).
template <int LOG, class Swap, class Out>
__device__ __forceinline__ void es_line(double2 (&z)[8], int t, const double2 *tw, double sg,
                                        Swap &&swap, Out &&out) {
    constexpr int N = 1 << LOG, A = N >= 8 ? 8 : 4, B = N / A;
    es_dft<A, 1>(z, sg);
    if constexpr (B == 1) {
#pragma unroll
        for (int k = 0; k < A; ++k) out(0, k, z[k]);
    } else {
        *swap(t, 0) = z[0];
#pragma unroll
        for (int k = 1; k < A; ++k) {
            const double2 w = tw[t * k];
            const double wy = sg * w.y;
            *swap(t, B * k) = make_double2(__builtin_fma(z[k].x, w.x, -(z[k].y * wy)),
                                           __builtin_fma(z[k].x, wy, z[k].y * w.x));
        }
        // a wave's LDS operations are done in order: its reads see its writes
        __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
        __builtin_amdgcn_wave_barrier();
        // 8/B transforms of B points: k = t, t + B, ..; point n of the r-th in
        // z[r + (8/B) n]
        constexpr int R = A / B;
#pragma unroll
        for (int r = 0; r < R; ++r)
#pragma unroll
            for (int n = 0; n < B; ++n) z[r + R * n] = *swap(B * t, n + B * B * r);
#pragma unroll
        for (int r = 0; r < R; ++r) es_dft<B, R>(z + r, sg);
        __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
        __builtin_amdgcn_wave_barrier();
#pragma unroll
        for (int r = 0; r < R; ++r)
#pragma unroll
            for (int n = 0; n < B; ++n) out(t, B * r + A * n, z[r + R * n]);
    }
}

template <int K, bool F32, int BZ>
__global__ __launch_bounds__(ES_T) void k_es_step(EsStep a) {
    constexpr int HL = Shape<K>::HL;
    extern __shared__ __align__(16) char es_smem[];
    __shared__ double red[2 * ES_WAVES];
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    const int nx = a.nx, ny = a.ny, mx = nx - 1, my = ny - 1, m = nx * ny;
    // LDS: the grid (complex), the twiddles (nx along x, then ny along y), the
    // spectral tables, the FP32 state's field, the charge grid
    double2 *X = reinterpret_cast<double2 *>(es_smem);
    double2 *tw = X + m;
    const int nq = (nx / 2 + 1) * ny;
    double2 *tk = tw + nx + ny;  // (kx, ky)/k2 times the solve's scale
    float2 *ef = reinterpret_cast<float2 *>(tk + nq);
    const int pe = nx + ES_EPAD;  // its row pitch: eight rows' words on all banks
    char *tiles = reinterpret_cast<char *>(F32 ? ef + pe * ny : ef);
    int *itile = reinterpret_cast<int *>(tiles);
    double *dtile = reinterpret_cast<double *>(tiles);
    const bool gather = a.mode != 0, deposit = a.mode != 2;
    const SegF64 &s = a.s64;
    // Node (i, j) sits at word i ^ f(j) of row j: the 16 lanes an LDS access of
    // 16-byte words serves at once are two rows (or columns) of eight, which
    // the flipped bit puts on different halves of the banks, in every pass.
    const int sw = nx >= 16 ? 8 : 0;
    auto at = [&](int i, int j) { return j * nx + (i ^ (-((j ^ (j >> 3)) & 1) & sw)); };

    // every global load of the launch's first phase is issued here, so that
    // their latencies overlap: this thread's first particle (used after the
    // solve), its points of the charge, the spectral tables
    // blocks [0, nbp) move the particles; block nbp, launched with the solve,
    // writes the field energy (and the last field) instead
    const bool field = (int)blockIdx.x == a.nbp;
    int64_t p = field ? a.n : (int64_t)blockIdx.x * ES_T + tid;
    const int64_t stride = (int64_t)a.nbp * ES_T;
    int pc = 0;
    float4 po = make_float4(0.0f, 0.0f, 0.0f, 0.0f);
    double px = 0.0, py = 0.0, pvx = 0.0, pvy = 0.0, pw = 0.0;
    if (p < a.n) {
        if (F32) {
            pc = a.cell[p];
            po = a.ov[p];
        } else {
            px = s.x[p];
            py = s.y[p];
            pvx = s.vx[p];
            pvy = s.vy[p];
            pw = s.w ? s.w[p] : s.w0;
        }
    }
    // lines along x: lane group tx of T = N/8 lanes works row jr; along y: the
    // groups of a wave interleave, so that its lanes are neighbouring columns
    const int ltx = max(a.lognx - 3, 0), lty = max(a.logny - 3, 0);
    const int jr = tid >> ltx, tx = tid & ((1 << ltx) - 1), dxp = 1 << ltx;
    const int lcw = 6 - lty;  // log2 of the columns of a wave
    const int col = (wave << lcw) + (lane & ((1 << lcw) - 1)), ty = lane >> lcw, dyp = 1 << lty;
    const int npx = min(nx, 8), npy = min(ny, 8);  // points per lane
    double2 z[8];
    if (a.solve) {
        // real rows j and j + ny/2 packed as one complex line
#pragma unroll
        for (int r = 0; r < 8; ++r) {
            z[r] = make_double2(0.0, 0.0);
            if (jr < ny / 2 && r < npx) {
                const int g = jr * nx + tx + dxp * r, g2 = g + (ny / 2) * nx;
                if (F32) {
                    const long long *q = reinterpret_cast<const long long *>(a.rin);
                    z[r] = make_double2((double)q[g], (double)q[g2]);
                } else {
                    const double *q = reinterpret_cast<const double *>(a.rin);
                    z[r] = make_double2(q[g], q[g2]);
                }
            }
        }
        for (int k = tid; k < nq; k += ES_T) {
            tk[k] = make_double2(a.kxk2[k] * a.scale, a.kyk2[k] * a.scale);
        }
        for (int k = tid; k < nx + ny; k += ES_T) tw[k] = a.tw[k];
    }
    if (deposit && !field)
        for (int t = tid; t < m; t += ES_T) {
            if (F32) itile[t] = 0;
            else dtile[t] = 0.0;
        }
    if (a.rclr) {
        const int lo = (int)((int64_t)m * blockIdx.x / gridDim.x);
        const int hi = (int)((int64_t)m * (blockIdx.x + 1) / gridDim.x);
        for (int t = lo + tid; t < hi; t += ES_T)
            reinterpret_cast<unsigned long long *>(a.rclr)[t] = 0ull;
    }
    __syncthreads();

    if (a.solve) {
        if (F32) {
#pragma unroll
            for (int r = 0; r < 8; ++r) z[r] = make_double2(z[r].x * a.unit, z[r].y * a.unit);
        }
        auto line = [&](int log, int t, const double2 *w, double sg, auto &&word, auto &&out) {
            switch (log) {
                case 6: es_line<6>(z, t, w, sg, word, out); break;
                case 5: es_line<5>(z, t, w, sg, word, out); break;
                case 4: es_line<4>(z, t, w, sg, word, out); break;
                case 3: es_line<3>(z, t, w, sg, word, out); break;
                default: es_line<2>(z, t, w, sg, word, out); break;
            }
        };
        // word t + c: only bit 3 (and along y bit 0) of c meets the flipped bit
        auto in_row = [&](int t, int c) { return X + (at(t + (c & 8), jr) + (c & ~8)); };
        auto in_col = [&](int t, int c) { return X + (at(col, t + (c & 9)) + (c & ~9) * nx); };
        // forward along x of the packed rows
        if (jr < ny / 2)
            line(a.lognx, tx, tw, 1.0, in_row,
                 [&](int t, int c, double2 v) { *in_row(t, c) = v; });
        __syncthreads();
        // forward along y of columns 0 .. nx/2, split on the way in into the
        // transforms of rows j, j + ny/2: (Z[k] + conj Z[-k]) / 2, (Z[k] - conj
        // Z[-k]) / 2i
        if (col <= nx / 2) {
#pragma unroll
            for (int r = 0; r < 4; ++r) {
                if (2 * r >= npy) break;
                const int j = ty + dyp * r;
                const double2 zk = X[at(col, j)], zm = X[at((nx - col) & mx, j)];
                z[r] = make_double2(0.5 * (zk.x + zm.x), 0.5 * (zk.y - zm.y));
                const double2 b = make_double2(0.5 * (zk.y + zm.y), -0.5 * (zk.x - zm.x));
                if (npy == 8) z[r + 4] = b;
                else z[(r + 2) & 7] = b;
            }
            line(a.logny, ty, tw + nx, 1.0, in_col,
                 [&](int t, int c, double2 v) { *in_col(t, c) = v; });
        }
        __syncthreads();
        // f + 1i g of (f, g) = -1i (kx, ky)/k2 R, columns past nx/2 the
        // conjugates of their mirrors.  The self-conjugate columns 0 and nx/2
        // hold the transforms of real columns, R(-j) = conj R(j): the Hermitian
        // part of f there is 0, and that of g is g but for its own mirrors 0
        // and ny/2, where it is 0 (R[0,0] -> 0 with them).
        if (col < nx) {
            const bool mir = col > nx / 2;
            const int ih = mir ? nx - col : col;
            const bool self = ih == 0 || 2 * ih == nx;
            const double sm = mir ? -1.0 : 1.0;
#pragma unroll
            for (int r = 0; r < 8; ++r) {
                if (r >= npy) break;
                const int jk = ty + dyp * r, jh = mir ? (ny - jk) & my : jk;
                const double2 R = X[at(ih, jh)];
                double2 k = tk[ih + (nx / 2 + 1) * jh];
                if (self) {
                    k.x = 0.0;
                    if ((jh & (ny / 2 - 1)) == 0) k.y = 0.0;
                }
                z[r] = make_double2(__builtin_fma(k.x, R.y, sm * (k.y * R.x)),
                                    __builtin_fma(k.y, R.y, -sm * (k.x * R.x)));
            }
        }
        __syncthreads();  // every column read before any is written
        if (col < nx)
            line(a.logny, ty, tw + nx, -1.0, in_col,
                 [&](int t, int c, double2 v) { *in_col(t, c) = v; });
        __syncthreads();
        // back along x: (ex, ey) = (Re, Im)
        if (jr < ny) {
#pragma unroll
            for (int r = 0; r < 8; ++r)
                if (r < npx) z[r] = X[at(tx + dxp * r, jr)];
            float2 *er = ef + jr * pe;
            line(a.lognx, tx, tw, -1.0, in_row, [&](int t, int c, double2 v) {
                if (F32 && !field) er[t + c] = make_float2((float)v.x, (float)v.y);
                else *in_row(t, c) = v;
            });
        }
        __syncthreads();
        if (field) {
            double sx = 0.0, sy = 0.0;
            for (int t = tid; t < m; t += ES_T) {
                const double2 v = X[at(t & mx, t >> a.lognx)];
                sx += v.x * v.x;
                sy += v.y * v.y;
                if (a.write_e) {
                    a.ex[t] = v.x;
                    a.ey[t] = v.y;
                    a.e32[t] = make_float2((float)v.x, (float)v.y);
                }
            }
            if (a.slot < 0) return;
            // fixed-order sums: wave trees, then the waves in order
            for (int o = 32; o > 0; o >>= 1) {
                sx += __shfl_xor(sx, o);
                sy += __shfl_xor(sy, o);
            }
            if (lane == 0) {
                red[wave] = sx;
                red[ES_WAVES + wave] = sy;
            }
            __syncthreads();
            if (tid == 0) {
                sx = sy = 0.0;
                for (int k = 0; k < ES_WAVES; ++k) {
                    sx += red[k];
                    sy += red[ES_WAVES + k];
                }
                a.hist[2 * a.slot] = sx * a.dxdy;
                a.hist[2 * a.slot + 1] = sy * a.dxdy;
            }
            return;
        }
    }

    while (p < a.n) {
        if (F32) {
            int ci = pc & mx, cj = pc >> a.lognx;
            float fx = po.x, fy = po.y, ux = po.z, uy = po.w;
            if (gather) {
                float e1, e2, b3 = 0.0f;
                interp32<K, BZ>(
                    fx, fy, ci, cj,
                    [&](int u, int v) {
                        return ef[((cj - HL + v) & my) * pe + ((ci - HL + u) & mx)];
                    },
                    [&](int, int) { return 0.0f; }, e1, e2, b3);
                kick32<BZ>(a.hdt, a.bz0, e1, e2, b3, ux, uy);
            }
            float nfx, nfy;
            const int si = drift1s(fx, ux, a.dtdx, nfx);
            const int sj = drift1s(fy, uy, a.dtdy, nfy);
            ci = (ci + si) & mx;
            cj = (cj + sj) & my;
            fx = nfx;
            fy = nfy;
            a.cell[p] = ci + nx * cj;
            a.ov[p] = make_float4(fx, fy, ux, uy);
            if (deposit)
                charge32_fixed<K>(fx, fy, ci, cj, a.wu, a.R, a.conserve != 0,
                                  [&](int u, int v, int q) {
                                      __hip_atomic_fetch_add(
                                          &itile[((cj - HL + v) & my) * nx + ((ci - HL + u) & mx)],
                                          q, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
                                  });
        } else {
            if (gather) {
                double fx, fy;
                const int ci = ref_cell_s(px, s.dx, nx, false, fx);
                const int cj = ref_cell_s(py, s.dy, ny, false, fy);
                double e1, e2, b3 = 0.0;
                interp64<K, BZ>(
                    fx, fy, ci, cj,
                    [&](int u, int v) {
                        return X[at((ci - HL + u) & mx, (cj - HL + v) & my)];
                    },
                    [&](int, int) { return 0.0; }, e1, e2, b3);
                kick64<BZ>(s, e1, e2, b3, pvx, pvy);
                s.vx[p] = pvx;
                s.vy[p] = pvy;
            }
            if (a.mode == 1) drift64<2>(s, pvx, pvy, px, py);
            else drift64<1>(s, pvx, pvy, px, py);
            s.x[p] = px;
            s.y[p] = py;
            if (deposit) {
                double fx, fy;
                const int ci = ref_cell_s(px, s.dx, nx, K == PIC_CIC, fx);
                const int cj = ref_cell_s(py, s.dy, ny, K == PIC_CIC, fy);
                charge64<K>(fx, fy, ci, cj, pw, [&](int u, int v, double q) {
                    __hip_atomic_fetch_add(
                        &dtile[((cj - HL + v) & my) * nx + ((ci - HL + u) & mx)], q,
                        __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
                });
            }
        }
        p += stride;
        if (p < a.n) {
            if (F32) {
                pc = a.cell[p];
                po = a.ov[p];
            } else {
                px = s.x[p];
                py = s.y[p];
                pvx = s.vx[p];
                pvy = s.vy[p];
                pw = s.w ? s.w[p] : s.w0;
            }
        }
    }
    if (!deposit || field) return;
    __syncthreads();
    // each block starts at its own node, so that the blocks' atomics spread
    // over the grid instead of meeting at the same addresses (measured: 0.7
    // us less per launch on 64 x 64)
    const int off = (int)((int64_t)blockIdx.x * m / a.nbp);
    for (int t0 = tid; t0 < m; t0 += ES_T) {
        const int t = (t0 + off) & (m - 1);
        if (F32) {
            const int q = itile[t];
            if (q) atomicAdd(reinterpret_cast<unsigned long long *>(a.racc) + t,
                             (unsigned long long)(long long)q);
        } else {
            const double q = dtile[t];
            if (q != 0.0) unsafeAtomicAdd(reinterpret_cast<double *>(a.racc) + t, q);
        }
    }
}

// Twiddles exp(-2 pi i k / N) of the transforms along x (k < nx), then y.
__global__ void k_es_twiddles(int nx, int ny, int lognx, int logny, double2 *tw) {
    const int k = threadIdx.x;
    if (k >= nx + ny) return;
    const bool along_x = k < nx;
    const int kk = along_x ? k : k - nx;
    double sn, cs;
    sincospi(ldexp((double)(-2 * kk), -(along_x ? lognx : logny)), &sn, &cs);
    tw[k] = make_double2(cs, sn);
}

// The raw charge of an accumulator buffer as FP64 (FP32 state: quanta times
// the unit).
__global__ void k_es_raw(const void *__restrict__ buf, int quanta, double unit, int64_t m,
                         double *__restrict__ out) {
    const int64_t k = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (k >= m) return;
    out[k] = quanta ? (double)reinterpret_cast<const long long *>(buf)[k] * unit
                    : reinterpret_cast<const double *>(buf)[k];
}

static bool pow2_within(int n, int lo, int hi) {
    return n >= lo && n <= hi && (n & (n - 1)) == 0;
}

static int log2_of(int n) {
    int l = 0;
    while ((1 << l) < n) ++l;
    return l;
}

bool es_step_ok(const Ctx *c) {
    return c->fused_step && pow2_within(c->nx, 4, ES_MAX_SIDE) &&
           pow2_within(c->ny, 4, ES_MAX_SIDE) && c->bz_mode != PIC_BZ_GRID &&
           (c->state == PIC_STATE_F64 || c->f32_acc == 2);
}

static size_t es_lds(const Ctx *c) {
    const size_t nx = c->nx, ny = c->ny;
    return (nx * ny + nx + ny) * sizeof(double2) + 2 * (nx / 2 + 1) * ny * sizeof(double) +
           (c->state == PIC_STATE_F32 ? (nx + ES_EPAD) * ny * sizeof(float2) + nx * ny * 4
                                      : nx * ny * 8);
}

template <int K, bool F32>
static int es_launch(const Ctx *c, const EsStep &a, size_t sm) {
    const int nb = a.nbp + (a.solve ? 1 : 0);
    auto go = [&](auto kern) -> int {
        PIC_HIP(hipFuncSetAttribute(reinterpret_cast<const void *>(kern),
                                    hipFuncAttributeMaxDynamicSharedMemorySize, (int)sm));
        hipLaunchKernelGGL(kern, dim3((unsigned)nb), dim3(ES_T), sm, c->stream, a);
        PIC_HIP(hipGetLastError());
        return PIC_OK;
    };
    if (c->bz_mode == PIC_BZ_UNIFORM && a.mode != 0) return go(k_es_step<K, F32, PIC_BZ_UNIFORM>);
    return go(k_es_step<K, F32, PIC_BZ_NONE>);
}

// pic_run's loop (pic_run.hip) as one launch per iteration: a prologue
// launch (drift dt/2 + deposit), then launch s solves the deposit of launch
// s - 1, records energy s and moves the particles on (the last one without
// deposit).  Leaves rho of the last solve's deposit (finalize_rho), ex, ey
// and e32 of the last solve.
int es_run(Ctx *c, int kernel, double dt, int nsteps) {
    const int64_t m = (int64_t)c->nx * c->ny;
    // three raw charge buffers, then the twiddles
    const size_t ntw = (size_t)(c->nx + c->ny);
    if (!c->es_buf) PIC_HIP(hipMalloc(&c->es_buf, (size_t)(3 * m) * 8 + ntw * sizeof(double2)));
    if (c->pending_perm) PIC_TRY(settle_state(c));
    const bool f32 = c->state == PIC_STATE_F32;
    // particle blocks: ~ES_BLOCK_PARTICLES each, one per CU at most, one CU
    // left to the field block
    int nb = (int)std::min<int64_t>(c->ncu - 1, (c->n + ES_BLOCK_PARTICLES - 1) / ES_BLOCK_PARTICLES);
    if (nb < 1) nb = 1;
    EsStep a = {};
    a.nx = c->nx;
    a.ny = c->ny;
    a.lognx = log2_of(c->nx);
    a.logny = log2_of(c->ny);
    a.nbp = nb;
    double2 *tw = reinterpret_cast<double2 *>(c->es_buf + 3 * m);
    hipLaunchKernelGGL(k_es_twiddles, dim3(1), dim3(2 * ES_MAX_SIDE), 0, c->stream, a.nx, a.ny, a.lognx,
                       a.logny, tw);
    PIC_HIP(hipGetLastError());
    a.tw = tw;
    a.n = c->n;
    SegF64 &s = a.s64;
    s.x = c->x; s.y = c->y; s.vx = c->vx; s.vy = c->vy;
    s.w = c->uniform_w ? nullptr : c->w;
    s.w0 = c->w0;
    s.bz0 = c->bz0;
    s.nx = c->nx; s.ny = c->ny; s.ncells = (int)m;
    s.dx = picd::Div(c->dx); s.dy = picd::Div(c->dy); s.dimx = c->dimx; s.dimy = c->dimy;
    s.dt = dt;
    s.dtd = 0.5 * dt;
    a.cell = c->cell;
    a.ov = c->ov32;
    a.hdt = (float)(0.5 * dt);
    a.bz0 = (float)c->bz0;
    if (f32) {
        // one quantum for every block: the largest particle count of a block
        const int64_t per_round = (int64_t)nb * ES_T;
        const int64_t count = (c->n + per_round - 1) / per_round * ES_T;
        const float w = (float)c->w0;
        double qmax = 1.0;
        PIC_SHAPE_SWITCH(kernel, qmax = Shape<KK>::QMAX);
        const int qe = fixed_exponent(w, qmax, count);
        a.wu = ldexpf(fabsf(w), -qe);
        a.conserve = count <= CONSERVE_MAX_COUNT;
        a.R = a.conserve ? (int)rintf(a.wu) : 0;
        a.unit = (a.conserve && a.R != 0) ? (double)w / a.R : copysign(ldexp(1.0, qe), (double)w);
    }
    a.kxk2 = c->kx_k2;
    a.kyk2 = c->ky_k2;
    a.scale = 1.0 / ((double)c->nx * (double)c->ny * c->dx * c->dy);
    a.dxdy = c->dx * c->dy;
    a.ex = c->ex;
    a.ey = c->ey;
    a.e32 = reinterpret_cast<float2 *>(c->e32);
    a.hist = c->energy_hist;
    const size_t sm = es_lds(c);
    double *buf[3] = {c->es_buf, c->es_buf + m, c->es_buf + 2 * m};
    auto launch = [&](const EsStep &e) -> int {
        int rc = PIC_OK;
        PIC_SHAPE_SWITCH(kernel, rc = f32 ? es_launch<KK, true>(c, e, sm)
                                          : es_launch<KK, false>(c, e, sm));
        return rc;
    };
    PIC_TRY(launch_fill(c, buf[0], 0.0, m));
    particles_moved(c, nsteps);
    // prologue: drift dt/2 and deposit into buffer 0, buffer 1 cleared
    EsStep e = a;
    e.mode = 0;
    e.solve = 0;
    e.slot = -1;
    e.dtdx = (float)(0.5 * dt / c->dx);
    e.dtdy = (float)(0.5 * dt / c->dy);
    e.racc = buf[0];
    e.rclr = buf[1];
    PIC_TRY(launch(e));
    std::vector<hipEvent_t> ev;
    int rc = PIC_OK;
    for (int st = 0; st < nsteps && rc == PIC_OK; ++st) {
        const bool last = st == nsteps - 1;
        e = a;
        e.mode = last ? 2 : 1;
        e.solve = 1;
        e.slot = st;
        e.write_e = last;
        // FP32: one drift of dt (mode 1) or dt/2; FP64 drifts by dt/2 once or twice
        const double dtd = last ? 0.5 * dt : dt;
        e.dtdx = (float)(dtd / c->dx);
        e.dtdy = (float)(dtd / c->dy);
        e.rin = buf[st % 3];
        e.racc = buf[(st + 1) % 3];
        e.rclr = buf[(st + 2) % 3];
        // events around every timing_every-th launch
        const bool timed = c->timing && st % c->timing_every == 0;
        auto mark = [&]() -> int {
            hipEvent_t h;
            if (hipEventCreate(&h) != hipSuccess) return fail(PIC_ERR_HIP, "event create failed");
            ev.push_back(h);
            (void)hipEventRecord(h, c->stream);
            return PIC_OK;
        };
        if (timed) rc = mark();
        if (rc == PIC_OK) rc = launch(e);
        if (rc == PIC_OK && timed) rc = mark();
    }
    if (c->timing && rc == PIC_OK && !ev.empty() &&
        hipEventSynchronize(ev.back()) == hipSuccess) {
        for (size_t k = 0; k + 1 < ev.size(); k += 2) {
            float ms = 0.0f;
            (void)hipEventElapsedTime(&ms, ev[k], ev[k + 1]);
            c->t_pass_ms += ms;
            c->t_passes += 1;
        }
    }
    for (hipEvent_t h : ev) (void)hipEventDestroy(h);
    PIC_TRY(rc);
    // the charge the last solve read, as the raw accumulator, then rho
    const void *last_in = nsteps > 0 ? buf[(nsteps - 1) % 3] : buf[0];
    hipLaunchKernelGGL(k_es_raw, dim3((unsigned)((m + 255) / 256)), dim3(256), 0, c->stream,
                       last_in, f32 ? 1 : 0, a.unit, m, c->rho_acc);
    PIC_HIP(hipGetLastError());
    return finalize_rho(c, kernel);
}

}  // namespace pic

using namespace pic;

extern "C" int pic_set_fused_step(pic_ctx *ctx, int fused) {
    PIC_CHECK(ctx, PIC_ERR_ARG, "null context");
    ctx_of(ctx)->fused_step = fused != 0;
    return PIC_OK;
}
