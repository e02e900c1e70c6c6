// pic_deposit.hip -- the charge deposit of particles in any order, with the
// whole grid's charge in LDS.
//
// Particles that are not sorted by cell put their charge anywhere, and one
// FP64 global atomic per stencil node is what that costs: measured on MI355X 20
// to 23e9/s (1,000,000 particles on 128 x 128 to 400 x 400 nodes, CIC and M6),
// 1.6 ms for 1,000,000 M6 particles.  Here block (chunk, r) takes a chunk of the
// particles and sums the nodes of part r of the grid in LDS (one part up to
// 20,480 nodes, at most DEP_PARTS_MAX), then stores its copy of that part
// without atomics; k_deposit_reduce adds the copies in chunk order, and sums the
// grid for the neutralising shift on the way.  Measured, the whole call:
// 1,000,000 unsorted M6 particles on 100 x 100 nodes 59 us, on 256 x 256 (four
// parts) 99, on 400 x 400 (eight) 167.
//
// With R parts every chunk is read and its weights formed R times, so past
// DEP_PARTS_MAX parts the chunk kernels of pic_step.hip serve; and for particles
// near their cells' order (particles_near_order), whose chunks cover small boxes:
// measured on lane-sorted M6 particles they take as long as one part does
// (10,000,000 on 128 x 128: 195 against 174 us; 300,000 CIC on 100 x 100: 28
// against 36) and less than several (2,000,000 on 400 x 400: 71 us against 363).
#include <algorithm>

#include "pic_internal.h"
#include "pic_push64.h"

namespace pic {

namespace {

constexpr int DT = 1024;
constexpr size_t DEP_LDS = 160 * 1024;

// How a position gives a cell and an in-cell offset, and where the weights go.
//   DEP_REF     compute_rho(p, kernel, mesh): pushers_cic.jl:84-105 (trunc for
//               CIC), pushers_m6.jl:246-338 (floor)
//   DEP_MF      the MeshFields M6 deposit at the residue x - x0 mod dimx
//               (compute_rho_m6.jl:70-81), in [0, dimx]
//   DEP_COMPAT  the same with the reference's neighbour indices of
//               compute_rho_m6!(fields, particles) (:216-227), every
//               off-centre weight one node low
// The residue is formed here from the position as given, or given itself
// (UA): a position put back into the domain, residue + x0, has lost the
// residue's last bits (128 x 64 cells, x0 = xmax: charge 1e-14 off normwise
// instead of 1e-16).
enum { DEP_REF, DEP_MF, DEP_COMPAT };

struct DepArgs {
    int64_t n;
    const double *x, *y, *w;  // w null: w0
    double w0, x0, y0, dimx, dimy, dx, dy;
    int residues;             // x, y are residues (DEP_MF)
    int nx, ny;
    double *copies;           // chunk c's grid at c * nx * ny
    int chunks, parts, len;   // len nodes per part
};

template <int K, int HOW, bool SPLIT>
__global__ __launch_bounds__(DT) void k_deposit_lds(DepArgs a) {
    extern __shared__ double lds[];
    constexpr int S = Shape<K>::S, HL = Shape<K>::HL;
    const int nx = a.nx, ny = a.ny, tid = threadIdx.x;
    const int chunk = SPLIT ? blockIdx.x / a.parts : blockIdx.x;
    const int r0 = SPLIT ? blockIdx.x - chunk * a.parts : 0;
    const int lo = r0 * a.len, len = min(a.len, nx * ny - lo);
    const int64_t p0 = a.n * chunk / a.chunks, p1 = a.n * (chunk + 1) / a.chunks;
    double x = 0.0, y = 0.0, w = 0.0;
    auto load = [&](int64_t k) {
        x = a.x[k];
        y = a.y[k];
        w = a.w ? a.w[k] : a.w0;
    };
    if (p0 + tid < p1) load(p0 + tid);
    for (int t = tid; t < len; t += DT) lds[t] = 0.0;
    __syncthreads();
    for (int64_t k = p0 + tid; k < p1; k += DT) {
        double fx, fy;
        int ci, cj;
        if (HOW == DEP_REF) {
            ci = ref_cell_s(x, a.dx, nx, K == PIC_CIC, fx);
            cj = ref_cell_s(y, a.dy, ny, K == PIC_CIC, fy);
        } else {
            const double px = (a.residues ? x : picd::jl_mod_pos(x - a.x0, a.dimx)) / a.dx;
            const double py = (a.residues ? y : picd::jl_mod_pos(y - a.y0, a.dimy)) / a.dy;
            ci = (int)px;
            cj = (int)py;
            fx = px - (double)ci;
            fy = py - (double)cj;
        }
        const double wk = w;
        if (k + DT < p1) load(k + DT);
        int col[S], row[S];
#pragma unroll
        for (int u = 0; u < S; ++u) {
            const int o = u - HL - (HOW == DEP_COMPAT && u != HL ? 1 : 0);
            col[u] = picd::wrap2(ci + o, nx);
            row[u] = picd::wrap2(cj + o, ny);
            // a position outside the domain (NaN, or one no call wrapped)
            // must not leave the grid
            if (HOW != DEP_REF) {
                col[u] = min(max(col[u], 0), nx - 1);
                row[u] = min(max(row[u], 0), ny - 1);
            }
            row[u] = row[u] * nx - lo;
        }
        charge64<K>(fx, fy, ci, cj, wk, [&](int u, int v, double q) {
            const int t = row[v] + col[u];
            if (SPLIT && (unsigned)t >= (unsigned)len) return;
            __hip_atomic_fetch_add(&lds[t], q, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
        });
    }
    __syncthreads();
    double *out = a.copies + (size_t)chunk * nx * ny + lo;
    for (int t = tid; t < len; t += DT) out[t] = lds[t];
}

// acc[t] = the copies' sum, W waves to 64 nodes, each taking every W-th chunk,
// the waves' sums added in order; *total = the sum of acc (each wave's nodes in
// order, a wave butterfly, then the waves and the blocks in a fixed order by the
// last block to arrive).  At most RD_BLOCKS blocks, which walk the grid: every
// block pays for its arrival, a fence and an atomic on one counter (measured on
// MI355X, 400 x 400 nodes: 73 us with a block per 64 nodes, whatever the number
// of copies).
constexpr int RD_T = 512, RD_BLOCKS = 256;
template <int W>
__global__ __launch_bounds__(RD_T) void k_deposit_reduce(const double *__restrict__ copies,
                                                         int chunks, int m,
                                                         double *__restrict__ acc, double *part,
                                                         unsigned *count, double *total) {
    constexpr int G = RD_T / 64 / W;  // groups of 64 nodes a block works at once
    __shared__ double sh[RD_T];
    __shared__ bool last;
    const int tid = threadIdx.x, lane = tid & 63, wv = tid >> 6, q = wv % W;
    double sum = 0.0;
    for (int g0 = blockIdx.x * G; g0 * 64 < m; g0 += gridDim.x * G) {
        const int t = (g0 + wv / W) * 64 + lane;
        double s = 0.0;
        if (t < m) {
#pragma unroll 8
            for (int b = q; b < chunks; b += W) s += copies[(size_t)b * m + t];
        }
        if (W > 1) {
            sh[tid] = s;
            __syncthreads();
            if (q == 0)
                for (int k = 1; k < W; ++k) s += sh[tid + 64 * k];
            __syncthreads();
        }
        if (q == 0 && t < m) {
            acc[t] = s;
            sum += s;
        }
    }
    for (int o = 32; o > 0; o >>= 1) sum += __shfl_xor(sum, o);
    if (lane == 0) sh[wv] = sum;
    __syncthreads();
    if (tid == 0) {
        for (int k = W; k < RD_T / 64; k += W) sum += sh[k];
        part[blockIdx.x] = sum;
        __threadfence();
        last = atomicAdd(count, 1u) == gridDim.x - 1;
    }
    __syncthreads();
    if (!last) return;
    __threadfence();
    sum = 0.0;
    for (int k = tid; k < (int)gridDim.x; k += RD_T)
        sum += __hip_atomic_load(&part[k], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    for (int o = 32; o > 0; o >>= 1) sum += __shfl_xor(sum, o);
    if (lane == 0) sh[wv] = sum;
    __syncthreads();
    if (tid == 0) {
        for (int k = 1; k < RD_T / 64; ++k) sum += sh[k];
        *total = sum;
        *count = 0u;
    }
}

// Residues back into the domain.
__global__ void k_residues_back(int64_t n, double *x, double *y, double x0, double y0) {
    const int64_t k = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (k >= n) return;
    x[k] += x0;
    y[k] += y0;
}

constexpr int DEP_PARTS_MAX = 8;

template <int K, int HOW>
int launch(Ctx *c, const DepArgs &a) {
    const size_t lds = (size_t)a.len * 8;
    auto go = [&](auto kern) -> int {
        PIC_HIP(hipFuncSetAttribute(reinterpret_cast<const void *>(kern),
                                    hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds));
        hipLaunchKernelGGL(kern, dim3((unsigned)(a.chunks * a.parts)), dim3(DT), lds, c->stream, a);
        PIC_HIP(hipGetLastError());
        return PIC_OK;
    };
    return a.parts == 1 ? go(k_deposit_lds<K, HOW, false>) : go(k_deposit_lds<K, HOW, true>);
}

int parts_of(const Ctx *c) {
    const int64_t m = (int64_t)c->nx * c->ny, room = (int64_t)(DEP_LDS / 8);
    return (int)std::min<int64_t>((m + room - 1) / room, DEP_PARTS_MAX + 1);
}

// One block per compute unit, and enough particles per thread that few of
// them do not pay for many copies of a large grid: measured on MI355X, 30,000
// particles on 400 x 400 nodes (eight parts), CIC and M6, 49.4 and 52.5 us with
// one per thread, 40.4 and 50.7 with four.
int chunks_of(const Ctx *c, int parts) {
    const int64_t per = DT * std::max(1, parts / 2);
    return (int)std::max<int64_t>(1, std::min<int64_t>((c->n + per - 1) / per, c->ncu / parts));
}

int deposit(Ctx *c, int kernel, int how, double x0, double y0, bool residues) {
    const int64_t m = (int64_t)c->nx * c->ny;
    DepArgs a;
    a.n = c->n;
    a.x = c->x;
    a.y = c->y;
    // the MeshFields deposits give every particle w0, as Particles.w is one
    // number (particles.jl:12-35), whatever the grid and so the kernel
    a.w = c->uniform_w || how != DEP_REF ? nullptr : c->w;
    a.w0 = c->w0;
    a.x0 = x0;
    a.y0 = y0;
    a.residues = residues;
    a.dimx = c->dimx;
    a.dimy = c->dimy;
    a.dx = c->dx;
    a.dy = c->dy;
    a.nx = c->nx;
    a.ny = c->ny;
    a.parts = parts_of(c);
    a.len = (int)((m + a.parts - 1) / a.parts);
    a.chunks = chunks_of(c, a.parts);
    a.copies = c->copies;
    int rc = PIC_OK;
    if (how == DEP_REF) {
        PIC_SHAPE_SWITCH(kernel, rc = (launch<KK, DEP_REF>(c, a)));
    } else if (how == DEP_MF) {
        rc = launch<PIC_M6, DEP_MF>(c, a);
    } else {
        rc = launch<PIC_M6, DEP_COMPAT>(c, a);
    }
    PIC_TRY(rc);
    double *part = c->copies + (size_t)a.chunks * m, *total = c->red_part + 2 * RED_BLOCKS;
    auto reduce = [&](auto kern, int w) {
        const int64_t per = RD_T / w;  // nodes a block takes at once
        const int64_t blocks = std::min<int64_t>((m + per - 1) / per, RD_BLOCKS);
        hipLaunchKernelGGL(kern, dim3((unsigned)blocks), dim3(RD_T), 0, c->stream,
                           (const double *)c->copies, a.chunks, (int)m, c->rho_acc, part,
                           c->red_count, total);
    };
    // More waves to a node read more copies at once but need more blocks.
    // Measured on MI355X, the whole call with CIC, us at 1 / 2 / 8 waves: 32 x 32
    // nodes and 30 copies 24.0 / 23.7 / 22.5, 64 x 64 and 59 25.9 / 25.0 / 24.5,
    // 100 x 100 and 63 29.5 / 27.8 / 28.8, 143 x 143 and 16 copies 27.4 / 27.1 /
    // 31.0, 256 x 256 and 64 39.3 / 42.1 / 46.6; 100 x 100 and 256 copies 44.9 /
    // 38.2 / 34.9, 143 x 143 and 256 49.3 / 43.5 / 47.9, 200 x 200 and 128 42.9 /
    // 43.2 / 47.0.
    if (m <= 10240 && a.chunks > (m <= 4096 ? 8 : 64)) reduce(k_deposit_reduce<8>, 8);
    else if (a.chunks > 64) reduce(k_deposit_reduce<2>, 2);
    else reduce(k_deposit_reduce<1>, 1);
    PIC_HIP(hipGetLastError());
    return shift_rho(c, kernel);
}

// The samples of the particles' order, a block each.
__global__ __launch_bounds__(256) void k_order(const double *__restrict__ x,
                                               const double *__restrict__ y, int64_t n, int nx,
                                               int ny, double dx, double dy, int64_t nch,
                                               Order *out) {
    const int s = blockIdx.x;
    picd::order_sample(out, s, s * nch / gridDim.x * STEP_CHUNK, n, nx, ny, dx, dy,
                       [&](int64_t k, double &a, double &b) {
                           a = x[k];
                           b = y[k];
                       });
}

}  // namespace

// Particles as a sort by cell left them, and as callers hand them back later,
// fill small boxes chunk by chunk, and the chunk kernels are then the faster
// ones.  So are they told from others by the chunks' extents: taken while
// particles are handed in, in the kernel that unpacks them, or by a kernel of
// their own when they are not known; a sort's order, and a verdict, are asked
// again after ORDER_MOVES moves.  A chunk whose stencils' box does not fit its
// tile pays for global atomics: one in sixteen of them may (for 2,000,000 M6
// particles 0.2 of 3.1 ms, as much as the LDS deposit takes).
// On grids of ORDER_ANY nodes and fewer the LDS deposit serves any order: measured on lane-sorted
// particles, chunk kernels and LDS, 10,000 CIC on 32 x 32 nodes 26 and 22 us,
// 300,000 M6 on 64 x 64 35 and 31 (sorted by cell alone 114 and 78); 300,000 CIC
// on 100 x 100 28 and 36.
int particles_near_order(Ctx *c, int kernel, bool *near) {
    *near = false;
    if ((int64_t)c->nx * c->ny <= ORDER_ANY) return PIC_OK;
    const int64_t nch = order_chunks(c->n);
    const int samples = (int)std::min<int64_t>(nch, ORDER_SAMPLES);
    if (c->order_known == Ctx::ORDER_UNKNOWN || c->order_moves >= ORDER_MOVES) {
        PIC_TRY(ensure_w_host(c));
        hipLaunchKernelGGL(k_order, dim3((unsigned)samples), dim3(256), 0, c->stream,
                           (const double *)c->x, (const double *)c->y, c->n, c->nx, c->ny, c->dx,
                           c->dy, nch, &c->w_host->order);
        PIC_HIP(hipGetLastError());
        PIC_HIP(hipStreamSynchronize(c->stream));
        c->order_known = Ctx::ORDER_JUDGED;
        c->order_moves = 0;
    }
    *near = true;
    if (c->order_known == Ctx::ORDER_SORTED) return PIC_OK;
    int span = 6;
    PIC_SHAPE_SWITCH(kernel, span = Shape<KK>::S);
    int far = 0;
    for (int s = 0; s < samples; ++s)
        far += (int64_t)(c->w_host->order.extent[s].x + span - 1) *
                   (c->w_host->order.extent[s].y + span - 1) > STEP_CAP64;
    *near = 16 * far <= samples;
    return PIC_OK;
}

int ensure_copies(Ctx *c, int64_t count) {
    if (count <= c->copies_cap) return PIC_OK;
    if (c->copies) (void)hipFree(c->copies);
    c->copies = nullptr;
    c->copies_cap = 0;
    PIC_HIP(hipMalloc(&c->copies, (size_t)count * 8));
    c->copies_cap = count;
    return PIC_OK;
}

bool deposit_lds_ok(Ctx *c) {
    const int parts = parts_of(c);
    if (c->n == 0 || parts > DEP_PARTS_MAX) return false;
    const int64_t m = (int64_t)c->nx * c->ny;
    if (ensure_copies(c, chunks_of(c, parts) * m + RD_BLOCKS) == PIC_OK) return true;
    (void)hipGetLastError();  // no room for the copies: the kernels without them
    return false;
}

// Against the chunk kernels on unsorted particles, measured on MI355X (the whole
// call): equal or faster from 300 particles on with M6, TSC and M4 and with CIC
// on up to six parts (30,000 on 300 x 300 nodes 35.0 against 37.7 us); on seven
// and eight, CIC's four shares a particle pay for the copies from about five
// particles to eight nodes on (400 x 400: 20,000 39.2 against 39.0, 50,000 44.2
// against 40.0, 100,000 46.9 against 48.1, 300,000 50.9 against 86.0).
bool deposit_lds_pays(Ctx *c, int kernel) {
    if (kernel == PIC_CIC && parts_of(c) > 6 && 8 * c->n < 5 * (int64_t)c->nx * c->ny) return false;
    return deposit_lds_ok(c);
}

int deposit_rho(Ctx *c, int kernel) { return deposit(c, kernel, DEP_REF, 0.0, 0.0, false); }

int deposit_rho_mf(Ctx *c, double x0, double y0, bool compat) {
    return deposit(c, PIC_M6, compat ? DEP_COMPAT : DEP_MF, x0, y0, false);
}

int deposit_rho_residues(Ctx *c) {
    PIC_TRY(deposit(c, PIC_M6, DEP_MF, 0.0, 0.0, true));
    if (c->n && (c->xmin != 0.0 || c->ymin != 0.0)) {
        hipLaunchKernelGGL(k_residues_back, dim3((unsigned)((c->n + 255) / 256)), dim3(256), 0,
                           c->stream, c->n, c->x, c->y, c->xmin, c->ymin);
        PIC_HIP(hipGetLastError());
    }
    return PIC_OK;
}

}  // namespace pic
