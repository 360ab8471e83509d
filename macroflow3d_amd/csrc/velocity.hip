// Darcy face velocities from head (FP64), gfx950.
//
// One launch covers every face, interior and boundary, in either layout: each
// thread owns cell (i,j,k) and writes its lower x-, y- and z-faces, plus the
// upper boundary face when the cell touches xmax/ymax/zmax. The reference
// launches 9 kernels on the legacy default stream and then syncs a different
// stream (src/physics/flow/velocity_from_head.cu:637-690); here everything is
// on the caller's stream.
//
// Formulas (velocity_from_head.cu:102-381):
//   interior face: q = -K_h (h_R - h_L) / dx, K_h = 2 Ka Kb / (Ka + Kb)
//   Dirichlet face: q = -K_C (h_in - h_bc) / (dx/2) (lower face),
//                   q = -K_C (h_bc - h_in) / (dx/2) (upper face)
//   Neumann face: 0; periodic face: harmonic mean across the wrap.

#include <algorithm>

#include "kernels.hpp"
#include "reduce.hpp"

namespace mf3d {
namespace {

constexpr int kBlock = 256;

__device__ inline double hmean_v(double a, double b) { return 2.0 * a * b / (a + b); }

struct FaceIdx {
    int nx, ny, nz;
    bool padded;
    __device__ long pidx(int i, int j, int k) const {
        return (long)k * (long)(ny + 1) * (long)(nx + 1) + (long)j * (long)(nx + 1) + (long)i;
    }
    __device__ long U(int i, int j, int k) const {
        return padded ? pidx(i, j, k) : (long)i + (long)(nx + 1) * ((long)j + (long)ny * k);
    }
    __device__ long V(int i, int j, int k) const {
        return padded ? pidx(i, j, k) : (long)i + (long)nx * ((long)j + (long)(ny + 1) * k);
    }
    __device__ long W(int i, int j, int k) const {
        return padded ? pidx(i, j, k) : (long)i + (long)nx * ((long)j + (long)ny * k);
    }
};

__global__ void __launch_bounds__(kBlock)
    velocity_kernel(FaceIdx fi, double dx, double dy, double dz, mf3d_bc bc,
                    const double* __restrict__ H, const double* __restrict__ K,
                    double* __restrict__ U, double* __restrict__ V, double* __restrict__ W) {
    const int nx = fi.nx, ny = fi.ny, nz = fi.nz;
    const long o = (long)blockIdx.x * blockDim.x + threadIdx.x;
    if (o >= (long)nx * ny * nz) return;
    const int i = (int)(o % nx);
    const long q = o / nx;
    const int j = (int)(q % ny);
    const int k = (int)(q / ny);
    const long sy = nx, sz = (long)nx * ny;
    const double Hc = H[o], Kc = K[o];

    // ---- x faces ----
    if (i > 0) {
        const long l = o - 1;
        U[fi.U(i, j, k)] = -hmean_v(K[l], Kc) * (Hc - H[l]) / dx;
    } else {  // kernel_U_west (velocity_from_head.cu:196-227)
        double u = 0.0;
        if (bc.type[0] == MF3D_BC_DIRICHLET) {
            u = -Kc * (Hc - bc.value[0]) / (dx * 0.5);
        } else if (bc.type[0] == MF3D_BC_PERIODIC) {
            const long w = o + (nx - 1);
            u = -hmean_v(K[w], Kc) * (Hc - H[w]) / dx;
        }
        U[fi.U(0, j, k)] = u;
    }
    if (i == nx - 1) {  // kernel_U_east (velocity_from_head.cu:232-258)
        double u = 0.0;
        if (bc.type[1] == MF3D_BC_DIRICHLET) {
            u = -Kc * (bc.value[1] - Hc) / (dx * 0.5);
        } else if (bc.type[1] == MF3D_BC_PERIODIC) {
            const long w = o - (nx - 1);
            u = -hmean_v(Kc, K[w]) * (H[w] - Hc) / dx;
        }
        U[fi.U(nx, j, k)] = u;
    }
    // ---- y faces ----
    if (j > 0) {
        const long s = o - sy;
        V[fi.V(i, j, k)] = -hmean_v(K[s], Kc) * (Hc - H[s]) / dy;
    } else {
        double v = 0.0;
        if (bc.type[2] == MF3D_BC_DIRICHLET) {
            v = -Kc * (Hc - bc.value[2]) / (dy * 0.5);
        } else if (bc.type[2] == MF3D_BC_PERIODIC) {
            const long w = o + (long)(ny - 1) * sy;
            v = -hmean_v(K[w], Kc) * (Hc - H[w]) / dy;
        }
        V[fi.V(i, 0, k)] = v;
    }
    if (j == ny - 1) {
        double v = 0.0;
        if (bc.type[3] == MF3D_BC_DIRICHLET) {
            v = -Kc * (bc.value[3] - Hc) / (dy * 0.5);
        } else if (bc.type[3] == MF3D_BC_PERIODIC) {
            const long w = o - (long)(ny - 1) * sy;
            v = -hmean_v(Kc, K[w]) * (H[w] - Hc) / dy;
        }
        V[fi.V(i, ny, k)] = v;
    }
    // ---- z faces ----
    if (k > 0) {
        const long b = o - sz;
        W[fi.W(i, j, k)] = -hmean_v(K[b], Kc) * (Hc - H[b]) / dz;
    } else {
        double w = 0.0;
        if (bc.type[4] == MF3D_BC_DIRICHLET) {
            w = -Kc * (Hc - bc.value[4]) / (dz * 0.5);
        } else if (bc.type[4] == MF3D_BC_PERIODIC) {
            const long t = o + (long)(nz - 1) * sz;
            w = -hmean_v(K[t], Kc) * (Hc - H[t]) / dz;
        }
        W[fi.W(i, j, 0)] = w;
    }
    if (k == nz - 1) {
        double w = 0.0;
        if (bc.type[5] == MF3D_BC_DIRICHLET) {
            w = -Kc * (bc.value[5] - Hc) / (dz * 0.5);
        } else if (bc.type[5] == MF3D_BC_PERIODIC) {
            const long t = o - (long)(nz - 1) * sz;
            w = -hmean_v(Kc, K[t]) * (H[t] - Hc) / dz;
        }
        W[fi.W(i, j, nz)] = w;
    }
}

// ---- velocity diagnostics (velocity_diagnostics.cu:46-177) -------------------
// Everything but the divergence is differences of cell-centred means (u: of the
// cell's two x faces, and so on), so a cell needs its own six faces and its
// neighbours' means. A workgroup owns 64 x 16 columns (a wave a row; rows 0 and 15
// only supply means: 64 x 14 cells a tile) and marches kz planes up: each thread
// forms its column's means from five loads a plane, two planes ahead of their use,
// keeps them for three planes (z differences) and shares plane k's through LDS (two
// buffers, one barrier a plane).
// Bound: HBM, the three padded components read once and the three cell fields
// written once, 48 bytes a cell. 250x190x130: with 17 loads a cell and plane, each
// plane's waited for at once, 105 us (2.8 TB/s); now 77 us (3.9 TB/s), 94 with
// ordinary stores, which push the velocities out of the Infinity Cache.
constexpr int kDiagX = 64, kDiagRows = 16, kDiagY = kDiagRows - 2;
constexpr int kDiagBlock = kDiagX * kDiagRows;
constexpr int kDiagQ = 9;  // per-workgroup partials: (min, max, sum) x 3 fields

// the number of z-chunks that makes the fewest steps with one workgroup a CU
struct Tiles {
    int tx, ty, kz;
    long nblocks;
};
Tiles tiles_of(int nx, int ny, int nz) {
    Tiles t{(nx + kDiagX - 1) / kDiagX, (ny + kDiagY - 1) / kDiagY, 0, 0};
    long best = -1;
    for (int c = 1; c <= nz; ++c) {
        const int kz = (nz + c - 1) / c, chunks = (nz + kz - 1) / kz;
        const long nb = (long)t.tx * t.ty * chunks;
        const long steps = (nb + 255) / 256 * (kz + 2);  // two planes before the first step
        if (best < 0 || steps < best) best = steps, t.kz = kz, t.nblocks = nb;
    }
    return t;
}

struct DiagDims {
    int nx, ny, nz;
    Tiles t;
    double ix, iy, iz;
    int curl;      // all dimensions >= 3
};

// padded_idx (src/physics/flow/padded_layout.cuh:30-33)
__device__ __forceinline__ long pad_idx(const DiagDims& d, int i, int j, int k) {
    return ((long)k * (d.ny + 1) + j) * (long)(d.nx + 1) + i;
}

struct MinMaxSum {
    double lo, hi, sum;
    __device__ void init() {
        lo = __builtin_huge_val();
        hi = -__builtin_huge_val();
        sum = 0.0;
    }
    __device__ void add(double v) {
        lo = fmin(lo, v);
        hi = fmax(hi, v);
        sum += v;
    }
};

// min, max and sum over the workgroup (BS threads), valid in thread 0;
// wv: LDS of 3 * BS / 64 doubles
template <int BS>
__device__ inline void block_mms(MinMaxSum& a, double* wv) {
#pragma unroll
    for (int off = 32; off > 0; off >>= 1) {
        a.lo = fmin(a.lo, __shfl_xor(a.lo, off, 64));
        a.hi = fmax(a.hi, __shfl_xor(a.hi, off, 64));
        a.sum += __shfl_xor(a.sum, off, 64);
    }
    constexpr int W = BS / 64;
    const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
    __syncthreads();  // wv may still be read by a previous call
    if (lane == 0) {
        wv[w] = a.lo;
        wv[W + w] = a.hi;
        wv[2 * W + w] = a.sum;
    }
    __syncthreads();
    if (threadIdx.x == 0) {
        for (int q = 1; q < W; ++q) {
            a.lo = fmin(a.lo, wv[q]);
            a.hi = fmax(a.hi, wv[W + q]);
        }
        double s = wv[2 * W];
        for (int q = 1; q < W; ++q) s += wv[2 * W + q];
        a.sum = s;
    }
}

__global__ void __launch_bounds__(kDiagBlock)
    diag_kernel(DiagDims d, const double* __restrict__ U, const double* __restrict__ V,
                const double* __restrict__ W, double* __restrict__ dv, double* __restrict__ om,
                double* __restrict__ he, double* __restrict__ partials) {
    constexpr int kRow = kDiagX + 2;
    __shared__ double mu[2][kDiagRows][kRow], mv[2][kDiagRows][kRow], mw[2][kDiagRows][kRow];
    const long blk = xcd_block(d.t.nblocks);
    if (blk < 0) return;  // padding block: uniform exit before the barriers
    const long tiles = (long)d.t.tx * d.t.ty;
    const int tile = (int)(blk % tiles), chunk = (int)(blk / tiles);
    const int lane = (int)(threadIdx.x & 63), row = (int)(threadIdx.x >> 6);
    const int i = tile % d.t.tx * kDiagX + lane, j = tile / d.t.tx * kDiagY - 1 + row;
    const int k0 = chunk * d.t.kz, k1 = min(k0 + d.t.kz, d.nz);
    const bool active = i < d.nx && j >= 0 && j < d.ny && row > 0 && row < kDiagRows - 1;
    // every load stays inside the padded arrays: columns clamped to the grid, planes
    // to [0, nz] (a clamped column's means are not used)
    const int ic = min(i, d.nx - 1), jc = min(max(j, 0), d.ny - 1);
    const bool colin = d.curl && i >= 1 && i <= d.nx - 2 && j >= 1 && j <= d.ny - 2;
    const double hx = 0.5 * d.ix, hy = 0.5 * d.iy, hz = 0.5 * d.iz;
    // the columns beyond the tile: the left one for lanes 0..31, the right one for the
    // others, every lane loading so that all loads are in flight together
    const bool left = lane < kDiagX / 2, edge = lane == 0 || lane == kDiagX - 1;
    const int ie = min(max(i - lane + (left ? -1 : kDiagX), 0), d.nx - 1);
    const int eslot = left ? 0 : kRow - 1;
    const long sp = (long)(d.nx + 1) * (d.ny + 1);
    const long o = pad_idx(d, ic, jc, 0), oe = pad_idx(d, ie, jc, 0);
    const int yp = d.nx + 1;

    struct Plane {  // plane k as loaded; w: of plane k + 1
        double ua, ub, va, vb, w, ea, eb, ew;
    };
    auto load = [&](int k) {
        const long q = sp * min(max(k, 0), d.nz), qw = sp * min(max(k + 1, 0), d.nz);
        return Plane{U[q + o], U[q + o + 1], V[q + o],       V[q + o + yp],
                     W[qw + o], V[q + oe],    V[q + oe + yp], W[qw + oe]};
    };
    double w0 = W[sp * k0 + o], ew0 = W[sp * k0 + oe];
    Plane below = load(k0 - 1), cur = load(k0), nxt = load(k0 + 1);
    double u0 = 0.5 * (below.ua + below.ub), v0 = 0.5 * (below.va + below.vb);

    MinMaxSum sd, so, sh;
    sd.init();
    so.init();
    sh.init();
    for (int k = k0; k < k1; ++k) {
        const Plane ahead = load(k + 2);  // (the chunk's last ones unused)
        const int buf = k & 1;
        const double uc = 0.5 * (cur.ua + cur.ub), vc = 0.5 * (cur.va + cur.vb),
                     wc = 0.5 * (w0 + cur.w);
        const double u2 = 0.5 * (nxt.ua + nxt.ub), v2 = 0.5 * (nxt.va + nxt.vb);
        mu[buf][row][lane + 1] = uc;
        mv[buf][row][lane + 1] = vc;
        mw[buf][row][lane + 1] = wc;
        if (edge) {
            mv[buf][row][eslot] = 0.5 * (cur.ea + cur.eb);
            mw[buf][row][eslot] = 0.5 * (ew0 + cur.ew);
        }
        lds_barrier();
        if (active) {
            const double divv = (cur.ub - cur.ua) * d.ix + (cur.vb - cur.va) * d.iy +
                                (cur.w - w0) * d.iz;
            double omv = 0.0, hev = 0.0;
            if (colin && k >= 1 && k <= d.nz - 2) {
                const double wx = (mw[buf][row + 1][lane + 1] - mw[buf][row - 1][lane + 1]) * hy -
                                  (v2 - v0) * hz;
                const double wy = (u2 - u0) * hz -
                                  (mw[buf][row][lane + 2] - mw[buf][row][lane]) * hx;
                const double wz = (mv[buf][row][lane + 2] - mv[buf][row][lane]) * hx -
                                  (mu[buf][row + 1][lane + 1] - mu[buf][row - 1][lane + 1]) * hy;
                omv = sqrt(wx * wx + wy * wy + wz * wz);
                hev = uc * wx + vc * wy + wc * wz;
            }
            const long c = (long)i + (long)d.nx * ((long)j + (long)d.ny * k);
            __builtin_nontemporal_store(divv, dv + c);
            __builtin_nontemporal_store(omv, om + c);
            __builtin_nontemporal_store(hev, he + c);
            if (partials) {
                sd.add(divv);
                so.add(omv);
                sh.add(hev);
            }
        }
        u0 = uc, v0 = vc, w0 = cur.w, ew0 = cur.ew;
        cur = nxt, nxt = ahead;
    }
    if (!partials) return;  // uniform across the grid
    __shared__ double wv[3 * kDiagBlock / 64];
    block_mms<kDiagBlock>(sd, wv);
    block_mms<kDiagBlock>(so, wv);
    block_mms<kDiagBlock>(sh, wv);
    if (threadIdx.x == 0) {
        const MinMaxSum* f[3] = {&sd, &so, &sh};
        for (int q = 0; q < 3; ++q) {
            partials[(3 * q + 0) * d.t.nblocks + blk] = f[q]->lo;
            partials[(3 * q + 1) * d.t.nblocks + blk] = f[q]->hi;
            partials[(3 * q + 2) * d.t.nblocks + blk] = f[q]->sum;
        }
    }
}

// compute_field_stats first stage (stochastic.cu:369-414): min, max and sum of
// 2048 consecutive values per workgroup (8 per thread, strided by kBlock);
// partials[q * nblocks + block] for q = min, max, sum
__global__ void __launch_bounds__(kBlock)
    stats_kernel(const double* __restrict__ x, long n, double* __restrict__ partials) {
    constexpr int kPer = 8;
    const long base = (long)blockIdx.x * kPer * kBlock + threadIdx.x;
    double v[kPer];
#pragma unroll
    for (int u = 0; u < kPer; ++u) v[u] = x[min(base + (long)u * kBlock, n - 1)];
    MinMaxSum a;
    a.init();
#pragma unroll
    for (int u = 0; u < kPer; ++u)
        if (base + (long)u * kBlock < n) a.add(v[u]);
    __shared__ double wv[3 * kBlock / 64];
    block_mms<kBlock>(a, wv);
    if (threadIdx.x == 0) {
        partials[blockIdx.x] = a.lo;
        partials[gridDim.x + blockIdx.x] = a.hi;
        partials[2 * (long)gridDim.x + blockIdx.x] = a.sum;
    }
}

// second stage, a workgroup per field with its (min, max, sum) partials of np blocks;
// out[3q..3q+2] = min, max, sum / n (fixed summation order)
__global__ void __launch_bounds__(kBlock)
    stats_final_kernel(const double* __restrict__ partials, long np, double n,
                       double* __restrict__ out) {
    __shared__ double wv[3 * kBlock / 64];
    const int q = (int)blockIdx.x;
    const double* lo = partials + (3 * q + 0) * np;
    const double* hi = partials + (3 * q + 1) * np;
    const double* sm = partials + (3 * q + 2) * np;
    MinMaxSum a;
    a.init();
    for (long b = threadIdx.x; b < np; b += kBlock) {
        a.lo = fmin(a.lo, lo[b]);
        a.hi = fmax(a.hi, hi[b]);
        a.sum += sm[b];
    }
    block_mms<kBlock>(a, wv);
    if (threadIdx.x == 0) {
        out[3 * q + 0] = a.lo;
        out[3 * q + 1] = a.hi;
        out[3 * q + 2] = a.sum / n;
    }
}

DiagDims diag_dims(const mf3d_grid& g) {
    DiagDims d{};
    d.nx = g.nx;
    d.ny = g.ny;
    d.nz = g.nz;
    d.t = tiles_of(g.nx, g.ny, g.nz);
    d.ix = 1.0 / g.dx;
    d.iy = 1.0 / g.dy;
    d.iz = 1.0 / g.dz;
    d.curl = g.nx >= 3 && g.ny >= 3 && g.nz >= 3;
    return d;
}

}  // namespace

namespace kern {

size_t diag_partials(const mf3d_grid& g) { return (size_t)kDiagQ * diag_dims(g).t.nblocks; }

int velocity_diagnostics(hipStream_t s, const mf3d_grid& g, const double* U, const double* V,
                         const double* W, double* div, double* omag, double* hel,
                         double* partials, double* stats) {
    const DiagDims d = diag_dims(g);
    diag_kernel<<<xcd_round((size_t)d.t.nblocks), kDiagBlock, 0, s>>>(d, U, V, W, div, omag, hel,
                                                                     stats ? partials : nullptr);
    MF3D_HIP_TRY(hipGetLastError());
    if (stats) {
        stats_final_kernel<<<3, kBlock, 0, s>>>(partials, d.t.nblocks, (double)cells(g), stats);
        MF3D_HIP_TRY(hipGetLastError());
    }
    return MF3D_OK;
}

size_t stats_partials(size_t n) { return 3 * ((n + 2047) / 2048); }

int field_stats(hipStream_t s, const double* x, size_t n, double* partials, double* out) {
    const long nb = (long)((n + 2047) / 2048);
    stats_kernel<<<(unsigned)nb, kBlock, 0, s>>>(x, (long)n, partials);
    MF3D_HIP_TRY(hipGetLastError());
    stats_final_kernel<<<1, kBlock, 0, s>>>(partials, nb, (double)n, out);
    MF3D_HIP_TRY(hipGetLastError());
    return MF3D_OK;
}

int velocity(hipStream_t s, const mf3d_grid& g, const mf3d_bc& bc, const double* h,
             const double* K, double* U, double* V, double* W, bool padded) {
    const size_t n = cells(g);
    FaceIdx fi{g.nx, g.ny, g.nz, padded};
    velocity_kernel<<<(unsigned)((n + kBlock - 1) / kBlock), kBlock, 0, s>>>(
        fi, g.dx, g.dy, g.dz, bc, h, K, U, V, W);
    MF3D_HIP_TRY(hipGetLastError());
    return MF3D_OK;
}

}  // namespace kern
}  // namespace mf3d
