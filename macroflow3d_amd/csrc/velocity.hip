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
#include <type_traits>

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
// neighbours' means. A workgroup owns 64 columns by 4, 8 or 16 rows (a wave a row; the
// first and last row only supply means unless the tile holds every row) and marches
// kz planes up: each thread forms its column's means from five loads a plane, two
// planes ahead of their use, keeps them for three planes (z differences) and shares
// plane k's through LDS (two buffers, one barrier a plane).
// Bound: HBM, the three padded components read once and the three cell fields
// written once, 48 bytes a cell. 250x190x130, with the statistics' second stage: with 17
// loads a cell and plane, each plane's waited for at once, 112 us; now 62 (the kernel
// 55, 5.4 TB/s). With ordinary stores, which push the velocities out of the Infinity
// Cache, 84.
constexpr int kDiagX = 64;
constexpr int kDiagQ = 9;  // per-workgroup partials: (min, max, sum) x 3 fields

struct Tiles {
    int tx, ty, kz;
    int rows;
    int halo;  // rows that only supply means, at either end: none where a tile needs none
    long nblocks;
    long steps;
};
// Tiles of `rows` rows and as many z-chunks as make the fewest steps with 16 waves a
// CU: one, two, ... rounds of workgroups, (planes of a chunk and two before the first
// step) each.
Tiles tiles_of_rows(int nx, int ny, int nz, int rows, bool curl) {
    Tiles best{};
    const int halo = curl && ny > rows ? 1 : 0, own = rows - 2 * halo;
    const int tx = (nx + kDiagX - 1) / kDiagX, ty = (ny + own - 1) / own;
    const long tiles = (long)tx * ty, flight = 256 * 16 / rows;
    for (long r = (tiles + flight - 1) / flight, c = 0; c < 32; ++r, ++c) {
        const int most = (int)std::min((long)nz, r * flight / tiles), kz = (nz + most - 1) / most;
        const long nb = tiles * ((nz + kz - 1) / kz);
        const long steps = (nb + flight - 1) / flight * (kz + 2);
        if (c == 0 || steps < best.steps) best = Tiles{tx, ty, kz, rows, halo, nb, steps};
        if (kz == 1) break;
    }
    return best;
}
// 8 rows, 6 of them stored, with two workgroups a CU; 16 where that saves over a sixth of
// the steps (it waits longer at its barriers and ends a launch in larger pieces); 4
// where they hold every row. With 16 always, us: 32^3 9.8 for 8.1, 512x512x16 57.9
// for 49.5, 250x190x130 66.5 for 62.3; with 8 always: 256^3 226 for 215, 1568x84x220 375
// for 335, 1000x14x600 88 for 76. 1024x1x1024 in 4, 8, 16: 26, 41, 72.
// Without the curl (a dimension below 3) nothing is shared between rows: 4.
Tiles tiles_of(int nx, int ny, int nz, bool curl) {
    if (ny <= 4 || !curl) return tiles_of_rows(nx, ny, nz, 4, curl);
    const Tiles t8 = tiles_of_rows(nx, ny, nz, 8, curl), t16 = tiles_of_rows(nx, ny, nz, 16, curl);
    return 6 * t16.steps < 5 * t8.steps ? t16 : t8;
}

struct DiagDims {
    int nx, ny, nz;
    Tiles t;
    double ix, iy, iz;
    bool curl;     // all dimensions >= 3
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

// one of min (0), max (1), sum (2)
__device__ __forceinline__ double mms_op(int kind, double a, double b) {
    return kind == 0 ? fmin(a, b) : kind == 1 ? fmax(a, b) : a + b;
}
// the value of the lane N places on in the row of 16 (rotated), by DPP
template <int N>
__device__ __forceinline__ double row_ror(double v) {
    const int2 u = __builtin_bit_cast(int2, v);
    return __builtin_bit_cast(
        double, int2{__builtin_amdgcn_update_dpp(0, u.x, 0x120 + N, 0xf, 0xf, false),
                     __builtin_amdgcn_update_dpp(0, u.y, 0x120 + N, 0xf, 0xf, false)});
}
__device__ __forceinline__ double row_mms(int kind, double v) {
    v = mms_op(kind, v, row_ror<8>(v));
    v = mms_op(kind, v, row_ror<4>(v));
    v = mms_op(kind, v, row_ror<2>(v));
    return mms_op(kind, v, row_ror<1>(v));
}
// min, max and sum of F fields over the workgroup of BS threads: out(q, v) for q = 3
// field + (0 min, 1 max, 2 sum), each from one thread. Rows of 16 lanes reduce by
// DPP, their values meet in LDS and the waves share the q's. (As wave-wide shuffles
// and a serial end, three fields of 1024 threads took about 6 us a workgroup, LDS
// bandwidth, as long as a thin tile's march.)
template <int BS, int F, typename Out>
__device__ __forceinline__ void block_mms(const MinMaxSum (&a)[F], Out&& out) {
    constexpr int E = BS / 16, W = BS / 64;
    static_assert(E <= 64, "a lane per row");
    __shared__ double wv[3 * F][E];
    const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
#pragma unroll
    for (int f = 0; f < F; ++f) {
        const double v[3] = {row_mms(0, a[f].lo), row_mms(1, a[f].hi), row_mms(2, a[f].sum)};
#pragma unroll
        for (int q = 0; q < 3; ++q)
            if (!(lane & 15)) wv[3 * f + q][threadIdx.x >> 4] = v[q];
    }
    __syncthreads();
    for (int q = w; q < 3 * F; q += W) {
        const int kind = q % 3;
        double v = kind == 0 ? __builtin_huge_val() : kind == 1 ? -__builtin_huge_val() : 0.0;
        if (lane < E) v = wv[q][lane];
        v = row_mms(kind, v);
        v = mms_op(kind, v, __shfl_xor(v, 16, 64));
        v = mms_op(kind, v, __shfl_xor(v, 32, 64));
        if (lane == 0) out(q, v);
    }
}

template <int ROWS, bool CURL>
__global__ void __launch_bounds__(kDiagX* ROWS, 4)
    diag_kernel(DiagDims d, const double* __restrict__ U, const double* __restrict__ V,
                const double* __restrict__ W, double* __restrict__ dv, double* __restrict__ om,
                double* __restrict__ he, double* __restrict__ partials) {
    constexpr int kRow = kDiagX + 2;
    constexpr int S = CURL ? ROWS : 1;
    __shared__ double mu[2][S][kRow], mv[2][S][kRow], mw[2][S][kRow];
    const long blk = xcd_block(d.t.nblocks);
    if (blk < 0) return;  // padding block: uniform exit before the barriers
    const long tiles = (long)d.t.tx * d.t.ty;
    const int tile = (int)(blk % tiles), chunk = (int)(blk / tiles);
    const int lane = (int)(threadIdx.x & 63), row = (int)(threadIdx.x >> 6);
    const int i = tile % d.t.tx * kDiagX + lane, j = tile / d.t.tx * (ROWS - 2 * d.t.halo) - d.t.halo + row;
    const int k0 = chunk * d.t.kz, k1 = min(k0 + d.t.kz, d.nz);
    const bool active = i < d.nx && j >= 0 && j < d.ny && row >= d.t.halo &&
                        row < ROWS - d.t.halo;
    // every load stays inside the padded arrays: columns clamped to the grid, planes
    // to [0, nz) (a clamped column's means are not used)
    const int ic = min(i, d.nx - 1), jc = min(max(j, 0), d.ny - 1);
    const bool colin = CURL && i >= 1 && i <= d.nx - 2 && j >= 1 && j <= d.ny - 2;
    const double hx = 0.5 * d.ix, hy = 0.5 * d.iy, hz = 0.5 * d.iz;
    // the columns beyond the tile: the left one for lanes 0..31, the right one for the
    // others, every lane loading so that all loads are in flight together
    const bool left = lane < kDiagX / 2, edge = lane == 0 || lane == kDiagX - 1;
    const int ie = min(max(i - lane + (left ? -1 : kDiagX), 0), d.nx - 1);
    const int eslot = left ? 0 : kRow - 1;
    const long sp = (long)(d.nx + 1) * (d.ny + 1);
    const long o = pad_idx(d, ic, jc, 0), oe = pad_idx(d, ie, jc, 0);
    const int yp = d.nx + 1;

    // the planes that are needed (others repeat the nearest one, unused): those either
    // side of the chunk for the curl's z differences only
    const int klo = CURL ? max(k0 - 1, 0) : k0, khi = CURL ? min(k1, d.nz - 1) : k1 - 1;

    struct Plane {  // plane k as loaded; w: of plane k + 1
        double ua, ub, va, vb, w, ea, eb, ew;
    };
    auto load = [&](int k) {
        k = min(max(k, klo), khi);
        const long q = sp * k, qw = sp * (k + 1);
        Plane p{U[q + o], U[q + o + 1], V[q + o], V[q + o + yp], W[qw + o]};
        if (CURL) p.ea = V[q + oe], p.eb = V[q + oe + yp], p.ew = W[qw + oe];
        return p;
    };
    double w0 = W[sp * k0 + o], ew0 = W[sp * k0 + oe];
    Plane below = load(k0 - 1), cur = load(k0), nxt = load(k0 + 1);
    double u0 = 0.5 * (below.ua + below.ub), v0 = 0.5 * (below.va + below.vb);

    MinMaxSum a[3];
    for (MinMaxSum& f : a) f.init();
    for (int k = k0; k < k1; ++k) {
        const Plane ahead = load(k + 2);
        const int buf = k & 1;
        const double uc = 0.5 * (cur.ua + cur.ub), vc = 0.5 * (cur.va + cur.vb),
                     wc = 0.5 * (w0 + cur.w);
        const double u2 = 0.5 * (nxt.ua + nxt.ub), v2 = 0.5 * (nxt.va + nxt.vb);
        if (CURL) {
            mu[buf][row][lane + 1] = uc;
            mv[buf][row][lane + 1] = vc;
            mw[buf][row][lane + 1] = wc;
            if (edge) {
                mv[buf][row][eslot] = 0.5 * (cur.ea + cur.eb);
                mw[buf][row][eslot] = 0.5 * (ew0 + cur.ew);
            }
            lds_barrier();
        }
        if (active) {
            const double divv = (cur.ub - cur.ua) * d.ix + (cur.vb - cur.va) * d.iy +
                                (cur.w - w0) * d.iz;
            double omv = 0.0, hev = 0.0;
            if (CURL && colin && k >= 1 && k <= d.nz - 2) {
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
                a[0].add(divv);
                a[1].add(omv);
                a[2].add(hev);
            }
        }
        u0 = uc, v0 = vc, w0 = cur.w, ew0 = cur.ew;
        cur = nxt, nxt = ahead;
    }
    if (!partials) return;  // uniform across the grid
    block_mms<kDiagX * ROWS>(a, [&](int q, double v) { partials[q * d.t.nblocks + blk] = v; });
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
    MinMaxSum a[1];
    a[0].init();
#pragma unroll
    for (int u = 0; u < kPer; ++u)
        if (base + (long)u * kBlock < n) a[0].add(v[u]);
    block_mms<kBlock>(a, [&](int q, double v) { partials[q * (long)gridDim.x + blockIdx.x] = v; });
}

// second stage, a workgroup per field with its (min, max, sum) partials of np blocks;
// out[3q..3q+2] = min, max, sum / n (fixed summation order)
__global__ void __launch_bounds__(kBlock)
    stats_final_kernel(const double* __restrict__ partials, long np, double n,
                       double* __restrict__ out) {
    const int q = (int)blockIdx.x;
    const double* lo = partials + (3 * q + 0) * np;
    const double* hi = partials + (3 * q + 1) * np;
    const double* sm = partials + (3 * q + 2) * np;
    MinMaxSum a[1];
    a[0].init();
    for (long b = threadIdx.x; b < np; b += kBlock) {
        a[0].lo = fmin(a[0].lo, lo[b]);
        a[0].hi = fmax(a[0].hi, hi[b]);
        a[0].sum += sm[b];
    }
    block_mms<kBlock>(a, [&](int e, double v) { out[3 * q + e] = e == 2 ? v / n : v; });
}

DiagDims diag_dims(const mf3d_grid& g) {
    DiagDims d{};
    d.nx = g.nx;
    d.ny = g.ny;
    d.nz = g.nz;
    d.curl = g.nx >= 3 && g.ny >= 3 && g.nz >= 3;
    d.t = tiles_of(g.nx, g.ny, g.nz, d.curl);
    d.ix = 1.0 / g.dx;
    d.iy = 1.0 / g.dy;
    d.iz = 1.0 / g.dz;
    return d;
}

}  // namespace

namespace kern {

size_t diag_partials(const mf3d_grid& g) { return (size_t)kDiagQ * diag_dims(g).t.nblocks; }

int velocity_diagnostics(hipStream_t s, const mf3d_grid& g, const double* U, const double* V,
                         const double* W, double* div, double* omag, double* hel,
                         double* partials, double* stats) {
    const DiagDims d = diag_dims(g);
    const unsigned nb = xcd_round((size_t)d.t.nblocks);
    double* const part = stats ? partials : nullptr;
    auto launch = [&](auto rows) {
        constexpr int R = decltype(rows)::value;
        diag_kernel<R, true><<<nb, kDiagX * R, 0, s>>>(d, U, V, W, div, omag, hel, part);
    };
    if (!d.curl)
        diag_kernel<4, false><<<nb, kDiagX * 4, 0, s>>>(d, U, V, W, div, omag, hel, part);
    else if (d.t.rows == 4) launch(std::integral_constant<int, 4>{});
    else if (d.t.rows == 8) launch(std::integral_constant<int, 8>{});
    else launch(std::integral_constant<int, 16>{});
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
