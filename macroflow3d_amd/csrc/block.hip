// Fused smoothing of the V-cycle's small levels, gfx950: up to two red-black
// Gauss-Seidel iterations (gsrb_3d.cu:29-366) with what precedes or follows them
// (prolongation; residual + restriction; PCG's (r, z)) in one launch.
//
// Bound: below about 64^3 cells a half-sweep's work is a microsecond and its
// launch, its first loads and its drain four, and a V(2,2) level is nine dependent
// launches. Here a workgroup loads a window of 16^3 cells, keeps it in LDS and
// registers, runs the half-sweeps with a barrier between them and stores the inner
// 8^3. Values at the window's rim lack neighbours and go wrong by one cell a
// half-sweep: four of them, or three and the residual (the first half-sweep from
// zero reads no neighbours), eat exactly the four rim cells. The recomputed rim is
// eight times the work, which is still cheaper than the launches while the windows
// fit the chip (kBlockMaxWindows, solver.hip).
//
// A thread owns a brick of 2 x 1 x 2 cells, two of each colour, so that every lane
// works in every half-sweep without divergence; the faces inside a brick are
// computed once and its own cells' values are read from registers, leaving four of
// a cell's six neighbours in LDS (stored by colour: conflict-free). The diagonal's
// reciprocal is taken once per cell and the quotients are corrected by their
// remainder. The kernel reads one copy of x and writes another: a window's rim is
// another window's inside. Per cell the FP32 sums are the half-sweep kernels'
// (gs_value) bit for bit, on every storage: colour-split or natural, stored faces
// or h = 1 / (2 K); the FP64 ones differ by the order of the x terms.
//
// MI355X, V(2,2) level in us, nine (16^3: three) launches before, two now:
//   FP32  64^3 36 -> 19   32^3 41 -> 12   16^3 28 -> 15
//   FP64  72x56x40 42 -> 36   32^3 with r update and (r, z) 37 -> 24   16^3 30 -> 15
// (a first version with a cell of each colour four times per thread and six LDS
// neighbours took 42, 20 and 21 in FP32: half the lanes idled in every half-sweep.)

#include <algorithm>
#include <type_traits>

#include "faces.hpp"
#include "reduce.hpp"
#include "split32.hpp"

namespace mf3d {
namespace {

constexpr int kW = 16, kRim = 4, kIn = kW - 2 * kRim;  // window, rim, stored cells per axis
constexpr int kThreads = kW * kW * kW / 4;
// LDS slots of a colour: x pair + 8 (y + 16 z), padded by a plane for the rim's reads
constexpr int kRow = kW / 2, kPlane = kRow * kW, kColour = kPlane * (kW + 2);

enum { START_ZERO = 0, START_PLAIN = 1, START_PROLONG = 2 };
enum { END_NONE = 0, END_RESTRICT = 1, END_RZ = 2 };

// the cells (i, i+1) x j x (k, k+1), i and k even; q: pair index (i / 2) + (nx / 2)
// (j + ny k). On plane s the cell of colour c sits at x position c ^ a(s).
struct Brick {
    int i, j, k, q;
    __device__ int a(int s) const { return (j + k + s) & 1; }
};
// Faces by plane s and colour c: between a plane's two cells, the other x face,
// y+, y-, between the planes (by the lower cell's colour), the other z face
template <typename T>
struct BFaces {
    T mid[2], out[2][2], yp[2][2], ym[2][2], zmid[2], zout[2][2];
};

__device__ __forceinline__ int split_index(int nx, int ny, int nz, int i, int j, int k) {
    const int h = nx >> 1;
    return ((i + j + k) & 1) * (h * ny * nz) + (i >> 1) + h * (j + ny * k);
}
__device__ __forceinline__ int natural_index(int nx, int ny, int i, int j, int k) {
    return i + nx * (j + ny * k);
}

// ---- storages: element type, index of a brick's cell, faces ---------------------
template <typename TC>
struct Split32 {  // FP32 colour-split level
    typedef float T;
    static constexpr bool kRedOnly = true;  // the residual's black cells vanish
    Dims d;
    SFaces<TC> F;
    __device__ int half() const { return (d.nx >> 1) * d.ny * d.nz; }
    __device__ int at(const Brick& b, int s, int c) const {
        return c * half() + b.q + s * (d.nx >> 1) * d.ny;
    }
    __device__ void faces(const BcTypes&, const Brick& b, BFaces<float>& f) const {
        const int h = d.nx >> 1, pl = h * d.ny, hf = half();
        const bool xu = b.i + 2 < d.nx, yu = b.j + 1 < d.ny, zu = b.k + 2 < d.nz;
#pragma unroll
        for (int s = 0; s < 2; ++s) {
            const int q = b.q + s * pl, a = b.a(s), k = b.k + s;
            // the pair's inner face belongs to its odd cell, of colour 1 ^ a
            f.mid[s] = cvt(F.lx[(1 ^ a) * hf + q]);
#pragma unroll
            for (int c = 0; c < 2; ++c) {
                const int own = c * hf + q, opp = (c ^ 1) * hf + q, pos = c ^ a;
                f.out[s][c] = cvt(!pos ? F.lx[own] : xu ? F.lx[opp + 1] : F.ux[b.j + d.ny * k]);
                f.ym[s][c] = cvt(F.ly[own]);
                f.yp[s][c] = cvt(yu ? F.ly[opp + h] : F.uy[b.i + pos + d.nx * k]);
                if (s == 0) {
                    f.zout[s][c] = cvt(F.lz[own]);
                    f.zmid[c] = cvt(F.lz[opp + pl]);
                } else {
                    f.zout[s][c] = cvt(zu ? F.lz[opp + pl] : F.uz[b.i + pos + d.nx * b.j]);
                }
            }
        }
    }
};
template <typename TT, typename TC>
struct Natural {  // natural order, faces on the MAC grid
    typedef TT T;
    static constexpr bool kRedOnly = false;
    Dims d;
    const TC* FX;
    const TC* FY;
    const TC* FZ;
    __device__ int at(const Brick& b, int s, int c) const {
        return 2 * (b.q + s * (d.nx >> 1) * d.ny) + (c ^ b.a(s));
    }
    __device__ void faces(const BcTypes&, const Brick& b, BFaces<T>& f) const {
        const int sy = d.nx * (d.ny + 1), sz = d.nx * d.ny;
#pragma unroll
        for (int s = 0; s < 2; ++s) {
            const int a = b.a(s), k = b.k + s;
            const int ox = b.i + (d.nx + 1) * (b.j + d.ny * k), oy = b.i + d.nx * b.j + sy * k,
                      oz = b.i + d.nx * b.j + sz * k;
            f.mid[s] = (T)cload(FX, ox + 1);
#pragma unroll
            for (int c = 0; c < 2; ++c) {
                const int pos = c ^ a;
                f.out[s][c] = (T)cload(FX, ox + 2 * pos);
                f.ym[s][c] = (T)cload(FY, oy + pos);
                f.yp[s][c] = (T)cload(FY, oy + pos + d.nx);
                f.zout[s][c] = (T)cload(FZ, oz + pos + s * sz);
                if (s == 0) f.zmid[c] = (T)cload(FZ, oz + pos + sz);
            }
        }
    }
};
struct Split64 {  // FP64 colour-split level, faces from h
    typedef double T;
    static constexpr bool kRedOnly = true;
    Dims d;
    const double* hs;
    __device__ int half() const { return (d.nx >> 1) * d.ny * d.nz; }
    __device__ int at(const Brick& b, int s, int c) const {
        return c * half() + b.q + s * (d.nx >> 1) * d.ny;
    }
    __device__ void faces(const BcTypes& bc, const Brick& b, BFaces<double>& f) const {
        const int h = d.nx >> 1, pl = h * d.ny, hf = half();
        // neighbours on the far side of a domain boundary are loaded wrapped and
        // used on a periodic axis only
        const bool xl = b.i > 0, xu = b.i + 2 < d.nx, yl = b.j > 0, yu = b.j + 1 < d.ny,
                   zl = b.k > 0, zu = b.k + 2 < d.nz;
        const int oxl = xl ? -1 : h - 1, oxu = xu ? 1 : 1 - h;
        const int oyl = yl ? -h : pl - h, oyu = yu ? h : h - pl;
        const int ozl = zl ? -pl : (d.nz - 1) * pl, ozu = zu ? pl : -(d.nz - 1) * pl;
        const Side sxl = side(xl, 0, bc.t[0], 0), sxu = side(xu, 0, bc.t[1], 0),
                   syl = side(yl, 0, bc.t[2], 0), syu = side(yu, 0, bc.t[3], 0),
                   szl = side(zl, 0, bc.t[4], 0), szu = side(zu, 0, bc.t[5], 0);
        double H[2][2], hx[2][2], hyl[2][2], hyu[2][2], hz[2][2];
#pragma unroll
        for (int s = 0; s < 2; ++s)
#pragma unroll
            for (int c = 0; c < 2; ++c) {
                const int q = b.q + s * pl, opp = (c ^ 1) * hf + q;
                H[s][c] = hs[c * hf + q];
                hx[s][c] = hs[opp + ((c ^ b.a(s)) ? oxu : oxl)];
                hyl[s][c] = hs[opp + oyl];
                hyu[s][c] = hs[opp + oyu];
                hz[s][c] = hs[opp + (s ? ozu : ozl)];
            }
#pragma unroll
        for (int s = 0; s < 2; ++s) {
            f.mid[s] = rcp_nr(H[s][0] + H[s][1]);
#pragma unroll
            for (int c = 0; c < 2; ++c) {
                const bool odd = (c ^ b.a(s)) != 0;
                const Side sx{0, odd ? sxu.nb : sxl.nb, odd ? sxu.face : sxl.face};
                f.out[s][c] = hface(sx, H[s][c], hx[s][c]);
                f.ym[s][c] = hface(syl, H[s][c], hyl[s][c]);
                f.yp[s][c] = hface(syu, H[s][c], hyu[s][c]);
                f.zout[s][c] = hface(s ? szu : szl, H[s][c], hz[s][c]);
                if (s == 0) f.zmid[c] = rcp_nr(H[0][c] + H[1][c ^ 1]);
            }
        }
    }
};

template <typename T>
struct BArgs {
    BcTypes bc;
    int pin, iters;
    int tx, ty, tz;  // windows
    T bs, rs;
    const T* xin;
    T* xout;
    const T* b;
    const T* xc;   // START_PROLONG: coarse correction
    T* bcoarse;    // END_RESTRICT
    int csplit;    // order of xc / bcoarse
    double* z;     // END_RZ: natural-order result instead of xout
    const double* r;
    double* partials;
};

// (FP32: eight waves per SIMD, two workgroups per CU)
template <class A, int START, int END>
__global__ void __launch_bounds__(kThreads, sizeof(typename A::T) == 4 ? 8 : 4)
    block_kernel(A st, BArgs<typename A::T> g) {
    typedef typename A::T T;
    constexpr bool F32 = sizeof(T) == 4;
    __shared__ T xs[2 * kColour];
    const long nblk = (long)g.tx * g.ty * g.tz;
    const int blk = (int)xcd_block(nblk);
    if (blk < 0) return;  // whole workgroup
    const int nx = st.d.nx, ny = st.d.ny, nz = st.d.nz;
    const int t = (int)threadIdx.x;
    // window coordinates of the brick and the domain's (before wrapping)
    const int P = t & 7, ly = (t >> 3) & 15, Z = t >> 7;
    const int i = blk % g.tx * kIn - kRim + 2 * P, j = blk / g.tx % g.ty * kIn - kRim + ly,
              k = blk / (g.tx * g.ty) * kIn - kRim + 2 * Z;
    // wrapped on a periodic axis; outside another one the brick is inactive (x = 0,
    // the ghost value of every boundary). Sizes are even, so bricks wrap whole and
    // keep their colours.
    bool act = true;
    auto coord = [&](int c, int n, int top, int type) {
        if (type == MF3D_BC_PERIODIC) return ((c % n) + n) % n;
        act = act && c >= 0 && c < n;
        return min(max(c, 0), top);
    };
    Brick B;
    B.i = coord(i, nx, nx - 2, g.bc.t[0]);
    B.j = coord(j, ny, ny - 1, g.bc.t[2]);
    B.k = coord(k, nz, nz - 2, g.bc.t[4]);
    B.q = (B.i >> 1) + (nx >> 1) * (B.j + ny * B.k);
    T bl[2][2], x[2][2];
    T add = T(0);  // the four cells share a parent
    if (START == START_PROLONG) {
        const int I = B.i >> 1, J = B.j >> 1, K = B.k >> 1;
        add = g.xc[g.csplit ? split_index(nx >> 1, ny >> 1, nz >> 1, I, J, K)
                            : natural_index(nx >> 1, ny >> 1, I, J, K)];
    }
#pragma unroll
    for (int s = 0; s < 2; ++s)
#pragma unroll
        for (int c = 0; c < 2; ++c) {
            const int o = st.at(B, s, c);
            bl[s][c] = g.b[o];
            x[s][c] = START != START_ZERO ? g.xin[o] : T(0);
        }
    BFaces<T> f;
    st.faces(g.bc, B, f);
    const int l0 = kPlane + P + kRow * (ly + kW * 2 * Z);  // plane s: l0 + s kPlane
#pragma unroll
    for (int s = 0; s < 2; ++s)
#pragma unroll
        for (int c = 0; c < 2; ++c) {
            if (START == START_PROLONG) x[s][c] += add;
            if (!act) x[s][c] = T(0);
            xs[c * kColour + l0 + s * kPlane] = x[s][c];
        }
    // f and neighbour values of a cell in the order of the sums: x+, x-, y+, y-, z+,
    // z- (FP64: the x terms as they come)
    auto coef = [&](int s, int c, T (&w)[6]) {
        const bool swap = F32 && (c ^ B.a(s));
        w[0] = swap ? f.out[s][c] : f.mid[s];
        w[1] = swap ? f.mid[s] : f.out[s][c];
        w[2] = f.yp[s][c];
        w[3] = f.ym[s][c];
        w[4] = s ? f.zout[s][c] : f.zmid[c];
        w[5] = s ? f.zmid[c ^ 1] : f.zout[s][c];
    };
    auto nbs = [&](int s, int c, T (&v)[6]) {
        const T* o = xs + (c ^ 1) * kColour + l0 + s * kPlane;
        const bool odd = (c ^ B.a(s)) != 0;
        const T m = x[s][c ^ 1], e = o[odd ? 1 : -1];
        v[0] = F32 && odd ? e : m;
        v[1] = F32 && odd ? m : e;
        v[2] = o[kRow];
        v[3] = o[-kRow];
        v[4] = s ? o[kPlane] : x[1][c ^ 1];
        v[5] = s ? x[0][c ^ 1] : o[-kPlane];
    };
    const bool pin0 = g.pin && act && B.q == 0;  // cell (0, 0, 0): plane 0, colour 0
    T dg[2][2], rd[2][2];
#pragma unroll
    for (int s = 0; s < 2; ++s)
#pragma unroll
        for (int c = 0; c < 2; ++c) {
            T w[6];
            coef(s, c, w);
            dg[s][c] = w[0] + w[1] + w[2] + w[3] + w[4] + w[5];
            if (s == 0 && c == 0 && pin0) dg[s][c] *= T(2);
            rd[s][c] = recip_of(dg[s][c]);
        }
    __syncthreads();
    for (int it = 0; it < g.iters; ++it) {
#pragma unroll
        for (int c = 0; c < 2; ++c) {
            if (act) {
#pragma unroll
                for (int s = 0; s < 2; ++s) {
                    T w[6], v[6];
                    T sum = T(0);
                    if (!(START == START_ZERO && c == 0 && it == 0)) {
                        coef(s, c, w);
                        nbs(s, c, v);
                        sum = v[0] * w[0];
#pragma unroll
                        for (int q = 1; q < 6; ++q) sum = fma(v[q], w[q], sum);
                    }
                    x[s][c] = quot_by(fma(-bl[s][c], g.bs, sum), dg[s][c], rd[s][c]);
                    xs[c * kColour + l0 + s * kPlane] = x[s][c];
                }
            }
            __syncthreads();
        }
    }
    // the inner cells, each owned by one window
    const bool mine = P >= kRim / 2 && P < (kW - kRim) / 2 && ly >= kRim && ly < kW - kRim &&
                      Z >= kRim / 2 && Z < (kW - kRim) / 2 && i < nx && j < ny && k < nz;
    if (END == END_RESTRICT) {
        // r = b - A x (smoother convention, residual_3d.cu:30-376); after a red-black
        // iteration the split levels take the black cells' as zero
        T r[2][2];
#pragma unroll
        for (int s = 0; s < 2; ++s)
#pragma unroll
            for (int c = 0; c < (A::kRedOnly ? 1 : 2); ++c) {
                T w[6], v[6];
                coef(s, c, w);
                nbs(s, c, v);
                T sum = w[0] * (x[s][c] - v[0]);
#pragma unroll
                for (int q = 1; q < 6; ++q) sum = fma(w[q], x[s][c] - v[q], sum);
                if (s == 0 && c == 0 && pin0)
                    sum = fma(w[0] + w[1] + w[2] + w[3] + w[4] + w[5], x[s][c], sum);
                r[s][c] = fma(sum, g.rs, bl[s][c]);
            }
        // a parent's eight children lie in this brick and the next row's, eight lanes up
        T sum = T(0);
#pragma unroll
        for (int s = 0; s < 2; ++s) {
            if (A::kRedOnly) {  // children (0,0,0), (1,1,0), (1,0,1), (0,1,1)
                sum += r[s][0];
                sum += __shfl_xor(r[s][0], 8);
            } else {
                const int a = B.a(s);
                const T e = a ? r[s][1] : r[s][0], o = a ? r[s][0] : r[s][1];
                sum += e;
                sum += o;
                sum += __shfl_xor(e, 8);
                sum += __shfl_xor(o, 8);
            }
        }
        if (mine && !(ly & 1)) {
            const int I = i >> 1, J = j >> 1, K = k >> 1;
            g.bcoarse[g.csplit ? split_index(nx >> 1, ny >> 1, nz >> 1, I, J, K)
                               : natural_index(nx >> 1, ny >> 1, I, J, K)] = sum / T(8);
        }
    }
    double acc = 0.0;
    if (mine) {
#pragma unroll
        for (int s = 0; s < 2; ++s) {
            if (END == END_RZ) {
                const int a = B.a(s), n = 2 * (B.q + s * (nx >> 1) * ny);
                const double e = (double)(a ? x[s][1] : x[s][0]), o = (double)(a ? x[s][0] : x[s][1]);
                *reinterpret_cast<double2*>(g.z + n) = make_double2(e, o);
                if (g.partials) {
                    const double2 rv = *reinterpret_cast<const double2*>(g.r + n);
                    acc += rv.x * e;
                    acc += rv.y * o;
                }
            } else {
#pragma unroll
                for (int c = 0; c < 2; ++c) g.xout[st.at(B, s, c)] = x[s][c];
            }
        }
    }
    if (END == END_RZ && g.partials) {  // uniform
        const double s = block_sum_dyn(acc);
        if (t == 0) g.partials[blk] = s;
    }
}

// r -= alpha Ap (skipped once stopped) with the (r, r) partials, and b = r in
// colour-split order (nx even): the windows read b at their rims, so the update cannot
// ride on them. One partial per 2048 cells.
template <bool UPD>
__global__ void __launch_bounds__(256) r_to_split64_kernel(Dims d, RUpd ru, double* __restrict__ b) {
    const long n = (long)d.nx * d.ny * d.nz, half = n >> 1;
    const bool go = UPD && !ru.st->stop;
    const double alpha = UPD ? ru.st->alpha : 0.0;
    double acc = 0.0;
#pragma unroll
    for (int u = 0; u < 4; ++u) {
        const long e = (long)blockIdx.x * 2048 + 512 * u + 2 * threadIdx.x;
        if (e >= n) continue;
        double2 rv = *reinterpret_cast<const double2*>(ru.r + e);
        if (go) {
            const double2 av = *reinterpret_cast<const double2*>(ru.Ap + e);
            rv.x = -alpha * av.x + rv.x;
            rv.y = -alpha * av.y + rv.y;
            *reinterpret_cast<double2*>(ru.r + e) = rv;
        }
        if (UPD) {
            acc += rv.x * rv.x;
            acc += rv.y * rv.y;
        }
        const unsigned row = (unsigned)((unsigned long)e / (unsigned)d.nx);
        const unsigned k = row / (unsigned)d.ny, j = row - k * (unsigned)d.ny;
        const long c0 = (j + k) & 1u;
        b[c0 * half + (e >> 1)] = rv.x;
        b[(c0 ^ 1) * half + (e >> 1)] = rv.y;
    }
    if (UPD) {
        const double s = block_sum<256>(acc);
        if (threadIdx.x == 0) ru.partials[blockIdx.x] = s;
    }
}

inline int windows(int n) { return (n + kIn - 1) / kIn; }

template <class A>
int launch(hipStream_t s, const A& a, const mf3d_grid& g, const kern::BlockPass<typename A::T>& p,
           const BcTypes& bc, bool pin) {
    typedef typename A::T T;
    BArgs<T> q{};
    q.bc = bc;
    q.pin = pin ? 1 : 0;
    q.iters = p.iters;
    q.tx = windows(g.nx), q.ty = windows(g.ny), q.tz = windows(g.nz);
    q.bs = (T)p.bs, q.rs = (T)p.rs;
    q.xin = p.xin, q.xout = p.xout, q.b = p.b, q.xc = p.xc, q.bcoarse = p.bcoarse;
    q.csplit = p.corder == ORDER_SPLIT;
    q.z = p.z, q.r = p.r, q.partials = p.partials;
    const unsigned nb = xcd_round((size_t)q.tx * q.ty * q.tz);
    if (p.iters < 1 || p.iters > 2 || (p.xin && p.xin == p.xout) ||
        (p.bcoarse && p.xin && p.iters > 1))
        return fail(MF3D_ERR_INVALID_ARGUMENT, "small-level pass: iterations or buffers");
    if (p.z && (!p.xin || !std::is_same<T, double>::value))
        return fail(MF3D_ERR_UNSUPPORTED, "small-level pass: z comes from FP64 post-smoothing");
    if (p.xc && p.bcoarse)
        return fail(MF3D_ERR_UNSUPPORTED, "small-level pass: both transfers");
    if (!p.xin) {
        if (p.bcoarse) block_kernel<A, START_ZERO, END_RESTRICT><<<nb, kThreads, 0, s>>>(a, q);
        else block_kernel<A, START_ZERO, END_NONE><<<nb, kThreads, 0, s>>>(a, q);
    } else if (p.bcoarse) {
        block_kernel<A, START_PLAIN, END_RESTRICT><<<nb, kThreads, 0, s>>>(a, q);
    } else if (p.z) {
        if constexpr (std::is_same<T, double>::value) {
            if (p.xc) block_kernel<A, START_PROLONG, END_RZ><<<nb, kThreads, 0, s>>>(a, q);
            else block_kernel<A, START_PLAIN, END_RZ><<<nb, kThreads, 0, s>>>(a, q);
        }
    } else if (p.xc) {
        block_kernel<A, START_PROLONG, END_NONE><<<nb, kThreads, 0, s>>>(a, q);
    } else {
        block_kernel<A, START_PLAIN, END_NONE><<<nb, kThreads, 0, s>>>(a, q);
    }
    MF3D_HIP_TRY(hipGetLastError());
    return MF3D_OK;
}

template <typename TC>
int launch32(hipStream_t s, const mf3d_grid& g, const BcTypes& bc, bool pin, const FaceSet& F,
             const kern::BlockPass<float>& p) {
    const Dims d{g.nx, g.ny, g.nz};
    if (F.split)
        return launch(s, Split32<TC>{d, SFaces<TC>{(const TC*)F.fx, (const TC*)F.fy,
                                                   (const TC*)F.fz, (const TC*)F.ux,
                                                   (const TC*)F.uy, (const TC*)F.uz}},
                      g, p, bc, pin);
    return launch(s, Natural<float, TC>{d, (const TC*)F.fx, (const TC*)F.fy, (const TC*)F.fz}, g, p,
                  bc, pin);
}

}  // namespace

namespace kern {

unsigned block_windows(const mf3d_grid& g) {
    return (unsigned)windows(g.nx) * (unsigned)windows(g.ny) * (unsigned)windows(g.nz);
}

int block_pass(hipStream_t s, const mf3d_grid& g, const BcTypes& bc, bool pin, const FaceSet& F,
               const BlockPass<float>& p) {
    switch (F.type) {
    case COEF_F32: return launch32<float>(s, g, bc, pin, F, p);
    case COEF_BF16: return launch32<__hip_bfloat16>(s, g, bc, pin, F, p);
    case COEF_F16: return launch32<__half>(s, g, bc, pin, F, p);
    default: return fail(MF3D_ERR_UNSUPPORTED, "FP32 smoothing needs 32- or 16-bit faces");
    }
}

int block_pass(hipStream_t s, const mf3d_grid& g, const BcTypes& bc, bool pin, const FaceSet& F,
               const double* hs, const BlockPass<double>& p) {
    const Dims d{g.nx, g.ny, g.nz};
    if (hs) return launch(s, Split64{d, hs}, g, p, bc, pin);
    if (F.type != COEF_F64) return fail(MF3D_ERR_UNSUPPORTED, "FP64 smoothing needs FP64 faces");
    return launch(s, Natural<double, double>{d, (const double*)F.fx, (const double*)F.fy,
                                             (const double*)F.fz}, g, p, bc, pin);
}

int r_to_split64(hipStream_t s, const mf3d_grid& g, const double* r, const RUpd* ru, double* b) {
    const Dims d{g.nx, g.ny, g.nz};
    const unsigned nb = (unsigned)((cells(g) + 2047) / 2048);
    if (ru) r_to_split64_kernel<true><<<nb, 256, 0, s>>>(d, *ru, b);
    else
        r_to_split64_kernel<false><<<nb, 256, 0, s>>>(
            d, RUpd{nullptr, nullptr, const_cast<double*>(r), nullptr}, b);
    MF3D_HIP_TRY(hipGetLastError());
    return MF3D_OK;
}

}  // namespace kern
}  // namespace mf3d
