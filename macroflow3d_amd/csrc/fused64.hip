// Fused smoothing passes of the FP64 V-cycle's large colour-split levels, gfx950.
//
// Two red-black Gauss-Seidel iterations (four half-sweeps, gsrb_3d.cu:29-366) with
// what precedes or follows them in the V-cycle (prolongation; residual +
// restriction; PCG's (r, z)) in ONE pass over the level, as fused32.hip does in
// FP32.
//
// Bound: one by one the half-sweeps stream 20 bytes a cell each (the other
// colour's x, b, h of both colours, the own x) at 4.9 TB/s, four of them and the
// residual 100 bytes. Fused, x, b and h cross HBM once: 21 bytes a cell for
// pre-smoothing + restriction, 29 for prolongation + post-smoothing. What bounds
// the pass instead is vector instructions: about 75 FP64 ones a cell, half of them
// for the faces (1 / (h_a + h_b)) and the diagonals' reciprocals.
//
// A workgroup owns a tile of 16 places x 32 rows (32 x 32 cells; a thread one
// place: a red and a black cell of each plane) and marches up in z, the half-sweeps
// pipelined over the planes: when plane k arrives, half-sweep s updates plane
// k - s. A cell's z neighbours are its own thread's values of adjacent planes
// (registers), its x partner the thread's other cell, and the three remaining
// neighbours lie in planes the previous step finished: values are exchanged through
// LDS with one barrier a step (two buffers in turn). The faces of a plane are
// formed once, a step after its h arrived (LDS, with a halo of one cell), and stay
// with b in registers until the last half-sweep, in a ring indexed at compile time
// by unrolling the march. 512 threads, so that a thread can hold them: two waves a
// SIMD, whose four half-sweeps are independent chains.
//
// Values at the tile's rim lack neighbours; a wrong value travels one cell a
// half-sweep, so the outer 2 places and 4 rows (and 4 or 5 planes around a z-chunk)
// are computed and dropped: 12 x 24 of 16 x 32 places are stored. The kernel reads
// one copy of x and writes another, since a tile's rim is another tile's interior.
// A red half-sweep reads black values only, so only those are read.
//
// A place outside the domain carries x = 0, the ghost value of every boundary, and
// the h that makes the boundary's face: 0 on a Dirichlet side (1 / h_C = 2 K_C),
// 1e300 on a Neumann side (a face of 1e-300, which vanishes in the sum).
//
// MI355X, 256^3: pre-smoothing + restriction 240 us and the r update before it 84
// (438 as half-sweeps, with the r update), prolongation + post-smoothing + (r, z) 237
// (327). 45 % of the vector issue slots are used; the rest waits on LDS and the
// chains of the quotients with two waves a SIMD. (One iteration a pass, 1024 threads,
// would stream 28 bytes a cell for the two half-sweeps' 40.)

#include <algorithm>
#include <type_traits>

#include "faces.hpp"
#include "reduce.hpp"
#include "split32.hpp"

namespace mf3d {
namespace {

constexpr int kTX = 16, kTY = 32;              // places x rows of a tile
constexpr int kHX = 2, kHY = 4;                // rim dropped on either side
constexpr int kIX = kTX - 2 * kHX, kIY = kTY - 2 * kHY;
constexpr int kThreads = kTX * kTY;
constexpr int kRow = kTX + 2, kSlots = kRow * (kTY + 2);  // LDS plane with its halo
constexpr int kHalo = 4 * kTX + 2 * kTY;       // h beyond the tile: 2 rows, 2 columns

enum { START_ZERO = 0, START_PROLONG = 1 };
enum { END_NONE = 0, END_RESTRICT = 1, END_RZ = 2 };

struct FGeo {
    int h, ny, nz;
    long half;
    int tx, ty;      // tiles
    int kz, chunks;  // planes per chunk (even)
};

// load / store at a 32-bit byte offset from a uniform base
template <typename T>
__device__ __forceinline__ T ldo(const void* base, unsigned byte) {
    return *reinterpret_cast<const T*>(static_cast<const char*>(base) + (size_t)byte);
}
template <typename T>
__device__ __forceinline__ void sto(void* base, unsigned byte, T v) {
    *reinterpret_cast<T*>(static_cast<char*>(base) + (size_t)byte) = v;
}

struct FArgs {
    BcTypes bc;
    int pin;
    double bs, rs;
    const double *xin, *b, *hs, *xc;
    double *xout, *bcoarse, *z, *partials;
};

template <int START, int END>
struct Fused64 {
    static constexpr bool XIN = START != START_ZERO;
    static constexpr int STAGES = 4;
    static constexpr int R = END == END_RESTRICT ? 8 : 6;  // ring: planes k .. k - R + 1
    // planes computed below a chunk: a stored value depends on 4 planes below (from
    // zero: 3, and the lowest plane's lower faces), the restricted residual on one more
    static constexpr int WARM = 4 + (END == END_RESTRICT ? 1 : 0);
    static constexpr int LAST = STAGES + (END == END_RESTRICT ? 1 : 0);
    static constexpr int AHEAD = 2;  // planes on their way
    // where the ring does not fit the registers (with a restriction it is a plane
    // longer), b and the red cells' y faces of planes k - 1 .. k - 5 wait in LDS (own
    // values, no barrier). With 34 of the 256 registers spilled instead, their reloads
    // waited for the planes on their way, and the pass took 417 us for 240.
    static constexpr bool PARK = END != END_RZ;
    static constexpr int kPark = 5;

    struct Lds {
        double x[STAGES + 1][2][kSlots];  // [s]: values half-sweep s left (0: black on arrival)
        double h[2][2][kSlots];           // [buffer][colour]
        double part[kThreads / 64];
        double ring[PARK ? 4 : 1][PARK ? kPark : 1][PARK ? kThreads : 1];
    };
    struct In {  // one plane on its way (b: of the plane below)
        double hr, hb, he, xb, par, br, bb;
    };

    static __device__ __forceinline__ void run(Lds& L, const FGeo& G, const FArgs& A, int bx,
                                               int by, int bz, long blk) {
        const int tid = (int)threadIdx.x;
        const int tx = tid & (kTX - 1), ty = tid / kTX;
        const int h = G.h, ny = G.ny, nz = G.nz;
        const int m0 = bx * kIX - kHX, j0 = by * kIY - kHY;
        const int m = m0 + tx, j = j0 + ty;
        const BcTypes& bc = A.bc;
        const bool px = bc.t[0] == MF3D_BC_PERIODIC, py = bc.t[2] == MF3D_BC_PERIODIC,
                   pz = bc.t[4] == MF3D_BC_PERIODIC;
        const int k0 = bz * G.kz, k1 = min(nz, k0 + G.kz);
        // a place in the domain: wrapped, or clamped with in = false; ghost: the h
        // that an outside place stands for
        auto wrap_x = [&](int a) { return px ? ((a % h) + h) % h : min(max(a, 0), h - 1); };
        auto wrap_y = [&](int a) { return py ? ((a % ny) + ny) % ny : min(max(a, 0), ny - 1); };
        auto in_xy = [&](int a, int c) {
            return (px || (unsigned)a < (unsigned)h) && (py || (unsigned)c < (unsigned)ny);
        };
        auto ghost_of = [&](int t) { return t == MF3D_BC_DIRICHLET ? 0.0 : 1e300; };
        auto ghost_xy = [&](int a, int c) {
            const int t = !px && a < 0 ? bc.t[0] : !px && a >= h ? bc.t[1] : c < 0 ? bc.t[2] : bc.t[3];
            return ghost_of(t);
        };
        const bool inside = in_xy(m, j);
        const double ghost = ghost_xy(m, j);
        const int mc = wrap_x(m), jc = wrap_y(j);
        const bool store = tx >= kHX && tx < kTX - kHX && ty >= kHY && ty < kTY - kHY && m < h &&
                           j < ny;
        const unsigned pl0 = (unsigned)mc + (unsigned)h * (unsigned)jc;
        const long half = G.half, hn = (long)h * ny;
        const long HC = half >> 3;  // one colour of the coarse level
        const unsigned hc = (unsigned)h >> 1, nyc = (unsigned)ny >> 1;
        // h beyond the tile, one value for each of the first kHalo threads: both
        // colours of the row below (0 .. 2 kTX) and above, then the odd cells of the
        // place to the left and the even ones to the right. (Every thread loads, so
        // that all waves have the same number of loads in flight.)
        const bool halo = tid < kHalo;
        const int e = tid & (kHalo - 1);
        const bool erow = e < 4 * kTX;
        const int ec = e - 4 * kTX;
        const int ex = erow ? e & (kTX - 1) : ec < kTY ? -1 : kTX;
        const int ey = erow ? (e < 2 * kTX ? -1 : kTY) : ec & (kTY - 1);
        const bool ein = in_xy(m0 + ex, j0 + ey);
        const double eghost = ghost_xy(m0 + ex, j0 + ey);
        const unsigned pe = (unsigned)wrap_x(m0 + ex) + (unsigned)h * (unsigned)wrap_y(j0 + ey);
        const int eslot = (ey + 1) * kRow + ex + 1;
        // colour of the halo cell on plane k: fixed in a row, by parity in a column
        // (position 1 to the left, 0 to the right)
        const int epar = (ec < kTY ? 1 : 0) + j0 + ey;
        auto ecol = [&](int k) { return erow ? (e / kTX) & 1 : (epar + k) & 1; };
        // the stored plane of a march index (-nz <= k < 2 nz), and whether it exists
        auto plane = [&](int k) {
            if (pz) return k < 0 ? k + nz : k >= nz ? k - nz : k;
            return min(max(k, 0), nz - 1);
        };
        auto kin = [&](int k) { return pz || (unsigned)k < (unsigned)nz; };

        // ring by plane: h, the faces of the red (r) and the black (b) cell (the one
        // between them, the outer x one, y+, y-, z-), b and x
        double hr[R], hb[R], mid[R], xor_[R], xob[R], yur[R], yub[R], ylr[R], ylb[R], zlr[R],
            zlb[R], br[R], bb[R], xr[R], xb[R];
#pragma unroll
        for (int q = 0; q < R; ++q) {
            hr[q] = hb[q] = mid[q] = xor_[q] = xob[q] = yur[q] = yub[q] = ylr[q] = ylb[q] = 0.0;
            zlr[q] = zlb[q] = br[q] = bb[q] = xr[q] = xb[q] = 0.0;
        }
        double acc = 0.0;
        double even = 0.0;  // END_RESTRICT: the pair of rows' residuals in the even plane

        int pk = 0;  // PARK: slot of plane k - 1
        In in[AHEAD];
        auto fetch = [&](In& n, int k) {
            const int kc = plane(k), kb = plane(k - 1);
            const double* hk = A.hs + hn * kc;
            n.hr = ldo<double>(hk, 8u * pl0);
            n.hb = ldo<double>(hk + half, 8u * pl0);
            n.he = hk[(ecol(k) ? half : 0L) + pe];
            const double* bk = A.b + hn * kb;
            n.br = ldo<double>(bk, 8u * pl0);
            n.bb = ldo<double>(bk + half, 8u * pl0);
            if (XIN) n.xb = ldo<double>(A.xin + half + hn * kc, 8u * pl0);
            if (XIN) {  // both cells of a place have parent (m, j/2, k/2)
                const unsigned J = (unsigned)jc >> 1, K = (unsigned)kc >> 1;
                const bool c = ((unsigned)mc + J + K) & 1u;
                n.par = A.xc[(c ? HC : 0L) + (long)hc * nyc * K + (((unsigned)mc >> 1) + hc * J)];
            }
        };

        const int kbeg = k0 - WARM, kend = k1 - 1 + LAST;
        fetch(in[0], kbeg);
        fetch(in[1], kbeg + 1);

        // one step: plane k arrives (ring slot U), half-sweep s updates plane k - s
        auto step = [&](auto uc, int k) {
            constexpr int U = decltype(uc)::value;
            auto sl = [](int back) constexpr { return (U - back + 2 * R) % R; };
            const int cur = k & 1, prv = cur ^ 1;
            In& nxt = in[U % AHEAD];
            const bool ki = kin(k);
            const double zghost = ghost_of(k < 0 ? bc.t[4] : bc.t[5]);
            hr[U] = !inside ? ghost : ki ? nxt.hr : zghost;
            hb[U] = !inside ? ghost : ki ? nxt.hb : zghost;
            double he = ein ? nxt.he : eghost;
            double br1 = nxt.br, bb1 = nxt.bb;
            if (PARK) pk = pk == kPark - 1 ? 0 : pk + 1;  // plane k - 1
            else br[sl(1)] = br1, bb[sl(1)] = bb1;
            xr[U] = xb[U] = 0.0;
            if (XIN) {
                xb[U] = inside && ki ? nxt.xb + nxt.par : 0.0;
            }
            // (all of the plane is waited for here, so that the number of younger loads
            // is known at compile time)
            asm volatile("" : "+v"(hr[U]), "+v"(hb[U]), "+v"(he), "+v"(xb[U]));
            asm volatile("" : "+v"(br1), "+v"(bb1));
            fetch(nxt, min(k + AHEAD, kend));
            const int at = (ty + 1) * kRow + tx + 1;
            L.h[cur][0][at] = hr[U];
            L.h[cur][1][at] = hb[U];
            if (halo) L.h[cur][ecol(k)][eslot] = he;
            if (XIN) L.x[0][cur][at] = xb[U];
            // p: which cell of the place half-sweep s updates in plane k - s (0: i = 2m)
            const int p = (j + k + 1) & 1;
            const int side = at + (p ? 1 : -1), other = at - (p ? 1 : -1);
            {  // the faces of plane k - 1, and those between it and plane k
                constexpr int a = sl(1);
                const double(&H)[2][kSlots] = L.h[prv];
                mid[a] = rcp_nr(hr[a] + hb[a]);
                xor_[a] = rcp_nr(hr[a] + H[1][side]);
                xob[a] = rcp_nr(hb[a] + H[0][other]);
                yur[a] = rcp_nr(hr[a] + H[1][at + kRow]);
                ylr[a] = rcp_nr(hr[a] + H[1][at - kRow]);
                if (PARK) {
                    L.ring[0][pk][tid] = br1;
                    L.ring[1][pk][tid] = bb1;
                    L.ring[2][pk][tid] = yur[a];
                    L.ring[3][pk][tid] = ylr[a];
                }
                yub[a] = rcp_nr(hb[a] + H[0][at + kRow]);
                ylb[a] = rcp_nr(hb[a] + H[0][at - kRow]);
                zlb[U] = rcp_nr(hb[U] + hr[a]);
                zlr[U] = rcp_nr(hr[U] + hb[a]);
            }
            // value w of plane k - back
            auto park = [&](int w, int back) {
                const int q = pk - (back - 1);
                return L.ring[w][PARK ? (q < 0 ? q + kPark : q) : 0][PARK ? tid : 0];
            };
            auto b_of = [&](int c, int back, double reg) {
                return !PARK ? reg : back == 1 ? (c ? bb1 : br1) : park(c, back);
            };
            // cell 0 or a wrapped copy of it
            auto pin0 = [&](int q) {
                return A.pin && (q == 0 || (pz && q == nz)) && p == 0 && pl0 == 0u && inside;
            };
            auto red_faces = [&](int a, int up, int back, double (&f)[6]) {
                f[0] = mid[a], f[1] = xor_[a], f[4] = zlb[up], f[5] = zlr[a];
                f[2] = PARK && back > 1 ? park(2, back) : yur[a];
                f[3] = PARK && back > 1 ? park(3, back) : ylr[a];
            };
            auto black_faces = [&](int a, int up, double (&f)[6]) {
                f[0] = mid[a], f[1] = xob[a], f[2] = yub[a], f[3] = ylb[a], f[4] = zlr[up],
                f[5] = zlb[a];
            };
            auto nbs = [&](int s, double own, double up, double down, double (&v)[6]) {
                v[0] = own;
                v[1] = L.x[s][prv][side];
                v[2] = L.x[s][prv][at + kRow];
                v[3] = L.x[s][prv][at - kRow];
                v[4] = up;
                v[5] = down;
            };
            auto gs = [&](const double (&f)[6], const double (&v)[6], bool zero, double b,
                          bool pinned) {
                double d = ((f[0] + f[1]) + (f[2] + f[3])) + (f[4] + f[5]);
                if (pinned) d *= 2.0;
                double n = 0.0;
                if (!zero) {
                    n = v[0] * f[0];
#pragma unroll
                    for (int q = 1; q < 6; ++q) n = fma(v[q], f[q], n);
                }
                return quot_by(fma(-b, A.bs, n), d, rcp_nr(d));
            };
            double f[6], v[6];
            if (kin(k - 1)) {  // 1: red of plane k - 1
                constexpr int a = sl(1), up = sl(0), dn = sl(2);
                red_faces(a, up, 1, f);
                if (XIN) nbs(0, xb[a], xb[up], xb[dn], v);
                const double x = gs(f, v, !XIN, PARK ? br1 : br[a], pin0(k - 1));
                xr[a] = inside ? x : 0.0;
                L.x[1][cur][at] = xr[a];
            }
            if (kin(k - 2)) {  // 2: black of plane k - 2
                constexpr int a = sl(2), up = sl(1), dn = sl(3);
                black_faces(a, up, f);
                nbs(1, xr[a], xr[up], xr[dn], v);
                const double x = gs(f, v, false, b_of(1, 2, bb[a]), false);
                xb[a] = inside ? x : 0.0;
                L.x[2][cur][at] = xb[a];
            }
            if (kin(k - 3)) {  // 3: red of plane k - 3
                constexpr int a = sl(3), up = sl(2), dn = sl(4);
                red_faces(a, up, 3, f);
                nbs(2, xb[a], xb[up], xb[dn], v);
                const double x = gs(f, v, false, b_of(0, 3, br[a]), pin0(k - 3));
                xr[a] = inside ? x : 0.0;
                L.x[3][cur][at] = xr[a];
            }
            if (kin(k - 4)) {  // 4: black of plane k - 4, which is then final
                constexpr int a = sl(4), up = sl(3), dn = sl(5);
                black_faces(a, up, f);
                nbs(3, xr[a], xr[up], xr[dn], v);
                const double x = gs(f, v, false, b_of(1, 4, bb[a]), false);
                xb[a] = inside ? x : 0.0;
                if (END == END_RESTRICT) L.x[4][cur][at] = xb[a];
                const int q = k - 4;
                if (store && q >= k0 && q < k1) {
                    if (END == END_RZ) {  // the black cell of plane k - 4 is at position p
                        *reinterpret_cast<double2*>(A.z + 2 * (hn * q + (long)pl0)) =
                            p ? make_double2(xr[a], xb[a]) : make_double2(xb[a], xr[a]);
                        acc += br[a] * xr[a];
                        acc += bb[a] * xb[a];
                    } else {
                        // (what follows a restriction starts from the black values alone)
                        if (END == END_NONE) sto(A.xout + hn * q, 8u * pl0, xr[a]);
                        sto(A.xout + half + hn * q, 8u * pl0, xb[a]);
                    }
                }
            }
            if (END == END_RESTRICT) {
                // residual of the red cell of plane k - 5 (the black ones' vanish after a
                // black half-sweep up to rounding) and the average over the coarse
                // cell's four red children: two rows (lanes kTX apart) of two planes
                constexpr int a = sl(5), up = sl(4), dn = sl(6);
                const int q = k - 5;
                red_faces(a, up, 5, f);
                nbs(4, xb[a], xb[up], xb[dn], v);
                const double x = xr[a];
                double s = f[0] * (x - v[0]);
#pragma unroll
                for (int w = 1; w < 6; ++w) s = fma(f[w], x - v[w], s);
                if (pin0(q)) s = fma(((f[0] + f[1]) + (f[2] + f[3])) + (f[4] + f[5]), x, s);
                const double res = fma(s, A.rs, b_of(0, 5, br[a]));
                const double oth = __shfl_xor(res, kTX, 64);
                if (!(q & 1)) {
                    even = res + oth;
                } else if (store && !(j & 1) && q > k0 && q < k1) {
                    const unsigned J = (unsigned)j >> 1, K = (unsigned)q >> 1;
                    const unsigned c = ((unsigned)m + J + K) & 1u;
                    A.bcoarse[(c ? HC : 0L) + (long)hc * nyc * K + (((unsigned)m >> 1) + hc * J)] =
                        ((even + res) + oth) / 8.0;
                }
            }
            lds_barrier();
        };
        for (int k = kbeg; k <= kend; k += R) {
            step(std::integral_constant<int, 0>{}, k);
            if (k + 1 > kend) break;
            step(std::integral_constant<int, 1>{}, k + 1);
            if (k + 2 > kend) break;
            step(std::integral_constant<int, 2>{}, k + 2);
            if (k + 3 > kend) break;
            step(std::integral_constant<int, 3>{}, k + 3);
            if (k + 4 > kend) break;
            step(std::integral_constant<int, 4>{}, k + 4);
            if (k + 5 > kend) break;
            step(std::integral_constant<int, 5>{}, k + 5);
            if constexpr (R > 6) {
                if (k + 6 > kend) break;
                step(std::integral_constant<int, 6>{}, k + 6);
                if (k + 7 > kend) break;
                step(std::integral_constant<int, 7>{}, k + 7);
            }
        }
        if (END == END_RZ && A.partials) {  // uniform
#pragma unroll
            for (int off = 32; off > 0; off >>= 1) acc += __shfl_xor(acc, off, 64);
            if ((tid & 63) == 0) L.part[tid >> 6] = acc;
            __syncthreads();
            if (tid == 0) {
                double s = 0.0;
                for (int w = 0; w < kThreads / 64; ++w) s += L.part[w];
                A.partials[blk] = s;
            }
        }
    }
};

template <int START, int END>
__global__ void __launch_bounds__(kThreads, 2) fused64_kernel(FGeo G, FArgs A) {
    __shared__ typename Fused64<START, END>::Lds L;
    const long blk = xcd_block((long)G.tx * G.ty * G.chunks);
    if (blk < 0) return;  // whole workgroup
    const int t = (int)(blk % ((long)G.tx * G.ty)), bz = (int)(blk / ((long)G.tx * G.ty));
    const int by = t / G.tx, bx = t - by * G.tx;
    Fused64<START, END>::run(L, G, A, bx, by, bz, blk);
}

constexpr int kExtra = 10;  // planes around a chunk
long steps_of(int tiles, int chunks, int kz) {
    return ((long)tiles * chunks + 255) / 256 * (kz + kExtra);
}

FGeo fgeo_of(const mf3d_grid& g) {
    FGeo G;
    G.h = g.nx / 2, G.ny = g.ny, G.nz = g.nz;
    G.half = (long)G.h * g.ny * g.nz;
    G.tx = (G.h + kIX - 1) / kIX;
    G.ty = (g.ny + kIY - 1) / kIY;
    // One workgroup runs on a CU at a time (its registers): as many chunks of planes
    // as make the fewest steps, (256 workgroups in flight) x (planes of a chunk and
    // the kExtra around it); more chunks read more rims, so only for a twentieth less
    long best = -1;
    for (int c = 1; c <= std::max(1, g.nz / 16); ++c) {
        const int kz = ((g.nz + c - 1) / c + 1) / 2 * 2, chunks = (g.nz + kz - 1) / kz;
        const long t = steps_of(G.tx * G.ty, chunks, kz);
        if (best < 0 || 20 * t < 19 * best) best = t, G.kz = kz, G.chunks = chunks;
    }
    return G;
}

}  // namespace

namespace kern {

// even sizes whose coarse level is even too (colour-split); planes beyond a periodic
// end at most one wrap away; 32-bit offsets within a plane
bool fused64_ok(const mf3d_grid& g) {
    return g.nx % 4 == 0 && g.ny % 4 == 0 && g.nz % 4 == 0 && g.nz >= 8 &&
           (size_t)g.nx * g.ny < ((size_t)1 << 28);
}

// A step takes 1.7 us; the half-sweeps, the residual and the transfers that the two
// passes replace take 41 ps a cell at 256^3 and nine launches (128^3: 115 us). Domains
// whose tiles end badly (1024x128x128: 43 x 6 of them, 210 steps, 350 us a pass for
// 250) stay with the half-sweeps.
bool fused64_pays(const mf3d_grid& g) {
    const FGeo G = fgeo_of(g);
    return steps_of(G.tx * G.ty, G.chunks, G.kz) <= (long)(cells(g) / 100000) + 10;
}

unsigned fused64_partials(const mf3d_grid& g) {
    const FGeo G = fgeo_of(g);
    return (unsigned)(G.tx * G.ty * G.chunks);
}

int fused64_pass(hipStream_t s, const mf3d_grid& g, const BcTypes& bc, bool pin,
                 const double* hs, const BlockPass<double>& p) {
    const bool pre = !p.xin && p.bcoarse && !p.xc && !p.z, post = p.xin && p.xc && !p.bcoarse;
    if (!fused64_ok(g) || p.iters != 2 || p.corder != ORDER_SPLIT || (!pre && !post) ||
        p.xin == p.xout)
        return fail(MF3D_ERR_UNSUPPORTED, "fused smoothing: sizes or combination");
    const FGeo G = fgeo_of(g);
    const FArgs a{bc, pin ? 1 : 0, p.bs, p.rs, p.xin, p.b, hs, p.xc, p.xout, p.bcoarse, p.z,
                  p.partials};
    const unsigned nb = xcd_round((size_t)G.tx * G.ty * G.chunks);
    if (pre) fused64_kernel<START_ZERO, END_RESTRICT><<<nb, kThreads, 0, s>>>(G, a);
    else if (p.z) fused64_kernel<START_PROLONG, END_RZ><<<nb, kThreads, 0, s>>>(G, a);
    else fused64_kernel<START_PROLONG, END_NONE><<<nb, kThreads, 0, s>>>(G, a);
    MF3D_HIP_TRY(hipGetLastError());
    return MF3D_OK;
}

}  // namespace kern
}  // namespace mf3d
