// Fused smoothing passes of the FP32 V-cycle's large colour-split levels, gfx950.
//
// Two red-black Gauss-Seidel iterations (four half-sweeps, gsrb_3d.cu:29-366)
// and what follows or precedes them in the V-cycle (v_cycle.cu:36-74: residual
// and restriction, or prolongation) in ONE pass over the level.
//
// Bound: the half-sweeps one by one stream the level's faces four times (12
// bytes a cell each, 48 together, and 12.5 more for the residual), and on
// levels beyond the caches HBM is what they wait for. Fused, a cell's faces, b
// and x cross HBM once: 12.5 bytes a cell for pre-smoothing + restriction,
// 16.5 for prolongation + post-smoothing. What bounds the fused pass instead is
// vector instructions (about 45 a half-sweep and cell).
//
// A workgroup owns a tile of 32 places x 32 rows (64 x 32 cells; a thread one
// place: a red and a black cell of each plane) and marches up in z, the
// half-sweeps pipelined over the planes: when plane k arrives, half-sweep s
// updates plane k - s. A cell's z neighbours are then its own thread's values
// of adjacent planes (registers), its x partner the thread's other cell, and
// the three remaining neighbours lie in planes the previous step finished, so
// values are exchanged through LDS with one barrier a step (two buffers in
// turn). Faces and b stay in registers for the five or six planes between
// arrival and last use, in a ring indexed at compile time by unrolling the
// march (shifting them instead would cost as much as a half-sweep).
//
// Values at the tile's rim lack neighbours; a wrong value travels one cell a
// half-sweep, so the outer 2 places and 4 rows (and 4 or 5 planes around a
// z-chunk) are computed and dropped: 28 x 24 of 32 x 32 places are stored. The
// kernel reads one copy of x and writes another, since a tile's rim is another
// tile's interior. Every stored value is the half-sweep kernels' bit for bit:
// same faces, same sums in the same order (gs_value).
//
// The level's faces are kept a second time for it (pack_faces): one 12-byte
// record per place with the red and the black cell's lower x, y and z faces in
// 16 bits each, on a grid one place, row and plane larger whose last ones hold
// the upper boundary's faces. A plane of faces is one load per thread at an
// offset that never changes (the plane moves the uniform base), boundaries
// included; with the six half-sweep arrays it was six loads and about 25 more
// vector instructions a step. b and the restricted residual are (red, black)
// pairs per place for the same reason.
//
// MI355X, bf16 faces, this pass against the half-sweeps (and residual) it replaces:
//   512^3 pre + restriction 702 us (1240), post 746 us (1286);
//   256^3 99 us (123), 86 us (124).
// About two thirds of the vector issue slots are used; at 512^3 the misses of the
// tiles' rims (1.4 times the bytes) take 4.8 TB/s.

#include <algorithm>
#include <type_traits>

#include "faces.hpp"
#include "reduce.hpp"
#include "split32.hpp"

namespace mf3d {
namespace {

constexpr int kTX = 32, kTY = 32;              // places x rows of a tile
constexpr int kHX = 2, kHY = 4;                // rim dropped on either side
constexpr int kIX = kTX - 2 * kHX, kIY = kTY - 2 * kHY;
constexpr int kThreads = kTX * kTY;
constexpr int kPadLds = kTX + 1;               // neighbours of the tile's rim read inside
constexpr int kSlots = kThreads + 2 * kPadLds;

enum { START_ZERO = 0, START_PROLONG = 1 };
enum { END_NONE = 0, END_RESTRICT = 1 };

struct FGeo {
    int h, ny, nz;
    long half;
    int tx, ty;      // tiles
    int kz, chunks;  // planes per chunk (even)
    int bcp;         // the coarse b: 1 (red, black) pairs, 0 colour by colour
};

// two 16-bit coefficients of one place (red low, black high)
template <typename TC>
struct FP {
    unsigned w;
    // the compiler must not keep the converted values of one half-sweep for the
    // next ones (twice the registers): hide that the word is the same
    __device__ void again() { asm("" : "+v"(w)); }
    __device__ float red() const {
        if (std::is_same<TC, __hip_bfloat16>::value) return __builtin_bit_cast(float, w << 16);
        return cvt(__builtin_bit_cast(TC, (unsigned short)(w & 0xffffu)));
    }
    __device__ float black() const {
        if (std::is_same<TC, __hip_bfloat16>::value)
            return __builtin_bit_cast(float, w & 0xffff0000u);
        return cvt(__builtin_bit_cast(TC, (unsigned short)(w >> 16)));
    }
};
struct Rec {  // lower x, y, z faces of a place
    unsigned x, y, z;
};

// load at a 32-bit byte offset from a uniform base
template <typename T>
__device__ __forceinline__ T ldo(const void* base, unsigned byte) {
    return *reinterpret_cast<const T*>(static_cast<const char*>(base) + (size_t)byte);
}
template <typename T>
__device__ __forceinline__ void sto(void* base, unsigned byte, T v) {
    *reinterpret_cast<T*>(static_cast<char*>(base) + (size_t)byte) = v;
}

template <typename TC, int START, int END>
struct Fused {
    static constexpr bool XIN = START == START_PROLONG;
    static constexpr int STAGES = 4;
    static constexpr int R = END == END_RESTRICT ? 8 : 6;  // ring: planes k .. k - R + 1
    // planes computed below a chunk: a stored value depends on 4 planes below
    // (START_ZERO: the first half-sweep reads no neighbours), the restricted
    // residual on one more
    static constexpr int WARM = (XIN ? 4 : 3) + (END == END_RESTRICT ? 1 : 0);
    static constexpr int LAST = STAGES + (END == END_RESTRICT ? 1 : 0);
    static constexpr int AHEAD = 2;  // planes on their way
    using F = FP<TC>;

    struct Lds {
        float x[STAGES + 1][2][kSlots];  // [s]: values half-sweep s left (0: black on arrival)
        F fx[2][kSlots + kTY], fy[2][kSlots];  // fx: then the column beyond the tile
    };

    struct In {  // one plane on its way
        Rec f;
        unsigned e;       // faces beyond the tile (END_RESTRICT)
        float2 b;
        float xb, par;
    };

    static __device__ __forceinline__ void run(Lds& L, const FGeo& G, const BcTypes& bc, int pin,
                                               float bs, float rs, const float* __restrict__ xin,
                                               float* __restrict__ xout,
                                               const float2* __restrict__ b,
                                               const Rec* __restrict__ faces,
                                               const float* __restrict__ xc,
                                               float* __restrict__ bcoarse, int bx, int by,
                                               int bz) {
        const int tid = (int)threadIdx.x;
        const int tx = tid & (kTX - 1), ty = tid / kTX;
        const int h = G.h, ny = G.ny, nz = G.nz;
        const int m = bx * kIX - kHX + tx, j = by * kIY - kHY + ty;
        const bool px = bc.t[0] == MF3D_BC_PERIODIC, py = bc.t[2] == MF3D_BC_PERIODIC,
                   pz = bc.t[4] == MF3D_BC_PERIODIC;
        const int k0 = bz * G.kz, k1 = min(nz, k0 + G.kz);
        // this thread's place in the domain: wrapped, or clamped with inside = false
        // (x = 0 there: the ghost value of every boundary face)
        const bool inside = (px || (m >= 0 && m < h)) && (py || (j >= 0 && j < ny));
        const int mc = px ? ((m % h) + h) % h : min(max(m, 0), h - 1);
        const int jc = py ? ((j % ny) + ny) % ny : min(max(j, 0), ny - 1);
        const bool store = tx >= kHX && tx < kTX - kHX && ty >= kHY && ty < kTY - kHY && m < h &&
                           j < ny;
        const unsigned pl0 = (unsigned)mc + (unsigned)h * (unsigned)jc;
        const long half = G.half, hn = (long)h * ny;
        const long HC = half >> 3;  // one colour of the coarse level
        const unsigned hc = (unsigned)h >> 1, nyc = (unsigned)ny >> 1;
        // face records: the place and row just beyond a non-periodic upper side
        // hold its boundary faces
        auto rec = [&](int mm, int jj) {
            const int a = px ? ((mm % h) + h) % h : min(max(mm, 0), h);
            const int c = py ? ((jj % ny) + ny) % ny : min(max(jj, 0), ny);
            return 12u * ((unsigned)a + (unsigned)(h + 1) * (unsigned)c);
        };
        const unsigned of = rec(m, j);
        const long fplane = (long)(h + 1) * (ny + 1);
        // END_RESTRICT is one half-sweep longer than the rim at the upper sides, where
        // the last place's and row's upper faces (lower faces of the next ones) are
        // already missing in the first: the first wave brings row 32's y faces (lanes
        // 0..31) and place 32's x faces (lanes 32..63). (Every wave loads, so that all
        // have the same number of loads in flight.)
        const bool extra = END == END_RESTRICT && tid < 2 * kTX;
        const bool ey = (tid & (2 * kTX - 1)) < kTX;
        const unsigned oe = ey ? rec(m, by * kIY - kHY + kTY) + 4u
                               : rec(bx * kIX - kHX + kTX, by * kIY - kHY + tx);
        // the stored plane of a march index (-nz <= k < 2 nz), and whether it exists
        auto plane = [&](int k) {
            if (pz) return k < 0 ? k + nz : k >= nz ? k - nz : k;
            return min(max(k, 0), nz - 1);
        };
        auto kin = [&](int k) { return pz || (unsigned)k < (unsigned)nz; };

        F lx[R], ly[R], lz[R], lyn[R];
        float lxn[R], br[R], bb[R], xr[R], xb[R];
#pragma unroll
        for (int q = 0; q < R; ++q) {
            lx[q] = ly[q] = lz[q] = lyn[q] = F{0u};
            lxn[q] = br[q] = bb[q] = xr[q] = xb[q] = 0.0f;
        }
        float even = 0.0f;  // END_RESTRICT: the pair of rows' residuals in the even plane

        In in[AHEAD];
        auto fetch = [&](In& n, int k) {
            const int kc = plane(k);
            const Rec* fk = faces + fplane * (!pz && k >= nz ? nz : kc);
            n.f = ldo<Rec>(fk, of);
            if (END == END_RESTRICT) n.e = ldo<unsigned>(fk, oe);
            n.b = ldo<float2>(b + hn * kc, 8u * pl0);
            if (XIN) n.xb = ldo<float>(xin + hn * kc, 4u * pl0);
            if (START == START_PROLONG) {  // both cells of a place have parent (m, j/2, k/2)
                const unsigned J = (unsigned)jc >> 1, K = (unsigned)kc >> 1;
                const bool c = ((unsigned)mc + J + K) & 1u;
                n.par = ldo<float>(xc + (long)hc * nyc * K,
                                   4u * ((c ? (unsigned)HC : 0u) + ((unsigned)mc >> 1) + hc * J));
            }
        };

        const int kbeg = k0 - WARM, kend = k1 - 1 + LAST;
        fetch(in[0], kbeg);
        if (AHEAD > 1) fetch(in[AHEAD - 1], kbeg + 1);

        // one step: plane k arrives (ring slot U), half-sweep s updates plane k - s
        auto step = [&](auto uc, int k) {
            constexpr int U = decltype(uc)::value;
            auto sl = [](int back) constexpr { return (U - back + 2 * R) % R; };
            const int cur = k & 1, prv = cur ^ 1;
            // arrival (later planes' loads go out before anything is computed)
            In& nxt = in[U % AHEAD];
            // Every value of the plane is waited for here, and a later plane is
            // requested on every path (the last one again): the number of younger
            // loads is then known at compile time. Left to their first uses,
            // half-sweeps later, the waits came out as "all loads done".
            lx[U].w = nxt.f.x, ly[U].w = nxt.f.y, lz[U].w = nxt.f.z;
            br[U] = nxt.b.x, bb[U] = nxt.b.y;
            xr[U] = xb[U] = 0.0f;
            if (XIN) {
                const float v = START == START_PROLONG ? nxt.xb + nxt.par : nxt.xb;
                xb[U] = inside && kin(k) ? v : 0.0f;
            }
            unsigned ext = 0u;
            if (END == END_RESTRICT) {
                ext = nxt.e;
                asm volatile("" : "+v"(ext));
            }
            asm volatile("" : "+v"(lx[U].w), "+v"(ly[U].w), "+v"(lz[U].w));
            asm volatile("" : "+v"(br[U]), "+v"(bb[U]), "+v"(xb[U]));
            fetch(nxt, min(k + AHEAD, kend));
            const int at = tid + kPadLds;
            L.fx[cur][at] = lx[U];
            L.fy[cur][at] = ly[U];
            if (END == END_RESTRICT && extra)
                (ey ? L.fy[cur][kPadLds + kThreads + tid] : L.fx[cur][kSlots + tid - kTX]) =
                    F{ext};
            if (XIN) L.x[0][cur][at] = xb[U];
            // p: which cell of the place half-sweep s updates in plane k - s (0: i = 2m)
            const int p = (j + k + 1) & 1;
            const int side = at + (p ? 1 : -1);
            {  // plane k - 1: the neighbours' faces (x+ of the place, y+)
                const F fn = L.fx[prv][END == END_RESTRICT && tx == kTX - 1 ? kSlots + ty : at + 1];
                lxn[sl(1)] = p ? fn.black() : fn.red();
                lyn[sl(1)] = L.fy[prv][at + kTX];
            }
            // cell 0 or a wrapped copy of it
            auto pin0 = [&](int q) {
                return pin && (q == 0 || (pz && q == nz)) && p == 0 && pl0 == 0u && inside;
            };
            auto red_faces = [&](int a, int up, float (&f)[6]) {
                lx[a].again(), ly[a].again(), lz[a].again(), lyn[a].again(), lz[up].again();
                f[0] = p ? lxn[a] : lx[a].black();
                f[1] = lx[a].red();
                f[2] = lyn[a].black();
                f[3] = ly[a].red();
                f[4] = lz[up].black();
                f[5] = lz[a].red();
            };
            auto black_faces = [&](int a, int up, float (&f)[6]) {
                lx[a].again(), ly[a].again(), lz[a].again(), lyn[a].again(), lz[up].again();
                f[0] = p ? lxn[a] : lx[a].red();
                f[1] = lx[a].black();
                f[2] = lyn[a].red();
                f[3] = ly[a].black();
                f[4] = lz[up].red();
                f[5] = lz[a].black();
            };
            auto nbs = [&](int s, float own, float up, float down, float (&v)[6]) {
                const float o = L.x[s][prv][side];
                v[0] = p ? o : own;
                v[1] = p ? own : o;
                v[2] = L.x[s][prv][at + kTX];
                v[3] = L.x[s][prv][at - kTX];
                v[4] = up;
                v[5] = down;
            };
            float f[6], v[6];
            if (kin(k - 1)) {  // 1: red of plane k - 1
                constexpr int a = sl(1), up = sl(0), dn = sl(2);
                red_faces(a, up, f);
                if (XIN) {
                    nbs(0, xb[a], xb[up], xb[dn], v);
                } else {
#pragma unroll
                    for (int q = 0; q < 6; ++q) v[q] = 0.0f;
                }
                const float x = gs_value(f, v, br[a], bs, pin0(k - 1));
                xr[a] = inside ? x : 0.0f;
                L.x[1][cur][at] = xr[a];
            }
            if (kin(k - 2)) {  // 2: black of plane k - 2
                constexpr int a = sl(2), up = sl(1), dn = sl(3);
                black_faces(a, up, f);
                nbs(1, xr[a], xr[up], xr[dn], v);
                const float x = gs_value(f, v, bb[a], bs, false);
                xb[a] = inside ? x : 0.0f;
                L.x[2][cur][at] = xb[a];
            }
            if (kin(k - 3)) {  // 3: red of plane k - 3
                constexpr int a = sl(3), up = sl(2), dn = sl(4);
                red_faces(a, up, f);
                nbs(2, xb[a], xb[up], xb[dn], v);
                const float x = gs_value(f, v, br[a], bs, pin0(k - 3));
                xr[a] = inside ? x : 0.0f;
                L.x[3][cur][at] = xr[a];
            }
            if (kin(k - 4)) {  // 4: black of plane k - 4, which is then final
                constexpr int a = sl(4), up = sl(3), dn = sl(5);
                black_faces(a, up, f);
                nbs(3, xr[a], xr[up], xr[dn], v);
                const float x = gs_value(f, v, bb[a], bs, false);
                xb[a] = inside ? x : 0.0f;
                if (END == END_RESTRICT) L.x[4][cur][at] = xb[a];
                const int q = k - 4;
                if (store && q >= k0 && q < k1) {
                    // (post-smoothing starts from the black values alone)
                    if (XIN) {
                        sto(xout + hn * q, 4u * pl0, xr[a]);
                        sto(xout + half + hn * q, 4u * pl0, xb[a]);
                    } else {
                        sto(xout + hn * q, 4u * pl0, xb[a]);
                    }
                }
            }
            if (END == END_RESTRICT) {
                // residual of the red cell of plane k - 5 (the black ones' vanish after a
                // black half-sweep up to rounding) and the average over the coarse
                // cell's four red children: two rows (lanes 32 apart) of two planes
                constexpr int a = sl(5), up = sl(4), dn = sl(6);
                const int q = k - 5;
                red_faces(a, up, f);
                nbs(4, xb[a], xb[up], xb[dn], v);
                const float x = xr[a];
                float s = f[0] * (x - v[0]);  // fma as in gs_value
                s = fma(f[1], x - v[1], s);
                s = fma(f[2], x - v[2], s);
                s = fma(f[3], x - v[3], s);
                s = fma(f[4], x - v[4], s);
                s = fma(f[5], x - v[5], s);
                if (pin0(q)) s = fma(f[0] + f[1] + f[2] + f[3] + f[4] + f[5], x, s);
                const float res = fma(s, rs, br[a]);
                const float other = __shfl_xor(res, 32, 64);
                if (!(q & 1)) {
                    even = res + other;
                } else if (store && !(j & 1) && q > k0 && q < k1) {
                    const unsigned J = (unsigned)j >> 1, K = (unsigned)q >> 1;
                    const unsigned c = ((unsigned)m + J + K) & 1u;
                    const long pc = (long)(((unsigned)m >> 1) + hc * (J + nyc * K));
                    bcoarse[G.bcp ? 2 * pc + c : (c ? HC : 0L) + pc] =
                        ((even + res) + other) / 8.0f;
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
    }
};

template <typename TC, int START, int END>
__global__ void __launch_bounds__(kThreads)
    fused_kernel(FGeo G, BcTypes bc, int pin, float bs, float rs, const float* __restrict__ xin,
                 float* __restrict__ xout, const float2* __restrict__ b,
                 const Rec* __restrict__ faces, const float* __restrict__ xc,
                 float* __restrict__ bcoarse) {
    __shared__ typename Fused<TC, START, END>::Lds L;
    const long blk = xcd_block((long)G.tx * G.ty * G.chunks);
    if (blk < 0) return;  // whole workgroup
    const int t = (int)(blk % ((long)G.tx * G.ty)), bz = (int)(blk / ((long)G.tx * G.ty));
    const int by = t / G.tx, bx = t - by * G.tx;
    Fused<TC, START, END>::run(L, G, bc, pin, bs, rs, xin, xout, b, faces, xc, bcoarse, bx, by, bz);
}

// face records of a level from its half-sweep arrays
template <typename TC>
__global__ void __launch_bounds__(256)
    pack_faces_kernel(Dims d, SFaces<TC> F, Rec* __restrict__ out) {
    const int h = d.nx >> 1;
    const long total = (long)(h + 1) * (d.ny + 1) * (d.nz + 1);
    const long t = (long)blockIdx.x * 256 + threadIdx.x;
    if (t >= total) return;
    const unsigned row = (unsigned)(t / (h + 1));
    const int m = (int)(t - (long)row * (h + 1));
    const int k = (int)(row / (unsigned)(d.ny + 1)), j = (int)(row - (unsigned)k * (d.ny + 1));
    const long half = (long)h * d.ny * d.nz;
    const long pl = (long)m + (long)h * ((long)j + (long)d.ny * k);
    const int odd = (j + k) & 1;  // 1: the place's second cell is red
    auto bits = [](TC v) { return (unsigned)__builtin_bit_cast(unsigned short, v); };
    auto two = [&](TC r, TC b) { return bits(r) | (bits(b) << 16); };
    const bool im = m < h, ij = j < d.ny, ik = k < d.nz;
    Rec o{0u, 0u, 0u};
    if (ij && ik) {
        // beyond the row both halves hold the boundary face (the reader takes one)
        const TC u = F.ux[j + (long)d.ny * k];
        o.x = im ? two(F.lx[pl], F.lx[half + pl]) : two(u, u);
    }
    if (im && ik) {
        const long u = 2L * m + (long)d.nx * k;
        o.y = ij ? two(F.ly[pl], F.ly[half + pl]) : two(F.uy[u + odd], F.uy[u + 1 - odd]);
    }
    if (im && ij) {
        const long u = 2L * m + (long)d.nx * j;
        o.z = ik ? two(F.lz[pl], F.lz[half + pl]) : two(F.uz[u + odd], F.uz[u + 1 - odd]);
    }
    out[t] = o;
}

// b = (float) r as (red, black) pairs of a place. UPD: r -= alpha Ap first, in
// place (pcg_update_r_kernel's form, skipped once stopped), with the (r, r)
// partials; the fused pass that follows reads b at its tiles' rims too, so it
// could not update r itself. Pairs (2m, 2m + 1) of a row, 64 in a row per wave
// and access; a workgroup covers 2048 cells. Streams 28 bytes a cell: 512^3
// 578 us (6.5 TB/s).
template <bool UPD>
__global__ void __launch_bounds__(256)
    r_to_b_kernel(Dims d, RUpd ru, float2* __restrict__ b) {
    const long n = (long)d.nx * d.ny * d.nz;
    const long nb = (n + 2047) / 2048;
    const long blk = xcd_block(nb);
    if (blk < 0) return;
    const long e0 = blk * 2048 + (long)(threadIdx.x >> 6) * 512 + 2L * (threadIdx.x & 63);
    const bool go = UPD && !ru.st->stop;
    const double alpha = UPD ? ru.st->alpha : 0.0;
    double2 rv[4], av[4];
#pragma unroll
    for (int u = 0; u < 4; ++u) {
        const long e = min(e0 + 128L * u, n - 2);
        rv[u] = ldnt(ru.r + e);
        if (UPD) av[u] = ldnt(ru.Ap + e);
    }
    double acc = 0.0;
#pragma unroll
    for (int u = 0; u < 4; ++u) {
        const long e = e0 + 128L * u;
        if (e < n) {
            const unsigned row = (unsigned)((unsigned long)e / (unsigned)d.nx);
            const unsigned k = row / (unsigned)d.ny, j = row - k * (unsigned)d.ny;
            const bool odd = (j + k) & 1u;
            if (UPD) {
                if (go) {
                    rv[u].x = -alpha * av[u].x + rv[u].x;
                    rv[u].y = -alpha * av[u].y + rv[u].y;
                    stnt(ru.r + e, rv[u].x, rv[u].y);
                }
                acc += rv[u].x * rv[u].x;
                acc += rv[u].y * rv[u].y;
            }
            const float f0 = (float)rv[u].x, f1 = (float)rv[u].y;
            b[e >> 1] = odd ? make_float2(f1, f0) : make_float2(f0, f1);
        }
    }
    if (UPD) {
        const double s = block_sum<256>(acc);
        if (threadIdx.x == 0) ru.partials[blk] = s;
    }
}

constexpr int kExtra = 9;  // planes around a chunk
// one workgroup runs on a CU at a time (its registers): 256 in flight
long steps_of(int tiles, int chunks, int kz) {
    return ((long)tiles * chunks + 255) / 256 * (kz + kExtra);
}

FGeo fgeo_of(const mf3d_grid& g) {
    FGeo G;
    G.ny = g.ny, G.nz = g.nz;
    G.bcp = 0;
    G.h = g.nx / 2;
    G.half = (long)G.h * g.ny * g.nz;
    G.tx = (G.h + kIX - 1) / kIX;
    G.ty = (g.ny + kIY - 1) / kIY;
    // as many chunks of planes as make the fewest steps; more chunks read more rims,
    // so only for a twentieth less
    long best = -1;
    for (int c = 1; c <= std::max(1, g.nz / 32); ++c) {
        const int kz = ((g.nz + c - 1) / c + 1) / 2 * 2, chunks = (g.nz + kz - 1) / kz;
        const long t = steps_of(G.tx * G.ty, chunks, kz);
        if (best < 0 || 20 * t < 19 * best) best = t, G.kz = kz, G.chunks = chunks;
    }
    return G;
}

template <typename TC, int START, int END>
int launch(hipStream_t s, const FGeo& G, const BcTypes& bc, bool pin, double bs, double rs,
           const float* xin, float* xout, const float* b, const void* faces, const float* xc,
           float* bcoarse) {
    const long nb = (long)G.tx * G.ty * G.chunks;
    fused_kernel<TC, START, END><<<xcd_round((size_t)nb), kThreads, 0, s>>>(
        G, bc, pin ? 1 : 0, (float)bs, (float)rs, xin, xout, reinterpret_cast<const float2*>(b),
        static_cast<const Rec*>(faces), xc, bcoarse);
    MF3D_HIP_TRY(hipGetLastError());
    return MF3D_OK;
}

int check(const mf3d_grid& g, CoefType t) {
    return kern::fused32_ok(g, t) ? MF3D_OK
                                  : fail(MF3D_ERR_UNSUPPORTED, "fused smoothing: sizes or faces");
}

}  // namespace

namespace kern {

// 16-bit faces (a thread's ring of 32-bit ones does not fit its registers); even
// sizes whose coarse level is even too (colour-split); planes beyond a periodic
// end at most one wrap away; 32-bit offsets within a plane and a colour of the
// coarse level
bool fused32_ok(const mf3d_grid& g, CoefType t) {
    return (t == COEF_BF16 || t == COEF_F16) && g.nx % 4 == 0 && g.ny % 4 == 0 && g.nz % 4 == 0 &&
           g.nz >= 8 && (size_t)g.nx * g.ny < ((size_t)1 << 28) &&
           cells(g) < ((size_t)1 << 32);
}

// From 2^23 cells, where the tiles and z-chunks occupy most of the 256 CUs (256^3: 220
// workgroups, 187 us a level for 271 us of half-sweeps; a 128^3 level would have 72
// workgroups of 41 planes, about 100 us for 56 us of launch-bound half-sweeps), and
// where the tiles are full enough: a step takes 2.4 us, what it replaces 20 ps a cell.
// V-cycles with the passes and with half-sweeps, by cells a step: 8x1024x1024 39 000
// 602 us for 241; 16x1024x512 74 000 376 for 259; 1024x8x1024 94 000 296 for 243;
// 8192x32x32 102 000 300 for 318; 2048x512x8 123 000 248 for 290; 256^3 230 000 378 for
// 499.
bool fused32_pays(const mf3d_grid& g) {
    const FGeo G = fgeo_of(g);
    return cells(g) >= ((size_t)1 << 23) &&
           steps_of(G.tx * G.ty, G.chunks, G.kz) <= (long)(cells(g) / 100000);
}

size_t fused32_face_bytes(const mf3d_grid& g) {
    return sizeof(Rec) * (size_t)(g.nx / 2 + 1) * (g.ny + 1) * (g.nz + 1);
}

int fused32_pack(hipStream_t s, const mf3d_grid& g, const FaceSet& F, void* faces) {
    MF3D_TRY(check(g, F.type));
    if (!F.split) return fail(MF3D_ERR_UNSUPPORTED, "face records come from colour-split faces");
    const unsigned nb = (unsigned)((fused32_face_bytes(g) / sizeof(Rec) + 255) / 256);
    const Dims d{g.nx, g.ny, g.nz};
    Rec* o = static_cast<Rec*>(faces);
    if (F.type == COEF_BF16) {
        typedef __hip_bfloat16 T;
        pack_faces_kernel<T><<<nb, 256, 0, s>>>(
            d, SFaces<T>{(const T*)F.fx, (const T*)F.fy, (const T*)F.fz, (const T*)F.ux,
                             (const T*)F.uy, (const T*)F.uz}, o);
    } else {
        typedef __half T;
        pack_faces_kernel<T><<<nb, 256, 0, s>>>(
            d, SFaces<T>{(const T*)F.fx, (const T*)F.fy, (const T*)F.fz, (const T*)F.ux,
                             (const T*)F.uy, (const T*)F.uz}, o);
    }
    MF3D_HIP_TRY(hipGetLastError());
    return MF3D_OK;
}

int fused32_pre(hipStream_t s, const mf3d_grid& g, const BcTypes& bc, bool pin, double bs,
                double rs, float* xb, const float* b, CoefType t, const void* faces,
                float* bcoarse, bool pairs) {
    MF3D_TRY(check(g, t));
    FGeo G = fgeo_of(g);
    G.bcp = pairs ? 1 : 0;
    if (t == COEF_BF16)
        return launch<__hip_bfloat16, START_ZERO, END_RESTRICT>(s, G, bc, pin, bs, rs, nullptr, xb,
                                                                b, faces, nullptr, bcoarse);
    return launch<__half, START_ZERO, END_RESTRICT>(s, G, bc, pin, bs, rs, nullptr, xb, b, faces,
                                                    nullptr, bcoarse);
}

int fused32_post(hipStream_t s, const mf3d_grid& g, const BcTypes& bc, bool pin, double bs,
                 const float* xb, float* x, const float* b, CoefType t, const void* faces,
                 const float* xc) {
    MF3D_TRY(check(g, t));
    const FGeo G = fgeo_of(g);
    if (t == COEF_BF16)
        return launch<__hip_bfloat16, START_PROLONG, END_NONE>(s, G, bc, pin, bs, 0.0, xb, x, b,
                                                               faces, xc, nullptr);
    return launch<__half, START_PROLONG, END_NONE>(s, G, bc, pin, bs, 0.0, xb, x, b, faces, xc,
                                                   nullptr);
}

int r_to_b(hipStream_t s, const mf3d_grid& g, const double* r, const RUpd* ru, float* b) {
    const size_t n = cells(g);
    const unsigned nb = xcd_round((n + 2047) / 2048);
    const Dims d{g.nx, g.ny, g.nz};
    if (ru)
        r_to_b_kernel<true><<<nb, 256, 0, s>>>(d, *ru, reinterpret_cast<float2*>(b));
    else  // (reads r only)
        r_to_b_kernel<false><<<nb, 256, 0, s>>>(
            d, RUpd{nullptr, nullptr, const_cast<double*>(r), nullptr},
            reinterpret_cast<float2*>(b));
    MF3D_HIP_TRY(hipGetLastError());
    return MF3D_OK;
}

}  // namespace kern
}  // namespace mf3d
