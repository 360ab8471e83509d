// Learned warm start for the head solve: a 3-D convolutional encoder-decoder
// that maps ln K to an initial head, trained and run with BF16 MFMA kernels
// (FP32 accumulation) on gfx950. No counterpart in MacroFlow3D.
//
// The network runs on the grid coarsened 4x per axis (block statistics of K
// in, a smooth correction out): MG-PCG removes high-frequency error in one
// V-cycle, so only the smooth part of a guess shortens the solve, and the
// coarse grid makes inference 64x cheaper and the receptive field 4x wider.
// Network (3 levels at 4x, 8x and 16x coarsening, 16/32/64 channels, 3^3
// kernels, zero padding), on the coarse grid G (cell V = a 4x4x4 block):
//   x0  = [<lnK>/2, log<K>/2, -log<1/K>/2, 2 (I + 1/2)/NX - 1]  (4 channels, stored as 16)
//   e0  = relu(conv_a(x0))          4 -> 16  G
//   e1  = relu(conv_b(pool(e0)))   16 -> 32  G/2
//   e2  = relu(conv_c(pool(e1)))   32 -> 64  G/4
//   e2b = relu(conv_d(e2))         64 -> 64  G/4
//   d1  = relu(conv_e(up(e2b)) + e1)   64 -> 32  G/2
//   d0  = relu(conv_f(up(d1)) + e0)    32 -> 16  G
//   y   = conv_g(d0)               16 -> 1   G  (FP32)
//   h0  = h_lin + J trilinear(y),  h_lin linear between the x faces, J = (h_W - h_E) / nx
// (<.> = mean over the block, pool = mean of 2x2x2 children, up = copy to the
// 8 children). Training minimises mean over G of (y - <(h - h_lin) / J>)^2
// with Adam on FP32 master weights.
//
// Activations are BF16, channels-last: a[v * C + c], v = i + nx (j + ny k),
// C a multiple of 16. Convolution = implicit GEMM: for 16 output channels x
// 16 voxels, K runs over (tap, input channel) pairs, tap = dx + 3 dy + 9 dz
// (d = -1, 0, 1 offsets + 1), k = tap * Cin + c, 32 per MFMA.
#include <hip/hip_bf16.h>
#include <hip/hip_runtime.h>

#include <algorithm>
#include <cmath>
#include <cstring>
#include <string>
#include <vector>

#include "common.hpp"

namespace mf3d {
namespace {

typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef float f32x4 __attribute__((ext_vector_type(4)));

constexpr int kVT = 4;  // 16-voxel tiles per wave in the convolution (large grids)
constexpr long kConvWaves = 2048;  // fewer tiles per wave below this many waves

__device__ __forceinline__ float bf2f(__hip_bfloat16 v) { return __bfloat162float(v); }
__device__ __forceinline__ __hip_bfloat16 f2bf(float v) { return __float2bfloat16(v); }

struct Geo {
    int nx, ny, nz;
    __device__ long n() const { return (long)nx * ny * nz; }
};

__device__ __forceinline__ bf16x8 load8(const __hip_bfloat16* p) {
    const uint4 u = *reinterpret_cast<const uint4*>(p);
    return __builtin_bit_cast(bf16x8, u);
}

// ---- convolution (forward, and backward-data with transposed weights) --------
// W: [Cout_pad][Kpad] BF16, Kpad = 32 * ceil(27 Cin / 32), zero beyond 27 Cin
// and for output channels >= Cout. FLIP reads the taps mirrored (backward
// data with the forward tap order in W). Epilogue, per output (v, c):
//   s = acc + bias[c] (if bias) + R[v*Cs + c] (if R); s = relu(s) (if relu);
//   s *= (M[v*Cs + c] > 0) (if M); stored to out (BF16 or FP32) for c < Cs.
// up: X holds the grid of half the size and a voxel reads its parent (the copy
// to the 8 children is never stored).
//
// KS waves of a workgroup share one wave's output tile and split its k steps;
// their accumulators meet in LDS, summed in wave order, and each of the KS waves
// finishes some of the tile's CT x VT fragments. The deep layers are a chain of
// 14-54 dependent k steps on few voxels: 8^3 voxels x 64 channels are 32 tiles,
// so with KS = 1 the launch was 32 waves on 256 CUs and the latency of the chain
// its whole time (8^3, 64 -> 64 channels: 33.8 us with KS = 1, 9.4 us with 16).
template <int CT, int VT, bool F32OUT, int KS>
__global__ void __launch_bounds__(KS > 4 ? KS * 64 : 256)
    conv_kernel(Geo g, int cin, int kpad, int cs, int up, const __hip_bfloat16* __restrict__ X,
                const __hip_bfloat16* __restrict__ W, const float* __restrict__ bias,
                const __hip_bfloat16* __restrict__ R, const __hip_bfloat16* __restrict__ M,
                int relu, int flip, void* __restrict__ out) {
    constexpr int WPB = KS > 4 ? KS : 4;  // waves per workgroup
    // (voxel indices are 32-bit: a grid has at most 4e9 cells, and a 64-bit
    // division is hundreds of instructions)
    const unsigned nvox = (unsigned)g.n();
    const int lane = threadIdx.x & 63;
    const int wv = (int)(threadIdx.x >> 6);
    const int part = wv % KS;  // this wave's share of the k steps
    const unsigned tile = blockIdx.x * (WPB / KS) + wv / KS;
    const unsigned vbase = tile * (16 * VT);
    if (KS == 1 && vbase >= nvox) return;  // whole wave (KS > 1: the workgroup meets below)
    const int col = lane & 15;   // voxel within a tile / output channel row of A
    const int grp = lane >> 4;   // k group: k = 8 grp .. 8 grp + 7 of each 32-chunk

    int vi[VT], vj[VT], vk[VT];
    bool live[VT];
#pragma unroll
    for (int t = 0; t < VT; ++t) {
        const unsigned v = vbase + 16 * t + col;
        live[t] = v < nvox;
        const unsigned vv = live[t] ? v : 0;
        const unsigned q = vv / (unsigned)g.nx;
        vi[t] = (int)(vv - q * g.nx);
        vk[t] = (int)(q / (unsigned)g.ny);
        vj[t] = (int)(q - vk[t] * (unsigned)g.ny);
    }
    f32x4 acc[VT][CT];
#pragma unroll
    for (int t = 0; t < VT; ++t)
#pragma unroll
        for (int c = 0; c < CT; ++c) acc[t][c] = f32x4{0.f, 0.f, 0.f, 0.f};

    const int K = 27 * cin;
    const int sx = g.nx >> up, sy = g.ny >> up;  // the stored grid of X
    const bf16x8 zero8 = __builtin_bit_cast(bf16x8, uint4{0u, 0u, 0u, 0u});
    // the operands of one 32-wide k step: weight rows (A) and the tap's
    // input channels at each voxel (B, zero outside the grid or past K). The
    // addresses are chosen without branches (an outside voxel reads voxel 0 and
    // is zeroed): a load under a per-lane branch would be waited for inside it
    auto load_step = [&](int k0, bf16x8 (&a)[CT], bf16x8 (&b)[VT]) {
        const int k = k0 + 8 * grp;
#pragma unroll
        for (int c = 0; c < CT; ++c) a[c] = load8(W + (long)(c * 16 + col) * kpad + k);
        const bool ok = k < K;
        int tap = ok ? k / cin : 0;
        const int c0 = ok ? k - tap * cin : 0;
        if (flip) tap = 26 - tap;
        const int dx = tap % 3 - 1, dy = (tap / 3) % 3 - 1, dz = tap / 9 - 1;
#pragma unroll
        for (int t = 0; t < VT; ++t) {
            const int ii = vi[t] + dx, jj = vj[t] + dy, kk = vk[t] + dz;
            const bool in = ok && live[t] && (unsigned)ii < (unsigned)g.nx &&
                            (unsigned)jj < (unsigned)g.ny && (unsigned)kk < (unsigned)g.nz;
            const long o = in ? (long)(ii >> up) + (long)sx * ((jj >> up) + (long)sy * (kk >> up)) : 0;
            const bf16x8 x = load8(X + o * cin + c0);
            b[t] = in ? x : zero8;
        }
    };
    // the next step's operands are loaded before this step's products are
    // issued, so the load latency overlaps the MFMAs (same accumulation order)
    const int steps = kpad / 32;
    const int kb = 32 * (steps * part / KS), ke = 32 * (steps * (part + 1) / KS);
    bf16x8 a[CT], b[VT];
    if (kb < ke) load_step(kb, a, b);
    for (int k0 = kb; k0 < ke; k0 += 32) {
        bf16x8 an[CT], bn[VT];
        if (k0 + 32 < ke) load_step(k0 + 32, an, bn);
#pragma unroll
        for (int t = 0; t < VT; ++t)
#pragma unroll
            for (int c = 0; c < CT; ++c)
                acc[t][c] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a[c], b[t], acc[t][c], 0, 0, 0);
        if (k0 + 32 < ke) {
#pragma unroll
            for (int c = 0; c < CT; ++c) a[c] = an[c];
#pragma unroll
            for (int t = 0; t < VT; ++t) b[t] = bn[t];
        }
    }
    // acc[t][c][r] = out(channel c*16 + 4 grp + r, voxel vbase + 16 t + col)
    __shared__ f32x4 red[KS > 1 ? WPB * VT * CT * 64 : 1];
    if (KS > 1) {
#pragma unroll
        for (int t = 0; t < VT; ++t)
#pragma unroll
            for (int c = 0; c < CT; ++c) red[((wv * VT + t) * CT + c) * 64 + lane] = acc[t][c];
        __syncthreads();
    }
#pragma unroll
    for (int t = 0; t < VT; ++t) {
        const long v = vbase + 16 * t + col;
#pragma unroll
        for (int c = 0; c < CT; ++c) {
            const int ch0 = c * 16 + 4 * grp;
            if (KS > 1) {
                if ((t * CT + c) % KS != part) continue;  // another wave's fragment (uniform)
                const int w0 = wv - part;
                f32x4 s = red[((w0 * VT + t) * CT + c) * 64 + lane];
#pragma unroll
                for (int w = 1; w < KS; ++w)
                    s += red[(((w0 + w) * VT + t) * CT + c) * 64 + lane];
                acc[t][c] = s;
            }
            if (!live[t] || ch0 >= cs) continue;
            float s[4];
#pragma unroll
            for (int r = 0; r < 4; ++r) {
                float x = acc[t][c][r];
                if (bias) x += bias[ch0 + r];
                if (R) x += bf2f(R[v * cs + ch0 + r]);
                if (relu) x = fmaxf(x, 0.0f);
                if (M) x = bf2f(M[v * cs + ch0 + r]) > 0.0f ? x : 0.0f;
                s[r] = x;
            }
            if (F32OUT) {
                float* o = static_cast<float*>(out) + v * cs + ch0;
                *reinterpret_cast<float4*>(o) = make_float4(s[0], s[1], s[2], s[3]);
            } else {
                __hip_bfloat16* o = static_cast<__hip_bfloat16*>(out) + v * cs + ch0;
                o[0] = f2bf(s[0]);
                o[1] = f2bf(s[1]);
                o[2] = f2bf(s[2]);
                o[3] = f2bf(s[3]);
            }
        }
    }
}

// ---- weight and bias gradients -------------------------------------------------
// dW[co][tap*Cin + ci] = sum_v dY[v][co] X[v + d(tap)][ci]: the voxels are the
// MFMA's K dimension, so a lane wants 8 consecutive voxels of one channel. Gathering
// them from the channels-last tensors cost 8 two-byte loads with their own address
// and bounds checks per operand (32^3, 16 x 16 channels: 66.9 us). Instead one
// launch copies every operand of every layer into a channel-first form with zero
// borders (Planar): each lane's 8 voxels are then one 16-byte load at any tap, and
// no bounds are checked. One more launch holds all layers' products (a wave per
// layer, tap and slice of the voxels; the layers are small enough that only
// together they fill the chip), and one sums the slices in order, straight into
// the master layout. 128^3 training sample: 28 launches of 408 us became 3 of
// 63 us (46.7 of them the products).

// channel-first copy of an [N][ch] tensor: voxel (i, j, k) of channel c at
// c * plane + lead + ((k + 1) (ny + 2) + j + 1) row + i, everything else zero.
// row = ceil8(nx) + 8 leaves at least 8 zeros after a row, which also serve as
// the next row's border at i = -1; lead covers the first row's.
constexpr int kPlanarLead = 16;
struct Planar {
    int row;       // row stride
    long slab;     // plane of one z: row (ny + 2)
    long plane;    // one channel
    int gpr;       // 8-voxel groups per row
    long groups;   // over all rows of the grid
    int nx, ny;
};
Planar planar_of(const mf3d_grid& g) {
    Planar P;
    const int n8 = (g.nx + 7) / 8;
    P.row = 8 * n8 + 8;
    P.slab = (long)P.row * (g.ny + 2);
    P.plane = P.slab * (g.nz + 2) + 2 * kPlanarLead;
    P.gpr = n8;
    P.groups = (long)n8 * g.ny * g.nz;
    P.nx = g.nx, P.ny = g.ny;
    return P;
}

struct PlanarCopy {
    const __hip_bfloat16* src;
    __hip_bfloat16* dst;
    int ch, up;  // up: src is on the half-size grid (a voxel copies its parent)
    Geo g;
    Planar P;
    int block0;   // first workgroup of this tensor
    int vblocks;  // workgroups per 8 channels
};
constexpr int kMaxCopies = 14, kMaxWLayers = 7;
struct PlanarCopies {
    PlanarCopy c[kMaxCopies];
    int n;
};
// a thread copies 8 channels of one voxel
__global__ void __launch_bounds__(256) planar_kernel(PlanarCopies D) {
    int e = 0;
    while (e + 1 < D.n && D.c[e + 1].block0 <= (int)blockIdx.x) ++e;
    const PlanarCopy& C = D.c[e];
    const unsigned nv = (unsigned)C.g.n();
    const int b = (int)blockIdx.x - C.block0, c8 = b / C.vblocks;
    const unsigned v = (unsigned)(b - c8 * C.vblocks) * 256 + threadIdx.x;
    if (v >= nv) return;
    const unsigned q = v / (unsigned)C.g.nx;
    const int i = (int)(v - q * C.g.nx);
    const int k = (int)(q / (unsigned)C.g.ny), j = (int)(q - k * (unsigned)C.g.ny);
    const int u = C.up;
    const long sv = (long)(i >> u) + (long)(C.g.nx >> u) * ((j >> u) + (long)(C.g.ny >> u) * (k >> u));
    const bf16x8 val = load8(C.src + sv * C.ch + 8 * c8);
    __bf16* d = reinterpret_cast<__bf16*>(C.dst) + (long)8 * c8 * C.P.plane + kPlanarLead +
                (long)(k + 1) * C.P.slab + (long)(j + 1) * C.P.row + i;
#pragma unroll
    for (int c = 0; c < 8; ++c) d[(long)c * C.P.plane] = val[c];
}

__global__ void __launch_bounds__(256) zero_kernel(uint4* __restrict__ p, long n) {
    const long e = (long)blockIdx.x * 256 + threadIdx.x;
    if (e < n) p[e] = uint4{0u, 0u, 0u, 0u};
}

struct WLayer {
    const __hip_bfloat16* dY;  // planar, 16 ct channels
    const __hip_bfloat16* X;   // planar, 16 it channels
    Planar P;
    int ct, it;
    int slices, steps;  // slices of `steps` 32-voxel steps each
    int wave0;          // first wave of this layer in the launch
    float* part;        // [slice][16 ct][27 * 16 it]
    float* bpart;       // [slice][16 ct]
    // reduction into the master layout
    int cin, cout;
    float* gw;
    float* gb;
    int elem0;  // first element of this layer in the reduction
};
struct WLayers {
    WLayer l[kMaxWLayers];
    int n, waves, elems;
};

template <int CT, int IT>
__device__ __forceinline__ void wgrad_body(const WLayer& L, int tap, int slice) {
    const int lane = threadIdx.x & 63, col = lane & 15, grp = lane >> 4;
    const int dx = tap % 3 - 1, dy = (tap / 3) % 3 - 1, dz = tap / 9 - 1;
    const long shift = (long)dy * L.P.row + (long)dz * L.P.slab;
    const bool bias = tap == 13;
    const __bf16 one = (__bf16)1.0f;
    const bf16x8 ones = {one, one, one, one, one, one, one, one};
    const bf16x8 zero8 = __builtin_bit_cast(bf16x8, uint4{0u, 0u, 0u, 0u});
    f32x4 acc[CT][IT], accb[CT];
#pragma unroll
    for (int c = 0; c < CT; ++c) {
        accb[c] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
        for (int i = 0; i < IT; ++i) acc[c][i] = f32x4{0.f, 0.f, 0.f, 0.f};
    }
    const __hip_bfloat16* A0 = L.dY + (long)col * L.P.plane + kPlanarLead;
    const __hip_bfloat16* B0 = L.X + (long)col * L.P.plane + kPlanarLead + shift;
    // this lane's 8 voxels of a step: group g0 + 4 st + grp of the grid's rows,
    // its place carried from step to step (past the end: zeros)
    int q = slice * L.steps * 4 + grp;
    int x8 = q % L.P.gpr, j = q / L.P.gpr % L.P.ny;
    long o = (long)(q / L.P.gpr / L.P.ny + 1) * L.P.slab + (long)(j + 1) * L.P.row + 8 * x8;
    const int groups = (int)L.P.groups;
    // The tap's shift along x is made in registers from an aligned load and the
    // 4 bytes next to it: 16-byte loads at odd element offsets took 68 us
    // for the launch instead of 51.
    // Products that are not part of the sum are 0 x 0 (the other factor may be infinite):
    // X is zeroed past the end, and where dx = -1 would bring a row's last value
    // beside the zero after its dY (the row's last group, element nx & 7, if it has one).
    const int tail = dx < 0 ? (L.P.nx & 7) : 0;
    uint4 keep{~0u, ~0u, ~0u, ~0u};
    if (tail) {  // uniform
        const unsigned half = tail & 1 ? 0x0000ffffu : 0xffff0000u;
        const int w = tail >> 1;
        keep = uint4{w == 0 ? half : ~0u, w == 1 ? half : ~0u, w == 2 ? half : ~0u,
                     w == 3 ? half : ~0u};
    }
    auto load = [&](bool mine, bf16x8 (&a)[CT], bf16x8 (&b)[IT]) {
        const bool ok = mine && q < groups, last = x8 == L.P.gpr - 1;
        const long oo = ok ? o : L.P.slab + L.P.row;
#pragma unroll
        for (int c = 0; c < CT; ++c) {
            a[c] = load8(A0 + (long)16 * c * L.P.plane + oo);
            if (!ok) a[c] = zero8;
        }
#pragma unroll
        for (int i = 0; i < IT; ++i) {
            const __hip_bfloat16* p = B0 + (long)16 * i * L.P.plane + oo;
            uint4 d = *reinterpret_cast<const uint4*>(p);
            if (dx > 0) {  // uniform
                const unsigned n = *reinterpret_cast<const unsigned*>(p + 8);
                d = uint4{__builtin_amdgcn_alignbit(d.y, d.x, 16), __builtin_amdgcn_alignbit(d.z, d.y, 16),
                          __builtin_amdgcn_alignbit(d.w, d.z, 16), __builtin_amdgcn_alignbit(n, d.w, 16)};
            } else if (dx < 0) {
                const unsigned n = *reinterpret_cast<const unsigned*>(p - 2);
                d = uint4{__builtin_amdgcn_alignbit(d.x, n, 16), __builtin_amdgcn_alignbit(d.y, d.x, 16),
                          __builtin_amdgcn_alignbit(d.z, d.y, 16), __builtin_amdgcn_alignbit(d.w, d.z, 16)};
                if (tail && last) d.x &= keep.x, d.y &= keep.y, d.z &= keep.z, d.w &= keep.w;
            }
            b[i] = ok ? __builtin_bit_cast(bf16x8, d) : zero8;
        }
        q += 4, x8 += 4, o += 32;
        while (x8 >= L.P.gpr) {  // rows end with 8 zeros; the next z skips the border rows
            x8 -= L.P.gpr, o += 8;
            if (++j == L.P.ny) j = 0, o += 2L * L.P.row;
        }
    };
    // U steps' loads are issued together: the chain of steps is latency
    constexpr int U = CT + IT <= 3 ? 4 : 1;
    for (int st = 0; st < L.steps; st += U) {
        bf16x8 a[U][CT], b[U][IT];
#pragma unroll
        for (int u = 0; u < U; ++u) load(st + u < L.steps, a[u], b[u]);
#pragma unroll
        for (int u = 0; u < U; ++u)
#pragma unroll
            for (int c = 0; c < CT; ++c) {
                if (bias)
                    accb[c] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a[u][c], ones, accb[c], 0, 0, 0);
#pragma unroll
                for (int i = 0; i < IT; ++i)
                    acc[c][i] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a[u][c], b[u][i], acc[c][i],
                                                                        0, 0, 0);
            }
    }
    // acc[c][i][r] = dW(co = c*16 + 4 grp + r, ci = i*16 + col)
    const long K = 27L * 16 * IT;
    float* p = L.part + (long)slice * (CT * 16) * K + (long)tap * (16 * IT) + col;
#pragma unroll
    for (int c = 0; c < CT; ++c)
#pragma unroll
        for (int r = 0; r < 4; ++r) {
            const int co = c * 16 + 4 * grp + r;
#pragma unroll
            for (int i = 0; i < IT; ++i) p[(long)co * K + i * 16] = acc[c][i][r];
            if (bias && col == 0) L.bpart[slice * (CT * 16) + co] = accb[c][r];
        }
}

__global__ void __launch_bounds__(256, 3) wgrad_kernel(WLayers D) {
    const int wave = (int)blockIdx.x * 4 + (int)(threadIdx.x >> 6);
    if (wave >= D.waves) return;
    int e = 0;
    while (e + 1 < D.n && D.l[e + 1].wave0 <= wave) ++e;
    const WLayer& L = D.l[e];
    const int w = wave - L.wave0, tap = w % 27, slice = w / 27;
    switch (L.ct * 8 + L.it) {
    case 8 + 1: wgrad_body<1, 1>(L, tap, slice); break;
    case 8 + 2: wgrad_body<1, 2>(L, tap, slice); break;
    case 16 + 1: wgrad_body<2, 1>(L, tap, slice); break;
    case 16 + 4: wgrad_body<2, 4>(L, tap, slice); break;
    case 32 + 2: wgrad_body<4, 2>(L, tap, slice); break;
    default: wgrad_body<4, 4>(L, tap, slice); break;
    }
}

// gw[co][tap][ci] and gb[co] (master layout): the slices' sums in slice order
__global__ void __launch_bounds__(256) wgrad_reduce_kernel(WLayers D) {
    const int t = (int)(blockIdx.x * 256 + threadIdx.x);
    if (t >= D.elems) return;
    int e = 0;
    while (e + 1 < D.n && D.l[e + 1].elem0 <= t) ++e;
    const WLayer& L = D.l[e];
    const int q = t - L.elem0, nw = L.cout * 27 * L.cin;
    const int cop = 16 * L.ct, cip = 16 * L.it;
    const float* p;
    long stride;
    if (q < nw) {
        const int ci = q % L.cin, r = q / L.cin, tap = r % 27, co = r / 27;
        p = L.part + (long)co * 27 * cip + tap * cip + ci;
        stride = (long)cop * 27 * cip;
    } else {
        p = L.bpart + (q - nw);
        stride = cop;
    }
    float s = 0.0f;
    int sl = 0;
    for (; sl + 8 <= L.slices; sl += 8) {  // 8 loads in flight
        float v[8];
#pragma unroll
        for (int u = 0; u < 8; ++u) v[u] = p[(sl + u) * stride];
#pragma unroll
        for (int u = 0; u < 8; ++u) s += v[u];
    }
    for (; sl < L.slices; ++sl) s += p[sl * stride];
    if (q < nw) L.gw[q] = s;
    else L.gb[q - nw] = s;
}

// ---- pooling / upsampling (channels-last), factor kF per axis ------------------
constexpr int kS = 4;  // fine cells per network cell, per axis
constexpr int kF = 2;
constexpr float kInvF3 = 1.0f / (kF * kF * kF);

__device__ __forceinline__ int parent_of(const Geo& g, int v) {
    const int q = v / g.nx, i = v - q * g.nx;
    const int k = q / g.ny, j = q - k * g.ny;
    return i / kF + (g.nx / kF) * ((j / kF) + (g.ny / kF) * (k / kF));
}

// sum over the kF^3 children of coarse cell V (fine g), channel c
__device__ __forceinline__ float child_sum(const Geo& g, int ch, const __hip_bfloat16* X, int V,
                                           int c) {
    const int NX = g.nx / kF, NY = g.ny / kF;
    const int q = V / NX, I = V - q * NX;
    const int K = q / NY, J = q - K * NY;
    float s = 0.0f;
    for (int dz = 0; dz < kF; ++dz)
        for (int dy = 0; dy < kF; ++dy)
            for (int dx = 0; dx < kF; ++dx)
                s += bf2f(X[((long)(kF * I + dx) +
                             (long)g.nx * ((kF * J + dy) + (long)g.ny * (kF * K + dz))) * ch + c]);
    return s;
}

// pool: Y[V][c] = mean of the children of coarse cell V (fine g)
__global__ void __launch_bounds__(256)
    pool_kernel(Geo g, int ch, const __hip_bfloat16* __restrict__ X, __hip_bfloat16* __restrict__ Y) {
    const int e = (int)(blockIdx.x * blockDim.x + threadIdx.x);
    if (e >= g.n() / (kF * kF * kF) * ch) return;
    Y[e] = f2bf(child_sum(g, ch, X, e / ch, e % ch) * kInvF3);
}

// pool backward with the skip gradient and the ReLU mask of the pooled input:
// dX[v][c] = (dY[parent][c] / kF^3 + (S ? S[v][c] : 0)) * (M[v][c] > 0)
__global__ void __launch_bounds__(256)
    pool_bwd_kernel(Geo g, int ch, const __hip_bfloat16* __restrict__ dY,
                    const __hip_bfloat16* __restrict__ S, const __hip_bfloat16* __restrict__ M,
                    __hip_bfloat16* __restrict__ dX) {
    const int e = (int)(blockIdx.x * blockDim.x + threadIdx.x);
    if (e >= g.n() * ch) return;
    const int c = e % ch;
    float s = bf2f(dY[parent_of(g, e / ch) * ch + c]) * kInvF3;
    if (S) s += bf2f(S[e]);
    if (M) s = bf2f(M[e]) > 0.0f ? s : 0.0f;
    dX[e] = f2bf(s);
}

// up backward with the ReLU mask of the coarse input:
// dX[V][c] = sum of dY over the children, times (M[V][c] > 0)
__global__ void __launch_bounds__(256)
    up_bwd_kernel(Geo g, int ch, const __hip_bfloat16* __restrict__ dY,
                  const __hip_bfloat16* __restrict__ M, __hip_bfloat16* __restrict__ dX) {
    const int e = (int)(blockIdx.x * blockDim.x + threadIdx.x);
    if (e >= g.n() / (kF * kF * kF) * ch) return;
    float s = child_sum(g, ch, dY, e / ch, e % ch);
    if (M) s = bf2f(M[e]) > 0.0f ? s : 0.0f;
    dX[e] = f2bf(s);
}

// ---- input, output, loss -------------------------------------------------------
// x0 on the coarse grid from the fine K (or ln K) of the kS^3 block of each cell:
// 0.5 mean ln K, 0.5 ln mean K, -0.5 ln mean 1/K, the x coordinate in [-1, 1].
// The features end in BF16, so they are accumulated in FP32. A workgroup holds
// 64 coarse cells x kS z-slices (one thread each); the slices' sums are added
// in LDS in a fixed order.
__global__ void __launch_bounds__(256)
    input_kernel(Geo g, const double* __restrict__ K, int is_log, __hip_bfloat16* __restrict__ x0) {
    static_assert(kS == 4, "64 cells x 4 slices per workgroup");
    const int NX = g.nx / kS, NY = g.ny / kS, NZ = g.nz / kS;
    const long nv = (long)NX * NY * NZ;
    const int lane = (int)(threadIdx.x & 63), dz = (int)(threadIdx.x >> 6);
    const long V = (long)blockIdx.x * 64 + lane;
    float sl = 0.0f, sk = 0.0f, si = 0.0f;
    int I = 0, J = 0, Kc = 0;
    if (V < nv) {
        I = (int)(V % NX);
        const long q = V / NX;
        J = (int)(q % NY);
        Kc = (int)(q / NY);
#pragma unroll
        for (int dy = 0; dy < kS; ++dy)
#pragma unroll
            for (int dx = 0; dx < kS; ++dx) {
                const long o = (long)(kS * I + dx) +
                               (long)g.nx * ((kS * J + dy) + (long)g.ny * (kS * Kc + dz));
                const float v = (float)K[o];
                const float l = is_log ? v : __logf(v);
                const float kv = is_log ? __expf(v) : v;
                sl += l;
                sk += kv;
                si += 1.0f / kv;
            }
    }
    __shared__ float part[3][kS][64];
    part[0][dz][lane] = sl;
    part[1][dz][lane] = sk;
    part[2][dz][lane] = si;
    __syncthreads();
    if (dz != 0 || V >= nv) return;
    sl = ((part[0][0][lane] + part[0][1][lane]) + part[0][2][lane]) + part[0][3][lane];
    sk = ((part[1][0][lane] + part[1][1][lane]) + part[1][2][lane]) + part[1][3][lane];
    si = ((part[2][0][lane] + part[2][1][lane]) + part[2][2][lane]) + part[2][3][lane];
    const float w = 1.0f / (kS * kS * kS);
    __hip_bfloat16* o = x0 + V * 16;
    o[0] = f2bf(0.5f * sl * w);
    o[1] = f2bf(0.5f * __logf(sk * w));
    o[2] = f2bf(-0.5f * __logf(si * w));
    o[3] = f2bf((float)(2.0 * (I + 0.5) / NX - 1.0));
#pragma unroll
    for (int c = 4; c < 16; ++c) o[c] = f2bf(0.0f);
}

// linear interpolation weights of fine index i on a coarse axis of n cells
// (cell centres at (I + 1/2) kS; constant beyond the outer centres)
__device__ __forceinline__ void lin_axis(int i, int n, int& i0, int& i1, float& w1) {
    const float u = (i + 0.5f) / kS - 0.5f;
    if (u <= 0.0f) {
        i0 = i1 = 0;
        w1 = 0.0f;
    } else if (u >= n - 1) {
        i0 = i1 = n - 1;
        w1 = 0.0f;
    } else {
        i0 = (int)u;
        i1 = i0 + 1;
        w1 = u - i0;
    }
}

__global__ void __launch_bounds__(256)
    channel0_kernel(const float* __restrict__ y, int ych, long n, float* __restrict__ yd) {
    const long v = (long)blockIdx.x * blockDim.x + threadIdx.x;
    if (v < n) yd[v] = y[v * ych];
}

// h0 = h_lin + J trilinear(yd) on the fine grid g (yd: the coarse field's
// channel 0, stored densely). A thread writes 4 consecutive cells of a row
// (two 16-byte stores; the network's sizes are multiples of 16); the coarse
// values it interpolates, at most 3 along x for each of the 4 y/z corner rows,
// are read directly (the coarse field is 1/64 of the fine one and stays in L2).
__global__ void __launch_bounds__(256)
    output_kernel(Geo g, double hw, double he, double inv_nx, const float* __restrict__ yd,
                  double* __restrict__ h) {
    const int q4 = g.nx / 4;
    const long total = (long)q4 * g.ny * g.nz;
    const long t = (long)blockIdx.x * 256 + threadIdx.x;
    if (t >= total) return;
    const int q = (int)(t % q4);
    const long row = t / q4;
    const int j = (int)(row % g.ny), k = (int)(row / g.ny);
    const int NX = g.nx / kS, NY = g.ny / kS, NZ = g.nz / kS;
    int y0, y1, z0, z1;
    float wy, wz;
    lin_axis(j, NY, y0, y1, wy);
    lin_axis(k, NZ, z0, z1, wz);
    const float* r00 = yd + (long)NX * (y0 + (long)NY * z0);
    const float* r10 = yd + (long)NX * (y1 + (long)NY * z0);
    const float* r01 = yd + (long)NX * (y0 + (long)NY * z1);
    const float* r11 = yd + (long)NX * (y1 + (long)NY * z1);
    const double J = (hw - he) * inv_nx;
    double out[4];
#pragma unroll
    for (int e = 0; e < 4; ++e) {
        const int i = 4 * q + e;
        int x0, x1;
        float wx;
        lin_axis(i, NX, x0, x1, wx);
        const float c00 = r00[x0] * (1.f - wx) + r00[x1] * wx;
        const float c10 = r10[x0] * (1.f - wx) + r10[x1] * wx;
        const float c01 = r01[x0] * (1.f - wx) + r01[x1] * wx;
        const float c11 = r11[x0] * (1.f - wx) + r11[x1] * wx;
        const float c0 = c00 * (1.f - wy) + c10 * wy, c1 = c01 * (1.f - wy) + c11 * wy;
        const float yi = c0 * (1.f - wz) + c1 * wz;
        out[e] = hw + (he - hw) * ((i + 0.5) * inv_nx) + J * (double)yi;
    }
    double* o = h + row * g.nx + 4L * q;
    *reinterpret_cast<double2*>(o) = make_double2(out[0], out[1]);
    *reinterpret_cast<double2*>(o + 2) = make_double2(out[2], out[3]);
}

// per coarse cell V: target t = mean over its block of (h - h_lin) / J;
// dOut[V][0] = 2 (y - t) / N_coarse (channels 1..15 zero); loss partials. A
// workgroup holds 64 coarse cells x kS z-slices (one thread each, as
// input_kernel: four times the loads in flight of a thread per cell); the
// slices' sums are added in LDS in a fixed order.
__global__ void __launch_bounds__(256)
    loss_kernel(Geo g, double hw, double he, const float* __restrict__ y,
                const double* __restrict__ h, __hip_bfloat16* __restrict__ dOut,
                float* __restrict__ partials) {
    static_assert(kS == 4, "64 cells x 4 slices per workgroup");
    const int NX = g.nx / kS, NY = g.ny / kS, NZ = g.nz / kS;
    const long nc = (long)NX * NY * NZ;
    const int lane = (int)(threadIdx.x & 63), dz = (int)(threadIdx.x >> 6);
    const long V = (long)blockIdx.x * 64 + lane;
    const double Jg = (hw - he) / g.nx;
    double st = 0.0;
    if (V < nc) {
        const int I = (int)(V % NX);
        const long q = V / NX;
        const int J = (int)(q % NY), Kc = (int)(q / NY);
        double hl[kS];
#pragma unroll
        for (int dx = 0; dx < kS; ++dx) hl[dx] = hw + (he - hw) * (kS * I + dx + 0.5) / g.nx;
#pragma unroll
        for (int dy = 0; dy < kS; ++dy)
#pragma unroll
            for (int dx = 0; dx < kS; ++dx)
                st += h[(long)(kS * I + dx) +
                        (long)g.nx * ((kS * J + dy) + (long)g.ny * (kS * Kc + dz))] - hl[dx];
    }
    __shared__ double part[kS][64];
    part[dz][lane] = st;
    __syncthreads();
    if (dz != 0) return;  // whole waves
    float e2 = 0.0f;
    if (V < nc) {
        st = ((part[0][lane] + part[1][lane]) + part[2][lane]) + part[3][lane];
        const float t = (float)(st / Jg / (kS * kS * kS));
        const float d = y[V * 16] - t;
        e2 = d * d;
        uint4* o = reinterpret_cast<uint4*>(dOut + V * 16);
        const unsigned first = __builtin_bit_cast(unsigned short, f2bf(2.0f * d / (float)nc));
        o[0] = uint4{first, 0u, 0u, 0u};
        o[1] = uint4{0u, 0u, 0u, 0u};
    }
#pragma unroll
    for (int off = 32; off > 0; off >>= 1) e2 += __shfl_xor(e2, off, 64);
    if (lane == 0) partials[blockIdx.x] = e2;
}

// ---- parameters ------------------------------------------------------------------
// master weights of a layer: w[co][tap][ci] (FP32, tap as above), bias[co]
// W  [Cout_pad][Kpad]: W[co][tap*Cin_pad + ci] = w[co][tap][ci] (zero padded)
// Wt [Cin_pad][Kpad_t]: Wt[ci][tap*Cout_pad + co] = w[co][tap][ci], used with
//   FLIP (tap mirrored) for the data gradient
struct PackLayer {
    const float* w;
    int cin, cout, cin_pad, cout_pad, kpad, kpad_t;
    __hip_bfloat16* W;
    __hip_bfloat16* Wt;
    int block0;  // first workgroup of the layer
};
struct PackLayers {
    PackLayer l[kMaxWLayers];
    int n;
};
__global__ void __launch_bounds__(256) pack_kernel(PackLayers D) {
    int q = 0;
    while (q + 1 < D.n && D.l[q + 1].block0 <= (int)blockIdx.x) ++q;
    const PackLayer& L = D.l[q];
    const int e = ((int)blockIdx.x - L.block0) * 256 + (int)threadIdx.x;
    if (e < L.cout_pad * L.kpad) {
        const int co = e / L.kpad, k = e % L.kpad;
        const int tap = k / L.cin_pad, ci = k % L.cin_pad;
        float v = 0.0f;
        if (co < L.cout && tap < 27 && ci < L.cin) v = L.w[(co * 27 + tap) * L.cin + ci];
        L.W[e] = f2bf(v);
    }
    if (e < L.cin_pad * L.kpad_t) {
        const int ci = e / L.kpad_t, k = e % L.kpad_t;
        const int tap = k / L.cout_pad, co = k % L.cout_pad;
        float v = 0.0f;
        if (ci < L.cin && tap < 27 && co < L.cout) v = L.w[(co * 27 + tap) * L.cin + ci];
        L.Wt[e] = f2bf(v);
    }
}

// Adam (Kingma & Ba 2015) with bias correction folded into the step size
__global__ void __launch_bounds__(256)
    adam_kernel(float* __restrict__ p, const float* __restrict__ gr, float* __restrict__ m,
                float* __restrict__ v, long n, float lr_t, float b1, float b2, float eps) {
    const long e = (long)blockIdx.x * blockDim.x + threadIdx.x;
    if (e >= n) return;
    const float g = gr[e];
    const float mm = b1 * m[e] + (1.0f - b1) * g;
    const float vv = b2 * v[e] + (1.0f - b2) * g * g;
    m[e] = mm;
    v[e] = vv;
    p[e] -= lr_t * mm / (sqrtf(vv) + eps);
}

inline unsigned blocks(long n, int b = 256) { return (unsigned)((n + b - 1) / b); }

}  // namespace

// ===========================================================================
// host side
// ===========================================================================
namespace cnn {

struct LayerDef {
    int cin, cout, level;
};
// conv_a .. conv_g
constexpr LayerDef kLayers[7] = {{4, 16, 0},  {16, 32, 1}, {32, 64, 2}, {64, 64, 2},
                                 {64, 32, 1}, {32, 16, 0}, {16, 1, 0}};
constexpr int kNumLayers = 7;

inline int pad16(int c) { return (c + 15) & ~15; }
inline int kpad_of(int cin_pad) { return (27 * cin_pad + 31) / 32 * 32; }

long param_count() {
    long n = 0;
    for (const LayerDef& L : kLayers) n += 27L * L.cin * L.cout + L.cout;
    return n;
}

}  // namespace cnn
}  // namespace mf3d

using namespace mf3d;
using namespace mf3d::cnn;

// Weight gradients of up to kMaxWLayers layers: channel-first operand copies
// (zeroed) and per-slice partial sums in one allocation
struct WeightScratch {
    void* mem = nullptr;
    PlanarCopies copies{};
    int copy_blocks = 0;
    WLayers layers{};
};

struct mf3d_wsnet {
    float* params = nullptr;  // FP32 master: per layer w then bias
    float* grads = nullptr;
    float* adam_m = nullptr;
    float* adam_v = nullptr;
    long nparam = 0;
    long step = 0;
    long woff[kNumLayers], boff[kNumLayers];
    int cin_pad[kNumLayers], cout_pad[kNumLayers], kpad[kNumLayers], kpad_t[kNumLayers];
    __hip_bfloat16* W[kNumLayers] = {};
    __hip_bfloat16* Wt[kNumLayers] = {};
    bool packed = false;
    // activations for the current grid
    int gx = 0, gy = 0, gz = 0;
    std::vector<void*> act;
    __hip_bfloat16 *x0 = nullptr, *e0 = nullptr, *p1 = nullptr, *e1 = nullptr, *p2 = nullptr,
                   *e2 = nullptr, *e2b = nullptr, *d1 = nullptr, *d0 = nullptr;
    float* y = nullptr;  // [N0][16] FP32 (channel 0 used)
    float* yd = nullptr; // [N0] channel 0 of y, dense (read by the output interpolation)
    // backward: the layers' pre-activation gradients (kept until the weight
    // gradients, which run for all layers at once) and upsampled ones
    __hip_bfloat16 *g0a = nullptr, *g0b = nullptr, *g0c = nullptr, *g0d = nullptr, *g1a = nullptr,
                   *g1b = nullptr, *g1c = nullptr, *g2a = nullptr, *g2b = nullptr, *g2c = nullptr;
    WeightScratch wg;
    float* lpart = nullptr;
    float* host_lpart = nullptr;
    long lpart_cap = 0;
};

namespace {

int net_alloc(void** p, size_t bytes) {
    MF3D_HIP_TRY(hipMalloc(p, bytes ? bytes : 8));
    return MF3D_OK;
}

void free_acts(mf3d_wsnet* net) {
    for (void* p : net->act) (void)hipFree(p);
    net->act.clear();
    net->gx = net->gy = net->gz = 0;
    if (net->wg.mem) (void)hipFree(net->wg.mem);
    net->wg = WeightScratch{};
    if (net->lpart) (void)hipFree(net->lpart);
    if (net->host_lpart) (void)hipHostFree(net->host_lpart);
    net->lpart = net->host_lpart = nullptr;
    net->lpart_cap = 0;
}

int check_grid(const mf3d_grid* g) {
    MF3D_TRY(validate_grid(g));
    constexpr int q = kS * kF * kF;
    if ((g->nx % q) || (g->ny % q) || (g->nz % q))
        return fail(MF3D_ERR_UNSUPPORTED, "warm-start network needs sizes divisible by 16");
    return MF3D_OK;
}

// one layer whose weight gradient is wanted (dY, X: channels-last, 16 ct and 16
// it channels; up: X on the half-size grid)
struct WeightTask {
    mf3d_grid g;
    const __hip_bfloat16* dY;
    const __hip_bfloat16* X;
    int ct, it, up, cin, cout;
    float* gw;
    float* gb;
};

// Slices of a layer: 16 steps (512 voxels) a wave amortise its partial sums;
// fewer steps where the layer would otherwise have under 8 slices (27 taps x 8
// waves), more above 64 slices (whose partial sums would grow with the grid).
// out is written last, once all of it is ready: a scratch with memory counts as
// usable, so a failed zeroing must leave none. The zeroing goes to the stream of
// the gradients that need it and waits for nothing.
int make_scratch(hipStream_t s, WeightScratch& out, const WeightTask* T, int n) {
    WeightScratch S;
    S.layers.n = n;
    size_t bytes = 0;
    auto take = [&](size_t b) {
        const size_t at = bytes;
        bytes += (b + 255) / 256 * 256;
        return at;
    };
    std::vector<size_t> at;
    for (int e = 0; e < n; ++e) {  // the operand copies first: they are zeroed
        const WeightTask& t = T[e];
        WLayer& L = S.layers.l[e];
        L.P = planar_of(t.g);
        L.ct = t.ct, L.it = t.it;
        at.push_back(take((size_t)16 * L.ct * L.P.plane * 2));
        at.push_back(take((size_t)16 * L.it * L.P.plane * 2));
    }
    const size_t copies = bytes;
    for (int e = 0; e < n; ++e) {
        const WeightTask& t = T[e];
        WLayer& L = S.layers.l[e];
        const long steps = (L.P.groups + 3) / 4;
        L.steps = (int)std::max({1L, std::min(16L, steps / 8), (steps + 63) / 64});
        L.slices = (int)((steps + L.steps - 1) / L.steps);
        L.wave0 = S.layers.waves;
        S.layers.waves += 27 * L.slices;
        L.cin = t.cin, L.cout = t.cout, L.gw = t.gw, L.gb = t.gb;
        L.elem0 = S.layers.elems;
        S.layers.elems += 27 * t.cin * t.cout + t.cout;
        at.push_back(take((size_t)L.slices * 16 * L.ct * 27 * 16 * L.it * 4));
        at.push_back(take((size_t)L.slices * 16 * L.ct * 4));
        for (int q = 0; q < 2; ++q) {
            PlanarCopy& C = S.copies.c[S.copies.n++];
            C.src = q ? t.X : t.dY;
            C.ch = 16 * (q ? t.it : t.ct);
            C.up = q ? t.up : 0;
            C.g = Geo{t.g.nx, t.g.ny, t.g.nz};
            C.P = L.P;
            C.block0 = S.copy_blocks;
            C.vblocks = (int)blocks((long)cells(t.g));
            S.copy_blocks += C.vblocks * (C.ch / 8);
        }
    }
    MF3D_TRY(net_alloc(&S.mem, bytes));
    // the copies' borders stay zero: planar_kernel writes the voxels only
    zero_kernel<<<blocks((long)(copies / 16)), 256, 0, s>>>(static_cast<uint4*>(S.mem),
                                                           (long)(copies / 16));
    const hipError_t err = hipGetLastError();
    if (err != hipSuccess) {
        (void)hipFree(S.mem);
        return fail(MF3D_ERR_HIP, std::string("weight-gradient scratch: ") + hipGetErrorString(err));
    }
    char* m = static_cast<char*>(S.mem);
    for (int e = 0; e < n; ++e) {
        WLayer& L = S.layers.l[e];
        __hip_bfloat16* d[2] = {(__hip_bfloat16*)(m + at[2 * e]), (__hip_bfloat16*)(m + at[2 * e + 1])};
        L.dY = d[0], L.X = d[1];
        S.copies.c[2 * e].dst = d[0];
        S.copies.c[2 * e + 1].dst = d[1];
        L.part = (float*)(m + at[2 * n + 2 * e]);
        L.bpart = (float*)(m + at[2 * n + 2 * e + 1]);
    }
    out = S;
    return MF3D_OK;
}

int run_weight_grads(hipStream_t s, const WeightScratch& S) {
    planar_kernel<<<S.copy_blocks, 256, 0, s>>>(S.copies);
    wgrad_kernel<<<(S.layers.waves + 3) / 4, 256, 0, s>>>(S.layers);
    wgrad_reduce_kernel<<<blocks(S.layers.elems), 256, 0, s>>>(S.layers);
    MF3D_HIP_TRY(hipGetLastError());
    return MF3D_OK;
}

int ensure_acts(mf3d_wsnet* net, const mf3d_grid& g) {
    if (net->gx == g.nx && net->gy == g.ny && net->gz == g.nz) return MF3D_OK;
    free_acts(net);
    const size_t n0 = cells(g), n1 = n0 / (kF * kF * kF), n2 = n1 / (kF * kF * kF);
    auto bf = [&](__hip_bfloat16** p, size_t elems) -> int {
        void* q = nullptr;
        MF3D_TRY(net_alloc(&q, elems * sizeof(__hip_bfloat16)));
        net->act.push_back(q);
        *p = static_cast<__hip_bfloat16*>(q);
        return MF3D_OK;
    };
    MF3D_TRY(bf(&net->x0, n0 * 16));
    MF3D_TRY(bf(&net->e0, n0 * 16));
    MF3D_TRY(bf(&net->p1, n1 * 16));
    MF3D_TRY(bf(&net->e1, n1 * 32));
    MF3D_TRY(bf(&net->p2, n2 * 32));
    MF3D_TRY(bf(&net->e2, n2 * 64));
    MF3D_TRY(bf(&net->e2b, n2 * 64));
    MF3D_TRY(bf(&net->d1, n1 * 32));
    MF3D_TRY(bf(&net->d0, n0 * 16));
    MF3D_TRY(bf(&net->g0a, n0 * 32));
    MF3D_TRY(bf(&net->g0b, n0 * 32));
    MF3D_TRY(bf(&net->g0c, n0 * 16));
    MF3D_TRY(bf(&net->g0d, n0 * 16));
    MF3D_TRY(bf(&net->g1c, n1 * 16));
    MF3D_TRY(bf(&net->g2c, n2 * 32));
    MF3D_TRY(bf(&net->g1a, n1 * 64));
    MF3D_TRY(bf(&net->g1b, n1 * 64));
    MF3D_TRY(bf(&net->g2a, n2 * 64));
    MF3D_TRY(bf(&net->g2b, n2 * 64));
    void* q = nullptr;
    MF3D_TRY(net_alloc(&q, n0 * 16 * sizeof(float)));
    net->act.push_back(q);
    net->y = static_cast<float*>(q);
    MF3D_TRY(net_alloc(&q, n0 * sizeof(float)));
    net->act.push_back(q);
    net->yd = static_cast<float*>(q);
    const long nb = ((long)n0 + 63) / 64;  // workgroups of loss_kernel
    MF3D_TRY(net_alloc((void**)&net->lpart, nb * sizeof(float)));
    MF3D_HIP_TRY(hipHostMalloc((void**)&net->host_lpart, nb * sizeof(float), hipHostMallocDefault));
    net->lpart_cap = nb;
    net->gx = g.nx;
    net->gy = g.ny;
    net->gz = g.nz;
    return MF3D_OK;
}

// appends a layer to D; returns the workgroups so far
int add_pack(PackLayers& D, int block0, const float* w, int cin, int cout, int cin_pad,
             int cout_pad, __hip_bfloat16* W, __hip_bfloat16* Wt) {
    const int kp = kpad_of(cin_pad), kpt = kpad_of(cout_pad);
    D.l[D.n++] = PackLayer{w, cin, cout, cin_pad, cout_pad, kp, kpt, W, Wt, block0};
    return block0 + (int)blocks(std::max((long)cout_pad * kp, (long)cin_pad * kpt));
}

int pack(mf3d_wsnet* net, hipStream_t s) {
    PackLayers D{};
    int nb = 0;
    for (int l = 0; l < kNumLayers; ++l)
        nb = add_pack(D, nb, net->params + net->woff[l], kLayers[l].cin, kLayers[l].cout,
                      net->cin_pad[l], net->cout_pad[l], net->W[l], net->Wt[l]);
    pack_kernel<<<nb, 256, 0, s>>>(D);
    MF3D_HIP_TRY(hipGetLastError());
    net->packed = true;
    return MF3D_OK;
}

// one convolution: out[v][0..cs) from X[v][0..cin_ch) with W (cout_pad rows)
int conv(hipStream_t s, const mf3d_grid& g, int cin_ch, int cout_pad, int kp, int cs,
         const __hip_bfloat16* X, const __hip_bfloat16* W, const float* bias,
         const __hip_bfloat16* R, const __hip_bfloat16* M, bool relu, bool flip, void* out,
         bool f32out, bool up = false) {
    const Geo G{g.nx, g.ny, g.nz};
    // 16-voxel tiles per wave: kVT on large grids, fewer where that would
    // leave the launch with fewer than kConvWaves waves (the small grids of
    // the deeper layers; same products and order per output either way); below
    // that, waves share a tile's k steps (kConvWaves / 4 tiles and fewer: 4, a
    // sixteenth and fewer: 16)
    const long nv = (long)cells(g);
    const int vt = (nv + 16 * kVT - 1) / (16 * kVT) >= kConvWaves ? kVT
                   : (nv + 31) / 32 >= kConvWaves                   ? 2
                                                                    : 1;
    const long tiles = (nv + 16L * vt - 1) / (16L * vt);
    const int ks = vt > 1 ? 1 : tiles <= kConvWaves / 16 ? 16 : tiles <= kConvWaves / 4 ? 4 : 1;
    const int wpb = ks > 4 ? ks : 4;
    const unsigned nb = (unsigned)((tiles * ks + wpb - 1) / wpb);
    const int ct = cout_pad / 16;
#define MF3D_CONV(CTV, VTV, F32, KSV)                                                          \
    conv_kernel<CTV, VTV, F32, KSV><<<nb, wpb * 64, 0, s>>>(                                    \
        G, cin_ch, kp, cs, up ? 1 : 0, X, W, bias, R, M, relu ? 1 : 0, flip ? 1 : 0, out)
#define MF3D_CONV_VT(CTV, F32)                                                                 \
    do {                                                                                       \
        if (vt == kVT) MF3D_CONV(CTV, kVT, F32, 1);                                            \
        else if (vt == 2) MF3D_CONV(CTV, 2, F32, 1);                                           \
        else if (ks == 1) MF3D_CONV(CTV, 1, F32, 1);                                           \
        else if (ks == 4) MF3D_CONV(CTV, 1, F32, 4);                                           \
        else MF3D_CONV(CTV, 1, F32, 16);                                                       \
    } while (0)
    if (f32out) {
        if (ct != 1) return fail(MF3D_ERR_UNSUPPORTED, "FP32 output only for 16 channels");
        MF3D_CONV_VT(1, true);
    } else if (ct == 1) MF3D_CONV_VT(1, false);
    else if (ct == 2) MF3D_CONV_VT(2, false);
    else if (ct == 4) MF3D_CONV_VT(4, false);
    else return fail(MF3D_ERR_UNSUPPORTED, "convolution: unsupported channel count");
#undef MF3D_CONV_VT
#undef MF3D_CONV
    MF3D_HIP_TRY(hipGetLastError());
    return MF3D_OK;
}

mf3d_grid coarse(const mf3d_grid& g, int f) {
    mf3d_grid c = g;
    c.nx /= f;
    c.ny /= f;
    c.nz /= f;
    return c;
}

// forward pass for the fine grid gf (the network runs on gf / kS)
int forward(mf3d_wsnet* net, hipStream_t s, const mf3d_grid& gf, const double* K, int is_log) {
    const mf3d_grid g = coarse(gf, kS);
    MF3D_TRY(ensure_acts(net, g));
    if (!net->packed) MF3D_TRY(pack(net, s));
    const mf3d_grid g1 = coarse(g, kF), g2 = coarse(g, kF * kF);
    const Geo G0{g.nx, g.ny, g.nz}, G1{g1.nx, g1.ny, g1.nz};
    const long n0 = (long)cells(g), n1 = (long)cells(g1), n2 = (long)cells(g2);
    float* P = net->params;
    input_kernel<<<(unsigned)((n0 + 63) / 64), 256, 0, s>>>(Geo{gf.nx, gf.ny, gf.nz}, K, is_log,
                                                          net->x0);
    MF3D_TRY(conv(s, g, 16, 16, net->kpad[0], 16, net->x0, net->W[0], P + net->boff[0], nullptr,
                  nullptr, true, false, net->e0, false));
    pool_kernel<<<blocks(n1 * 16), 256, 0, s>>>(G0, 16, net->e0, net->p1);
    MF3D_TRY(conv(s, g1, 16, 32, net->kpad[1], 32, net->p1, net->W[1], P + net->boff[1], nullptr,
                  nullptr, true, false, net->e1, false));
    pool_kernel<<<blocks(n2 * 32), 256, 0, s>>>(G1, 32, net->e1, net->p2);
    MF3D_TRY(conv(s, g2, 32, 64, net->kpad[2], 64, net->p2, net->W[2], P + net->boff[2], nullptr,
                  nullptr, true, false, net->e2, false));
    MF3D_TRY(conv(s, g2, 64, 64, net->kpad[3], 64, net->e2, net->W[3], P + net->boff[3], nullptr,
                  nullptr, true, false, net->e2b, false));
    MF3D_TRY(conv(s, g1, 64, 32, net->kpad[4], 32, net->e2b, net->W[4], P + net->boff[4], net->e1,
                  nullptr, true, false, net->d1, false, true));
    MF3D_TRY(conv(s, g, 32, 16, net->kpad[5], 16, net->d1, net->W[5], P + net->boff[5], net->e0,
                  nullptr, true, false, net->d0, false, true));
    MF3D_TRY(conv(s, g, 16, 16, net->kpad[6], 16, net->d0, net->W[6], P + net->boff[6], nullptr,
                  nullptr, false, false, net->y, true));
    MF3D_HIP_TRY(hipGetLastError());
    return MF3D_OK;
}

// loss and all parameter gradients (net->grads) for target head h
int backward(mf3d_wsnet* net, hipStream_t s, const mf3d_grid& gf, double hw, double he,
             const double* h, double* loss) {
    const mf3d_grid g = coarse(gf, kS);
    const mf3d_grid g1 = coarse(g, kF), g2 = coarse(g, kF * kF);
    const Geo G0{g.nx, g.ny, g.nz}, G1{g1.nx, g1.ny, g1.nz};
    const long n0 = (long)cells(g), n1 = (long)cells(g1), n2 = (long)cells(g2);
    const unsigned lb = (unsigned)((n0 + 63) / 64);
    float* GR = net->grads;
    // dY of conv_g (16 channels, channel 0 live) -> g0c
    loss_kernel<<<lb, 256, 0, s>>>(Geo{gf.nx, gf.ny, gf.nz}, hw, he, net->y, h, net->g0c,
                                   net->lpart);
    // conv_g: data gradient masked by d0 > 0 -> dPre_f (g0b, 16 ch), also e0's skip gradient
    MF3D_TRY(conv(s, g, 16, 16, net->kpad_t[6], 16, net->g0c, net->Wt[6], nullptr, nullptr,
                  net->d0, false, true, net->g0b, false));
    MF3D_TRY(conv(s, g, 16, 32, net->kpad_t[5], 32, net->g0b, net->Wt[5], nullptr, nullptr,
                  nullptr, false, true, net->g0a, false));  // du0 (32 ch)
    // up bwd into d1, masked by d1 > 0 -> dPre_e (g1a, 32 ch)
    up_bwd_kernel<<<blocks(n1 * 32), 256, 0, s>>>(G0, 32, net->g0a, net->d1, net->g1a);
    MF3D_TRY(conv(s, g1, 32, 64, net->kpad_t[4], 64, net->g1a, net->Wt[4], nullptr, nullptr,
                  nullptr, false, true, net->g1b, false));  // du1 (64 ch)
    // up bwd into e2b, masked -> dPre_d (g2a)
    up_bwd_kernel<<<blocks(n2 * 64), 256, 0, s>>>(G1, 64, net->g1b, net->e2b, net->g2a);
    MF3D_TRY(conv(s, g2, 64, 64, net->kpad_t[3], 64, net->g2a, net->Wt[3], nullptr, nullptr,
                  net->e2, false, true, net->g2b, false));  // dPre_c (64 ch)
    MF3D_TRY(conv(s, g2, 64, 32, net->kpad_t[2], 32, net->g2b, net->Wt[2], nullptr, nullptr,
                  nullptr, false, true, net->g2c, false));  // dp2 (32 ch)
    // pool bwd into e1 + skip gradient (g1a), masked by e1 -> dPre_b (g1b, 32 ch)
    pool_bwd_kernel<<<blocks(n1 * 32), 256, 0, s>>>(G1, 32, net->g2c, net->g1a, net->e1, net->g1b);
    MF3D_TRY(conv(s, g1, 32, 16, net->kpad_t[1], 16, net->g1b, net->Wt[1], nullptr, nullptr,
                  nullptr, false, true, net->g1c, false));  // dp1 (16 ch)
    // pool bwd into e0 + skip gradient (g0b), masked by e0 -> dPre_a (g0d, 16 ch)
    pool_bwd_kernel<<<blocks(n0 * 16), 256, 0, s>>>(G0, 16, net->g1c, net->g0b, net->e0, net->g0d);
    MF3D_HIP_TRY(hipGetLastError());
    if (!net->wg.mem) {
        const struct {
            const mf3d_grid* g;
            const __hip_bfloat16 *dY, *X;
            int up;
        } in[kNumLayers] = {{&g, net->g0d, net->x0, 0},   {&g1, net->g1b, net->p1, 0},
                            {&g2, net->g2b, net->p2, 0},  {&g2, net->g2a, net->e2, 0},
                            {&g1, net->g1a, net->e2b, 1}, {&g, net->g0b, net->d1, 1},
                            {&g, net->g0c, net->d0, 0}};
        WeightTask T[kNumLayers];
        for (int l = 0; l < kNumLayers; ++l)
            T[l] = WeightTask{*in[l].g, in[l].dY, in[l].X, net->cout_pad[l] / 16,
                              net->cin_pad[l] / 16, in[l].up, kLayers[l].cin, kLayers[l].cout,
                              GR + net->woff[l], GR + net->boff[l]};
        MF3D_TRY(make_scratch(s, net->wg, T, kNumLayers));
    }
    MF3D_TRY(run_weight_grads(s, net->wg));
    if (loss) {
        MF3D_HIP_TRY(hipMemcpyAsync(net->host_lpart, net->lpart, lb * sizeof(float),
                                    hipMemcpyDeviceToHost, s));
        MF3D_HIP_TRY(hipStreamSynchronize(s));
        double t = 0.0;
        for (unsigned b = 0; b < lb; ++b) t += net->host_lpart[b];
        *loss = t / (double)n0;
    }
    MF3D_HIP_TRY(hipGetLastError());
    return MF3D_OK;
}

int x_dirichlet(const mf3d_bc* bc, double* hw, double* he) {
    if (bc->type[0] != MF3D_BC_DIRICHLET || bc->type[1] != MF3D_BC_DIRICHLET)
        return fail(MF3D_ERR_UNSUPPORTED, "warm start needs Dirichlet x faces");
    if (bc->value[0] == bc->value[1])
        return fail(MF3D_ERR_UNSUPPORTED, "warm start needs h_west != h_east");
    *hw = bc->value[0];
    *he = bc->value[1];
    return MF3D_OK;
}

}  // namespace

// ===========================================================================
// C ABI
// ===========================================================================
extern "C" {

int mf3d_wsnet_destroy(mf3d_wsnet* net);

long mf3d_wsnet_param_count(void) { return param_count(); }

int mf3d_wsnet_create(mf3d_wsnet** out) {
    if (!out) return fail(MF3D_ERR_INVALID_ARGUMENT, "null output pointer");
    mf3d_wsnet* net = new mf3d_wsnet();
    long off = 0;
    for (int l = 0; l < kNumLayers; ++l) {
        const LayerDef& L = kLayers[l];
        net->woff[l] = off;
        off += 27L * L.cin * L.cout;
        net->boff[l] = off;
        off += L.cout;
        net->cin_pad[l] = pad16(L.cin);
        net->cout_pad[l] = pad16(L.cout);
        net->kpad[l] = kpad_of(net->cin_pad[l]);
        net->kpad_t[l] = kpad_of(net->cout_pad[l]);
    }
    net->nparam = off;
    int st = MF3D_OK;
    auto al = [&](float** p) {
        if (st == MF3D_OK) st = net_alloc((void**)p, off * sizeof(float));
    };
    al(&net->params);
    al(&net->grads);
    al(&net->adam_m);
    al(&net->adam_v);
    for (int l = 0; l < kNumLayers && st == MF3D_OK; ++l) {
        st = net_alloc((void**)&net->W[l], (size_t)net->cout_pad[l] * net->kpad[l] * 2);
        if (st == MF3D_OK)
            st = net_alloc((void**)&net->Wt[l], (size_t)pad16(net->cin_pad[l]) * net->kpad_t[l] * 2);
    }
    if (st == MF3D_OK) {
        hipError_t e = hipMemset(net->params, 0, off * sizeof(float));
        if (e == hipSuccess) e = hipMemset(net->adam_m, 0, off * sizeof(float));
        if (e == hipSuccess) e = hipMemset(net->adam_v, 0, off * sizeof(float));
        if (e != hipSuccess) st = fail(MF3D_ERR_HIP, hipGetErrorString(e));
    }
    if (st != MF3D_OK) {
        mf3d_wsnet_destroy(net);
        return st;
    }
    *out = net;
    return MF3D_OK;
}

int mf3d_wsnet_destroy(mf3d_wsnet* net) {
    if (!net) return MF3D_OK;
    free_acts(net);
    for (float* p : {net->params, net->grads, net->adam_m, net->adam_v})
        if (p) (void)hipFree(p);
    for (int l = 0; l < kNumLayers; ++l) {
        if (net->W[l]) (void)hipFree(net->W[l]);
        if (net->Wt[l]) (void)hipFree(net->Wt[l]);
    }
    delete net;
    return MF3D_OK;
}

int mf3d_wsnet_set_params(mf3d_wsnet* net, const float* host, long n) {
    if (!net || !host) return fail(MF3D_ERR_INVALID_ARGUMENT, "null pointer");
    if (n != net->nparam) return fail(MF3D_ERR_SIZE_MISMATCH, "parameter count");
    MF3D_HIP_TRY(hipMemcpy(net->params, host, n * sizeof(float), hipMemcpyHostToDevice));
    MF3D_HIP_TRY(hipMemset(net->adam_m, 0, n * sizeof(float)));
    MF3D_HIP_TRY(hipMemset(net->adam_v, 0, n * sizeof(float)));
    net->step = 0;
    net->packed = false;
    return MF3D_OK;
}

int mf3d_wsnet_get_params(const mf3d_wsnet* net, float* host, long n) {
    if (!net || !host) return fail(MF3D_ERR_INVALID_ARGUMENT, "null pointer");
    if (n != net->nparam) return fail(MF3D_ERR_SIZE_MISMATCH, "parameter count");
    MF3D_HIP_TRY(hipMemcpy(host, net->params, n * sizeof(float), hipMemcpyDeviceToHost));
    return MF3D_OK;
}

int mf3d_wsnet_get_grads(const mf3d_wsnet* net, float* host, long n) {
    if (!net || !host) return fail(MF3D_ERR_INVALID_ARGUMENT, "null pointer");
    if (n != net->nparam) return fail(MF3D_ERR_SIZE_MISMATCH, "parameter count");
    MF3D_HIP_TRY(hipMemcpy(host, net->grads, n * sizeof(float), hipMemcpyDeviceToHost));
    return MF3D_OK;
}

int mf3d_wsnet_predict(mf3d_wsnet* net, mf3d_stream stream, const mf3d_grid* grid,
                       const mf3d_bc* bc, const double* K, int k_is_log, double* h0, size_t n) {
    if (!net || !grid || !bc || !K || !h0) return fail(MF3D_ERR_INVALID_ARGUMENT, "null pointer");
    MF3D_TRY(check_grid(grid));
    if (n < cells(*grid)) return fail(MF3D_ERR_SIZE_MISMATCH, "h0/K shorter than the grid");
    double hw, he;
    MF3D_TRY(x_dirichlet(bc, &hw, &he));
    (void)hipGetLastError();
    hipStream_t s = reinterpret_cast<hipStream_t>(stream);
    MF3D_TRY(forward(net, s, *grid, K, k_is_log));
    // channel 0 densely first: the interpolation's 8 gathers per cell then
    // share cache lines between neighbouring cells
    const long n0 = cells(*grid) / ((long)kS * kS * kS);
    channel0_kernel<<<blocks(n0), 256, 0, s>>>(net->y, 16, n0, net->yd);
    // h0 must be 16-byte aligned for the paired stores (the network's sizes
    // make every row start so)
    if (reinterpret_cast<uintptr_t>(h0) & 15)
        return fail(MF3D_ERR_UNSUPPORTED, "warm-start output needs a 16-byte aligned head");
    const long quads = cells(*grid) / 4;
    output_kernel<<<(unsigned)((quads + 255) / 256), 256, 0, s>>>(
        Geo{grid->nx, grid->ny, grid->nz}, hw, he, 1.0 / grid->nx, net->yd, h0);
    MF3D_HIP_TRY(hipGetLastError());
    return MF3D_OK;
}

int mf3d_wsnet_gradients(mf3d_wsnet* net, mf3d_stream stream, const mf3d_grid* grid,
                         const mf3d_bc* bc, const double* K, int k_is_log, const double* h,
                         size_t n, double* loss) {
    if (!net || !grid || !bc || !K || !h) return fail(MF3D_ERR_INVALID_ARGUMENT, "null pointer");
    MF3D_TRY(check_grid(grid));
    if (n < cells(*grid)) return fail(MF3D_ERR_SIZE_MISMATCH, "h/K shorter than the grid");
    double hw, he;
    MF3D_TRY(x_dirichlet(bc, &hw, &he));
    (void)hipGetLastError();
    hipStream_t s = reinterpret_cast<hipStream_t>(stream);
    MF3D_TRY(forward(net, s, *grid, K, k_is_log));
    return backward(net, s, *grid, hw, he, h, loss);
}

int mf3d_wsnet_train_step(mf3d_wsnet* net, mf3d_stream stream, const mf3d_grid* grid,
                          const mf3d_bc* bc, const double* K, int k_is_log, const double* h,
                          size_t n, double lr, double* loss) {
    MF3D_TRY(mf3d_wsnet_gradients(net, stream, grid, bc, K, k_is_log, h, n, loss));
    hipStream_t s = reinterpret_cast<hipStream_t>(stream);
    const float b1 = 0.9f, b2 = 0.999f;
    net->step += 1;
    const double c1 = 1.0 - std::pow((double)b1, (double)net->step);
    const double c2 = 1.0 - std::pow((double)b2, (double)net->step);
    const float lr_t = (float)(lr * std::sqrt(c2) / c1);
    adam_kernel<<<blocks(net->nparam), 256, 0, s>>>(net->params, net->grads, net->adam_m,
                                                    net->adam_v, net->nparam, lr_t, b1, b2, 1e-8f);
    MF3D_HIP_TRY(hipGetLastError());
    net->packed = false;
    return MF3D_OK;
}

// single convolution layer for tests: X [N][cin] BF16 (cin a multiple of 8),
// w [cout][27][cin] FP32, bias [cout] FP32 (nullable), R [N][cout] (nullable,
// added before the ReLU), relu; Y [N][cout] BF16 (cout a multiple of 16, <= 64)
int mf3d_conv3d_forward(mf3d_stream stream, const mf3d_grid* grid, int cin, int cout,
                        const void* X, const float* w, const float* bias, const void* R,
                        int relu, void* Y) {
    if (!grid || !X || !w || !Y) return fail(MF3D_ERR_INVALID_ARGUMENT, "null pointer");
    MF3D_TRY(validate_grid(grid));
    if (cin % 8 || cin > 128 || cout % 16 || cout > 64)
        return fail(MF3D_ERR_UNSUPPORTED, "cin must be a multiple of 8, cout 16/32/64");
    (void)hipGetLastError();
    hipStream_t s = reinterpret_cast<hipStream_t>(stream);
    const int kp = kpad_of(cin), kpt = kpad_of(cout);
    __hip_bfloat16 *W = nullptr, *Wt = nullptr;
    MF3D_TRY(net_alloc((void**)&W, (size_t)cout * kp * 2));
    int st = net_alloc((void**)&Wt, (size_t)pad16(cin) * kpt * 2);
    if (st == MF3D_OK) {
        PackLayers D{};
        const int nb = add_pack(D, 0, w, cin, cout, cin, cout, W, Wt);
        pack_kernel<<<nb, 256, 0, s>>>(D);
        st = conv(s, *grid, cin, cout, kp, cout, (const __hip_bfloat16*)X, W, bias,
                  (const __hip_bfloat16*)R, nullptr, relu != 0, false, Y, false);
    }
    if (st == MF3D_OK) {
        const hipError_t e = hipStreamSynchronize(s);
        if (e != hipSuccess) st = fail(MF3D_ERR_HIP, hipGetErrorString(e));
    }
    (void)hipFree(W);
    if (Wt) (void)hipFree(Wt);
    return st;
}

// data gradient of a convolution: dX [N][cin] = sum over taps/cout of w and
// dY [N][cout], times (M > 0) if M [N][cin] is given (the ReLU of X)
int mf3d_conv3d_backward_data(mf3d_stream stream, const mf3d_grid* grid, int cin, int cout,
                              const void* dY, const float* w, const void* M, void* dX) {
    if (!grid || !dY || !w || !dX) return fail(MF3D_ERR_INVALID_ARGUMENT, "null pointer");
    MF3D_TRY(validate_grid(grid));
    if (cin % 16 || cin > 64 || cout % 16 || cout > 64)
        return fail(MF3D_ERR_UNSUPPORTED, "cin and cout must be 16/32/64");
    (void)hipGetLastError();
    hipStream_t s = reinterpret_cast<hipStream_t>(stream);
    const int kp = kpad_of(cin), kpt = kpad_of(cout);
    __hip_bfloat16 *W = nullptr, *Wt = nullptr;
    MF3D_TRY(net_alloc((void**)&W, (size_t)cout * kp * 2));
    int st = net_alloc((void**)&Wt, (size_t)cin * kpt * 2);
    if (st == MF3D_OK) {
        PackLayers D{};
        const int nb = add_pack(D, 0, w, cin, cout, cin, cout, W, Wt);
        pack_kernel<<<nb, 256, 0, s>>>(D);
        st = conv(s, *grid, cout, cin, kpt, cin, (const __hip_bfloat16*)dY, Wt, nullptr, nullptr,
                  (const __hip_bfloat16*)M, false, true, dX, false);
    }
    if (st == MF3D_OK) {
        const hipError_t e = hipStreamSynchronize(s);
        if (e != hipSuccess) st = fail(MF3D_ERR_HIP, hipGetErrorString(e));
    }
    (void)hipFree(W);
    if (Wt) (void)hipFree(Wt);
    return st;
}

// weight and bias gradients: gw [cout][27][cin] = sum_v dY[v][co] X[v + d][ci],
// gb [cout] = sum_v dY[v][co] (FP32)
int mf3d_conv3d_backward_weights(mf3d_stream stream, const mf3d_grid* grid, int cin, int cout,
                                 const void* X, const void* dY, float* gw, float* gb) {
    if (!grid || !X || !dY || !gw || !gb) return fail(MF3D_ERR_INVALID_ARGUMENT, "null pointer");
    MF3D_TRY(validate_grid(grid));
    if (cin % 16 || cin > 64 || cout % 16 || cout > 64)
        return fail(MF3D_ERR_UNSUPPORTED, "cin and cout must be 16/32/64");
    (void)hipGetLastError();
    hipStream_t s = reinterpret_cast<hipStream_t>(stream);
    const int ct = cout / 16, it = cin / 16;
    const bool known = (ct == 1 && it <= 2) || (ct == 2 && (it == 1 || it == 4)) ||
                       (ct == 4 && (it == 2 || it == 4));
    if (!known) return fail(MF3D_ERR_UNSUPPORTED, "weight gradient: unsupported channel counts");
    const WeightTask T{*grid, (const __hip_bfloat16*)dY, (const __hip_bfloat16*)X, ct, it, 0, cin,
                       cout, gw, gb};
    WeightScratch S;
    int st = make_scratch(s, S, &T, 1);
    if (st == MF3D_OK) st = run_weight_grads(s, S);
    if (st == MF3D_OK) {
        const hipError_t e = hipStreamSynchronize(s);
        if (e != hipSuccess) st = fail(MF3D_ERR_HIP, hipGetErrorString(e));
    }
    if (S.mem) (void)hipFree(S.mem);
    return st;
}

}  // extern "C"
