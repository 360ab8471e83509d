// Colour-split FP32 V-cycle levels: storage, faces and the Gauss-Seidel value,
// shared by the one-colour sweeps (faces.hip) and the fused smoothing passes
// (fused32.hip).
#pragma once

#include <hip/hip_bf16.h>
#include <hip/hip_fp16.h>

#include "hface.hpp"

namespace mf3d {

struct Dims {
    int nx, ny, nz;
    __device__ long fx(int i, int j, int k) const {
        return (long)i + (long)(nx + 1) * ((long)j + (long)ny * k);
    }
    __device__ long fy(int i, int j, int k) const {
        return (long)i + (long)nx * ((long)j + (long)(ny + 1) * k);
    }
    __device__ long fz(int i, int j, int k) const {
        return (long)i + (long)nx * ((long)j + (long)ny * k);
    }
};

// ---- coefficient storage conversions ---------------------------------------
__device__ __forceinline__ double cload(const double* p, long i) { return p[i]; }
__device__ __forceinline__ float cload(const float* p, long i) { return p[i]; }
__device__ __forceinline__ float cload(const __hip_bfloat16* p, long i) {
    return __bfloat162float(p[i]);
}
__device__ __forceinline__ float cload(const __half* p, long i) { return __half2float(p[i]); }

// GSRB cell value (sum f x_nb - b cs dx^2) / sum f, summed x+, x-, y+, y-,
// z+, z- as in gsrb_interior_kernel (gsrb_3d.cu:53-69); pin doubles the
// diagonal of cell 0 (gsrb_3d.cu:360-362). The multiply-adds are written as
// fma: the first product is rounded, each later one is fused into the running
// sum, and b bs into the last step. Left to contraction, the compiler may
// fuse either product of a pair depending on the code around a call, and two
// kernels calling this would then differ in the last bit.
// The quotient is the hardware reciprocal's, corrected once by its remainder (the
// rounded quotient: no other in 3e9 random pairs), with the hardware's fix-up for
// zeros and infinities: half the instructions of a division.
__device__ __forceinline__ float gs_quot(float n, float d) {
    const float r = __builtin_amdgcn_rcpf(d);
    const float q = n * r;
    return __builtin_amdgcn_div_fixupf(fmaf(fmaf(-q, d, n), r, q), d, n);
}
__device__ __forceinline__ double gs_quot(double n, double d) { return n / d; }
template <typename T>
__device__ __forceinline__ T gs_value(const T (&f)[6], const T (&v)[6], T b, T bs, bool pin0) {
    T result = v[0] * f[0];
    result = fma(v[1], f[1], result);
    result = fma(v[2], f[2], result);
    result = fma(v[3], f[3], result);
    result = fma(v[4], f[4], result);
    result = fma(v[5], f[5], result);
    T aC = f[0] + f[1] + f[2] + f[3] + f[4] + f[5];
    if (pin0) aC *= T(2);
    return gs_quot(fma(-b, bs, result), aC);
}

// faces (x+, x-, y+, y-, z+, z-) of cell (i,j,k) of a natural-order level
template <typename T, typename TC>
__device__ __forceinline__ void cell_faces(const Dims& d, const TC* FX, const TC* FY,
                                           const TC* FZ, int i, int j, int k, T (&f)[6]) {
    f[0] = (T)cload(FX, d.fx(i + 1, j, k));
    f[1] = (T)cload(FX, d.fx(i, j, k));
    f[2] = (T)cload(FY, d.fy(i, j + 1, k));
    f[3] = (T)cload(FY, d.fy(i, j, k));
    f[4] = (T)cload(FZ, d.fz(i, j, k + 1));
    f[5] = (T)cload(FZ, d.fz(i, j, k));
}

// ---- colour-split storage of the FP32 V-cycle levels -----------------------------
// With even nx, ny, nz a level's x and b may be stored colour by colour: the
// cells of colour c = (i+j+k) & 1 at c*N/2 + (i >> 1) + (nx/2)(j + ny k). A
// half-sweep then reads only the opposite colour's x and its own colour's b
// and writes only its own colour, all with unit stride.
// Every neighbour of a cell has the other colour: the y and z neighbours sit at
// the same (i >> 1) one row or plane away, the x neighbours at ((i +- 1) >> 1)
// of the same row.
// The face coefficients of such a level are stored the same way, each face
// with the cell on its upper side: LX/LY/LZ[split(i,j,k)] hold the faces
// between (i-1,j,k)|(i,j,k), (i,j-1,k)|(i,j,k), (i,j,k-1)|(i,j,k) (the MAC
// entries FX(i,j,k), FY(i,j,k), FZ(i,j,k)); the faces on the upper domain
// boundary, owned by no cell, go to UX[j + ny k], UY[i + nx k], UZ[i + nx j]
// (FX(nx,j,k), FY(i,ny,k), FZ(i,j,nz)). A cell's lower faces are then at its
// own index, its upper faces at its +x/+y/+z neighbours' indices.
struct Split {
    int h;       // nx / 2
    long half;   // N / 2
    __device__ long at(const Dims& d, int i, int j, int k) const {
        return (long)((i + j + k) & 1) * half + (long)(i >> 1) + (long)h * ((long)j + (long)d.ny * k);
    }
};
__device__ __forceinline__ Split split_of(const Dims& d) {
    return Split{d.nx >> 1, (long)(d.nx >> 1) * d.ny * d.nz};
}

// The FP64 Krylov vectors that the mixed-precision iteration's r-update sweep
// and x/p update touch (r, A p, x, p: 128 MiB each at 256^3) are each read or
// written once per kernel, so they move with non-temporal loads and stores:
// that keeps them from displacing the FP32 V-cycle's x, b and faces (224 MiB
// at 256^3) from the 256 MB Infinity Cache between that V-cycle's
// half-sweeps. (The (r, z) sweep's read of r measured faster without it.)
typedef double __attribute__((ext_vector_type(2))) ntd2;
__device__ __forceinline__ double2 ldnt(const double* p) {
    const ntd2 v = __builtin_nontemporal_load(reinterpret_cast<const ntd2*>(p));
    return make_double2(v.x, v.y);
}
__device__ __forceinline__ void stnt(double* p, double a, double b) {
    ntd2 v;
    v.x = a;
    v.y = b;
    __builtin_nontemporal_store(v, reinterpret_cast<ntd2*>(p));
}

template <typename TC>
struct SFaces {
    const TC* lx;
    const TC* ly;
    const TC* lz;
    const TC* ux;
    const TC* uy;
    const TC* uz;
};

__device__ __forceinline__ float cvt(float v) { return v; }
__device__ __forceinline__ float cvt(__hip_bfloat16 v) { return __bfloat162float(v); }
__device__ __forceinline__ float cvt(__half v) { return __half2float(v); }

// faces (x+, x-, y+, y-, z+, z-) of cell (i,j,k) of a colour-split level
template <typename TC>
__device__ __forceinline__ void cell_faces_split(const Dims& d, const Split& sp,
                                                 const SFaces<TC>& F, int i, int j, int k,
                                                 float (&f)[6]) {
    const long own = sp.at(d, i, j, k);
    f[1] = cvt(F.lx[own]);
    f[3] = cvt(F.ly[own]);
    f[5] = cvt(F.lz[own]);
    f[0] = i < d.nx - 1 ? cvt(F.lx[sp.at(d, i + 1, j, k)]) : cvt(F.ux[j + (long)d.ny * k]);
    f[2] = j < d.ny - 1 ? cvt(F.ly[sp.at(d, i, j + 1, k)]) : cvt(F.uy[i + (long)d.nx * k]);
    f[4] = k < d.nz - 1 ? cvt(F.lz[sp.at(d, i, j, k + 1)]) : cvt(F.uz[i + (long)d.nx * j]);
}

}  // namespace mf3d
