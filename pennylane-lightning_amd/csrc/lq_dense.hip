// Dense operators on three to six bits, one in-place pass per operator.
//
// Such an operator multiplies the 2^k amplitudes of every group that shares
// the other bits by one matrix: a 2^k x 2^k by 2^k x 2^(n-k) complex product
// of 8 2^k flops per amplitude, 32 bytes of HBM traffic per amplitude in
// complex128. A workgroup stages a tile of 2^11 amplitudes (the target bits
// and the lowest other bits, so HBM is read in contiguous runs) in LDS as a
// 2^k x 2^(11-k) panel. For k >= 4 the panel is the B operand of 16x16x4 MFMA
// instructions (FP64 for complex128, FP32 for complex64; complex products as
// four real ones) and each wave keeps its 16 rows of the matrix in registers
// over all tiles of the workgroup; for k = 3 (8 rows, half a matrix-core tile)
// one thread takes a column with scalar coefficients.
//
// Bound: HBM up to k = 5 in complex128 (256 flops per amplitude against 71.7
// TFLOP/s), the FP64 matrix rate for k = 6. Measured, 23 qubits complex128: a
// plain and a controlled operator of k = 3, 4, 5, 6 take 73, 56, 92, 186 us
// together (the plain k = 4 one at 6 TB/s, the plain k = 6 one at 29 TFLOP/s);
// interpreted as LDS ops of generic tile passes, twelve operators on one to
// six wires took 8229 us of kernel time, now 515.
#include <hip/hip_runtime.h>

#include <algorithm>

#include "lq_devcommon.hpp"
#include "lq_kernels.hpp"

namespace lqamd {
namespace {

using namespace dev;

constexpr int kTileAmps = 1 << kDenseTileBits;
constexpr int kPerThread = kTileAmps / kBlock;

template <typename T> struct Mfma;
template <> struct Mfma<double> {
    typedef double acc __attribute__((ext_vector_type(4)));
    static __device__ __forceinline__ acc mul(double a, double b, acc c) {
        return __builtin_amdgcn_mfma_f64_16x16x4f64(a, b, c, 0, 0, 0);
    }
    // D register v of lane l is row 4 v + l / 16
    static __device__ __forceinline__ uint32_t row(uint32_t v, uint32_t lq) { return 4u * v + lq; }
};
template <> struct Mfma<float> {
    typedef float acc __attribute__((ext_vector_type(4)));
    static __device__ __forceinline__ acc mul(float a, float b, acc c) {
        return __builtin_amdgcn_mfma_f32_16x16x4f32(a, b, c, 0, 0, 0);
    }
    // D register v of lane l is row 4 (l / 16) + v
    static __device__ __forceinline__ uint32_t row(uint32_t v, uint32_t lq) { return 4u * lq + v; }
};

template <typename T, int K>
__global__ __launch_bounds__(kBlock) void dense_tile_kernel(DenseTileArgs a, const double2 *__restrict__ U) {
    using V = typename VecT<T>::type;
    constexpr int R = 1 << K, CL = kDenseTileBits - K, C = 1 << CL;
    __shared__ __align__(16) V lds[kTileAmps];
    V *sv = static_cast<V *>(a.sv[blockIdx.y]);
    const uint32_t tid = threadIdx.x, lane = tid & 63u, lq = lane >> 4, lj = lane & 15u, wave = tid >> 6;

    // panel coordinate row * C + column, the column's low bits turned by the
    // row so that reading a run of amplitudes that are targets (one column,
    // many rows) and reading 16 columns of a row both spread over the banks
    auto at = [](uint32_t l) { return l ^ (((l >> CL) ^ (l >> (CL + 4) << 2)) & 15u); };
    // tile-local amplitude tid + 256 i: address offset and panel coordinate
    uint64_t off = 0;
    uint32_t pan = 0;
#pragma unroll
    for (int b = 0; b < 8; ++b) {
        off |= static_cast<uint64_t>((tid >> b) & 1u) << a.tb[b];
        pan |= ((tid >> b) & 1u) << a.lp[b];
    }
    auto off_i = [&](int i) {
        uint64_t o = 0;
#pragma unroll
        for (int b = 8; b < kDenseTileBits; ++b)
            if ((i >> (b - 8)) & 1) o |= 1ull << a.tb[b];
        return o;
    };
    auto pan_i = [&](int i) {
        uint32_t o = 0;
#pragma unroll
        for (int b = 8; b < kDenseTileBits; ++b)
            if ((i >> (b - 8)) & 1) o |= 1u << a.lp[b];
        return o;
    };

    // this wave's rows of the matrix: 16 rows, four columns per step
    constexpr int RB = R / 16 < 1 ? 1 : R / 16, STEPS = R / 4;
    const uint32_t rb = wave % RB;
    T ur[STEPS], ui[STEPS];
    if constexpr (K >= 4) {
#pragma unroll
        for (int s = 0; s < STEPS; ++s) {
            const double2 u = U[(rb * 16u + lj) * R + 4u * s + lq];
            ur[s] = static_cast<T>(u.x);
            ui[s] = static_cast<T>(u.y);
        }
    }

    for (uint64_t tile = blockIdx.x; tile < a.ntiles; tile += gridDim.x) {
        uint64_t base = a.ocval;
        for (int j = 0; j < a.nout; ++j) base |= ((tile >> j) & 1ull) << a.ob[j];
        V *p = sv + (base | off);
        T xr[kPerThread], xi[kPerThread];
#pragma unroll
        for (int i = 0; i < kPerThread; ++i) {
            const V v = p[off_i(i)];
            xr[i] = v.x;
            xi[i] = v.y;
        }
        __syncthreads(); // the last tile's amplitudes have left the panel
#pragma unroll
        for (int i = 0; i < kPerThread; ++i) lds[at(pan | pan_i(i))] = mk<T>(xr[i], xi[i]);
        __syncthreads();
        if constexpr (K >= 4) {
            using M = Mfma<T>;
            // 16-column blocks: eight (row block, column block) pairs over four waves
            constexpr int CBW = 2;
            const uint32_t cb0 = (wave / RB) * CBW;
            typename M::acc dr[CBW] = {}, di[CBW] = {};
#pragma unroll
            for (int s = 0; s < STEPS; ++s)
#pragma unroll
                for (int c = 0; c < CBW; ++c) {
                    const V b = lds[at((4u * s + lq) * C + (cb0 + c) * 16u + lj)];
                    dr[c] = M::mul(ur[s], b.x, dr[c]);
                    di[c] = M::mul(ur[s], b.y, di[c]);
                    dr[c] = M::mul(ui[s], -b.y, dr[c]);
                    di[c] = M::mul(ui[s], b.x, di[c]);
                }
            __syncthreads(); // every wave has read the whole panel
#pragma unroll
            for (int c = 0; c < CBW; ++c) {
                const uint32_t col = (cb0 + c) * 16u + lj;
                if ((col & a.ccmask) != a.ccval) continue; // controls inside the tile: unchanged
#pragma unroll
                for (int v = 0; v < 4; ++v)
                    lds[at((rb * 16u + M::row(v, lq)) * C + col)] = mk<T>(dr[c][v], di[c][v]);
            }
            __syncthreads();
        } else {
            if ((tid & a.ccmask) == a.ccval) { // the thread's own column: no barrier inside
                V in[R];
#pragma unroll
                for (int c = 0; c < R; ++c) in[c] = lds[at(c * C + tid)];
#pragma unroll
                for (int r = 0; r < R; ++r) {
                    T sr = T(0), si = T(0);
#pragma unroll
                    for (int c = 0; c < R; ++c) {
                        const V u = ld_coef<T>(U, r * R + c);
                        sr += u.x * in[c].x - u.y * in[c].y;
                        si += u.x * in[c].y + u.y * in[c].x;
                    }
                    lds[at(r * C + tid)] = mk<T>(sr, si);
                }
            }
            __syncthreads();
        }
#pragma unroll
        for (int i = 0; i < kPerThread; ++i) p[off_i(i)] = lds[at(pan | pan_i(i))];
    }
}

} // namespace

template <typename T> void launch_dense_tile(const DenseTileArgs &a, int k, int ns, const double2 *U, hipStream_t s) {
    // four workgroups per CU are resident: each keeps its matrix rows over its tiles
    const dim3 grid(static_cast<uint32_t>(std::min<uint64_t>(a.ntiles, 1024)), static_cast<uint32_t>(ns));
    switch (k) {
    case 3: hipLaunchKernelGGL((dense_tile_kernel<T, 3>), grid, dim3(kBlock), 0, s, a, U); break;
    case 4: hipLaunchKernelGGL((dense_tile_kernel<T, 4>), grid, dim3(kBlock), 0, s, a, U); break;
    case 5: hipLaunchKernelGGL((dense_tile_kernel<T, 5>), grid, dim3(kBlock), 0, s, a, U); break;
    default: hipLaunchKernelGGL((dense_tile_kernel<T, 6>), grid, dim3(kBlock), 0, s, a, U); break;
    }
}
template void launch_dense_tile<double>(const DenseTileArgs &, int, int, const double2 *, hipStream_t);
template void launch_dense_tile<float>(const DenseTileArgs &, int, int, const double2 *, hipStream_t);

} // namespace lqamd
