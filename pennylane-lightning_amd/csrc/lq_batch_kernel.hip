// Packed small-request kernel: one workgroup per request runs the request's
// whole program (forward, H lambda, energy, backward sweep) on its lambda and
// mu. Up to 12 qubits (complex128) both states live in LDS, so a request costs
// no HBM traffic besides its program; up to 16 they live in a global scratch
// area that only this workgroup touches. Ops run in program order with a
// workgroup barrier after each; dot ops reduce per wave, then across the
// waves, into the request's result slots.
#include <hip/hip_runtime.h>

#include <algorithm>

#include "lq_batch.hpp"
#include "lq_devcommon.hpp"

namespace lqamd {
namespace {

using namespace dev;

// A request is a serial chain of some 1500 ops, so a launch lasts as long as
// the ops of its longest request one after the other. An op used to wait twice
// for global memory, for its fields and then for its coefficients, and kept
// four waves busy with up to 16 amplitudes a thread: the fields are now loaded
// two ops ahead and the coefficients one op ahead, a word per lane (readlane
// gives them back as scalars), a workgroup has a thread per amplitude pair
// where it may (BLK), and the two states' loads are issued together: the longest
// launch of 64 requests of 10 to 15 qubits 5.4 -> 2.8 ms. What is left per op
// is the LDS traffic of the states (12 qubits: 1024 cycles a state).
//
// LDS: the states in dynamic LDS. Otherwise in `scratch` (only this
// workgroup touches them; the barrier between ops orders the global accesses
// of the workgroup's threads).
template <typename T, bool LDS, int BLK>
__global__ __launch_bounds__(BLK) void batch_kernel(const BReq *__restrict__ reqs, const BOp *__restrict__ ops,
                                                    const double2 *__restrict__ coef,
                                                    const PauliTerm *__restrict__ terms, double2 *__restrict__ out,
                                                    typename VecT<T>::type *__restrict__ scratch) {
    using V = typename VecT<T>::type;
    constexpr int kWaves = BLK / 64;
    extern __shared__ __align__(16) unsigned char smem_raw[];
    __shared__ double2 red[2][kWaves]; // alternating: a dot needs one barrier
    const BReq r = reqs[blockIdx.x];
    const uint32_t tid = threadIdx.x, lane = tid & 63u;
    const uint32_t N = 1u << r.n;
    V *S0 = LDS ? reinterpret_cast<V *>(smem_raw) : scratch + r.state_off;
    V *S1 = S0 + N;

    auto load_op = [&](uint32_t o) -> uint32_t {
        return o < r.op_end && lane < sizeof(BOp) / 4 ? reinterpret_cast<const uint32_t *>(ops + o)[lane] : 0u;
    };
    auto word = [](uint32_t w, int i) -> uint32_t { return __builtin_amdgcn_readlane(w, i); };
    auto load_coef = [&](uint32_t w) -> uint32_t {
        const uint32_t h = word(w, 0), kind = h & 255u, k = h >> 24;
        const uint32_t nw = kind == BOP_DENSE1   ? 16u
                            : kind == BOP_DENSE2 ? 64u
                            : kind == BOP_DIAG   ? 4u << k
                            : kind == BOP_PARITY ? 8u
                                                 : 0u;
        return lane < nw ? reinterpret_cast<const uint32_t *>(coef + word(w, 4))[lane] : 0u;
    };
    uint32_t w0 = load_op(r.op_begin), w1 = load_op(r.op_begin + 1);
    uint32_t c0 = load_coef(w0), c1 = 0u, w2 = 0u;
    for (uint32_t i = tid; i < N; i += BLK) {
        S0[i] = mk<T>(i == 0 ? T(1) : T(0), T(0));
        S1[i] = mk<T>(T(0), T(0));
    }
    __syncthreads();

    uint32_t par = 0;
    for (uint32_t o = r.op_begin; o < r.op_end; ++o, w0 = w1, w1 = w2, c0 = c1) {
        w2 = load_op(o + 2);
        c1 = load_coef(w1);
        const uint32_t h = word(w0, 0), kind = h & 255u, k = h >> 24;
        const uint32_t t0 = word(w0, 1) & 255u, t1 = (word(w0, 1) >> 8) & 255u;
        const uint32_t cmask = word(w0, 2), cval = word(w0, 3), arg = word(w0, 4), arg2 = word(w0, 5);
        const bool dot = ((h >> 8) & BOP_F_DOT) != 0;
        const bool s0 = ((h >> 16) & 1u) != 0, s1 = ((h >> 16) & 2u) != 0;
        auto co = [&](int i) -> V {
            return mk<T>(static_cast<T>(__hiloint2double(word(c0, 4 * i + 1), word(c0, 4 * i))),
                         static_cast<T>(__hiloint2double(word(c0, 4 * i + 3), word(c0, 4 * i + 2))));
        };
        double ar = 0.0, ai = 0.0;
        switch (kind) {
        case BOP_DENSE1: {
            const V m00 = co(0), m01 = co(1), m10 = co(2), m11 = co(3);
            const uint32_t tb = 1u << t0;
            for (uint32_t p = tid; p < (N >> 1); p += BLK) {
                const uint32_t i0 = insert_zero(p, t0), i1 = i0 | tb;
                if ((i0 & cmask) != cval) continue;
                if (dot) {
                    const V a0 = S0[i0], a1 = S0[i1], b0 = S1[i0], b1 = S1[i1];
                    acc_dot(ar, ai, b0, cmul2(m00, a0, m01, a1));
                    acc_dot(ar, ai, b1, cmul2(m10, a0, m11, a1));
                } else if (s0 && s1) {
                    const V a0 = S0[i0], a1 = S0[i1], b0 = S1[i0], b1 = S1[i1];
                    S0[i0] = cmul2(m00, a0, m01, a1);
                    S0[i1] = cmul2(m10, a0, m11, a1);
                    S1[i0] = cmul2(m00, b0, m01, b1);
                    S1[i1] = cmul2(m10, b0, m11, b1);
                } else {
                    V *S = s0 ? S0 : S1;
                    const V a0 = S[i0], a1 = S[i1];
                    S[i0] = cmul2(m00, a0, m01, a1);
                    S[i1] = cmul2(m10, a0, m11, a1);
                }
            }
            break;
        }
        case BOP_DENSE2: {
            V m[16];
#pragma unroll
            for (int i = 0; i < 16; ++i) m[i] = co(i);
            const uint32_t lo = t0 < t1 ? t0 : t1, hi = t0 < t1 ? t1 : t0;
            const uint32_t b0 = 1u << t0, b1 = 1u << t1;
            for (uint32_t p = tid; p < (N >> 2); p += BLK) {
                const uint32_t i00 = insert_zero(insert_zero(p, lo), hi);
                if ((i00 & cmask) != cval) continue;
                const uint32_t idx[4] = {i00, i00 | b1, i00 | b0, i00 | b0 | b1};
                if (dot) {
                    V a[4];
#pragma unroll
                    for (int c = 0; c < 4; ++c) a[c] = S0[idx[c]];
#pragma unroll
                    for (int rr = 0; rr < 4; ++rr) {
                        const V x = cmul2(m[4 * rr], a[0], m[4 * rr + 1], a[1]);
                        const V y = cmul2(m[4 * rr + 2], a[2], m[4 * rr + 3], a[3]);
                        acc_dot(ar, ai, S1[idx[rr]], mk<T>(x.x + y.x, x.y + y.y));
                    }
                    continue;
                }
#pragma unroll
                for (int s = 0; s < 2; ++s) {
                    if (!(s ? s1 : s0)) continue;
                    V *S = s ? S1 : S0;
                    V a[4];
#pragma unroll
                    for (int c = 0; c < 4; ++c) a[c] = S[idx[c]];
#pragma unroll
                    for (int rr = 0; rr < 4; ++rr) {
                        const V x = cmul2(m[4 * rr], a[0], m[4 * rr + 1], a[1]);
                        const V y = cmul2(m[4 * rr + 2], a[2], m[4 * rr + 3], a[3]);
                        S[idx[rr]] = mk<T>(x.x + y.x, x.y + y.y);
                    }
                }
            }
            break;
        }
        case BOP_DIAG:
        case BOP_PARITY: {
            const bool parity = kind == BOP_PARITY;
            const uint32_t nd = parity ? 2u : (1u << k);
            V d[4];
#pragma unroll
            for (uint32_t i = 0; i < 4; ++i) d[i] = i < nd ? co(i) : d[0];
            for (uint32_t i = tid; i < N; i += BLK) {
                if ((i & cmask) != cval) continue;
                uint32_t idx;
                if (parity) {
                    idx = __popc(i & arg2) & 1u;
                } else if (k == 0) {
                    idx = 0;
                } else if (k == 1) {
                    idx = (i >> t0) & 1u;
                } else {
                    idx = (((i >> t0) & 1u) << 1) | ((i >> t1) & 1u);
                }
                // select by index bits (a select chain on idx compiles to a
                // dynamically indexed private array in scratch memory)
                const V f01 = (idx & 1u) ? d[1] : d[0];
                const V f23 = (idx & 1u) ? d[3] : d[2];
                const V f = (idx & 2u) ? f23 : f01;
                if (dot) {
                    const V a = S0[i], b = S1[i];
                    acc_dot(ar, ai, b, cmul(f, a));
                } else if (s0 && s1) {
                    const V a = S0[i], b = S1[i];
                    S0[i] = cmul(f, a);
                    S1[i] = cmul(f, b);
                } else {
                    V *S = s0 ? S0 : S1;
                    S[i] = cmul(f, S[i]);
                }
            }
            break;
        }
        case BOP_HAM: {
            for (uint32_t i = tid; i < N; i += BLK) {
                double sr = 0.0, si = 0.0;
#pragma unroll 4
                for (uint32_t t = 0; t < arg2; ++t) {
                    const PauliTerm pt = terms[arg + t];
                    const V v = S0[i ^ static_cast<uint32_t>(pt.x)];
                    const double sg = (__popc(i & static_cast<uint32_t>(pt.yz)) & 1) ? -1.0 : 1.0;
                    const double cr = sg * pt.cre, ci = sg * pt.cim;
                    const double vx = v.x, vy = v.y;
                    sr += cr * vx - ci * vy;
                    si += cr * vy + ci * vx;
                }
                S1[i] = mk<T>(static_cast<T>(sr), static_cast<T>(si));
            }
            break;
        }
        case BOP_DOTID: {
            for (uint32_t i = tid; i < N; i += BLK) acc_dot(ar, ai, S1[i], S0[i]);
            break;
        }
        default: break;
        }
        if (dot) {
            wave_sum(ar, ai);
            if (lane == 0) red[par][tid >> 6] = make_double2(ar, ai);
        }
        __syncthreads();
        if (dot) {
            if (tid < 64) {
                double2 t = lane < kWaves ? red[par][lane] : make_double2(0.0, 0.0);
                wave_sum(t.x, t.y);
                if (tid == 0) out[r.out_off + arg2] = t;
            }
            par ^= 1u;
        }
    }
}

} // namespace

namespace {
__global__ __launch_bounds__(256) void copy16_kernel(const uint4 *__restrict__ src, uint4 *__restrict__ dst,
                                                     size_t n) {
    for (size_t i = static_cast<size_t>(blockIdx.x) * 256u + threadIdx.x; i < n;
         i += static_cast<size_t>(gridDim.x) * 256u)
        dst[i] = src[i];
}
} // namespace

void launch_copy16(const void *src, void *dst, size_t bytes, hipStream_t s) {
    const size_t n = bytes / 16;
    if (n == 0) return;
    const unsigned blocks = static_cast<unsigned>(std::min<size_t>((n + 255) / 256, 1024));
    hipLaunchKernelGGL(copy16_kernel, dim3(blocks), dim3(256), 0, s, static_cast<const uint4 *>(src),
                       static_cast<uint4 *>(dst), n);
}

void launch_batch(const BReq *reqs, const BOp *ops, const double2 *coef, const PauliTerm *terms, double2 *out,
                  void *scratch, uint32_t nreq, int max_n, bool in_lds, int dtype, hipStream_t s) {
    if (nreq == 0) return;
    const size_t elem = dtype ? 16 : 8;
    const size_t lds = in_lds ? 2 * (elem << max_n) : 0;
    // threads per workgroup: one per amplitude pair of the largest request, two
    // pairs where that would be 2048 (more waves than pairs only wait at the
    // barriers, and fewer workgroups then share a CU)
    const int blk = max_n >= 11 ? 1024 : max_n == 10 ? 512 : 256;
#define LQ_BATCH(T_, L_, B_)                                                                                 \
    hipLaunchKernelGGL((batch_kernel<T_, L_, B_>), dim3(nreq), dim3(B_), lds, s, reqs, ops, coef, terms, out, \
                       static_cast<typename VecT<T_>::type *>(scratch))
#define LQ_BATCH_T(T_)                                \
    if (!in_lds) LQ_BATCH(T_, false, 1024);           \
    else if (blk == 1024) LQ_BATCH(T_, true, 1024);   \
    else if (blk == 512) LQ_BATCH(T_, true, 512);     \
    else LQ_BATCH(T_, true, 256)
    if (dtype) {
        LQ_BATCH_T(double);
    } else {
        LQ_BATCH_T(float);
    }
#undef LQ_BATCH_T
#undef LQ_BATCH
}

} // namespace lqamd
