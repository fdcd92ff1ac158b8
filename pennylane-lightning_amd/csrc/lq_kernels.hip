// HIP kernels for gfx950 (MI355X): the LDS tile-program kernel that applies
// runs of gates (and reads generator inner products) in one HBM pass, plus
// the standalone reductions and fills around it.
//
// Amplitude layout: interleaved complex (double2 / float2), index bit n-1-w
// is wire w (lq/StateVectorLQubit.hpp:950). All sums are accumulated in
// double, also for complex64 states.
#include <hip/hip_runtime.h>

#include "lq_devcommon.hpp"
#include "lq_kernels.hpp"

namespace lqamd {
namespace {

using dev::VecT;
using dev::mk;
using dev::ld_coef;
using dev::cmul;
using dev::acc_dot;
using dev::OpView;
using dev::warm_program;
using dev::deposit_bits;
using dev::spread_bits;

__device__ __forceinline__ void block_reduce_store(double re, double im, double2 *red, double2 *dst) {
    dev::wave_sum(re, im);
    const uint32_t tid = threadIdx.x;
    if ((tid & 63u) == 0) red[tid >> 6] = make_double2(re, im);
    __syncthreads();
    if (tid == 0) {
        double2 s = red[0];
        for (int w = 1; w < kBlock / 64; ++w) {
            s.x += red[w].x;
            s.y += red[w].y;
        }
        *dst = s;
    }
}

// ---------------------------------------------------------------------------
// Small-tile kernel: the whole tile lives in LDS and every op sweeps it.
// Used for tiles of at most 2^10 amplitudes and for passes with more than two
// states; larger tiles run in tile_reg_kernel (lq_kernels_reg.hip). Bound by
// the latency of reading each op and of its sweep: heads are brought to the
// caches first and read one op ahead (OpView), and a state of one tile runs
// its whole program in one launch. 10 qubits, three layers of RX RY RZ + CNOT
// with ten dots: three passes of 37 us -> one of 80 us.
// ---------------------------------------------------------------------------
template <typename T, int NS>
__global__ __launch_bounds__(kBlock) void tile_pass_kernel(TilePassArgs a, const OpHead *__restrict__ heads,
                                                          const TileOp *__restrict__ ops,
                                                          const double2 *__restrict__ coef,
                                                          double2 *__restrict__ partials) {
    using V = typename VecT<T>::type;
    extern __shared__ __align__(16) unsigned char smem_raw[];
    V *lds = reinterpret_cast<V *>(smem_raw);
    __shared__ double2 red[kBlock / 64];

    const uint32_t tid = threadIdx.x;
    const uint64_t tile = static_cast<uint64_t>(blockIdx.x) + static_cast<uint64_t>(blockIdx.y) * gridDim.x;
    if (tile >= a.ntiles) return; // uniform over the block
    const int kt = a.g.kt;
    const uint32_t tsize = 1u << kt;
    if (a.ntiles <= kWarmTiles) warm_program(heads, a.nops * static_cast<uint32_t>(sizeof(OpHead)));

    const uint64_t base = deposit_bits(tile, a.g.ob, a.g.nout);

    // spread(l) = base offset of tile-local index l; separable over the bits
    // of l, so spread(tid + it*kBlock) = sp_tid | spread(it*kBlock).
    auto spread = [&](uint32_t l) -> uint64_t { return spread_bits(l, a.g.tb); };
    const uint64_t sp_tid = spread(tid < tsize ? tid : 0u);
    const uint32_t iters = (tsize + kBlock - 1) / kBlock;

#pragma unroll
    for (int s = 0; s < NS; ++s) {
        if (!((a.load_mask >> s) & 1u)) continue;
        const V *src = reinterpret_cast<const V *>(a.sv[s]);
        for (uint32_t it = 0; it < iters; ++it) {
            const uint32_t l = tid + it * kBlock;
            if (l < tsize) lds[s * tsize + l] = src[base | sp_tid | spread(it * kBlock)];
        }
    }
    __syncthreads();

    const V zero = mk<T>(T(0), T(0));
    OpView next = OpView::load(heads);
    for (uint32_t oi = 0; oi < a.nops; ++oi) {
        const OpView op = next;
        next = OpView::load(heads + (oi + 1 < a.nops ? oi + 1 : oi)); // in flight while this op runs
        const bool dot = (op.flags() & TF_DOT) != 0;
        double2 *dst = dot ? &partials[static_cast<uint64_t>(op.slot()) * a.ntiles + tile] : nullptr;
        if ((base & op.ocmask()) != op.ocval()) {
            // control bits outside the tile do not match: no-op for this tile
            if (dot) {
                if (tid == 0) *dst = make_double2(0.0, 0.0);
            } else if (op.flags() & TF_ZERO_UNCTRL) {
#pragma unroll
                for (int s = 0; s < NS; ++s)
                    if ((op.smask() >> s) & 1u)
                        for (uint32_t l = tid; l < tsize; l += kBlock) lds[s * tsize + l] = zero;
            }
            __syncthreads();
            continue;
        }
        double accr = 0.0, acci = 0.0;
        dev::lds_apply_op<T, NS, false>(op, ops[oi], lds, tsize, base, coef, accr, acci);
        if (dot) block_reduce_store(accr, acci, red, dst);
        __syncthreads();
    }

#pragma unroll
    for (int s = 0; s < NS; ++s) {
        if (!((a.store_mask >> s) & 1u)) continue;
        V *dstp = reinterpret_cast<V *>(a.sv[s]);
        for (uint32_t it = 0; it < iters; ++it) {
            const uint32_t l = tid + it * kBlock;
            if (l < tsize) dstp[base | sp_tid | spread(it * kBlock)] = lds[s * tsize + l];
        }
    }
}

// ---------------------------------------------------------------------------
// Reductions
// ---------------------------------------------------------------------------
// One block per slot; each thread keeps a Neumaier-compensated sum over a
// strided subset, then a fixed-order tree.
__global__ __launch_bounds__(kBlock) void reduce_slots_kernel(const double2 *partials, const SlotRange *ranges,
                                                             double2 *out) {
    __shared__ double2 red[kBlock / 64];
    const SlotRange r = ranges[blockIdx.x];
    double sr = 0.0, cr = 0.0, si = 0.0, ci = 0.0;
    for (uint64_t i = threadIdx.x; i < r.count; i += kBlock) {
        const double2 v = partials[r.off + i];
        double t = sr + v.x;
        cr += (fabs(sr) >= fabs(v.x)) ? (sr - t) + v.x : (v.x - t) + sr;
        sr = t;
        t = si + v.y;
        ci += (fabs(si) >= fabs(v.y)) ? (si - t) + v.y : (v.y - t) + si;
        si = t;
    }
    block_reduce_store(sr + cr, si + ci, red, &out[blockIdx.x]);
}

// Sum of Pauli words, bound by the reads of a[i ^ x]: one pass over the state
// per distinct x. A workgroup takes 256 U consecutive amplitudes, U per
// thread, so a term costs each thread one address and one sign for U loads in
// flight; term fields are scalar loads, the parts of sign and address that are
// uniform over the workgroup scalar arithmetic. The host sorts the terms by x:
// neighbouring terms then read the same region (a ^ high bits of x), and an
// XCD takes 2^wc_log consecutive blocks at a time, so part of the reads hits
// its L2; terms of equal x share their loads. Coefficients that are real or
// imaginary (all of a Hermitian sum) take two FMAs per amplitude. In MODE 0 a
// term with x != 0 pairs i with i ^ x, whose contributions are conjugates:
// only the i with the highest bit of x clear are read, the host doubles the
// coefficient. 24 qubits complex128, 200 random words (MODE 1): 6148 us with
// one amplitude per thread and terms as given; 6355 us with U = 4 unsorted,
// 4703 us sorted with a workgroup per block, 4151 us with 1024 workgroups that
// walk the blocks and wc_log = 6 (13 TB/s of mostly L2 misses; with x inside
// the workgroup's amplitudes 1.6 ms). 26 qubits, 40 words (MODE 0, 2048
// workgroups; 1024: 5% slower): 6034 -> 3016 us.
typedef __attribute__((address_space(4))) const PauliTerm KTerm;

template <typename T, int MODE, int U>
__global__ __launch_bounds__(kBlock) void pauli_sum_kernel(const typename VecT<T>::type *__restrict__ a,
                                                          typename VecT<T>::type *__restrict__ out,
                                                          const PauliTerm *__restrict__ terms, uint32_t nterms,
                                                          uint64_t N, uint64_t nblk, uint32_t wc_log,
                                                          double2 *__restrict__ partials) {
    using V = typename VecT<T>::type;
    __shared__ double2 red[kBlock / 64];
    const uint32_t tid = threadIdx.x;
    KTerm *kt = (KTerm *)terms;
    const bool in = tid < N; // states below 256 amplitudes
    double energy = 0.0;
    for (uint64_t lb = blockIdx.x; lb < nblk; lb += gridDim.x) {
        // XCD lb % 8 takes 2^wc_log consecutive blocks at a time
        const uint64_t q = lb >> 3, wm = (1ull << wc_log) - 1ull;
        const uint64_t blk = nblk < 8 ? lb : ((((q >> wc_log) << 3) | (lb & 7ull)) << wc_log) | (q & wm);
        const uint64_t base = blk * (static_cast<uint64_t>(kBlock) * U);
        V b[U], v[U];
        double sr[U], si[U];
#pragma unroll
        for (int u = 0; u < U; ++u) {
            sr[u] = si[u] = 0.0;
            b[u] = mk<T>(T(0), T(0));
            if (MODE == 0 && in) b[u] = a[base + u * kBlock + tid];
            v[u] = b[u];
        }
        uint64_t px = MODE == 0 ? 0ull : ~0ull; // the x that v holds
        for (uint32_t t = 0; t < nterms; ++t) {
            const uint64_t x = kt[t].x, yz = kt[t].yz;
            const double cre = kt[t].cre, cim = kt[t].cim;
            const uint64_t top = MODE == 0 && x ? 1ull << (63 - __builtin_clzll(x)) : 0ull;
            if (top >= static_cast<uint64_t>(kBlock) * U && (base & top)) continue; // the partner's term
            if (x != px) {
                px = x;
                const uint32_t lane = tid ^ (static_cast<uint32_t>(x) & (kBlock - 1u));
                const uint64_t xh = x & ~static_cast<uint64_t>(kBlock - 1);
#pragma unroll
                for (int u = 0; u < U; ++u)
                    if (in) v[u] = (a + ((base + u * kBlock) ^ xh))[lane];
            }
            const uint32_t sg = static_cast<uint32_t>(__popc(tid & static_cast<uint32_t>(yz) & (kBlock - 1u))) << 31;
            const bool real = (__double_as_longlong(cim) << 1) == 0, imag = (__double_as_longlong(cre) << 1) == 0;
#pragma unroll
            for (int u = 0; u < U; ++u) {
                const uint64_t iu = base + u * kBlock;
                if (MODE == 0 && (iu & top)) continue; // uniform; `top` below 256 is a lane bit
                const uint32_t s = sg ^ (static_cast<uint32_t>(__popcll(iu & yz)) << 31);
                const double vx = v[u].x, vy = v[u].y;
                auto sgn = [&](double c) { return __hiloint2double(__double2hiint(c) ^ static_cast<int>(s), __double2loint(c)); };
                if (MODE == 0) {
                    // Re(conj(b) c v)
                    const double bx = b[u].x, by = b[u].y;
                    double e = real ? bx * vx + by * vy : by * vx - bx * vy;
                    if (top && top < kBlock && (tid & static_cast<uint32_t>(top))) e = 0.0;
                    sr[u] += sgn(real ? cre : cim) * e;
                } else if (real) {
                    const double c = sgn(cre);
                    sr[u] += c * vx;
                    si[u] += c * vy;
                } else if (imag) {
                    const double c = sgn(cim);
                    sr[u] -= c * vy;
                    si[u] += c * vx;
                } else {
                    const double c = sgn(cre), d = sgn(cim);
                    sr[u] += c * vx - d * vy;
                    si[u] += c * vy + d * vx;
                }
            }
        }
#pragma unroll
        for (int u = 0; u < U; ++u) {
            if (MODE == 0) energy += sr[u];
            else if (in) out[base + u * kBlock + tid] = mk<T>(static_cast<T>(sr[u]), static_cast<T>(si[u]));
        }
    }
    if (MODE == 0) block_reduce_store(energy, 0.0, red, &partials[blockIdx.x]);
}

// The same sum of P_t a for large complex128 states. pauli_sum_kernel reads the
// state once for each x through the L2 (13 TB/s of mostly misses); here a
// workgroup brings a tile of 2^12 amplitudes (its own ^ the high bits of x) to
// LDS once for all terms that share those bits and takes a[i ^ x] from there,
// the next group's tile in flight meanwhile, its sums in registers (8
// amplitudes a thread, in the order of the terms as there); two workgroups of
// 64 KiB a CU. 24 qubits, 200 random words in 136 groups: 4.43 -> 3.40 ms (10.7
// TB/s). Groups of many terms are bound by the LDS reads instead, where the L1
// does as well.
__global__ __launch_bounds__(kPauliTileThreads) void pauli_tile_kernel(const double2 *__restrict__ a,
                                                                      double2 *__restrict__ out,
                                                                      const PauliTerm *__restrict__ terms,
                                                                      const uint32_t *__restrict__ ends,
                                                                      uint32_t ngroups, uint64_t ntiles) {
    using T = double;
    using V = double2;
    constexpr int U = (1 << kPauliTileBits) / kPauliTileThreads;
    extern __shared__ __align__(16) unsigned char smem_raw[];
    V *lds = reinterpret_cast<V *>(smem_raw);
    const uint32_t tid = threadIdx.x;
    KTerm *kt = (KTerm *)terms;
    typedef __attribute__((address_space(4))) const uint32_t KEnd;
    KEnd *ke = (KEnd *)ends;
    // XCD b % 8 takes an eighth of the tiles in order: its workgroups read
    // neighbouring tiles at a time (ntiles is a power of two, at least 8)
    const uint64_t tile = (blockIdx.x & 7ull) * (ntiles >> 3) + (blockIdx.x >> 3);
    const uint64_t base = tile << kPauliTileBits;
    T px[U], py[U]; // the tile in flight
    double sr[U], si[U];
    auto fetch = [&](uint64_t x) {
        const V *src = a + (base ^ (x >> kPauliTileBits << kPauliTileBits));
#pragma unroll
        for (int u = 0; u < U; ++u) {
            const V v = src[u * kPauliTileThreads + tid];
            px[u] = v.x;
            py[u] = v.y;
        }
    };
#pragma unroll
    for (int u = 0; u < U; ++u) sr[u] = si[u] = 0.0;
    fetch(kt[0].x);
    uint32_t t = 0;
    for (uint32_t g = 0; g < ngroups; ++g) {
        const uint32_t end = ke[g];
        __syncthreads(); // the last group's reads
#pragma unroll
        for (int u = 0; u < U; ++u) lds[u * kPauliTileThreads + tid] = mk<T>(px[u], py[u]);
        __syncthreads();
        if (g + 1 < ngroups) fetch(kt[end].x);
        for (; t < end; ++t) {
            const uint64_t yz = kt[t].yz;
            const uint32_t x = static_cast<uint32_t>(kt[t].x) & ((1u << kPauliTileBits) - 1u);
            const double cre = kt[t].cre, cim = kt[t].cim;
            const uint32_t sg = static_cast<uint32_t>(__popc(tid & static_cast<uint32_t>(yz))) << 31;
            const bool real = (__double_as_longlong(cim) << 1) == 0, imag = (__double_as_longlong(cre) << 1) == 0;
#pragma unroll
            for (int u = 0; u < U; ++u) {
                const uint32_t s = sg ^ (static_cast<uint32_t>(__popcll((base + u * kPauliTileThreads) & yz)) << 31);
                const V v = lds[(u * kPauliTileThreads + tid) ^ x];
                const double vx = v.x, vy = v.y;
                auto sgn = [&](double c) { return __hiloint2double(__double2hiint(c) ^ static_cast<int>(s), __double2loint(c)); };
                if (real) {
                    const double c = sgn(cre);
                    sr[u] += c * vx;
                    si[u] += c * vy;
                } else if (imag) {
                    const double c = sgn(cim);
                    sr[u] -= c * vy;
                    si[u] += c * vx;
                } else {
                    const double c = sgn(cre), d = sgn(cim);
                    sr[u] += c * vx - d * vy;
                    si[u] += c * vy + d * vx;
                }
            }
        }
    }
#pragma unroll
    for (int u = 0; u < U; ++u)
        out[base + u * kPauliTileThreads + tid] = mk<T>(static_cast<T>(sr[u]), static_cast<T>(si[u]));
}

template <typename T>
__global__ __launch_bounds__(kBlock) void norm2_kernel(const typename VecT<T>::type *a, uint64_t N, double2 *partials) {
    __shared__ double2 red[kBlock / 64];
    double s = 0.0;
    const uint64_t stride = static_cast<uint64_t>(gridDim.x) * kBlock;
    for (uint64_t i = static_cast<uint64_t>(blockIdx.x) * kBlock + threadIdx.x; i < N; i += stride) {
        const double x = a[i].x, y = a[i].y;
        s += x * x + y * y;
    }
    block_reduce_store(s, 0.0, red, &partials[blockIdx.x]);
}

// <a|b> of two states of either precision, accumulated in FP64
template <typename TA, typename TB>
__global__ __launch_bounds__(kBlock) void overlap_kernel(const typename VecT<TA>::type *__restrict__ a,
                                                         const typename VecT<TB>::type *__restrict__ b, uint64_t N,
                                                         double2 *partials) {
    __shared__ double2 red[kBlock / 64];
    double re = 0.0, im = 0.0;
    const uint64_t stride = static_cast<uint64_t>(gridDim.x) * kBlock;
    for (uint64_t i = static_cast<uint64_t>(blockIdx.x) * kBlock + threadIdx.x; i < N; i += stride) {
        const double ax = a[i].x, ay = a[i].y, bx = b[i].x, by = b[i].y;
        re += ax * bx + ay * by;
        im += ax * by - ay * bx;
    }
    block_reduce_store(re, im, red, &partials[blockIdx.x]);
}

// CSR operator rows over the state index (lq/utils/SparseLinAlg.hpp:42-63):
// v_i = sum_k values[k] a[indices[k]], k in [indptr[i], indptr[i+1]), in FP64.
// MODE 0: per-block partials of sum conj(a_i) v_i (partials[2b]) and
// sum |v_i|^2 (partials[2b+1].x); MODE 1: out[i] = v_i.
template <typename T, int MODE>
__global__ __launch_bounds__(kBlock) void sparse_rows_kernel(const typename VecT<T>::type *__restrict__ a,
                                                             typename VecT<T>::type *__restrict__ out,
                                                             const int64_t *__restrict__ indptr,
                                                             const int64_t *__restrict__ indices,
                                                             const typename VecT<T>::type *__restrict__ values,
                                                             uint64_t nrows, double2 *partials) {
    __shared__ double2 red[kBlock / 64];
    double re = 0.0, im = 0.0, sq = 0.0;
    const uint64_t stride = static_cast<uint64_t>(gridDim.x) * kBlock;
    for (uint64_t i = static_cast<uint64_t>(blockIdx.x) * kBlock + threadIdx.x; i < nrows; i += stride) {
        double vr = 0.0, vi = 0.0;
        const int64_t k1 = indptr[i + 1];
        for (int64_t k = indptr[i]; k < k1; ++k) {
            const typename VecT<T>::type h = values[k], x = a[indices[k]];
            const double hx = h.x, hy = h.y, xx = x.x, xy = x.y;
            vr += hx * xx - hy * xy;
            vi += hx * xy + hy * xx;
        }
        if (MODE == 1) {
            out[i] = mk<T>(static_cast<T>(vr), static_cast<T>(vi));
        } else {
            const double ax = a[i].x, ay = a[i].y;
            re += ax * vr + ay * vi;
            im += ax * vi - ay * vr;
            sq += vr * vr + vi * vi;
        }
    }
    if (MODE == 0) {
        block_reduce_store(re, im, red, &partials[2 * static_cast<uint64_t>(blockIdx.x)]);
        __syncthreads(); // red is reused
        block_reduce_store(sq, 0.0, red, &partials[2 * static_cast<uint64_t>(blockIdx.x) + 1]);
    }
}

struct BitList {
    int32_t b[64];
};

// Marginal probabilities, bound by the read of the state. The index splits
// into the low lb <= 8 bits (one thread each: every load is a contiguous run
// of 2^lb amplitudes) and the high bits: a workgroup fixes the measured high
// bits (and the split bits `sm` of the unmeasured ones), each thread sums its
// amplitudes over the remaining high bits `rm` in registers, and one
// cross-lane reduction over the unmeasured low bits ends the item. No
// histogram and no atomics, so any number of wires takes the same route and
// the sums do not depend on scheduling. 26 qubits complex128, 14 scattered
// wires: 3.19 ms (one thread per output gathering 2^12 scattered amplitudes)
// -> 0.16 ms, the read of 1 GiB at 6.5 TB/s. Where nearly all high bits are
// measured an item is one load a thread, so what an item costs besides counts:
// its bits are put in place by one ballot each (lane L answers for bit L of the
// index, then for bit L of the output), not by a loop over the bits, and a
// workgroup takes many items (24 qubits, the 16 high wires: 227 -> 101 us
// for the call; by gathers 174).
template <typename T>
__global__ __launch_bounds__(kBlock) void probs_kernel(const typename VecT<T>::type *__restrict__ a, int lb,
                                                      uint32_t wl, uint64_t wh, uint64_t sm, uint64_t rm,
                                                      uint64_t items, BitList bits, int nw,
                                                      double *__restrict__ out) {
    __shared__ double red[kBlock];
    const uint32_t tid = threadIdx.x;
    const uint32_t rest = ((1u << lb) - 1u) & ~wl; // unmeasured low bits, summed across threads
    const uint64_t count = 1ull << __popcll(rm);
    const uint32_t lane = tid & 63u;
    // the item's bit that stands at state bit `lane`: measured high bits
    // first, then the split bits
    const uint64_t below = (1ull << lane) - 1ull;
    const int mine = (wh >> lane) & 1ull   ? __popcll(wh & below)
                     : (sm >> lane) & 1ull ? __popcll(wh) + __popcll(sm & below)
                                           : -1;
    // the high state bit that output bit `lane` stands for
    const int from = lane < static_cast<uint32_t>(nw) && bits.b[lane] >= lb ? bits.b[lane] : -1;
    uint64_t olow = 0; // this thread's part of the output index
    for (int j = 0; j < nw; ++j)
        if (bits.b[j] < lb) olow |= static_cast<uint64_t>((tid >> bits.b[j]) & 1u) << j;
    for (uint64_t item = blockIdx.x; item < items; item += gridDim.x) {
        const uint64_t base = __ballot(mine >= 0 && ((item >> (mine & 63)) & 1ull));
        const uint64_t row = item >> __popcll(wh);
        double s0 = 0.0, s1 = 0.0, s2 = 0.0, s3 = 0.0;
        if (tid < (1u << lb)) {
            const typename VecT<T>::type *p = a + (base | tid);
            uint64_t r = 0; // runs through the subsets of rm
            auto term = [&](uint64_t at) {
                const typename VecT<T>::type v = p[at];
                const double vx = v.x, vy = v.y;
                return vx * vx + vy * vy;
            };
            uint64_t k = 0;
            for (; k + 4 <= count; k += 4) {
                const uint64_t r1 = (r - rm) & rm, r2 = (r1 - rm) & rm, r3 = (r2 - rm) & rm;
                s0 += term(r);
                s1 += term(r1);
                s2 += term(r2);
                s3 += term(r3);
                r = (r3 - rm) & rm;
            }
            for (; k < count; ++k, r = (r - rm) & rm) s0 += term(r);
        }
        double s = (s0 + s1) + (s2 + s3);
        for (int b = 0; b < 6; ++b)
            if ((rest >> b) & 1u) s += __shfl_xor(s, 1 << b, 64);
        if (rest >> 6) { // across waves
            red[tid] = s;
            __syncthreads();
            if (rest & 64u) s += red[tid ^ 64u];
            if (rest & 128u) {
                double t = red[tid ^ 128u];
                if (rest & 64u) t += red[tid ^ 192u];
                s += t;
            }
            __syncthreads(); // red is reused by the next item
        }
        const uint64_t ohigh = __ballot(from >= 0 && ((base >> (from & 63)) & 1ull));
        if (tid < (1u << lb) && (tid & rest) == 0) out[(row << nw) + (olow | ohigh)] = s;
    }
}

// out[col] = sum of the rows: 16 columns by 16 row groups per workgroup
// (with one thread per column, 512 rows of 1024 columns were a serial chain of
// 129 us; 20 qubits, 10 wires: reset, circuit and probs 1061 -> 957 us), each
// thread's sum compensated, then a fixed-order sum.
__global__ __launch_bounds__(kBlock) void reduce_rows_kernel(const double *__restrict__ partials, uint32_t nrows,
                                                            uint32_t ncols, double *__restrict__ out) {
    __shared__ double2 red[16][17];
    const uint32_t c = threadIdx.x & 15u, g = threadIdx.x >> 4;
    const uint32_t col = blockIdx.x * 16u + c;
    double s = 0.0, cmp = 0.0;
    if (col < ncols)
        for (uint32_t r = g; r < nrows; r += 16) {
            const double v = partials[static_cast<uint64_t>(r) * ncols + col];
            const double t = s + v;
            cmp += (fabs(s) >= fabs(v)) ? (s - t) + v : (v - t) + s;
            s = t;
        }
    red[g][c] = make_double2(s, cmp);
    __syncthreads();
    if (g == 0 && col < ncols) {
        for (int k = 1; k < 16; ++k) {
            const double2 v = red[k][c];
            const double t = s + v.x;
            cmp += ((fabs(s) >= fabs(v.x)) ? (s - t) + v.x : (v.x - t) + s) + v.y;
            s = t;
        }
        out[col] = s + cmp;
    }
}

// One workgroup per segment of 2^(lb + mb) amplitudes: the products over the
// low lb and the next mb bits are tables in LDS, the product over the
// segment's own bits one value; every amplitude is then two multiplies.
template <typename T>
__global__ __launch_bounds__(kBlock) void fill_product_kernel(typename VecT<T>::type *a, int n, int lb, int mb,
                                                             ProductFactors f) {
    __shared__ double2 lo[256], mid[256];
    __shared__ double2 seg;
    const uint32_t tid = threadIdx.x;
    auto prod = [&](uint64_t bits, int from, int count) {
        double2 p = make_double2(1.0, 0.0);
        for (int j = 0; j < count; ++j) {
            const double2 g = f.f[2 * (from + j) + ((bits >> j) & 1ull)];
            p = make_double2(p.x * g.x - p.y * g.y, p.x * g.y + p.y * g.x);
        }
        return p;
    };
    if (tid < (1u << lb)) lo[tid] = prod(tid, 0, lb);
    if (tid < (1u << mb)) mid[tid] = prod(tid, lb, mb);
    if (tid == 0) seg = prod(blockIdx.x, lb + mb, n - lb - mb);
    __syncthreads();
    const uint64_t base = static_cast<uint64_t>(blockIdx.x) << (lb + mb);
    const uint32_t per = 1u << (lb + mb);
    for (uint32_t i = tid; i < per; i += kBlock) {
        const double2 m = mid[i >> lb], l = lo[i & ((1u << lb) - 1u)];
        const double2 h = make_double2(seg.x * m.x - seg.y * m.y, seg.x * m.y + seg.y * m.x);
        a[base + i] = mk<T>(static_cast<T>(h.x * l.x - h.y * l.y), static_cast<T>(h.x * l.y + h.y * l.x));
    }
}

__global__ __launch_bounds__(kBlock) void stream_copy_kernel(const double2 *__restrict__ src, double2 *__restrict__ dst,
                                                            uint64_t N) {
    typedef double dvec __attribute__((ext_vector_type(2)));
    const uint64_t stride = static_cast<uint64_t>(gridDim.x) * kBlock * 4;
    for (uint64_t i = (static_cast<uint64_t>(blockIdx.x) * kBlock * 4) + threadIdx.x; i < N; i += stride) {
        dvec v[4];
#pragma unroll
        for (int u = 0; u < 4; ++u)
            if (i + u * kBlock < N) v[u] = __builtin_nontemporal_load(reinterpret_cast<const dvec *>(src + i + u * kBlock));
#pragma unroll
        for (int u = 0; u < 4; ++u)
            if (i + u * kBlock < N) __builtin_nontemporal_store(v[u], reinterpret_cast<dvec *>(dst + i + u * kBlock));
    }
}

// Dense 2^k x 2^k operator on k target bits (any k), out of place: one
// thread per output amplitude sums its matrix row against the 2^k amplitudes
// of its group (targets bits[0] = local MSB). Amplitudes whose control bits
// do not match are copied unchanged. M is row-major complex double.
template <typename T>
__global__ __launch_bounds__(kBlock) void dense_wide_kernel(const typename VecT<T>::type *__restrict__ in,
                                                           typename VecT<T>::type *__restrict__ out,
                                                           const double2 *__restrict__ M, BitList bits, int k,
                                                           uint64_t tmask, uint64_t cmask, uint64_t cval, uint64_t N) {
    const uint64_t stride = static_cast<uint64_t>(gridDim.x) * kBlock;
    const uint64_t d = 1ull << k;
    for (uint64_t i = static_cast<uint64_t>(blockIdx.x) * kBlock + threadIdx.x; i < N; i += stride) {
        if ((i & cmask) != cval) {
            out[i] = in[i];
            continue;
        }
        uint64_t r = 0;
        for (int j = 0; j < k; ++j) r |= ((i >> bits.b[j]) & 1ull) << (k - 1 - j);
        const uint64_t base = i & ~tmask;
        const double2 *row = M + r * d;
        double ar = 0.0, ai = 0.0;
        for (uint64_t c = 0; c < d; ++c) {
            uint64_t idx = base; // the group's amplitude with target bits c
            for (int j = 0; j < k; ++j) idx |= ((c >> (k - 1 - j)) & 1ull) << bits.b[j];
            const typename VecT<T>::type v = in[idx];
            const double2 m = row[c];
            const double vx = v.x, vy = v.y;
            ar += m.x * vx - m.y * vy;
            ai += m.x * vy + m.y * vx;
        }
        out[i] = mk<T>(static_cast<T>(ar), static_cast<T>(ai));
    }
}

template <typename T>
__global__ __launch_bounds__(kBlock) void scale_kernel(typename VecT<T>::type *a, uint64_t N, double re, double im) {
    const uint64_t stride = static_cast<uint64_t>(gridDim.x) * kBlock;
    const typename VecT<T>::type f = mk<T>(static_cast<T>(re), static_cast<T>(im));
    for (uint64_t i = static_cast<uint64_t>(blockIdx.x) * kBlock + threadIdx.x; i < N; i += stride)
        a[i] = cmul(f, a[i]);
}

template <typename T>
__global__ __launch_bounds__(kBlock) void collapse_kernel(typename VecT<T>::type *a, uint64_t N, int bit, int branch,
                                                         double factor) {
    const uint64_t stride = static_cast<uint64_t>(gridDim.x) * kBlock;
    const T f = static_cast<T>(factor);
    for (uint64_t i = static_cast<uint64_t>(blockIdx.x) * kBlock + threadIdx.x; i < N; i += stride) {
        if (static_cast<int>((i >> bit) & 1ull) != branch) a[i] = mk<T>(T(0), T(0));
        else a[i] = mk<T>(a[i].x * f, a[i].y * f);
    }
}

template <typename T>
__global__ __launch_bounds__(kBlock) void set_subspace_kernel(typename VecT<T>::type *a, const typename VecT<T>::type *src,
                                                             BitList bits, int nw) {
    const uint64_t i = static_cast<uint64_t>(blockIdx.x) * kBlock + threadIdx.x;
    if (i >= (1ull << nw)) return;
    uint64_t idx = 0;
    for (int j = 0; j < nw; ++j) idx |= ((i >> (nw - 1 - j)) & 1ull) << bits.b[j];
    a[idx] = src[i];
}

template <typename T>
__global__ __launch_bounds__(kBlock) void axpy_kernel(const typename VecT<T>::type *x, typename VecT<T>::type *y,
                                                     uint64_t N, double re, double im) {
    const uint64_t stride = static_cast<uint64_t>(gridDim.x) * kBlock;
    const typename VecT<T>::type f = mk<T>(static_cast<T>(re), static_cast<T>(im));
    for (uint64_t i = static_cast<uint64_t>(blockIdx.x) * kBlock + threadIdx.x; i < N; i += stride) {
        const typename VecT<T>::type v = cmul(f, x[i]);
        y[i] = mk<T>(y[i].x + v.x, y[i].y + v.y);
    }
}

__global__ __launch_bounds__(kBlock) void c128_to_c64_kernel(const double2 *s, float2 *d, uint64_t N) {
    const uint64_t stride = static_cast<uint64_t>(gridDim.x) * kBlock;
    for (uint64_t i = static_cast<uint64_t>(blockIdx.x) * kBlock + threadIdx.x; i < N; i += stride)
        d[i] = make_float2(static_cast<float>(s[i].x), static_cast<float>(s[i].y));
}
__global__ __launch_bounds__(kBlock) void c64_to_c128_kernel(const float2 *s, double2 *d, uint64_t N) {
    const uint64_t stride = static_cast<uint64_t>(gridDim.x) * kBlock;
    for (uint64_t i = static_cast<uint64_t>(blockIdx.x) * kBlock + threadIdx.x; i < N; i += stride)
        d[i] = make_double2(s[i].x, s[i].y);
}

uint32_t stream_blocks(uint64_t N) {
    const uint64_t b = (N + kBlock - 1) / kBlock;
    return static_cast<uint32_t>(b < 8192 ? (b ? b : 1) : 8192);
}

BitList to_bitlist(const int *bits, int nw) {
    BitList b{};
    for (int j = 0; j < nw && j < 64; ++j) b.b[j] = bits[j];
    return b;
}

} // namespace

// ---------------------------------------------------------------------------
// Launchers
// ---------------------------------------------------------------------------
template <typename T> void launch_tile_pass(const TilePassArgs &a, size_t lds_bytes, hipStream_t s) {
    const uint64_t nt = a.ntiles;
    const uint32_t gx = static_cast<uint32_t>(nt < 65536 ? nt : 65536);
    const uint32_t gy = static_cast<uint32_t>((nt + gx - 1) / gx);
    const dim3 grid(gx, gy);
    switch (a.ns) {
    case 1: hipLaunchKernelGGL((tile_pass_kernel<T, 1>), grid, dim3(kBlock), lds_bytes, s, a, a.heads, a.ops, a.coef, a.partials); break;
    case 2: hipLaunchKernelGGL((tile_pass_kernel<T, 2>), grid, dim3(kBlock), lds_bytes, s, a, a.heads, a.ops, a.coef, a.partials); break;
    case 3: hipLaunchKernelGGL((tile_pass_kernel<T, 3>), grid, dim3(kBlock), lds_bytes, s, a, a.heads, a.ops, a.coef, a.partials); break;
    default: hipLaunchKernelGGL((tile_pass_kernel<T, 4>), grid, dim3(kBlock), lds_bytes, s, a, a.heads, a.ops, a.coef, a.partials); break;
    }
}
template void launch_tile_pass<double>(const TilePassArgs &, size_t, hipStream_t);
template void launch_tile_pass<float>(const TilePassArgs &, size_t, hipStream_t);

void launch_reduce_slots(const double2 *partials, const SlotRange *ranges, uint32_t nslots, double2 *out,
                         hipStream_t s) {
    if (nslots == 0) return;
    hipLaunchKernelGGL(reduce_slots_kernel, dim3(nslots), dim3(kBlock), 0, s, partials, ranges, out);
}

// four amplitudes per thread once that still gives every CU a workgroup
static int pauli_unroll(int n) { return n >= 18 ? 4 : 1; }

uint32_t pauli_blocks(int n, int mode) {
    const uint64_t per = static_cast<uint64_t>(kBlock) * pauli_unroll(n), nb = (1ull << n) / per;
    const uint64_t cap = mode == 0 ? 2048 : 1024;
    return static_cast<uint32_t>(nb < 1 ? 1 : (nb < cap ? nb : cap));
}

template <typename T>
void launch_pauli_sum(const void *a, void *out, const PauliTerm *terms, uint32_t nterms, int n, int mode,
                      double2 *partials, hipStream_t s) {
    using V = typename VecT<T>::type;
    const uint64_t N = 1ull << n;
    const int unroll = pauli_unroll(n);
    const uint64_t per = static_cast<uint64_t>(kBlock) * unroll;
    const uint64_t nblk = N < per ? 1 : N / per;
    uint32_t wc = 0;
    while (wc < 6 && (16ull << wc) <= nblk) ++wc;
#define LQ_PAULI(M_, U_, G_)                                                                                   \
    hipLaunchKernelGGL((pauli_sum_kernel<T, M_, U_>), dim3(G_), dim3(kBlock), 0, s, static_cast<const V *>(a), \
                       static_cast<V *>(out), terms, nterms, N, nblk, wc, partials)
    const uint32_t grid = pauli_blocks(n, mode);
    if (mode == 0) {
        if (unroll == 4) LQ_PAULI(0, 4, grid);
        else LQ_PAULI(0, 1, grid);
    } else {
        if (unroll == 4) LQ_PAULI(1, 4, grid);
        else LQ_PAULI(1, 1, grid);
    }
#undef LQ_PAULI
}
template void launch_pauli_sum<double>(const void *, void *, const PauliTerm *, uint32_t, int, int, double2 *,
                                       hipStream_t);
template void launch_pauli_sum<float>(const void *, void *, const PauliTerm *, uint32_t, int, int, double2 *,
                                      hipStream_t);

void launch_pauli_tiles(const void *a, void *out, const PauliTerm *terms, const uint32_t *ends, uint32_t ngroups, int n,
                        hipStream_t s) {
    const uint64_t ntiles = 1ull << (n - kPauliTileBits);
    hipLaunchKernelGGL(pauli_tile_kernel, dim3(static_cast<uint32_t>(ntiles)), dim3(kPauliTileThreads),
                       sizeof(double2) << kPauliTileBits, s, static_cast<const double2 *>(a),
                       static_cast<double2 *>(out), terms, ends, ngroups, ntiles);
}

template <typename T> void launch_norm2(const void *a, int n, double2 *partials, uint32_t nblocks, hipStream_t s) {
    using V = typename VecT<T>::type;
    hipLaunchKernelGGL(norm2_kernel<T>, dim3(nblocks), dim3(kBlock), 0, s, static_cast<const V *>(a), 1ull << n,
                       partials);
}
template void launch_norm2<double>(const void *, int, double2 *, uint32_t, hipStream_t);
template void launch_norm2<float>(const void *, int, double2 *, uint32_t, hipStream_t);

void launch_overlap(const void *a, int dtype_a, const void *b, int dtype_b, int n, double2 *partials, uint32_t nblocks,
                    hipStream_t s) {
    const uint64_t N = 1ull << n;
#define LQ_OV(TA, TB)                                                                                          \
    hipLaunchKernelGGL((overlap_kernel<TA, TB>), dim3(nblocks), dim3(kBlock), 0, s,                          \
                       static_cast<const typename VecT<TA>::type *>(a), static_cast<const typename VecT<TB>::type *>(b), \
                       N, partials)
    if (dtype_a && dtype_b) LQ_OV(double, double);
    else if (dtype_a) LQ_OV(double, float);
    else if (dtype_b) LQ_OV(float, double);
    else LQ_OV(float, float);
#undef LQ_OV
}

template <typename T>
void launch_sparse_rows(const void *a, void *out, const int64_t *indptr, const int64_t *indices, const void *values,
                        uint64_t nrows, int mode, double2 *partials, uint32_t nblocks, hipStream_t s) {
    using V = typename VecT<T>::type;
    if (mode == 0)
        hipLaunchKernelGGL((sparse_rows_kernel<T, 0>), dim3(nblocks), dim3(kBlock), 0, s, static_cast<const V *>(a),
                           nullptr, indptr, indices, static_cast<const V *>(values), nrows, partials);
    else
        hipLaunchKernelGGL((sparse_rows_kernel<T, 1>), dim3(nblocks), dim3(kBlock), 0, s, static_cast<const V *>(a),
                           static_cast<V *>(out), indptr, indices, static_cast<const V *>(values), nrows, nullptr);
}
template void launch_sparse_rows<double>(const void *, void *, const int64_t *, const int64_t *, const void *, uint64_t,
                                         int, double2 *, uint32_t, hipStream_t);
template void launch_sparse_rows<float>(const void *, void *, const int64_t *, const int64_t *, const void *, uint64_t,
                                        int, double2 *, uint32_t, hipStream_t);

// Workgroups of a marginal: two rounds of the eight a CU holds; each then takes
// several items (22 and 24 qubits, the 16 high wires: 61 and 101 us with 2048,
// 63 and 101 with 4096, 75 and 104 with 16384).
constexpr uint64_t kProbsBlocks = 4096;

// High bits of a marginal: measured (wh) and not (rest), and how many of the
// unmeasured ones (the highest) are split over workgroups. Eight workgroups
// for each of the 256 CUs fill the chip, but an item keeps at least four
// loads per thread and there are at most 512 rows to add up.
static int probs_split(int n, const int *bits, int nw, int lb, uint64_t *wh, uint64_t *rest) {
    uint64_t w = 0;
    for (int j = 0; j < nw; ++j) w |= 1ull << bits[j];
    const uint64_t high = ((1ull << n) - 1ull) & ~((1ull << lb) - 1ull);
    *wh = w & high;
    *rest = ~w & high;
    const int nh = __builtin_popcountll(*wh), nr = __builtin_popcountll(*rest);
    int s = 0;
    while (s < 9 && nh + s < 11 && nr - s > 2) ++s;
    return s;
}

uint32_t probs_rows(int n, const int *bits, int nw) {
    uint64_t wh, rest;
    return 1u << probs_split(n, bits, nw, n < 8 ? n : 8, &wh, &rest);
}

template <typename T> void launch_probs(const void *a, int n, const int *bits, int nw, double *out, hipStream_t s) {
    using V = typename VecT<T>::type;
    const int lb = n < 8 ? n : 8;
    uint64_t wh, rest;
    const int split = probs_split(n, bits, nw, lb, &wh, &rest);
    uint64_t sm = 0, rm = rest;
    for (int k = 0; k < split; ++k) {
        const uint64_t top = 1ull << (63 - __builtin_clzll(rm));
        sm |= top;
        rm ^= top;
    }
    uint32_t wl = 0;
    for (int j = 0; j < nw; ++j)
        if (bits[j] < lb) wl |= 1u << bits[j];
    const uint64_t items = 1ull << (__builtin_popcountll(wh) + split);
    int from[64] = {}; // state bit of each output bit
    for (int j = 0; j < nw; ++j) from[nw - 1 - j] = bits[j];
    const uint32_t grid = static_cast<uint32_t>(std::min<uint64_t>(items, kProbsBlocks));
    hipLaunchKernelGGL(probs_kernel<T>, dim3(grid), dim3(kBlock), 0, s, static_cast<const V *>(a), lb, wl, wh, sm, rm,
                       items, to_bitlist(from, nw), nw, out);
}
template void launch_probs<double>(const void *, int, const int *, int, double *, hipStream_t);
template void launch_probs<float>(const void *, int, const int *, int, double *, hipStream_t);

void launch_reduce_rows(const double *partials, uint32_t nrows, uint32_t ncols, double *out, hipStream_t s) {
    hipLaunchKernelGGL(reduce_rows_kernel, dim3((ncols + 15) / 16), dim3(kBlock), 0, s, partials, nrows, ncols, out);
}

template <typename T> void launch_fill_product(void *a, int n, const ProductFactors &f, hipStream_t s) {
    using V = typename VecT<T>::type;
    const int lb = n < 8 ? n : 8;
    const int mb = (n - lb) < 8 ? (n - lb) : 8;
    const uint32_t segs = 1u << (n - lb - mb); // n <= 40: at most 2^24 segments
    hipLaunchKernelGGL(fill_product_kernel<T>, dim3(segs), dim3(kBlock), 0, s, static_cast<V *>(a), n, lb, mb, f);
}
template void launch_fill_product<double>(void *, int, const ProductFactors &, hipStream_t);
template void launch_fill_product<float>(void *, int, const ProductFactors &, hipStream_t);

void launch_stream_copy(const void *src, void *dst, uint64_t bytes, hipStream_t s) {
    const uint64_t N = bytes / 16;
    const uint64_t per = static_cast<uint64_t>(kBlock) * 4;
    const uint64_t b = (N + per - 1) / per;
    const uint32_t blocks = static_cast<uint32_t>(b < 16384 ? (b ? b : 1) : 16384);
    hipLaunchKernelGGL(stream_copy_kernel, dim3(blocks), dim3(kBlock), 0, s, static_cast<const double2 *>(src),
                       static_cast<double2 *>(dst), N);
}

template <typename T>
void launch_dense_wide(const void *in, void *out, const double2 *M, const int *bits, int k, uint64_t cmask,
                       uint64_t cval, int n, hipStream_t s) {
    using V = typename VecT<T>::type;
    const uint64_t N = 1ull << n;
    uint64_t tmask = 0;
    for (int j = 0; j < k; ++j) tmask |= 1ull << bits[j];
    hipLaunchKernelGGL(dense_wide_kernel<T>, dim3(stream_blocks(N)), dim3(kBlock), 0, s, static_cast<const V *>(in),
                       static_cast<V *>(out), M, to_bitlist(bits, k), k, tmask, cmask, cval, N);
}
template void launch_dense_wide<double>(const void *, void *, const double2 *, const int *, int, uint64_t, uint64_t,
                                        int, hipStream_t);
template void launch_dense_wide<float>(const void *, void *, const double2 *, const int *, int, uint64_t, uint64_t,
                                       int, hipStream_t);

template <typename T> void launch_scale(void *a, int n, double re, double im, hipStream_t s) {
    using V = typename VecT<T>::type;
    const uint64_t N = 1ull << n;
    hipLaunchKernelGGL(scale_kernel<T>, dim3(stream_blocks(N)), dim3(kBlock), 0, s, static_cast<V *>(a), N, re, im);
}
template void launch_scale<double>(void *, int, double, double, hipStream_t);
template void launch_scale<float>(void *, int, double, double, hipStream_t);

template <typename T> void launch_collapse(void *a, int n, int bit, int branch, double factor, hipStream_t s) {
    using V = typename VecT<T>::type;
    const uint64_t N = 1ull << n;
    hipLaunchKernelGGL(collapse_kernel<T>, dim3(stream_blocks(N)), dim3(kBlock), 0, s, static_cast<V *>(a), N, bit,
                       branch, factor);
}
template void launch_collapse<double>(void *, int, int, int, double, hipStream_t);
template void launch_collapse<float>(void *, int, int, int, double, hipStream_t);

template <typename T>
void launch_set_subspace(void *a, int n, const void *src, const int *bits, int nw, hipStream_t s) {
    using V = typename VecT<T>::type;
    (void)n;
    const uint64_t no = 1ull << nw;
    hipLaunchKernelGGL(set_subspace_kernel<T>, dim3(static_cast<uint32_t>((no + kBlock - 1) / kBlock)), dim3(kBlock), 0,
                       s, static_cast<V *>(a), static_cast<const V *>(src), to_bitlist(bits, nw), nw);
}
template void launch_set_subspace<double>(void *, int, const void *, const int *, int, hipStream_t);
template void launch_set_subspace<float>(void *, int, const void *, const int *, int, hipStream_t);

template <typename T> void launch_axpy(const void *x, void *y, double re, double im, int n, hipStream_t s) {
    using V = typename VecT<T>::type;
    const uint64_t N = 1ull << n;
    hipLaunchKernelGGL(axpy_kernel<T>, dim3(stream_blocks(N)), dim3(kBlock), 0, s, static_cast<const V *>(x),
                       static_cast<V *>(y), N, re, im);
}
template void launch_axpy<double>(const void *, void *, double, double, int, hipStream_t);
template void launch_axpy<float>(const void *, void *, double, double, int, hipStream_t);

void launch_c128_to_c64(const void *src, void *dst, uint64_t count, hipStream_t s) {
    hipLaunchKernelGGL(c128_to_c64_kernel, dim3(stream_blocks(count)), dim3(kBlock), 0, s,
                       static_cast<const double2 *>(src), static_cast<float2 *>(dst), count);
}
void launch_c64_to_c128(const void *src, void *dst, uint64_t count, hipStream_t s) {
    hipLaunchKernelGGL(c64_to_c128_kernel, dim3(stream_blocks(count)), dim3(kBlock), 0, s,
                       static_cast<const float2 *>(src), static_cast<double2 *>(dst), count);
}

} // namespace lqamd
