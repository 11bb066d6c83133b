// Device utilities for gfx950 (wave64): block reductions with a deterministic
// "last block finishes" step, number formats, and launch helpers.
#pragma once

#include <hip/hip_runtime.h>

#include <cmath>
#include <cstdint>

namespace owtk::dev {

constexpr int kWave = 64;
constexpr int kBlock = 256;          // threads per block for streaming kernels
constexpr int kWavesPerBlock = kBlock / kWave;
constexpr int kMaxReduceValues = 64; // values one reduction kernel may carry
constexpr int kMaxReduceBlocks = 16384;

// ------------------------------------------------------------ number types --
struct bf16 {
    std::uint16_t bits;
};

__host__ __device__ inline float bf16_to_float(std::uint16_t b)
{
    union {
        std::uint32_t u;
        float f;
    } v;
    v.u = static_cast<std::uint32_t>(b) << 16;
    return v.f;
}

// Round to nearest even; NaN stays NaN.
__host__ __device__ inline std::uint16_t float_to_bf16(float f)
{
    union {
        std::uint32_t u;
        float f;
    } v;
    v.f = f;
    if ((v.u & 0x7fffffffU) > 0x7f800000U) return static_cast<std::uint16_t>((v.u >> 16) | 0x40U);
    const std::uint32_t rounding = 0x7fffU + ((v.u >> 16) & 1U);
    return static_cast<std::uint16_t>((v.u + rounding) >> 16);
}

// Dense B x B blocks in the SELL-64 layout, elements in lane-interleaved
// pairs: elements 2g and 2g+1 (j = r*B + c) of the 64 slots of a wave sit in
// one contiguous run of 128 values, each lane's pair adjacent, so one load
// of a wave reads both elements of a pair (16 bytes a lane in FP64).  With
// B*B odd the last element is a run of 64 single values.  Element j of slot
// s is at (s & ~63) * B*B + dense_offset(s & 63, j, B*B).
__host__ __device__ constexpr std::int64_t dense_offset(std::int64_t lane, int j, int bb)
{
    return j < (bb & ~1) ? 128 * (j >> 1) + 2 * lane + (j & 1) : 64 * j + lane;
}
__host__ __device__ constexpr std::int64_t dense_index(std::int64_t slot, int j, int bb)
{
    return (slot & ~std::int64_t(63)) * bb + dense_offset(slot & 63, j, bb);
}
// The inverse within one wave's run of 64 * bb values: offset o holds
// element j of lane `lane`.
__host__ __device__ constexpr void dense_element(std::int64_t o, int bb, int& lane, int& j)
{
    if (o < 64 * (bb & ~1)) {
        lane = static_cast<int>((o & 127) >> 1);
        j = static_cast<int>(2 * (o >> 7) + (o & 1));
    } else {
        lane = static_cast<int>(o & 63);
        j = bb - 1;
    }
}

template<class V> __device__ inline float load_as_float(const V* p, std::int64_t i);
template<> __device__ inline float load_as_float<float>(const float* p, std::int64_t i) { return p[i]; }
template<> __device__ inline float load_as_float<std::uint16_t>(const std::uint16_t* p, std::int64_t i)
{
    return bf16_to_float(p[i]);
}

__device__ inline double dfma(double a, double b, double c) { return __builtin_fma(a, b, c); }
__device__ inline float dfma(float a, float b, float c) { return __builtin_fmaf(a, b, c); }

// ------------------------------------------------------------- reductions --
__device__ inline double wave_sum(double v)
{
#pragma unroll
    for (int offset = kWave / 2; offset > 0; offset >>= 1) v += __shfl_xor(v, offset, kWave);
    return v;
}

__device__ inline double wave_max(double v)
{
#pragma unroll
    for (int offset = kWave / 2; offset > 0; offset >>= 1) v = fmax(v, __shfl_xor(v, offset, kWave));
    return v;
}

// How a reduced value is combined: sum, or max of magnitudes (NaN-aware: a NaN
// anywhere yields NaN).
enum class Combine { sum, max };

template<Combine C>
__device__ inline double combine(double a, double b)
{
    if constexpr (C == Combine::sum) {
        return a + b;
    } else {
        if (a != a || b != b) return __builtin_nan("");
        return a > b ? a : b;
    }
}

template<Combine C>
__device__ inline double wave_combine(double v)
{
#pragma unroll
    for (int offset = kWave / 2; offset > 0; offset >>= 1) v = combine<C>(v, __shfl_xor(v, offset, kWave));
    return v;
}

// Reduce v[0..K) over the block; thread 0 gets the block totals in v.
// Bit k of max_mask set: value k is a max of magnitudes, else a sum.
template<int K>
__device__ inline void block_reduce(double (&v)[K], std::uint64_t max_mask)
{
    __shared__ double lds[kWavesPerBlock][K > 0 ? K : 1];
    const int lane = threadIdx.x & (kWave - 1);
    const int wave = threadIdx.x / kWave;
#pragma unroll
    for (int k = 0; k < K; ++k) {
        v[k] = ((max_mask >> k) & 1) ? wave_combine<Combine::max>(v[k])
                                     : wave_combine<Combine::sum>(v[k]);
    }
    if (lane == 0) {
#pragma unroll
        for (int k = 0; k < K; ++k) lds[wave][k] = v[k];
    }
    __syncthreads();
    if (threadIdx.x == 0) {
#pragma unroll
        for (int k = 0; k < K; ++k) {
            double acc = lds[0][k];
            for (int w = 1; w < kWavesPerBlock; ++w)
                acc = ((max_mask >> k) & 1) ? combine<Combine::max>(acc, lds[w][k])
                                            : combine<Combine::sum>(acc, lds[w][k]);
            v[k] = acc;
        }
    }
    __syncthreads();
}

// Partials of cross-block reductions: value k of block b lives at
// partials[k * stride + b], so a reduction over G blocks needs stride >= G.
// A context's buffer holds kMaxReduceValues rows of `stride` blocks and grows
// (at matrix creation) for kernels that launch more blocks than that.
struct ReduceScratch {
    double* partials;
    std::int64_t stride;
    // fused reductions (reduce_end): the count of blocks that are done, zero
    // between kernels; null: the partials go to a finisher launch
    unsigned int* ticket = nullptr;
};

// Largest grid whose last block finishes a reduction itself.  A finisher
// launch costs about 4 us; a block's fence and its atomic on the one counter
// cost less until the blocks queue up.  BiCGSTAB + Jacobi (four reductions an
// iteration), block 3, us per iteration fused / with finishers: 38 / 42 at
// 2,048 vertices (8 blocks), 39 / 46 at 8,192 (32), 45 / 47 at 32,768 (128),
// 59 / 51 at 64,800 (254).
constexpr unsigned int kFuseBlocks = 128;

// Cross-block reductions of more than kFuseBlocks blocks run in two launches
// (those of fewer end in the kernel itself, reduce_end).  The streaming kernel
// calls store_partials: each block reduces its values and writes one partial
// per value.  A one-block finisher (k_finish, launched right after on the same
// stream) then sums the partials in a fixed order, so results are
// deterministic for a fixed grid, and runs the caller's finalizer with all of
// its threads (totals in LDS, identical on every thread); single-thread state
// updates inside a finalizer are guarded by threadIdx.x == 0.  The kernel
// boundary makes the partials visible across XCDs without any fence or atomic
// inside the streaming kernel.
template<int K>
__device__ inline void store_partials(double (&v)[K], std::uint64_t max_mask, ReduceScratch scratch)
{
    block_reduce<K>(v, max_mask);
    if (threadIdx.x == 0) {
#pragma unroll
        for (int k = 0; k < K; ++k) scratch.partials[k * scratch.stride + blockIdx.x] = v[k];
    }
}

// Sums the partials of nblocks blocks in a fixed order; totals (LDS) on every
// thread (the last block of a kernel that ends its own reduction).
template<int K>
__device__ inline void finish_totals(double (&totals)[K], unsigned int nblocks, std::uint64_t max_mask,
                                     ReduceScratch scratch)
{
    // The partials were written by other XCDs, so each load waits a full
    // memory latency.  A thread issues all loads of a chunk (U blocks x K
    // values) before its first combine; the combine order per thread stays
    // b = t, t + 256, ..., so totals do not depend on U.
    constexpr int U = K >= 32 ? 1 : (K >= 16 ? 2 : 4);
    double acc[K];
#pragma unroll
    for (int k = 0; k < K; ++k) acc[k] = 0.0;
    for (unsigned int base = threadIdx.x; base < nblocks; base += U * blockDim.x) {
        double p[U][K];
#pragma unroll
        for (int u = 0; u < U; ++u) {
            const unsigned int b = base + u * blockDim.x;
#pragma unroll
            for (int k = 0; k < K; ++k) p[u][k] = b < nblocks ? scratch.partials[k * scratch.stride + b] : 0.0;
        }
#pragma unroll
        for (int u = 0; u < U; ++u) {
            if (base + u * blockDim.x >= nblocks) break;
#pragma unroll
            for (int k = 0; k < K; ++k)
                acc[k] = ((max_mask >> k) & 1) ? combine<Combine::max>(acc[k], p[u][k])
                                               : combine<Combine::sum>(acc[k], p[u][k]);
        }
    }
    block_reduce<K>(acc, max_mask);
    if (threadIdx.x == 0) {
#pragma unroll
        for (int k = 0; k < K; ++k) totals[k] = acc[k];
    }
    __syncthreads();
}

// A result the host waits for: after the values (pinned memory, written by one
// block) the block writes their number, which the host polls.  The wait for
// the stream itself costs several microseconds more.
struct Mail {
    unsigned long long* flag = nullptr;
    unsigned long long number = 0;
    // all threads of the block, after their stores
    __device__ void post() const
    {
        if (flag == nullptr) return;
        __syncthreads();
        if (threadIdx.x == 0) {
            __threadfence_system();
            __hip_atomic_store(flag, number, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
        }
    }
};

// Scratch of a kernel of g blocks: the ticket, if the caller's scratch has one,
// only where the kernel finishes its reduction itself.
inline ReduceScratch scratch_for(ReduceScratch s, unsigned int g)
{
    if (g > kFuseBlocks) s.ticket = nullptr;
    return s;
}

// Finalizers that read a vector which their own kernel wrote, or report to a
// host that may read it, say so: static constexpr bool kReadsStores = true.
template<class Fin>
constexpr bool reads_stores()
{
    if constexpr (requires { Fin::kReadsStores; }) return Fin::kReadsStores;
    else return false;
}

// Waits until the wave's stores have reached the XCD's L2.
__device__ inline void stores_in_l2()
{
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "workgroup");  // compiler order
    __builtin_amdgcn_s_waitcnt(0x0f70);                     // vmcnt(0)
}

// Ends a reducing kernel: the block's partials, and with a ticket the last
// block to arrive does the finisher's work (the same sums in the same order).
// Thread 0's fence before the counter writes the XCD's L2 back and so publishes
// what the block had stored there by then: the partials, which thread 0 stored
// itself, and where a vector of this kernel is read next (by block_norm's
// second pass, or by the host's other streams once it has the result) also the
// vector, because every wave then waits for its own stores before a barrier of
// the block (a barrier alone waits for LDS only).  The wait comes after the
// block's sums, which hide most of it.  (A release fence in every wave would
// write the L2 back four times a block: 47 -> 56 us an iteration of BiCGSTAB +
// Jacobi at 32,768 vertices.)
template<int K, class Fin>
__device__ inline void reduce_end(double (&v)[K], std::uint64_t max_mask, ReduceScratch scratch, const Fin& fin)
{
    store_partials<K>(v, max_mask, scratch);
    if (scratch.ticket == nullptr) return;
    if constexpr (reads_stores<Fin>()) {
        stores_in_l2();
        __syncthreads();
    }
    __shared__ double totals[K];
    __shared__ unsigned int arrived;
    if (threadIdx.x == 0) {
        __threadfence();
        arrived = atomicAdd(scratch.ticket, 1U);
    }
    __syncthreads();
    if (arrived != gridDim.x - 1) return;
    __threadfence();
    if (threadIdx.x == 0) *scratch.ticket = 0;
    finish_totals<K>(totals, gridDim.x, max_mask, scratch);
    fin(static_cast<const double*>(totals));
}

// One 16-wave block.  What bounds it is latency: the partials come from other
// XCDs, and nothing else runs.  The waves are dealt out to the values (16 / P
// waves each, P the power of two from K; in turns for K > 16), so a wave
// combines one value across its lanes instead of each wave all of them, and
// 16 loads are in flight per lane.  Three values of 8,192 blocks: 7.8 us, and
// 10 with four waves that each combined all values; BiCGSTAB + ILU(0) at 2M
// vertices, four finishers an iteration: 25.7 -> 25.4 ms a solve.
constexpr int kFinishThreads = 1024;

template<int K, class Fin>
__global__ __launch_bounds__(kFinishThreads) void k_finish(Fin fin, unsigned int nblocks, std::uint64_t max_mask,
                                                           ReduceScratch scratch, const int* stop, const int* need)
{
    if (stop != nullptr && *stop != 0) return;
    if (need != nullptr && *need == 0) return;
    constexpr int kWaves = kFinishThreads / kWave;
    constexpr int P = K <= 1 ? 1 : K <= 2 ? 2 : K <= 4 ? 4 : K <= 8 ? 8 : 16;
    constexpr int S = kWaves / P;  // waves per value
    constexpr int U = 16;
    __shared__ double parts[K][S];
    __shared__ double totals[K];
    const int wave = threadIdx.x / kWave;
    const unsigned int lane = threadIdx.x & (kWave - 1);
    const unsigned int first = (wave % S) * kWave + lane;
    for (int k = wave / S; k < K; k += P) {
        const double* row = scratch.partials + k * scratch.stride;
        auto sum = [&]<Combine C>() {
            double acc = 0.0;
            for (unsigned int base = first; base < nblocks; base += U * S * kWave) {
                double p[U];
#pragma unroll
                for (int u = 0; u < U; ++u) {
                    const unsigned int b = base + u * S * kWave;
                    p[u] = b < nblocks ? row[b] : 0.0;
                }
#pragma unroll
                for (int u = 0; u < U; ++u) acc = combine<C>(acc, p[u]);
            }
            return wave_combine<C>(acc);
        };
        const double v = ((max_mask >> k) & 1) ? sum.template operator()<Combine::max>()
                                               : sum.template operator()<Combine::sum>();
        if (lane == 0) parts[k][wave % S] = v;
    }
    __syncthreads();
    if (threadIdx.x < K) {
        const bool is_max = (max_mask >> threadIdx.x) & 1;
        double acc = parts[threadIdx.x][0];
        for (int w = 1; w < S; ++w)
            acc = is_max ? combine<Combine::max>(acc, parts[threadIdx.x][w])
                         : combine<Combine::sum>(acc, parts[threadIdx.x][w]);
        totals[threadIdx.x] = acc;
    }
    __syncthreads();
    fin(static_cast<const double*>(totals));
}

// stop: skip when *stop != 0; need (optional): skip when *need == 0.  Nothing
// to launch when the kernel finished its reduction itself.
template<int K, class Fin>
inline void launch_finish(hipStream_t st, const Fin& fin, unsigned int nblocks, std::uint64_t max_mask,
                          ReduceScratch scratch, const int* stop, const int* need = nullptr)
{
    if (scratch.ticket != nullptr) return;
    k_finish<K, Fin><<<1, kFinishThreads, 0, st>>>(fin, nblocks, max_mask, scratch, stop, need);
}

// ------------------------------------------- double-double (compensated) --
// Compensated reductions carry each sum as an unevaluated pair hi + lo.
// TwoSum (Knuth) gives s + e == a + b exactly; TwoProd by FMA gives the
// product's rounding error.  The kernels are built with -ffp-contract=off,
// so none of these operations is fused or reassociated.
__device__ inline void two_sum(double a, double b, double& s, double& e)
{
    s = a + b;
    const double bb = s - a;
    e = (a - (s - bb)) + (b - bb);
}

// (hi, lo) += a * b
__device__ inline void dd_fma(double& hi, double& lo, double a, double b)
{
    const double p = a * b;
    const double pe = __builtin_fma(a, b, -p);
    double s, e;
    two_sum(hi, p, s, e);
    hi = s;
    lo += e + pe;
}

// (h1, l1) += (h2, l2)
__device__ inline void dd_combine(double& h1, double& l1, double h2, double l2)
{
    double s, e;
    two_sum(h1, h2, s, e);
    h1 = s;
    l1 = (l1 + l2) + e;
}

// Block reduction of K pairs (hi[k], lo[k]); bit k of max_mask: value k is a
// max of magnitudes (carried in hi, lo stays 0).  Thread 0 gets the totals.
template<int K>
__device__ inline void block_reduce_dd(double (&hi)[K], double (&lo)[K], std::uint64_t max_mask)
{
    __shared__ double lds[kWavesPerBlock][2 * (K > 0 ? K : 1)];
    const int lane = threadIdx.x & (kWave - 1);
    const int wave = threadIdx.x / kWave;
#pragma unroll
    for (int k = 0; k < K; ++k) {
#pragma unroll
        for (int offset = kWave / 2; offset > 0; offset >>= 1) {
            const double h2 = __shfl_xor(hi[k], offset, kWave);
            const double l2 = __shfl_xor(lo[k], offset, kWave);
            if ((max_mask >> k) & 1) hi[k] = combine<Combine::max>(hi[k], h2);
            else dd_combine(hi[k], lo[k], h2, l2);
        }
    }
    if (lane == 0) {
#pragma unroll
        for (int k = 0; k < K; ++k) {
            lds[wave][k] = hi[k];
            lds[wave][K + k] = lo[k];
        }
    }
    __syncthreads();
    if (threadIdx.x == 0) {
#pragma unroll
        for (int k = 0; k < K; ++k) {
            double h = lds[0][k], l = lds[0][K + k];
            for (int w = 1; w < kWavesPerBlock; ++w) {
                if ((max_mask >> k) & 1) h = combine<Combine::max>(h, lds[w][k]);
                else dd_combine(h, l, lds[w][k], lds[w][K + k]);
            }
            hi[k] = h;
            lo[k] = l;
        }
    }
    __syncthreads();
}

// Compensated partials: value k of block b as hi at row k, lo at row K + k
// (2K <= kMaxReduceValues rows).
template<int K>
__device__ inline void store_partials_dd(double (&hi)[K], double (&lo)[K], std::uint64_t max_mask,
                                         ReduceScratch scratch)
{
    static_assert(2 * K <= kMaxReduceValues, "too many compensated values");
    block_reduce_dd<K>(hi, lo, max_mask);
    if (threadIdx.x == 0) {
#pragma unroll
        for (int k = 0; k < K; ++k) {
            scratch.partials[k * scratch.stride + blockIdx.x] = hi[k];
            scratch.partials[(K + k) * scratch.stride + blockIdx.x] = lo[k];
        }
    }
}

// Finisher of compensated partials: pairs combined in a fixed order (block
// b = t, t + 256, ... per thread, then the block tree); the finalizer gets
// hi + lo rounded once.
template<int K, class Fin>
__global__ __launch_bounds__(256) void k_finish_dd(Fin fin, unsigned int nblocks, std::uint64_t max_mask,
                                                   ReduceScratch scratch, const int* stop)
{
    if (stop != nullptr && *stop != 0) return;
    __shared__ double totals[K > 0 ? K : 1];
    double hi[K], lo[K];
#pragma unroll
    for (int k = 0; k < K; ++k) hi[k] = lo[k] = 0.0;
    for (unsigned int b = threadIdx.x; b < nblocks; b += blockDim.x) {
        double ph[K], pl[K];
#pragma unroll
        for (int k = 0; k < K; ++k) {
            ph[k] = scratch.partials[k * scratch.stride + b];
            pl[k] = scratch.partials[(K + k) * scratch.stride + b];
        }
#pragma unroll
        for (int k = 0; k < K; ++k) {
            if ((max_mask >> k) & 1) hi[k] = combine<Combine::max>(hi[k], ph[k]);
            else dd_combine(hi[k], lo[k], ph[k], pl[k]);
        }
    }
    block_reduce_dd<K>(hi, lo, max_mask);
    if (threadIdx.x == 0) {
#pragma unroll
        for (int k = 0; k < K; ++k) totals[k] = ((max_mask >> k) & 1) ? hi[k] : hi[k] + lo[k];
    }
    __syncthreads();
    fin(static_cast<const double*>(totals));
}

template<int K, class Fin>
inline void launch_finish_dd(hipStream_t st, const Fin& fin, unsigned int nblocks, std::uint64_t max_mask,
                             ReduceScratch scratch, const int* stop)
{
    k_finish_dd<K, Fin><<<1, kBlock, 0, st>>>(fin, nblocks, max_mask, scratch, stop);
}

// Sum over the block (any number of waves), result on every thread.
__device__ inline double block_sum_all(double v)
{
    __shared__ double lds[kFinishThreads / kWave];
    __shared__ double total;
    v = wave_combine<Combine::sum>(v);
    if ((threadIdx.x & (kWave - 1)) == 0) lds[threadIdx.x / kWave] = v;
    __syncthreads();
    if (threadIdx.x == 0) {
        double acc = lds[0];
        for (unsigned int w = 1; w < blockDim.x / kWave; ++w) acc += lds[w];
        total = acc;
    }
    __syncthreads();
    return total;
}

// 2-norm from a fused (sum of squares, max magnitude) pair, overflow and
// underflow safe with the semantics of detail::scaled_norm
// (reduction.hpp:64-89): NaN anywhere -> NaN, otherwise an infinite entry ->
// inf, all zero -> 0.  When the plain sum of squares over- or underflowed,
// the calling block re-reads v once and sums (v_i / max)^2.  Call with all
// threads of one block; every thread gets the result.
constexpr double kSafeSumOfSquares = 0x1.0p-960;

template<class X>
__device__ inline double block_norm(double sum_squares, double max_abs, const X* v, std::int64_t n)
{
    if (max_abs != max_abs) return __builtin_nan("");
    if (max_abs == 0.0) return 0.0;
    if (__builtin_isinf(max_abs)) return max_abs;
    if (__builtin_isfinite(sum_squares) && sum_squares >= kSafeSumOfSquares) return __builtin_sqrt(sum_squares);
    double acc = 0.0;
    for (std::int64_t i = threadIdx.x; i < n; i += blockDim.x) {
        const double r = static_cast<double>(v[i]) / max_abs;
        acc = __builtin_fma(r, r, acc);
    }
    return max_abs * __builtin_sqrt(block_sum_all(acc));
}

// Grid for streaming kernels over n items with `per_thread` items per thread.
inline unsigned int stream_grid(std::int64_t n, int per_thread = 1)
{
    std::int64_t blocks = (n + static_cast<std::int64_t>(kBlock) * per_thread - 1)
        / (static_cast<std::int64_t>(kBlock) * per_thread);
    if (blocks < 1) blocks = 1;
    if (blocks > kMaxReduceBlocks) blocks = kMaxReduceBlocks;
    return static_cast<unsigned int>(blocks);
}

} // namespace owtk::dev
