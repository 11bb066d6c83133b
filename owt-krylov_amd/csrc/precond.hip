// Jacobi, SSOR and ILU(k) preconditioners on the device.
//
// Symbolic work (block partition, ILU fill pattern, update lists, level
// schedules) runs once on the host at creation; numeric updates (value
// gather, ILU factorization, inverse diagonals) and every apply run on the
// GPU.  This is the reference's "symbolic once, numeric many" contract
// (IluLevelPreconditioner::update_values, preconditioner.hpp:269-311).
#include "precond.hpp"
#include "chain_rule.hpp"
#include "learned.hpp"
#include "kernels/blas1.hpp"
#include "kernels/spmv.hpp"
#include "host/host.hpp"

#include <algorithm>
#include <cmath>
#include <limits>
#include <map>
#include <numeric>

using namespace owtk;

namespace owtk {
namespace {

using dev::kBlock;

constexpr double kTol = 64.0 * std::numeric_limits<double>::epsilon();

enum Flag : int { flag_ok = 0, flag_zero_pivot = 1, flag_singular_diag = 2, flag_no_diag = 3 };

// ------------------------------------------------------------------ kernels --

// Gather matrix values through encoded sources: src >= 0 -> values[src + c*stride],
// src <= -2 -> diag[-2-src + c*stride], src == -1 -> 0.  out is [c][count].
__global__ __launch_bounds__(256) void k_gather(double* __restrict__ out, const std::int64_t* __restrict__ src,
                                                std::int64_t count, int bs, std::int64_t stride,
                                                const double* __restrict__ values, const double* __restrict__ diag,
                                                double scale)
{
    const std::int64_t total = count * bs;
    const std::int64_t step = static_cast<std::int64_t>(gridDim.x) * blockDim.x;
    for (std::int64_t t = static_cast<std::int64_t>(blockIdx.x) * blockDim.x + threadIdx.x; t < total; t += step) {
        const std::int64_t c = t / count;
        const std::int64_t e = t - c * count;
        const std::int64_t s = src[e];
        double v = 0.0;
        if (s >= 0) v = values[s + c * stride];
        else if (s <= -2) v = diag[(-2 - s) + c * stride];
        out[t] = scale == 1.0 ? v : scale * v;
    }
}

// Gather from a [c][nsrc] array by index (index < 0 -> 0).
__global__ __launch_bounds__(256) void k_gather_cm(double* __restrict__ out, const std::int64_t* __restrict__ src,
                                                   std::int64_t count, int bs, const double* __restrict__ in,
                                                   std::int64_t nsrc)
{
    const std::int64_t total = count * bs;
    const std::int64_t step = static_cast<std::int64_t>(gridDim.x) * blockDim.x;
    for (std::int64_t t = static_cast<std::int64_t>(blockIdx.x) * blockDim.x + threadIdx.x; t < total; t += step) {
        const std::int64_t c = t / count;
        const std::int64_t e = t - c * count;
        const std::int64_t s = src[e];
        out[t] = s >= 0 ? in[c * nsrc + s] : 0.0;
    }
}

// SSOR diagonal check (LocalSsorPreconditioner::update_values,
// preconditioner.hpp:142-174): finite and |d| > 64 eps.
__global__ __launch_bounds__(256) void k_check_diag(const double* __restrict__ d, std::int64_t n, double tol, int* flag)
{
    const std::int64_t step = static_cast<std::int64_t>(gridDim.x) * blockDim.x;
    for (std::int64_t i = static_cast<std::int64_t>(blockIdx.x) * blockDim.x + threadIdx.x; i < n; i += step) {
        const double v = d[i];
        if (!(__builtin_isfinite(v) && __builtin_fabs(v) > tol)) atomicExch(flag, static_cast<int>(flag_singular_diag));
    }
}

// Jacobi inverse (JacobiPreconditioner::update_values, preconditioner.hpp:55-71).
__global__ __launch_bounds__(256) void k_jacobi_inverse(double* __restrict__ inv, const std::int64_t* __restrict__ src,
                                                        std::int64_t rows, int bs, std::int64_t stride,
                                                        const double* __restrict__ values,
                                                        const double* __restrict__ diag, double minimum, int* flag)
{
    const std::int64_t total = rows * bs;
    const std::int64_t step = static_cast<std::int64_t>(gridDim.x) * blockDim.x;
    for (std::int64_t t = static_cast<std::int64_t>(blockIdx.x) * blockDim.x + threadIdx.x; t < total; t += step) {
        const std::int64_t row = t / bs;
        const std::int64_t c = t - row * bs;
        const std::int64_t s = src[row];
        const double v = s >= 0 ? values[s + c * stride] : diag[(-2 - s) + c * stride];
        if (!(__builtin_isfinite(v) && __builtin_fabs(v) > minimum)) atomicExch(flag, static_cast<int>(flag_singular_diag));
        inv[t] = 1.0 / v;
    }
}

template<class X, class V>
__global__ __launch_bounds__(256) void k_jacobi_apply(const V* __restrict__ inv, const X* __restrict__ in,
                                                      X* __restrict__ out, std::int64_t n, const int* stop)
{
    if (stop && *stop) return;
    const std::int64_t step = static_cast<std::int64_t>(gridDim.x) * blockDim.x;
    for (std::int64_t i = static_cast<std::int64_t>(blockIdx.x) * blockDim.x + threadIdx.x; i < n; i += step)
        out[i] = static_cast<X>(inv[i]) * in[i];
}

// Dense block-Jacobi: invert each bs x bs diagonal block by Gauss-Jordan with
// partial pivoting (thread per row).  No reference counterpart: the dense
// BSR form has no diagonal() (dense_block_csr.hpp).
template<int BS>
__global__ __launch_bounds__(256) void k_block_inverse(double* __restrict__ inv, const std::int64_t* __restrict__ slot,
                                                       std::int64_t rows, const double* __restrict__ values,
                                                       int* flag)
{
    const std::int64_t row = static_cast<std::int64_t>(blockIdx.x) * blockDim.x + threadIdx.x;
    if (row >= rows) return;
    double a[BS][BS], b[BS][BS];
    const std::int64_t ds = slot[row];
#pragma unroll
    for (int r = 0; r < BS; ++r)
#pragma unroll
        for (int c = 0; c < BS; ++c) {
            a[r][c] = values[dev::dense_index(ds, r * BS + c, BS * BS)];
            b[r][c] = r == c ? 1.0 : 0.0;
        }
    for (int k = 0; k < BS; ++k) {
        int p = k;
        for (int r = k + 1; r < BS; ++r)
            if (__builtin_fabs(a[r][k]) > __builtin_fabs(a[p][k])) p = r;
        if (!(__builtin_fabs(a[p][k]) > 0.0) || !__builtin_isfinite(a[p][k])) {
            atomicExch(flag, static_cast<int>(flag_singular_diag));
            return;
        }
        if (p != k)
            for (int c = 0; c < BS; ++c) {
                double t = a[k][c]; a[k][c] = a[p][c]; a[p][c] = t;
                t = b[k][c]; b[k][c] = b[p][c]; b[p][c] = t;
            }
        const double inv_p = 1.0 / a[k][k];
        for (int c = 0; c < BS; ++c) {
            a[k][c] *= inv_p;
            b[k][c] *= inv_p;
        }
        for (int r = 0; r < BS; ++r) {
            if (r == k) continue;
            const double f = a[r][k];
            for (int c = 0; c < BS; ++c) {
                a[r][c] = __builtin_fma(-f, a[k][c], a[r][c]);
                b[r][c] = __builtin_fma(-f, b[k][c], b[r][c]);
            }
        }
    }
    double* out = inv + row * (BS * BS);
#pragma unroll
    for (int r = 0; r < BS; ++r)
#pragma unroll
        for (int c = 0; c < BS; ++c) out[r * BS + c] = b[r][c];
}

template<int BS, class X, class V>
__global__ __launch_bounds__(256) void k_block_jacobi_apply(const V* __restrict__ inv, const X* __restrict__ in,
                                                            X* __restrict__ out, std::int64_t rows, const int* stop)
{
    if (stop && *stop) return;
    const std::int64_t row = static_cast<std::int64_t>(blockIdx.x) * blockDim.x + threadIdx.x;
    if (row >= rows) return;
    X r[BS];
#pragma unroll
    for (int c = 0; c < BS; ++c) r[c] = in[row * BS + c];
    const V* blk = inv + row * (BS * BS);
#pragma unroll
    for (int i = 0; i < BS; ++i) {
        X t = X(0);
#pragma unroll
        for (int c = 0; c < BS; ++c) t = dev::dfma(static_cast<X>(blk[i * BS + c]), r[c], t);
        out[row * BS + i] = t;
    }
}

// Dense-block SSOR in multicolour order (no reference counterpart: the
// reference's DenseBlockCsrMatrix has no SSOR).  Rows of one colour are
// independent, so each colour is one parallel launch:
//   forward  y_i = D_i^-1 (r_i - omega sum_(colour j < colour i) A_ij y_j)
//   backward z_i = D_i^-1 (s D_i y_i - omega sum_(colour j > colour i) A_ij z_j),
// s = omega (2 - omega), i.e. z = s (D + omega U)^-1 D (D + omega L)^-1 r in
// the colour-permuted order.  Ghost columns are dropped (rank-local, like the
// component-diagonal SSOR).  Entries are visited in the row's stored order.
template<int BS, class V, class X, class I, bool FWD>
__global__ __launch_bounds__(256) void k_mc_ssor(const std::int32_t* __restrict__ prow, std::int64_t seg0,
                                                 std::int64_t count, const std::int32_t* __restrict__ slice_ptr,
                                                 const std::int32_t* __restrict__ row_len,
                                                 const std::int32_t* __restrict__ cols, const V* __restrict__ vals,
                                                 const V* __restrict__ dvals, double omega, double scale,
                                                 const X* __restrict__ in, X* __restrict__ y, X* __restrict__ out,
                                                 const I* __restrict__ inv, const int* stop)
{
    using A = typename dev::acc_type<X>::type;
    if (stop && *stop) return;
    const std::int64_t t = static_cast<std::int64_t>(blockIdx.x) * blockDim.x + threadIdx.x;
    if (t >= count) return;
    const std::int64_t q = seg0 + t;  // copy row: consecutive threads read consecutive slots
    const std::int64_t i = prow[q];
    const A w = static_cast<A>(omega);
    A acc[BS];
    if constexpr (FWD) {
#pragma unroll
        for (int r = 0; r < BS; ++r) acc[r] = static_cast<A>(in[i * BS + r]);
    } else {
        A yi[BS];
#pragma unroll
        for (int r = 0; r < BS; ++r) yi[r] = static_cast<A>(y[i * BS + r]);
#pragma unroll
        for (int r = 0; r < BS; ++r) {
            A d = A(0);
#pragma unroll
            for (int c = 0; c < BS; ++c)
                d = dev::dfma(static_cast<A>(dev::load_value(dvals, dev::dense_index(q, r * BS + c, BS * BS))),
                              yi[c], d);
            acc[r] = d * static_cast<A>(scale);
        }
    }
    const std::int64_t base = slice_ptr[q >> 6];
    const int lane = static_cast<int>(q & 63);
    const int len = row_len[q];
    const X* src = FWD ? y : out;
    for (int k = 0; k < len; ++k) {
        const std::int64_t slot = base + 64 * k + lane;
        const std::int64_t j = cols[slot];
        A xj[BS];
#pragma unroll
        for (int c = 0; c < BS; ++c) xj[c] = static_cast<A>(src[j * BS + c]);
#pragma unroll
        for (int r = 0; r < BS; ++r)
#pragma unroll
            for (int c = 0; c < BS; ++c)
                acc[r] = dev::dfma(-(w * static_cast<A>(dev::load_value(vals, dev::dense_index(slot, r * BS + c,
                                                                                              BS * BS)))),
                                   xj[c], acc[r]);
    }
    X* dst = FWD ? y : out;
    const I* blk = inv + i * (BS * BS);
#pragma unroll
    for (int r = 0; r < BS; ++r) {
        A sum = A(0);
#pragma unroll
        for (int c = 0; c < BS; ++c) sum = dev::dfma(static_cast<A>(blk[r * BS + c]), acc[c], sum);
        dst[i * BS + r] = static_cast<X>(sum);
    }
}

// Copy slots' block values from the matrix: dst[dense_index(s, j, bb)] =
// src[dense_index(map[s], j, bb)] (0 for padding).  Thread t writes dst[t].
template<class V>
__global__ __launch_bounds__(256) void k_mc_gather(V* __restrict__ dst, const V* __restrict__ src,
                                                   const std::int64_t* __restrict__ map, std::int64_t slots, int bb)
{
    const std::int64_t total = slots * bb;
    const std::int64_t step = static_cast<std::int64_t>(gridDim.x) * blockDim.x;
    for (std::int64_t t = static_cast<std::int64_t>(blockIdx.x) * blockDim.x + threadIdx.x; t < total; t += step) {
        const std::int64_t slice = t / (64 * bb);
        int lane = 0, j = 0;
        dev::dense_element(t - slice * 64 * bb, bb, lane, j);
        const std::int64_t sl = slice * 64 + lane;
        const std::int64_t from = map[sl];
        dst[t] = from >= 0 ? src[dev::dense_index(from, j, bb)] : V(0);
    }
}

struct TriArgs {
    const std::int32_t* row0;
    const std::int32_t* nrows;
    const std::int32_t* flev;
    const std::int32_t* blev;
    const std::int32_t* flev_pos;
    const std::int32_t* blev_pos;
    const std::int32_t* frow;
    const std::int32_t* brow;
    const std::int64_t* fptr;
    const std::int64_t* bptr;
    const std::int32_t* fcol;
    const std::int32_t* bcol;
    std::int64_t fnnz, bnnz, rows;
    int bs;
};

// ILU(k) numeric factorization (IluLevelPreconditioner::factorize,
// preconditioner.hpp:439-485), one workgroup per (block, component), rows in
// forward level order.  F is the FP64 factor, [c][entry].
__global__ __launch_bounds__(256) void k_ilu_factor(TriArgs a, const std::int32_t* __restrict__ lvl_rows,
                                                    const std::int64_t* __restrict__ offsets,
                                                    const std::int64_t* __restrict__ diag_pos,
                                                    const std::int64_t* __restrict__ upd_ptr,
                                                    const std::int64_t* __restrict__ upd_target,
                                                    const std::int64_t* __restrict__ upd_upper,
                                                    const std::int64_t* __restrict__ columns_global,
                                                    double* __restrict__ F, std::int64_t nnz,
                                                    double* __restrict__ inv, int* flag)
{
    const int c = blockIdx.x % a.bs;
    const int b = blockIdx.x / a.bs;
    const std::int64_t r0 = a.row0[b];
    double* Fc = F + static_cast<std::int64_t>(c) * nnz;
    const int l_begin = a.flev[b], l_end = a.flev[b + 1] - 1;
    for (int l = l_begin; l < l_end; ++l) {
        const int p0 = a.flev_pos[l], p1 = a.flev_pos[l + 1];
        for (int p = p0 + threadIdx.x; p < p1; p += blockDim.x) {
            const std::int64_t row = r0 + lvl_rows[r0 + p];
            const std::int64_t dpos = diag_pos[row];
            for (std::int64_t e = offsets[row]; e < dpos; ++e) {
                const std::int64_t k = columns_global[e];
                const double pivot = Fc[diag_pos[k]];
                if (__builtin_fabs(pivot) <= kTol) atomicExch(flag, static_cast<int>(flag_zero_pivot));
                const double lv = Fc[e] / pivot;
                Fc[e] = lv;
                for (std::int64_t u = upd_ptr[e]; u < upd_ptr[e + 1]; ++u) {
                    const std::int64_t t = upd_target[u];
                    Fc[t] = __builtin_fma(-lv, Fc[upd_upper[u]], Fc[t]);
                }
            }
        }
        __syncthreads();
    }
    const std::int64_t n = a.nrows[b];
    for (std::int64_t i = threadIdx.x; i < n; i += blockDim.x) {
        const std::int64_t row = r0 + i;
        const double d = Fc[diag_pos[row]];
        if (!(__builtin_isfinite(d) && __builtin_fabs(d) > kTol)) atomicExch(flag, static_cast<int>(flag_zero_pivot));
        inv[static_cast<std::int64_t>(c) * a.rows + row] = 1.0 / d;
    }
}

// ILU(k) numeric factorization in 64-row chunks (the IKJ order of
// IluLevelPreconditioner::factorize, preconditioner.hpp:439-485, per row),
// one wave per (block, component), rows in natural order, one row per lane:
//   1. a lane loads its row's entries into LDS (rv[slot][lane]), and the
//      chunk's static program (IluChunkProgram) is staged in LDS;
//   2. it gathers the final values of earlier chunks that its lower entries
//      need (pivots u_kk and sources u_kj) in one batch (ga[t][lane]) and
//      applies those lower entries in column order;
//   3. the chunk's own lower entries run in 64 steps: at step s row s is
//      final, and every lane whose row has an entry in column s divides by
//      row s's pivot and updates its targets from row s's entries (read from
//      LDS), which keeps each row's column order;
//   4. the chunk's rows are stored, fenced for the next chunks' gathers.
// Each row sees the same operations in the same order as the reference's
// loop, so the factors are bitwise those of the level-scheduled kernel.
// This general form takes any number of updates per operation; with at most
// seven k_ilu_factor_rec runs.
struct IluChunkArgs {
    const std::int32_t* chunk_first;
    const std::int64_t* hdr;
    const std::int32_t* src_a;
    const std::uint32_t* op_a;
    const std::uint32_t* op_b;
    const std::uint16_t* upd_a;
    const std::uint16_t* upd_b;
    const std::uint32_t* rec;
    int kmax, max_src, max_a, max_nua, max_b, max_nub;
};

inline std::size_t ilu_chunk_lds(const IluChunkProgram& P)
{
    return static_cast<std::size_t>(64) * (8 * (P.kmax + P.max_src) + 4 * (P.max_a + P.max_b)
                                           + 2 * (P.max_a * P.max_nua + P.max_b * P.max_nub));
}

// count values load(j) -> store(j, v), eight loads in flight before their
// stores; load() gets only indices below count
template<class T, class Load, class Store>
__device__ inline void copy_batched(int count, Load load, Store store)
{
    for (int j0 = 0; j0 < count; j0 += 8) {
        T v[8];
#pragma unroll
        for (int u = 0; u < 8; ++u) v[u] = load(j0 + u < count ? j0 + u : count - 1);
#pragma unroll
        for (int u = 0; u < 8; ++u)
            if (j0 + u < count) store(j0 + u, v[u]);
    }
}

__global__ __launch_bounds__(64) void k_ilu_factor_chunks(IluChunkArgs P, const std::int64_t* __restrict__ offsets,
                                                          const std::int64_t* __restrict__ diag_pos,
                                                          const std::int32_t* __restrict__ row0,
                                                          const std::int32_t* __restrict__ nrows, int bs,
                                                          double* __restrict__ F, std::int64_t nnz,
                                                          std::int64_t rows, double* __restrict__ inv, int* flag)
{
    extern __shared__ double lds_d[];
    const int lane = static_cast<int>(threadIdx.x);
    const int c = static_cast<int>(blockIdx.x) % bs;
    const int b = static_cast<int>(blockIdx.x) / bs;
    double* Fc = F + static_cast<std::int64_t>(c) * nnz;
    double* rv = lds_d;                                   // [kmax][64]
    double* ga = rv + P.kmax * 64;                        // [max_src][64]
    auto* opa = reinterpret_cast<std::uint32_t*>(ga + P.max_src * 64);  // [max_a][64]
    std::uint32_t* opb = opa + P.max_a * 64;              // [max_b][64]
    auto* upa = reinterpret_cast<std::uint16_t*>(opb + P.max_b * 64);  // [max_a*max_nua][64]
    std::uint16_t* upb = upa + P.max_a * P.max_nua * 64;  // [max_b*max_nub][64]
    const int ch_end = P.chunk_first[b + 1];
    for (int ch = P.chunk_first[b]; ch < ch_end; ++ch) {
        const std::int64_t* h = P.hdr + static_cast<std::int64_t>(ch) * 12;
        const int cnt = static_cast<int>(h[1]), nsrc = static_cast<int>(h[3]);
        const std::int64_t src_off = h[2];
        const int na = static_cast<int>(h[5]), nua = static_cast<int>(h[7]);
        const int nb = static_cast<int>(h[9]), nub = static_cast<int>(h[11]);
        std::int64_t base = 0;
        int len = 0;
        const std::int64_t row_first = h[0];
        const std::int64_t opa_off = h[4], upa_off = h[6], opb_off = h[8], upb_off = h[10];
        if (lane < cnt) {
            base = offsets[row_first + lane];
            len = static_cast<int>(offsets[row_first + lane + 1] - base);
        }
        // 1. row values and the chunk's program, all loads independent and
        //    issued in batches (a plain loop would wait for each load before
        //    its LDS store)
        const int lastq = len > 0 ? len - 1 : 0;
        copy_batched<double>(P.kmax, [&](int q) { return Fc[base + (q < lastq ? q : lastq)]; },
                             [&](int q, double v) { rv[q * 64 + lane] = q < len ? v : 0.0; });
        copy_batched<std::uint32_t>(na, [&](int j) { return P.op_a[opa_off + j * 64 + lane]; },
                                    [&](int j, std::uint32_t v) { opa[j * 64 + lane] = v; });
        copy_batched<std::uint16_t>(na * nua, [&](int j) { return P.upd_a[upa_off + j * 64 + lane]; },
                                    [&](int j, std::uint16_t v) { upa[j * 64 + lane] = v; });
        copy_batched<std::uint32_t>(nb, [&](int j) { return P.op_b[opb_off + j * 64 + lane]; },
                                    [&](int j, std::uint32_t v) { opb[j * 64 + lane] = v; });
        copy_batched<std::uint16_t>(nb * nub, [&](int j) { return P.upd_b[upb_off + j * 64 + lane]; },
                                    [&](int j, std::uint16_t v) { upb[j * 64 + lane] = v; });
        // 2. earlier chunks: gather (source indices, then values, each batch
        //    in flight together), then the lower entries in column order
        for (int t0 = 0; t0 < nsrc; t0 += 8) {
            std::int32_t idx[8];
#pragma unroll
            for (int u = 0; u < 8; ++u) {
                const int t = t0 + u < nsrc ? t0 + u : nsrc - 1;
                idx[u] = P.src_a[src_off + t * 64 + lane];
            }
            double v[8];
#pragma unroll
            for (int u = 0; u < 8; ++u) v[u] = Fc[idx[u] >= 0 ? idx[u] : 0];
#pragma unroll
            for (int u = 0; u < 8; ++u)
                if (t0 + u < nsrc) ga[(t0 + u) * 64 + lane] = idx[u] >= 0 ? v[u] : 0.0;
        }
        for (int j = 0; j < na; ++j) {
            const std::uint32_t d = opa[j * 64 + lane];
            if (d == 0xffffffffu) continue;
            const int es = static_cast<int>(d & 255u), pt = static_cast<int>((d >> 8) & 255u);
            const int nu = static_cast<int>((d >> 16) & 255u);
            const double pivot = ga[pt * 64 + lane];
            if (__builtin_fabs(pivot) <= kTol) atomicExch(flag, static_cast<int>(flag_zero_pivot));
            const double lv = rv[es * 64 + lane] / pivot;
            rv[es * 64 + lane] = lv;
            for (int u = 0; u < nu; ++u) {
                const std::uint16_t w = upa[(j * nua + u) * 64 + lane];
                const int ts = w & 255, st = w >> 8;
                rv[ts * 64 + lane] = __builtin_fma(-lv, ga[st * 64 + lane], rv[ts * 64 + lane]);
            }
        }
        // 3. the chunk's own lower entries, one pivot row per step
        int jb = 0;
        std::uint32_t d = nb > 0 ? opb[lane] : 0xffffffffu;
        for (int s = 0; s < cnt; ++s) {
            __builtin_amdgcn_wave_barrier();
            if (d != 0xffffffffu && static_cast<int>(d & 255u) == s) {
                const int es = static_cast<int>((d >> 8) & 255u), ps = static_cast<int>((d >> 16) & 255u);
                const int nu = static_cast<int>(d >> 24);
                const double pivot = rv[ps * 64 + s];
                if (__builtin_fabs(pivot) <= kTol) atomicExch(flag, static_cast<int>(flag_zero_pivot));
                const double lv = rv[es * 64 + lane] / pivot;
                rv[es * 64 + lane] = lv;
                for (int u = 0; u < nu; ++u) {
                    const std::uint16_t w = upb[(jb * nub + u) * 64 + lane];
                    const int ts = w & 255, qs = w >> 8;
                    rv[ts * 64 + lane] = __builtin_fma(-lv, rv[qs * 64 + s], rv[ts * 64 + lane]);
                }
                ++jb;
                d = jb < nb ? opb[jb * 64 + lane] : 0xffffffffu;
            }
        }
        __builtin_amdgcn_wave_barrier();
        // 4. store; later chunks of this wave gather these values
        for (int q = 0; q < len; ++q) Fc[base + q] = rv[q * 64 + lane];
        __threadfence_block();
        __builtin_amdgcn_wave_barrier();
    }
    const std::int64_t r0 = row0[b], n = nrows[b];
    for (std::int64_t i = lane; i < n; i += 64) {
        const std::int64_t row = r0 + i;
        const double dg = Fc[diag_pos[row]];
        if (!(__builtin_isfinite(dg) && __builtin_fabs(dg) > kTol)) atomicExch(flag, static_cast<int>(flag_zero_pivot));
        inv[static_cast<std::int64_t>(c) * rows + row] = 1.0 / dg;
    }
}

// The same chunks with every operation as one record of LDS byte offsets
// (IluChunkProgram::rec): its own entry, its pivot, and NU (source, target)
// pairs.  A record is one load, its halves are the addresses, and a missing
// pair or lane names a trash entry and a constant one, so an operation has no
// branch, no count and no address arithmetic beyond unpacking.
//
// What bounds it: the chain of a chunk's 64 pivot rows, one after another on
// one wave.  A step is its reads (~100 clk), a correctly rounded division
// (~130), the update and the LDS write that the next step reads (65); the
// rest is issue at 4 clk an instruction.  The step of the general kernel
// unpacked bytes into addresses and tested a count per update: ~110
// instructions, 1,940 us for 68 blocks of 4,096 vertices and 3 components
// (64 chunks one after another); 1,048 us this way, ~600 clk a step.  Holding
// the next chunk's rows, records and sources in 140 registers was slower
// (1,327 us against 1,209 without any look-ahead); its header and row
// extents alone are worth loading early.
template<int NU> using IluRec = std::uint32_t __attribute__((ext_vector_type(1 + NU)));

constexpr std::size_t ilu_rec_fixed(int kmax, int max_src) { return static_cast<std::size_t>(kmax + 2 + max_src) * 512; }

inline std::size_t ilu_rec_lds(const IluChunkProgram& P)
{
    return ilu_rec_fixed(P.kmax, P.max_src) + static_cast<std::size_t>(P.max_a + P.max_b + 1) * 64 * 4 * (1 + P.nu);
}

// after_reads() runs once the operation's own reads are issued
template<int NU, class F>
__device__ inline void ilu_rec_op(unsigned char* lds, const IluRec<NU> r, double& lowest, F after_reads)
{
    auto at = [&](int k) -> double& {
        const std::uint32_t o = k & 1 ? r[k >> 1] >> 16 : r[k >> 1] & 0xffffu;
        return *reinterpret_cast<double*>(lds + o);
    };
    const double pivot = at(1);
    const double own = at(0);
    double src[NU], tgt[NU];
#pragma unroll
    for (int u = 0; u < NU; ++u) {
        src[u] = at(2 + 2 * u);
        tgt[u] = at(3 + 2 * u);
    }
    after_reads();
    lowest = __builtin_fmin(lowest, __builtin_fabs(pivot));
    const double lv = own / pivot;
    // the targets are distinct slots of the lane's own row, neither its own
    // lower entry nor the pivot row's: the order of these stores is free
#pragma unroll
    for (int u = 0; u < NU; ++u) at(3 + 2 * u) = __builtin_fma(-lv, src[u], tgt[u]);
    at(0) = lv;
}

template<int NU>
__global__ __launch_bounds__(64) void k_ilu_factor_rec(IluChunkArgs P, const std::int64_t* __restrict__ offsets,
                                                       const std::int64_t* __restrict__ diag_pos, int bs,
                                                       double* __restrict__ F, std::int64_t nnz, std::int64_t rows,
                                                       double* __restrict__ inv, int* flag)
{
    extern __shared__ __align__(16) unsigned char lds_b[];
    const int lane = static_cast<int>(threadIdx.x);
    const int c = static_cast<int>(blockIdx.x) % bs;
    const int b = static_cast<int>(blockIdx.x) / bs;
    double* Fc = F + static_cast<std::int64_t>(c) * nnz;
    double* invc = inv + static_cast<std::int64_t>(c) * rows;
    double* rv = reinterpret_cast<double*>(lds_b);  // [kmax][64], trash [64], ones [64]
    double* ga = rv + (P.kmax + 2) * 64;            // [max_src][64]
    auto* recs = reinterpret_cast<IluRec<NU>*>(ga + P.max_src * 64);
    rv[P.kmax * 64 + lane] = 0.0;
    rv[(P.kmax + 1) * 64 + lane] = 1.0;
    double lowest = 1.0;  // smallest |pivot| divided by
    bool bad = false;
    // a chunk's header and row extents, loaded one chunk ahead
    struct { std::int64_t row, base, end, diag, src_off, rec_off; int cnt, nsrc, na, nb; } h;
    auto header = [&](int ch) {
        const std::int64_t* p = P.hdr + static_cast<std::int64_t>(ch) * 12;
        h.cnt = static_cast<int>(p[1]);
        h.src_off = p[2];
        h.nsrc = static_cast<int>(p[3]);
        h.rec_off = p[4] * 64;
        h.na = static_cast<int>(p[5]);
        h.nb = static_cast<int>(p[9]);
        h.row = p[0] + (lane < h.cnt ? lane : h.cnt - 1);
        h.base = offsets[h.row];
        h.end = offsets[h.row + 1];
        h.diag = diag_pos[h.row];
    };
    const int ch_begin = P.chunk_first[b], ch_end = P.chunk_first[b + 1];
    if (ch_begin < ch_end) header(ch_begin);
    for (int ch = ch_begin; ch < ch_end; ++ch) {
        const int cnt = h.cnt, nsrc = h.nsrc, na = h.na, nb = h.nb;
        const std::int64_t row = h.row, base = h.base, src_off = h.src_off, rec_off = h.rec_off;
        const int len = lane < cnt ? static_cast<int>(h.end - base) : 0, dslot = static_cast<int>(h.diag - base);
        const int lastq = len > 0 ? len - 1 : 0;
        copy_batched<double>(P.kmax, [&](int q) { return Fc[base + (q < lastq ? q : lastq)]; },
                             [&](int q, double v) { rv[q * 64 + lane] = q < len ? v : 0.0; });
        const auto* rec = reinterpret_cast<const IluRec<NU>*>(P.rec) + rec_off + lane;
        copy_batched<IluRec<NU>>(na + nb + 1, [&](int j) { return rec[j * 64]; },
                                 [&](int j, IluRec<NU> r) { recs[j * 64 + lane] = r; });
        for (int t0 = 0; t0 < nsrc; t0 += 8) {
            std::int32_t idx[8];
            double v[8];
#pragma unroll
            for (int u = 0; u < 8; ++u) idx[u] = P.src_a[src_off + (t0 + u < nsrc ? t0 + u : nsrc - 1) * 64 + lane];
#pragma unroll
            for (int u = 0; u < 8; ++u) v[u] = Fc[idx[u] >= 0 ? idx[u] : 0];
#pragma unroll
            for (int u = 0; u < 8; ++u)
                if (t0 + u < nsrc) ga[(t0 + u) * 64 + lane] = v[u];
        }
        if (ch + 1 < ch_end) header(ch + 1);
        __builtin_amdgcn_wave_barrier();
        for (int j = 0; j < na; ++j) {
            const IluRec<NU> r = recs[j * 64 + lane];
            ilu_rec_op<NU>(lds_b, r, lowest, [] {});
        }
        // the chunk's own pivot rows; the record after a lane's last names
        // row 63, which no later row of the chunk can depend on
        const IluRec<NU>* next = recs + na * 64 + lane;
        IluRec<NU> r = *next;
        for (int s = 0; s < cnt - 1; ++s) {
            __builtin_amdgcn_wave_barrier();
            if (static_cast<int>((r[0] >> 19) & 63u) == s) {
                next += 64;
                IluRec<NU> following;
                ilu_rec_op<NU>(lds_b, r, lowest, [&] { following = *next; });
                r = following;
            }
        }
        __builtin_amdgcn_wave_barrier();
        // store; later chunks of this wave gather these values
        for (int q = 0; q < len; ++q) Fc[base + q] = rv[q * 64 + lane];
        if (lane < cnt) {
            const double dg = rv[dslot * 64 + lane];
            bad = bad || !(__builtin_isfinite(dg) && __builtin_fabs(dg) > kTol);
            invc[row] = 1.0 / dg;
        }
        __threadfence_block();
        __builtin_amdgcn_wave_barrier();
    }
    if (bad || lowest <= kTol) atomicExch(flag, static_cast<int>(flag_zero_pivot));
}

enum class TriMode { ilu, ssor };

template<class V> __device__ inline auto vload(const V* p, std::int64_t i)
{
    if constexpr (sizeof(V) == 2) return dev::bf16_to_float(p[i]);
    else return p[i];
}

// Level-scheduled triangular apply, one workgroup per (block, component).
//  ILU : forward y_i = r_i - sum_j<i l_ij y_j; backward x_i = (y_i - sum_j>i u_ij x_j) * inv_i
//        (IluLevelPreconditioner::apply, preconditioner.hpp:320-363)
//  SSOR: forward y_i = (r_i - sum_j<i (w a_ij) y_j) / d_i; backward
//        z_i = (d_i y_i - sum_j>i (w a_ij) z_j) / d_i, then * w(2-w) if w != 1
//        (preconditioner.hpp:181-239, split_block_csr.hpp:243-309)
// With LDS the block's component vector lives in LDS; otherwise it is kept in
// `out` (strided by bs).
template<TriMode MODE, class X, class V, bool LDS>
__global__ __launch_bounds__(256) void k_tri_apply(TriArgs a, const V* __restrict__ fval, const V* __restrict__ bval,
                                                   const X* __restrict__ dval, const X* in, X* out, X scale,
                                                   const int* stop)
{
    extern __shared__ unsigned char smem_raw[];
    if (stop && *stop) return;
    const int bs = a.bs;
    const int c = blockIdx.x % bs;
    const int b = blockIdx.x / bs;
    const std::int64_t r0 = a.row0[b];
    const std::int64_t nb = a.nrows[b];
    X* lds = reinterpret_cast<X*>(smem_raw);
    auto Y = [&](std::int64_t i) -> X& {
        if constexpr (LDS) return lds[i];
        else return out[(r0 + i) * bs + c];
    };
    if constexpr (LDS) {
        for (std::int64_t i = threadIdx.x; i < nb; i += blockDim.x) lds[i] = in[(r0 + i) * bs + c];
    } else {
        if (in != out)
            for (std::int64_t i = threadIdx.x; i < nb; i += blockDim.x) out[(r0 + i) * bs + c] = in[(r0 + i) * bs + c];
    }
    __syncthreads();
    const V* fv = fval + static_cast<std::int64_t>(c) * a.fnnz;
    const V* bv = bval + static_cast<std::int64_t>(c) * a.bnnz;
    const X* dv = dval + static_cast<std::int64_t>(c) * a.rows + r0;
    for (int l = a.flev[b]; l < a.flev[b + 1] - 1; ++l) {
        const int p0 = a.flev_pos[l], p1 = a.flev_pos[l + 1];
        for (int p = p0 + threadIdx.x; p < p1; p += blockDim.x) {
            const std::int64_t gp = r0 + p;
            const std::int32_t i = a.frow[gp];
            X acc = Y(i);
            for (std::int64_t e = a.fptr[gp]; e < a.fptr[gp + 1]; ++e)
                acc = dev::dfma(-static_cast<X>(vload(fv, e)), Y(a.fcol[e]), acc);
            if constexpr (MODE == TriMode::ssor) acc = acc / dv[i];
            Y(i) = acc;
        }
        __syncthreads();
    }
    for (int l = a.blev[b]; l < a.blev[b + 1] - 1; ++l) {
        const int p0 = a.blev_pos[l], p1 = a.blev_pos[l + 1];
        for (int p = p0 + threadIdx.x; p < p1; p += blockDim.x) {
            const std::int64_t gp = r0 + p;
            const std::int32_t i = a.brow[gp];
            X acc;
            if constexpr (MODE == TriMode::ssor) acc = dv[i] * Y(i);
            else acc = Y(i);
            for (std::int64_t e = a.bptr[gp]; e < a.bptr[gp + 1]; ++e)
                acc = dev::dfma(-static_cast<X>(vload(bv, e)), Y(a.bcol[e]), acc);
            if constexpr (MODE == TriMode::ssor) acc = acc / dv[i];
            else acc = acc * dv[i];
            Y(i) = acc;
        }
        __syncthreads();
    }
    if constexpr (LDS) {
        for (std::int64_t i = threadIdx.x; i < nb; i += blockDim.x) {
            X v = lds[i];
            if constexpr (MODE == TriMode::ssor)
                if (scale != X(1)) v = v * scale;
            out[(r0 + i) * bs + c] = v;
        }
    } else if constexpr (MODE == TriMode::ssor) {
        if (scale != X(1))
            for (std::int64_t i = threadIdx.x; i < nb; i += blockDim.x) out[(r0 + i) * bs + c] *= scale;
    }
}

// ------------------------------------------------------------ chain sweeps --
// Triangular sweeps over blocks whose rows form long dependency chains
// (Hilbert-ordered blocks of 4,096 rows have about 3,500 levels): one row
// after the other, at the latency of one instruction per row.
//
// A wave walks four chains, one (block, component) per DPP row of 16 lanes,
// in chunks of 16 rows in sweep order (ascending rows forward, descending
// backward), lane l of a group owning the chunk's l-th row.  The 15 in-chunk
// steps are one instruction each: step s broadcasts lane s's finished value
// within its group and every later lane subtracts it times its coefficient
// (v_fmac with row_newbcast: 16 clocks a step; a 64-row chunk per wave with
// the value broadcast through scalar registers took 23 and an LDS read).  A
// lone wave issues one instruction in four clocks, so a second wave of the
// workgroup, on another SIMD, prepares the next chunk: it scatters the
// in-chunk coefficients and gathers the old rows, and the first wave is left
// with its K near entries, the steps and the results.
//
// The host classifies every entry by where its solution value comes from
// (build_rows16), so a chunk is branch-free but for its far entries:
//   in-chunk  the coefficient goes to the LDS tile, tile[step][lane]; zeros
//             elsewhere keep a finished row's value;
//   near      a row of the last 27 chunks, from an LDS ring of the chunks'
//             results (the ring's zero for in-chunk entries and padding);
//   far       an older row (2% of the entries of a Hilbert-ordered grid, none
//             where a block's bandwidth is below 432 rows), gathered from the
//             solution P chunks ahead, when any lane of the wave has one, and
//             handed over in LDS.
// Entries fold in slot order, then the in-chunk steps, which for sorted rows
// is the reference's order in the forward sweep; backward sweeps take their
// entries in the order the rows finish.
//
// Measured (FP64, the earlier 64-row sweep in brackets; launches that a stopped
// solver skips left out): ILU(0) apply at 2M vertices, block 3, 4,096-row
// blocks 237 (307) us; 2,048 vertices, 512-row blocks 18.1 (27.4) us; SSOR of
// 1,296 components on a 32 x 32 grid 62.0 (94.5) us.  A lone chunk takes about
// 0.25 us, 243 clocks of it the steps, which bounds the small ones.  At 2M
// vertices the two sweeps' 512 chunks would take 128 us; there the padded
// values and codes bound it, about 1 GB an apply at 4.2 TB/s.  One wave doing
// all of this took 266 us where this form had 225 (a mean with skipped
// launches), and a third wave touching the coming chunks' lines 282 us.
template<class X>
__device__ inline X chain_finish(X acc, X, X, std::integral_constant<int, 0>)  // ILU forward: unit diagonal
{
    return acc;
}
template<class X>
__device__ inline X chain_finish(X acc, X d, X, std::integral_constant<int, 1>)  // ILU backward: inverse diagonal
{
    return acc * d;
}
// SSOR: acc / d from the reciprocal and one fma-based correction (Markstein:
// with rinv = RN(1/d) and q = RN(acc rinv), the residual acc - q d is exact
// and RN(q + residual rinv) is the correctly rounded quotient), which keeps
// the division's long latency off the step-to-step dependency chain.
template<class X>
__device__ inline X chain_finish(X acc, X d, X rinv, std::integral_constant<int, 2>)
{
    const X q = acc * rinv;
    const X r = dev::dfma(-q, d, acc);
    return dev::dfma(r, rinv, q);
}

template<TriMode MODE, bool FWD>
using FinishKind = std::integral_constant<int, MODE == TriMode::ssor ? 2 : (FWD ? 0 : 1)>;

// The 15 in-chunk steps: at step s every lane subtracts its coefficient times
// the finished value of its group's lane s (see chain_finish), rounded once.
// A DPP operand may not have been written by the two vector instructions
// before, hence the wait states; one block, because the compiler adds another
// to every inline statement it puts between.  (KIND as FinishKind.)
#define OWTK_STEP0(T, S) "s_nop 1\n\tv_fmac_" T "_dpp %0, -%0, %[c" #S "] row_newbcast:" #S " row_mask:0xf bank_mask:0xf\n\t"
#define OWTK_STEP1(T, S)                                                                                              \
    "v_mul_" T " %[t], %0, %[d]\n\ts_nop 1\n\tv_fmac_" T "_dpp %0, -%[t], %[c" #S "] row_newbcast:" #S             \
    " row_mask:0xf bank_mask:0xf\n\t"
#define OWTK_STEP2(T, S)                                                                                              \
    "v_mul_" T " %[t], %0, %[r]\n\tv_fma_" T " %[u], -%[t], %[d], %0\n\tv_fma_" T " %[t], %[u], %[r], %[t]\n\t"   \
    "s_nop 1\n\tv_fmac_" T "_dpp %0, -%[t], %[c" #S "] row_newbcast:" #S " row_mask:0xf bank_mask:0xf\n\t"
#define OWTK_STEPS(M, T)                                                                                              \
    M(T, 0) M(T, 1) M(T, 2) M(T, 3) M(T, 4) M(T, 5) M(T, 6) M(T, 7) M(T, 8) M(T, 9) M(T, 10) M(T, 11) M(T, 12) M(T, 13) \
        M(T, 14)
#define OWTK_COEFS                                                                                                    \
    [c0] "v"(c[0]), [c1] "v"(c[1]), [c2] "v"(c[2]), [c3] "v"(c[3]), [c4] "v"(c[4]), [c5] "v"(c[5]), [c6] "v"(c[6]),    \
        [c7] "v"(c[7]), [c8] "v"(c[8]), [c9] "v"(c[9]), [c10] "v"(c[10]), [c11] "v"(c[11]), [c12] "v"(c[12]),         \
        [c13] "v"(c[13]), [c14] "v"(c[14])
#define OWTK_CHAIN_STEPS(X, T)                                                                                        \
    template<int KIND>                                                                                                \
    __device__ inline void chain_steps(X& acc, const X (&c)[15], X d, X rinv)                                         \
    {                                                                                                                 \
        X t, u;                                                                                                       \
        if constexpr (KIND == 0) __asm__(OWTK_STEPS(OWTK_STEP0, T) : "+v"(acc) : OWTK_COEFS);                         \
        else if constexpr (KIND == 1)                                                                                 \
            __asm__(OWTK_STEPS(OWTK_STEP1, T) : "+v"(acc), [t] "=&v"(t) : OWTK_COEFS, [d] "v"(d));                    \
        else                                                                                                          \
            __asm__(OWTK_STEPS(OWTK_STEP2, T)                                                                         \
                    : "+v"(acc), [t] "=&v"(t), [u] "=&v"(u)                                                           \
                    : OWTK_COEFS, [d] "v"(d), [r] "v"(rinv));                                                         \
    }
OWTK_CHAIN_STEPS(double, "f64")
OWTK_CHAIN_STEPS(float, "f32")
#undef OWTK_STEP0
#undef OWTK_STEP1
#undef OWTK_STEP2
#undef OWTK_STEPS
#undef OWTK_COEFS
#undef OWTK_CHAIN_STEPS

// LDS of a workgroup, bytes.  Elements sit 8 bytes apart in either precision,
// so the host's codes serve both.  Per group: 28 ring entries of 16 results,
// the zero entry, then the far values [parity][K][16]; behind the groups, for
// even and odd chunks, the tile [15 steps and a spare row][64 lanes] and the
// right-hand side, diagonal and reciprocal [3][64 lanes].
constexpr int kRing16 = 28, kRingZero = kRing16 * 128, kFar16 = 4096;
constexpr int kGroup16 = 8192 + 128;  // the groups' entries start on different LDS banks
constexpr int kTile16 = 4 * kGroup16, kTileSpare = kTile16 + 15 * 512, kTileBytes = 16 * 512;
constexpr int kRow16 = kTile16 + 2 * kTileBytes, kRowBytes = 3 * 512, kLds16 = kRow16 + 2 * kRowBytes;
constexpr int chunks_ahead(int k) { return k <= 8 ? 4 : 2; }  // P, even
constexpr int kPadChunks16 = 16;  // idle chunks behind the last block: loads run ahead of the sweep

struct Rows16Args {
    const std::int32_t* row0;
    const std::int32_t* nrows;
    // per sweep, [chunk * 16 + lane][K]: LDS address of an entry's value (near,
    // within the group) and of its coefficient's tile entry (less the lane's
    // 8 bytes), and the block-local far row (-1 none)
    const std::uint16_t *fnear, *bnear, *ftile, *btile;
    const std::int16_t *ffar, *bfar;
    std::int64_t slots;         // values per component and sweep: chunks * K * 16
    std::int64_t rows;
    int chains, block_chunks;   // blocks * bs; chunks each block has room for
    int bs;
};

template<class V> struct alignas(2 * sizeof(V)) Pair { V v[2]; };
// a row's K 16-bit codes, two to a word (the low half first)
template<int K> struct Codes { std::uint32_t w[K / 2]; };
template<int K> __device__ inline unsigned int code_of(const Codes<K>& c, int k)
{
    return k & 1 ? c.w[k / 2] >> 16 : c.w[k / 2] & 0xffffU;
}

// What the two waves of a workgroup share in a sweep; pointers are the lane's.
template<class X, class V>
struct Rows16Sweep {
    const std::uint16_t* __restrict__ near;
    const std::uint16_t* __restrict__ tile;
    const std::int16_t* __restrict__ far;
    const V* __restrict__ val;
    const X* __restrict__ dv;  // diagonal of the chain's row 0
    const X* src;              // right-hand side
    X* y;                      // solution
    int first, last;           // byte offsets of the chain's first and last row in src and y
    int row_bytes;
    unsigned char* lds;
    int rows, stored;          // rows of the chain; rows to store (0: a group past the last chain)
    int chunks;                // of the wave's longest chain, rounded up to P
    int full;                  // chunks whose 64 rows are all stored
    int lane;
    __device__ X& at(unsigned int byte) const { return *reinterpret_cast<X*>(lds + byte); }
};

// One barrier a chunk.  LDS is handed over, and the results in memory that the
// preparing wave gathers many chunks later.  A workgroup's waves share one L1,
// which takes their accesses in order, so these fences wait for LDS alone and
// the loads of later chunks stay in flight (the code is the same as with
// fences for LDS only).
__device__ inline void chunk_barrier()
{
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "workgroup");
    __builtin_amdgcn_s_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "workgroup");
}

// The preparing wave: during chunk q it writes the tile, right-hand side and
// diagonal of chunk q + 2 (the solving wave reads chunk q + 1's then) and the
// far values of chunk q + 1.  Codes, values and rows of a chunk load P chunks
// ahead, the far rows' numbers 2P.  The rows of chunk q + P + 1 are gathered
// during chunk q, and a far row of it was stored in chunk q + P + 1 - kRing16
// or before: kFarBarriers barriers lie between, and the storing wave has
// waited for loads that it issued after that store (those of the chunk after
// it, used P + 1 chunks later).
template<int K> constexpr int kFarBarriers = kRing16 - chunks_ahead(K) - 1;
template<TriMode MODE, bool FWD, class X, class V, int K>
__device__ __attribute__((always_inline)) inline void rows16_prepare(const Rows16Sweep<X, V>& s)
{
    constexpr int P = chunks_ahead(K);
    constexpr bool kDiag = MODE == TriMode::ssor || !FWD;
    const int l = s.lane & 15;
    const unsigned int group = static_cast<unsigned int>(s.lane >> 4) * kGroup16;
    const unsigned int lane8 = static_cast<unsigned int>(s.lane) * 8;
    const auto* pc = reinterpret_cast<const Codes<K>*>(s.tile) + l;
    const auto* pf = reinterpret_cast<const Codes<K>*>(s.far) + l;
    const auto* pv = reinterpret_cast<const Pair<V>*>(s.val) + l;
    Codes<K> cc[P], fr[P];
    X cv[P][K], xo[P][K], rr[P], dd[P];
    unsigned int used[2][K];    // tile entries of the last chunk of each parity
    unsigned int far_mask = 0;  // bit t: stage t has far entries (wave-uniform)
    int p = l;                  // position and byte offset of the next chunk's row
    int off = FWD ? s.first + l * s.row_bytes : s.last - l * s.row_bytes;
#pragma unroll
    for (int k = 0; k < K; ++k) used[0][k] = used[1][k] = kTileSpare + lane8;
    auto load_far = [&](int t) {
        fr[t] = *pf;
        pf += 16;
    };
    // the next chunk into stage t, its far rows' numbers already there
    auto load_chunk = [&](int t) {
        std::uint32_t none = 0x80008000U;
#pragma unroll
        for (int k = 0; k < K / 2; ++k) none &= fr[t].w[k];
        far_mask &= ~(1U << t);
        if (__builtin_amdgcn_ballot_w64(none != 0x80008000U) != 0) {
            far_mask |= 1U << t;
#pragma unroll
            for (int k = 0; k < K; ++k) {
                const int code = static_cast<std::int16_t>(code_of<K>(fr[t], k));
                const unsigned int at = static_cast<unsigned int>(s.first + (code > 0 ? code : 0) * s.row_bytes);
                xo[t][k] = *reinterpret_cast<const X*>(reinterpret_cast<const char*>(s.y) + at);
            }
        }
        cc[t] = *pc;
        pc += 16;
#pragma unroll
        for (int j = 0; j < K / 2; ++j) {
            const Pair<V> u = pv[j * 16];
            cv[t][2 * j] = static_cast<X>(vload(u.v, 0));
            cv[t][2 * j + 1] = static_cast<X>(vload(u.v, 1));
        }
        pv += (K / 2) * 16;
        const int at = FWD ? min(off, s.last) : max(off, s.first);
        off = FWD ? off + 16 * s.row_bytes : off - 16 * s.row_bytes;
        rr[t] = *reinterpret_cast<const X*>(reinterpret_cast<const char*>(s.src) + static_cast<unsigned int>(at));
        dd[t] = X(1);
        if constexpr (kDiag) {
            const int q = min(p, s.rows - 1);
            dd[t] = s.dv[FWD ? q : s.rows - 1 - q];
            p += 16;
        }
    };
    // the far values of stage t's chunk; the solving wave reads them at the
    // start of that chunk, so they go out one chunk later than the tile
    auto hand_far = [&](int t) {
        if (far_mask >> t & 1U) {
#pragma unroll
            for (int k = 0; k < K; ++k) s.at(group + kFar16 + ((t & 1) * K + k) * 128 + l * 8) = xo[t][k];
        }
    };
    // the chunk of stage t into the LDS of its parity
    auto build = [&](int t) {
        const int par = t & 1;
#pragma unroll
        for (int k = 0; k < K; ++k) s.at(used[par][k]) = X(0);
#pragma unroll
        for (int k = 0; k < K; ++k) {
            used[par][k] = code_of<K>(cc[t], k) + (lane8 + par * kTileBytes);
            s.at(used[par][k]) = cv[t][k];
        }
        X r0 = rr[t];
        if constexpr (MODE == TriMode::ssor && !FWD) r0 = dd[t] * r0;
        s.at(kRow16 + par * kRowBytes + lane8) = r0;
        if constexpr (kDiag) s.at(kRow16 + par * kRowBytes + 512 + lane8) = dd[t];
        if constexpr (MODE == TriMode::ssor) s.at(kRow16 + par * kRowBytes + 1024 + lane8) = X(1) / dd[t];
    };
#pragma unroll
    for (int t = 0; t < P; ++t) load_far(t);
#pragma unroll
    for (int t = 0; t < P; ++t) {
        load_chunk(t);
        load_far(t);
    }
    build(0);
    __syncthreads();
    load_chunk(0);
    load_far(0);
    build(1);
    __syncthreads();  // the solving wave has read chunk 0's tile
    for (int q0 = 0; q0 < s.chunks; q0 += P) {
#pragma unroll
        for (int t = 0; t < P; ++t) {
            // stage t + 1 (chunk q0 + t + 1) is built: hand its far values over
            // and refill it, build chunk q0 + t + 2
            hand_far((t + 1) % P);
            load_chunk((t + 1) % P);
            load_far((t + 1) % P);
            build((t + 2) % P);
            chunk_barrier();
        }
    }
    // an empty tile for the next sweep
#pragma unroll
    for (int k = 0; k < K; ++k) {
        s.at(used[0][k]) = X(0);
        s.at(used[1][k]) = X(0);
    }
    __syncthreads();
}

// The solving wave.  It reads the next chunk's coefficients, right-hand side
// and diagonal during a chunk's steps, so a chunk starts with its near reads.
template<TriMode MODE, bool FWD, class X, class V, int K>
__device__ __attribute__((always_inline)) inline void rows16_solve(const Rows16Sweep<X, V>& s)
{
    constexpr int P = chunks_ahead(K);
    constexpr bool kDiag = MODE == TriMode::ssor || !FWD;
    const int l = s.lane & 15;
    const unsigned int group = static_cast<unsigned int>(s.lane >> 4) * kGroup16;
    const unsigned int lane8 = static_cast<unsigned int>(s.lane) * 8;
    const auto* pc = reinterpret_cast<const Codes<K>*>(s.near) + l;
    const auto* pv = reinterpret_cast<const Pair<V>*>(s.val) + l;
    Codes<K> cc[P];
    X cv[P][K];
    auto load_chunk = [&](int t) {
        cc[t] = *pc;
        pc += 16;
#pragma unroll
        for (int j = 0; j < K / 2; ++j) {
            const Pair<V> u = pv[j * 16];
            cv[t][2 * j] = static_cast<X>(vload(u.v, 0));
            cv[t][2 * j + 1] = static_cast<X>(vload(u.v, 1));
        }
        pv += (K / 2) * 16;
    };
    X coef[2][15], rhs[2], dd[2], ri[2];
    auto read_tile = [&](int par) {
        rhs[par] = s.at(kRow16 + par * kRowBytes + lane8);
        dd[par] = ri[par] = X(1);
        if constexpr (kDiag) dd[par] = s.at(kRow16 + par * kRowBytes + 512 + lane8);
        if constexpr (MODE == TriMode::ssor) ri[par] = s.at(kRow16 + par * kRowBytes + 1024 + lane8);
#pragma unroll
        for (int st = 0; st < 15; ++st) coef[par][st] = s.at(kTile16 + par * kTileBytes + st * 512 + lane8);
    };
#pragma unroll
    for (int t = 0; t < P; ++t) load_chunk(t);
    __syncthreads();
    read_tile(0);
    __syncthreads();
    const int step_bytes = FWD ? 16 * s.row_bytes : -16 * s.row_bytes;
    int off = FWD ? s.first + l * s.row_bytes : s.last - l * s.row_bytes;
    unsigned int ring = group + l * 8;  // ring entry of chunk q0, this lane
    int ring_q = 0;
    unsigned int na[K];  // near addresses of the coming chunk
#pragma unroll
    for (int k = 0; k < K; ++k) na[k] = code_of<K>(cc[0], k) + group;
    // MASKED: some row of the chunks may lie past its chain's end
    auto chunks = [&](int q0, auto masked) {
#pragma unroll
        for (int t = 0; t < P; ++t) {
            const int par = t & 1;
            // the ring's newest results first; chunk q + 1's tile (built
            // during chunk q - 1), chunk q + P's loads and chunk q + 1's near
            // addresses issue while they are on their way
            X xn[K], mine[K];
#pragma unroll
            for (int k = 0; k < K; ++k) xn[k] = s.at(na[k]);
            X acc = rhs[par];
            const X d = dd[par], rinv = ri[par];
            read_tile(1 - par);
#pragma unroll
            for (int k = 0; k < K; ++k) mine[k] = cv[t][k];
#pragma unroll
            for (int k = 0; k < K; ++k) na[k] = code_of<K>(cc[(t + 1) % P], k) + group;
            load_chunk(t);
            __builtin_amdgcn_sched_barrier(0);
#pragma unroll
            for (int k = 0; k < K; ++k) acc = dev::dfma(-mine[k], xn[k], acc);
            chain_steps<FinishKind<MODE, FWD>::value>(acc, coef[par], d, rinv);
            const X fin = chain_finish(acc, d, rinv, FinishKind<MODE, FWD>{});
            s.at(ring + t * 128) = fin;
            X* const out = reinterpret_cast<X*>(reinterpret_cast<char*>(s.y) + static_cast<unsigned int>(off));
            if constexpr (decltype(masked)::value) {
                if ((q0 + t) * 16 + l < s.stored) *out = fin;
            } else {
                *out = fin;
            }
            off += step_bytes;
            chunk_barrier();
        }
        ring_q = ring_q == kRing16 - P ? 0 : ring_q + P;
        ring = group + l * 8 + static_cast<unsigned int>(ring_q) * 128;
    };
    int q0 = 0;
    for (; q0 + P <= s.full; q0 += P) chunks(q0, std::false_type{});
    for (; q0 < s.chunks; q0 += P) chunks(q0, std::true_type{});
    __syncthreads();
}

template<TriMode MODE, class X, class V, int K>
__global__ __launch_bounds__(128) void k_tri_rows16(Rows16Args a, const V* __restrict__ fval,
                                                    const V* __restrict__ bval, const X* __restrict__ dval,
                                                    const X* in, X* out, X scale, const int* stop)
{
    constexpr int P = chunks_ahead(K);
    static_assert(2 * K * 128 <= kGroup16 - kFar16 && kTile16 + 16 * 512 <= 65536 && P % 2 == 0 && kRing16 % P == 0 && 3 * P + 2 <= kPadChunks16);
    static_assert(kRingZero + 128 <= kFar16);
    static_assert(kFarBarriers<K> >= P + 2, "a far row's store is waited for before its gather");
    static_assert(K <= kChainEntries && (2 * P + 2) * 16 <= kChainOverrun && kChainRows <= 32767);
    __shared__ __attribute__((aligned(16))) unsigned char lds[kLds16];
    if (stop && *stop) return;
    const int lane = static_cast<int>(threadIdx.x & 63);
    const bool solver = __builtin_amdgcn_readfirstlane(static_cast<int>(threadIdx.x >> 6)) == 0;
    for (int t = static_cast<int>(threadIdx.x); t < kLds16 / 8; t += 128) *reinterpret_cast<X*>(lds + 8 * t) = X(0);
    __syncthreads();
    // the component chains of a block side by side: they read the same codes
    const int first = static_cast<int>(kern::xcd_block(blockIdx.x, gridDim.x)) * 4;
    const int mine = first + (lane >> 4);
    const int chain = mine < a.chains ? mine : a.chains - 1;
    const int b = chain / a.bs, c = chain - b * a.bs;
    const int rows = a.nrows[b];
    const int r0 = a.row0[b], r0_first = a.row0[first / a.bs];
    int nch = (rows + 15) >> 4;
    nch = max(max(__builtin_amdgcn_readlane(nch, 0), __builtin_amdgcn_readlane(nch, 16)),
              max(__builtin_amdgcn_readlane(nch, 32), __builtin_amdgcn_readlane(nch, 48)));
    const std::int64_t start = static_cast<std::int64_t>(__builtin_amdgcn_readfirstlane(r0_first)) * a.bs;
    Rows16Sweep<X, V> s;
    s.row_bytes = a.bs * static_cast<int>(sizeof(X));
    s.first = (r0 - r0_first) * s.row_bytes + c * static_cast<int>(sizeof(X));
    s.last = s.first + (rows - 1) * s.row_bytes;
    s.lds = lds;
    s.rows = rows;
    s.stored = mine < a.chains ? rows : 0;
    s.chunks = (nch + P - 1) / P * P;
    s.full = s.stored >> 4;
    s.full = min(min(__builtin_amdgcn_readlane(s.full, 0), __builtin_amdgcn_readlane(s.full, 16)),
                 min(__builtin_amdgcn_readlane(s.full, 32), __builtin_amdgcn_readlane(s.full, 48)));
    s.lane = lane;
    s.dv = dval + static_cast<std::int64_t>(c) * a.rows + r0;
    s.y = out + start;
    const std::int64_t g0 = static_cast<std::int64_t>(b) * a.block_chunks * (K * 16);
    const std::int64_t v0 = static_cast<std::int64_t>(c) * a.slots + g0;
    s.src = in + start;
    s.near = a.fnear + g0;
    s.tile = a.ftile + g0;
    s.far = a.ffar + g0;
    s.val = fval + v0;
    if (solver) rows16_solve<MODE, true, X, V, K>(s);
    else rows16_prepare<MODE, true, X, V, K>(s);
    s.src = s.y;
    s.near = a.bnear + g0;
    s.tile = a.btile + g0;
    s.far = a.bfar + g0;
    s.val = bval + v0;
    if (solver) rows16_solve<MODE, false, X, V, K>(s);
    else rows16_prepare<MODE, false, X, V, K>(s);
    if (MODE == TriMode::ssor && scale != X(1) && solver) {
        X* o = reinterpret_cast<X*>(reinterpret_cast<char*>(s.y) + s.first);
        for (int i = lane & 15; i < s.stored; i += 16) o[static_cast<std::int64_t>(i) * a.bs] *= scale;
    }
}

// Sweep values from the chain-order values: dst[c][slot] = src[c][map[slot]] (0 for padding)
template<class V>
__global__ __launch_bounds__(256) void k_ell_gather(V* __restrict__ dst, const V* __restrict__ src,
                                                    const std::int64_t* __restrict__ map, std::int64_t slots,
                                                    std::int64_t nnz, int bs)
{
    const std::int64_t total = slots * bs;
    const std::int64_t step = static_cast<std::int64_t>(gridDim.x) * blockDim.x;
    for (std::int64_t t = static_cast<std::int64_t>(blockIdx.x) * blockDim.x + threadIdx.x; t < total; t += step) {
        const std::int64_t c = t / slots;
        const std::int64_t sl = t - c * slots;
        const std::int64_t e = map[sl];
        dst[t] = e >= 0 ? src[c * nnz + e] : V(0);
    }
}

// ---------------------------------------------------------------- symbolic --

// Encoded gather source of matrix value (row, CSR entry e): >= 0 index of
// component 0 in the value array; <= -2: diagonal array.
std::int64_t entry_source(owtk_matrix m, std::int64_t e) { return m->value_index(m->s.slot_of_entry[e], 0); }
std::int64_t diag_source(owtk_matrix m, std::int64_t row) { return -2 - m->diag_index(row, 0); }
std::int64_t comp_stride(owtk_matrix m) { return m->s.layout == Layout::sell ? 64 : 1; }

// Block-restricted local rows in the original CSR order (ghost columns and
// cross-block columns dropped), with each row's diagonal source.
struct LocalRows {
    std::vector<std::int64_t> off;
    std::vector<std::int64_t> col;
    std::vector<std::int64_t> src;
    std::vector<std::int64_t> diag_src; // -1 when the row has no diagonal
};

LocalRows local_rows(owtk_matrix m, std::int64_t block_nodes)
{
    LocalRows L;
    const std::int64_t n = m->owned;
    L.off.assign(n + 1, 0);
    L.diag_src.assign(n, -1);
    L.col.reserve(m->h_columns.size() + (m->has_diag_array() ? n : 0));
    L.src.reserve(L.col.capacity());
    for (std::int64_t row = 0; row < n; ++row) {
        const std::int64_t blk = block_nodes > 0 ? row / block_nodes : 0;
        if (m->has_diag_array()) L.diag_src[row] = diag_source(m, row);
        for (std::int32_t e = m->h_offsets[row]; e < m->h_offsets[row + 1]; ++e) {
            const std::int64_t c = m->h_columns[e];
            if (c >= n) continue;
            if (block_nodes > 0 && c / block_nodes != blk) continue;
            if (!m->has_diag_array() && c == row && L.diag_src[row] == -1) L.diag_src[row] = entry_source(m, e);
            L.col.push_back(c);
            L.src.push_back(entry_source(m, e));
        }
        if (m->has_diag_array()) {
            // the split diagonal is a separate array; keep it out of the edge list
        }
        L.off[row + 1] = static_cast<std::int64_t>(L.col.size());
    }
    return L;
}

template<class T>
void upload(DeviceArray<T>& d, const std::vector<T>& h)
{
    d.allocate(std::max<std::size_t>(h.size(), 1));
    if (!h.empty()) OWTK_HIP(hipMemcpy(d.get(), h.data(), h.size() * sizeof(T), hipMemcpyHostToDevice));
}

// Build the level schedule of one triangular pair.  lower(i)/upper(i) list
// the block-local entries of row i (global index space) in apply order.
struct TriHost {
    // per row: forward entries (col, src) and backward entries
    std::vector<std::int64_t> f_off, f_col, f_src, b_off, b_col, b_src;
};

// Codes and value maps of the chain sweeps (k_tri_rows16) from the chain
// layout: entry k of the row at position p (chunk q = p / 16, lane l) goes to
// value slot ((q * K / 2 + k / 2) * 16 + l) * 2 + k % 2 of its block.
void build_rows16(TriSchedule& tri, const std::vector<std::int64_t>& fptr, const std::vector<std::int32_t>& fcol,
                  const std::vector<std::int64_t>& bptr, const std::vector<std::int32_t>& bcol)
{
    if (!tri.chain) return;
    const std::int64_t n = tri.rows;
    std::int64_t need = 1;
    for (std::int64_t i = 0; i < n; ++i) need = std::max({need, fptr[i + 1] - fptr[i], bptr[i + 1] - bptr[i]});
    const int K = need <= 4 ? 4 : need <= 6 ? 6 : need <= 8 ? 8 : 16;
    // every block has room for the longest one's chunks: a wave's four chains
    // run as long as its longest block
    const std::int64_t per = (tri.max_block_rows + 15) / 16;
    const std::int64_t chunks = tri.blocks * per + kPadChunks16;
    for (int dir = 0; dir < 2; ++dir) {
        const auto& ptr = dir == 0 ? fptr : bptr;
        const auto& col = dir == 0 ? fcol : bcol;
        std::vector<std::uint16_t> near(static_cast<std::size_t>(chunks * K * 16), kRingZero), tile(near.size(), kTileSpare);
        std::vector<std::int16_t> far(near.size(), -1);
        std::vector<std::int64_t> map(near.size(), -1);
        for (std::int64_t b = 0; b < tri.blocks; ++b) {
            const std::int64_t r0 = tri.h_row0[b], nb = tri.h_nrows[b];
            for (std::int64_t p = 0; p < nb; ++p) {
                const std::int64_t q = p / 16, l = p % 16, g = b * per + q;
                for (std::int64_t e = ptr[r0 + p]; e < ptr[r0 + p + 1]; ++e) {
                    const int k = static_cast<int>(e - ptr[r0 + p]);
                    const std::size_t slot = static_cast<std::size_t>(((g * (K / 2) + k / 2) * 16 + l) * 2 + k % 2);
                    const std::int64_t pc = dir == 0 ? col[e] : nb - 1 - col[e];  // the column's position in the sweep
                    const std::int64_t qc = pc / 16;
                    const std::size_t at = static_cast<std::size_t>((g * 16 + l) * K + k);
                    if (pc >= p) throw std::logic_error("chain layout: entry on a later row");
                    if (qc == q) {
                        tile[at] = static_cast<std::uint16_t>(kTile16 + (pc % 16) * 512);
                    } else if (q - qc < kRing16) {
                        near[at] = static_cast<std::uint16_t>((qc % kRing16) * 128 + (pc % 16) * 8);
                    } else {
                        near[at] = static_cast<std::uint16_t>(kFar16 + ((q % 2) * K + k) * 128 + l * 8);
                        far[at] = static_cast<std::int16_t>(col[e]);
                    }
                    map[slot] = e;
                }
            }
        }
        upload(dir == 0 ? tri.fnear : tri.bnear, near);
        upload(dir == 0 ? tri.ftile : tri.btile, tile);
        upload(dir == 0 ? tri.ffar : tri.bfar, far);
        upload(dir == 0 ? tri.fmap : tri.bmap, map);
    }
    tri.k16 = K;
    tri.block_chunks = static_cast<int>(per);
    tri.slots16 = chunks * K * 16;
}

// Whether a row names a column more than once in one direction.  The chains'
// tile has one place for a (row, column of the chunk), so such rows take the
// level sets, which add the products up.
bool repeated_columns(const TriHost& t, std::int64_t n)
{
    for (std::int64_t i = 0; i < n; ++i)
        for (const auto* d : {&t.f_off, &t.b_off}) {
            const auto& col = d == &t.f_off ? t.f_col : t.b_col;
            for (std::int64_t e = (*d)[i]; e < (*d)[i + 1]; ++e)
                for (std::int64_t k = (*d)[i]; k < e; ++k)
                    if (col[k] == col[e]) return true;
        }
    return false;
}

void build_schedule(owtk_precond pc, const TriHost& t)
{
    auto& tri = pc->tri;
    const std::int64_t n = pc->m->owned;
    const std::int64_t bn = pc->block_nodes > 0 ? pc->block_nodes : n;
    tri.rows = n;
    tri.bs = pc->m->bs;
    tri.blocks = (n + bn - 1) / bn;
    tri.h_row0.assign(tri.blocks, 0);
    tri.h_nrows.assign(tri.blocks, 0);
    tri.h_flev.assign(tri.blocks + 1, 0);
    tri.h_blev.assign(tri.blocks + 1, 0);
    tri.h_flev_pos.clear();
    tri.h_blev_pos.clear();
    tri.max_block_rows = tri.max_flevels = tri.max_blevels = tri.max_level_width = 0;
    // pass 1: levels (forward from the top, backward from the bottom), depths, widths
    std::vector<std::int32_t> flevel(n, 0), blevel(n, 0);
    std::vector<int> fdepth(tri.blocks, 0), bdepth(tri.blocks, 0);
    int emax = 0;
    for (std::int64_t i = 0; i < n; ++i)
        emax = std::max<int>(emax, static_cast<int>(std::max(t.f_off[i + 1] - t.f_off[i], t.b_off[i + 1] - t.b_off[i])));
    std::int64_t depth_sum = 0;
    for (std::int64_t b = 0; b < tri.blocks; ++b) {
        const std::int64_t r0 = b * bn;
        const std::int64_t nb = std::min(bn, n - r0);
        tri.h_row0[b] = static_cast<std::int32_t>(r0);
        tri.h_nrows[b] = static_cast<std::int32_t>(nb);
        tri.max_block_rows = std::max(tri.max_block_rows, nb);
        for (std::int64_t i = r0; i < r0 + nb; ++i) {
            int lv = 0;
            for (std::int64_t e = t.f_off[i]; e < t.f_off[i + 1]; ++e) lv = std::max(lv, flevel[t.f_col[e]] + 1);
            flevel[i] = lv;
            fdepth[b] = std::max(fdepth[b], lv + 1);
        }
        for (std::int64_t i = r0 + nb; i-- > r0;) {
            int lv = 0;
            for (std::int64_t e = t.b_off[i]; e < t.b_off[i + 1]; ++e) lv = std::max(lv, blevel[t.b_col[e]] + 1);
            blevel[i] = lv;
            bdepth[b] = std::max(bdepth[b], lv + 1);
        }
        tri.max_flevels = std::max<std::int64_t>(tri.max_flevels, fdepth[b]);
        tri.max_blevels = std::max<std::int64_t>(tri.max_blevels, bdepth[b]);
        depth_sum += std::max(fdepth[b], bdepth[b]);
    }
    // Chain sweeps win when levels are narrow: a level then costs a barrier
    // (about 1.1 us) for a handful of rows, a chain 0.25 us per 16 rows.  The
    // line at an average width of 16 rows is on the safe side of the crossing:
    // RCM-ordered 512 x 512 grid, block 3, level sets / chains in us: 917 / 127
    // at width 8 (4,096-row blocks), 1,233 / 491 at width 30 (16,384); one
    // 8,192-row block in random order, width 585: 63 / 295.
    tri.emax = emax;
    const bool chain_ok = emax <= kChainEntries && tri.max_block_rows <= kChainRows;
    if (pc->schedule == 2 && !chain_ok)
        throw unsupported_error("chain sweeps need at most 16 entries per row and blocks of at most 16384 rows");
    tri.chain = (pc->schedule == 2 || (pc->schedule == 0 && chain_ok && depth_sum * 16 > n))
        && chain_offsets_fit(tri.blocks, tri.max_block_rows, tri.bs) && !repeated_columns(t, n);
    // pass 2: level lists and apply arrays
    std::vector<std::int32_t> frow(n), brow(n), frow_lvl(n);
    std::vector<std::int64_t> fptr(n + 1, 0), bptr(n + 1, 0);
    std::vector<std::int32_t> fcol, bcol;
    std::vector<std::int64_t> fsrc, bsrc;
    fcol.reserve(t.f_col.size());
    bcol.reserve(t.b_col.size());
    for (std::int64_t b = 0; b < tri.blocks; ++b) {
        const std::int64_t r0 = tri.h_row0[b];
        const std::int64_t nb = tri.h_nrows[b];
        for (int dir = 0; dir < 2; ++dir) {
            const auto& off = dir == 0 ? t.f_off : t.b_off;
            const auto& col = dir == 0 ? t.f_col : t.b_col;
            const auto& src = dir == 0 ? t.f_src : t.b_src;
            const auto& level = dir == 0 ? flevel : blevel;
            const int depth = dir == 0 ? fdepth[b] : bdepth[b];
            // counting sort by level, stable in row order (forward) / reverse row order (backward)
            std::vector<std::int64_t> count(depth + 1, 0);
            for (std::int64_t i = r0; i < r0 + nb; ++i) ++count[level[i] + 1];
            for (int l = 0; l < depth; ++l) count[l + 1] += count[l];
            auto& lev_pos = dir == 0 ? tri.h_flev_pos : tri.h_blev_pos;
            auto& lev = dir == 0 ? tri.h_flev : tri.h_blev;
            lev[b] = static_cast<std::int32_t>(lev_pos.size());
            for (int l = 0; l <= depth; ++l) lev_pos.push_back(static_cast<std::int32_t>(count[l]));
            for (int l = 0; l < depth; ++l) tri.max_level_width = std::max(tri.max_level_width, count[l + 1] - count[l]);
            lev[b + 1] = static_cast<std::int32_t>(lev_pos.size());
            std::vector<std::int64_t> next(count.begin(), count.end() - 1);
            std::vector<std::int32_t> lvl_map(nb);
            auto place = [&](std::int64_t i) { lvl_map[next[level[i]]++] = static_cast<std::int32_t>(i - r0); };
            if (dir == 0)
                for (std::int64_t i = r0; i < r0 + nb; ++i) place(i);
            else
                for (std::int64_t i = r0 + nb; i-- > r0;) place(i);
            if (dir == 0) std::copy(lvl_map.begin(), lvl_map.end(), frow_lvl.begin() + r0);
            auto& rowmap = dir == 0 ? frow : brow;
            for (std::int64_t p = 0; p < nb; ++p) {
                if (tri.chain) rowmap[r0 + p] = static_cast<std::int32_t>(dir == 0 ? p : nb - 1 - p);
                else rowmap[r0 + p] = lvl_map[p];
            }
            auto& ptr = dir == 0 ? fptr : bptr;
            auto& ocol = dir == 0 ? fcol : bcol;
            auto& osrc = dir == 0 ? fsrc : bsrc;
            std::vector<std::pair<int, std::int64_t>> inside;
            for (std::int64_t p = 0; p < nb; ++p) {
                const std::int64_t i = r0 + rowmap[r0 + p];
                if (!tri.chain) {
                    for (std::int64_t e = off[i]; e < off[i + 1]; ++e) {
                        ocol.push_back(static_cast<std::int32_t>(col[e] - r0));
                        osrc.push_back(src[e]);
                    }
                } else {
                    // chain layout: entries from rows before this chunk, then the
                    // in-chunk entries by the step that finishes their row
                    const std::int64_t cs = (p / 64) * 64;
                    inside.clear();
                    for (std::int64_t e = off[i]; e < off[i + 1]; ++e) {
                        const std::int64_t c = col[e] - r0;
                        const bool in_chunk = dir == 0 ? c >= cs : c <= nb - 1 - cs;
                        if (in_chunk) {
                            inside.push_back({static_cast<int>(dir == 0 ? c - cs : nb - 1 - cs - c), e});
                        } else {
                            ocol.push_back(static_cast<std::int32_t>(c));
                            osrc.push_back(src[e]);
                        }
                    }
                    std::sort(inside.begin(), inside.end());
                    for (const auto& [step, e] : inside) {
                        ocol.push_back(static_cast<std::int32_t>(col[e] - r0));
                        osrc.push_back(src[e]);
                    }
                }
                ptr[r0 + p + 1] = static_cast<std::int64_t>(ocol.size());
            }
        }
    }
    tri.fnnz = static_cast<std::int64_t>(fcol.size());
    tri.bnnz = static_cast<std::int64_t>(bcol.size());
    build_rows16(tri, fptr, fcol, bptr, bcol);
    upload(tri.row0, tri.h_row0);
    upload(tri.nrows, tri.h_nrows);
    upload(tri.flev, tri.h_flev);
    upload(tri.blev, tri.h_blev);
    upload(tri.flev_pos, tri.h_flev_pos);
    upload(tri.blev_pos, tri.h_blev_pos);
    upload(tri.frow_lvl, frow_lvl);
    if (!tri.chain) {  // the chains read codes instead
        upload(tri.frow, frow);
        upload(tri.brow, brow);
        upload(tri.fptr, fptr);
        upload(tri.bptr, bptr);
        upload(tri.fcol, fcol);
        upload(tri.bcol, bcol);
    }
    upload(tri.fsrc, fsrc);
    upload(tri.bsrc, bsrc);
}

TriArgs tri_args(const TriSchedule& t)
{
    return TriArgs{t.row0.get(), t.nrows.get(), t.flev.get(), t.blev.get(), t.flev_pos.get(), t.blev_pos.get(),
                   t.frow.get(), t.brow.get(), t.fptr.get(), t.bptr.get(), t.fcol.get(), t.bcol.get(),
                   t.fnnz, t.bnnz, t.rows, t.bs};
}

std::size_t lds_limit(owtk_precond pc)
{
    // device LDS limit per workgroup (cached per device)
    static thread_local int cached_device = -1;
    static thread_local std::size_t cached = 0;
    if (cached_device != pc->m->ctx->device) {
        hipDeviceProp_t prop;
        OWTK_HIP(hipGetDeviceProperties(&prop, pc->m->ctx->device));
        cached = prop.sharedMemPerBlock;
        cached_device = pc->m->ctx->device;
    }
    return cached;
}

void read_flag(owtk_precond pc, int* value)
{
    OWTK_HIP(hipMemcpyAsync(value, pc->flag.get(), sizeof(int), hipMemcpyDeviceToHost, pc->m->ctx->stream));
    pc->m->ctx->sync();
}

void clear_flag(owtk_precond pc) { kern::fill_zero_bytes(pc->m->ctx->stream, pc->flag.get(), sizeof(int) * 4); }

unsigned int grid_for(std::int64_t n) { return dev::stream_grid(n, 4); }

// Value arrays in the preconditioner's storage precision.
void refresh_storage(owtk_precond pc)
{
    auto& t = pc->tri;
    const hipStream_t st = pc->m->ctx->stream;
    const int bs = pc->m->bs;
    if (t.chain) {
        // the sweeps' value slots, FP64 from the chain-order factor, then the storage's copy
        const std::int64_t nv = t.slots16 * bs;
        if (!t.f16v64.get()) t.f16v64.allocate(nv);
        if (!t.b16v64.get()) t.b16v64.allocate(nv);
        k_ell_gather<double><<<grid_for(nv), kBlock, 0, st>>>(t.f16v64.get(), t.fval64.get(), t.fmap.get(), t.slots16,
                                                              t.fnnz, bs);
        k_ell_gather<double><<<grid_for(nv), kBlock, 0, st>>>(t.b16v64.get(), t.bval64.get(), t.bmap.get(), t.slots16,
                                                              t.bnnz, bs);
        OWTK_LAUNCH_CHECK();
        if (pc->storage == OWTK_F32) {
            if (!t.f16v32.get()) t.f16v32.allocate(nv);
            if (!t.b16v32.get()) t.b16v32.allocate(nv);
            kern::convert(st, t.f16v32.get(), t.f16v64.get(), static_cast<std::size_t>(nv));
            kern::convert(st, t.b16v32.get(), t.b16v64.get(), static_cast<std::size_t>(nv));
        } else if (pc->storage == OWTK_BF16) {
            if (!t.f16v16.get()) t.f16v16.allocate(nv);
            if (!t.b16v16.get()) t.b16v16.allocate(nv);
            kern::k_to_bf16<<<grid_for(nv), kBlock, 0, st>>>(t.f16v16.get(), t.f16v64.get(), nv);
            kern::k_to_bf16<<<grid_for(nv), kBlock, 0, st>>>(t.b16v16.get(), t.b16v64.get(), nv);
            OWTK_LAUNCH_CHECK();
        }
    }
    if (pc->storage == OWTK_F32 || pc->storage == OWTK_BF16) {
        const std::int64_t nd = t.rows * bs;
        if (!t.dval32.get()) t.dval32.allocate(std::max<std::int64_t>(nd, 1));
        kern::convert(st, t.dval32.get(), t.dval64.get(), static_cast<std::size_t>(nd));
    }
    if (t.chain) return;  // the flat copies are for the level sets alone
    if (pc->storage == OWTK_F32) {
        if (!t.fval32.get()) t.fval32.allocate(std::max<std::int64_t>(t.fnnz * bs, 1));
        if (!t.bval32.get()) t.bval32.allocate(std::max<std::int64_t>(t.bnnz * bs, 1));
        if (t.fnnz) kern::convert(st, t.fval32.get(), t.fval64.get(), static_cast<std::size_t>(t.fnnz * bs));
        if (t.bnnz) kern::convert(st, t.bval32.get(), t.bval64.get(), static_cast<std::size_t>(t.bnnz * bs));
    } else if (pc->storage == OWTK_BF16) {
        if (!t.fval16.get()) t.fval16.allocate(std::max<std::int64_t>(t.fnnz * bs, 1));
        if (!t.bval16.get()) t.bval16.allocate(std::max<std::int64_t>(t.bnnz * bs, 1));
        if (t.fnnz)
            kern::k_to_bf16<<<grid_for(t.fnnz * bs), kBlock, 0, st>>>(t.fval16.get(), t.fval64.get(), t.fnnz * bs);
        if (t.bnnz)
            kern::k_to_bf16<<<grid_for(t.bnnz * bs), kBlock, 0, st>>>(t.bval16.get(), t.bval64.get(), t.bnnz * bs);
        OWTK_LAUNCH_CHECK();
    }
}

// ------------------------------------------------------------------- Jacobi --
void jacobi_setup(owtk_precond pc)
{
    owtk_matrix m = pc->m;
    if (m->dense()) {
        if (m->bs > 8 || m->s.layout != Layout::sell)
            throw unsupported_error("dense block-Jacobi supports block sizes up to 4");
        std::vector<std::int64_t> slot(m->owned);
        for (std::int64_t row = 0; row < m->owned; ++row) {
            std::int64_t s = -1;
            for (std::int32_t e = m->h_offsets[row]; e < m->h_offsets[row + 1]; ++e)
                if (m->h_columns[e] == row) {
                    s = m->s.slot_of_entry[e];
                    break;
                }
            if (s < 0) throw std::invalid_argument("dense-block CSR row has no diagonal block");
            slot[row] = s;
        }
        upload(pc->tri.dsrc, slot);
        pc->inv64.allocate(static_cast<std::size_t>(m->owned) * m->bs * m->bs);
        return;
    }
    std::vector<std::int64_t> src(m->owned);
    for (std::int64_t row = 0; row < m->owned; ++row) {
        if (m->has_diag_array()) {
            src[row] = diag_source(m, row);
            continue;
        }
        std::int64_t s = std::numeric_limits<std::int64_t>::min();
        for (std::int32_t e = m->h_offsets[row]; e < m->h_offsets[row + 1]; ++e)
            if (m->h_columns[e] == row) {
                s = entry_source(m, e);
                break;
            }
        if (s == std::numeric_limits<std::int64_t>::min())
            throw std::invalid_argument("BlockCsrMatrix row has no diagonal");
        src[row] = s;
    }
    upload(pc->tri.dsrc, src);
    pc->inv64.allocate(static_cast<std::size_t>(m->owned) * m->bs);
}

void jacobi_numeric(owtk_precond pc)
{
    owtk_matrix m = pc->m;
    const hipStream_t st = m->ctx->stream;
    clear_flag(pc);
    if (m->dense()) {
        const unsigned int g = static_cast<unsigned int>((m->owned + 255) / 256);
        switch (m->bs) {
        case 1: k_block_inverse<1><<<g, kBlock, 0, st>>>(pc->inv64.get(), pc->tri.dsrc.get(), m->owned, m->v64.get(), pc->flag.get()); break;
        case 2: k_block_inverse<2><<<g, kBlock, 0, st>>>(pc->inv64.get(), pc->tri.dsrc.get(), m->owned, m->v64.get(), pc->flag.get()); break;
        case 3: k_block_inverse<3><<<g, kBlock, 0, st>>>(pc->inv64.get(), pc->tri.dsrc.get(), m->owned, m->v64.get(), pc->flag.get()); break;
        default: k_block_inverse<4><<<g, kBlock, 0, st>>>(pc->inv64.get(), pc->tri.dsrc.get(), m->owned, m->v64.get(), pc->flag.get()); break;
        }
        OWTK_LAUNCH_CHECK();
    } else {
        const double minimum = pc->minimum_diagonal > 0 ? pc->minimum_diagonal : kTol;
        k_jacobi_inverse<<<grid_for(m->owned * m->bs), kBlock, 0, st>>>(pc->inv64.get(), pc->tri.dsrc.get(),
                                                                       m->owned, m->bs, comp_stride(m),
                                                                       m->v64.get(), m->d64.get(), minimum,
                                                                       pc->flag.get());
        OWTK_LAUNCH_CHECK();
    }
    int flag = 0;
    read_flag(pc, &flag);
    if (flag != flag_ok) {
        if (m->dense()) throw std::invalid_argument("block-Jacobi preconditioner has a singular diagonal block");
        throw std::invalid_argument("Jacobi preconditioner has a singular diagonal");
    }
    if (pc->storage != OWTK_F64) {
        if (!pc->inv32.get()) pc->inv32.allocate(pc->inv64.count);
        kern::convert(st, pc->inv32.get(), pc->inv64.get(), pc->inv64.count);
    }
}

// --------------------------------------------------------------------- SSOR --
// Greedy colouring of the symmetrised owned-row graph in row order: each row
// takes the smallest colour none of its neighbours holds.
std::vector<std::int32_t> greedy_colours(owtk_matrix m)
{
    const std::int64_t n = m->owned;
    std::vector<std::vector<std::int32_t>> adj(n);
    for (std::int64_t i = 0; i < n; ++i)
        for (std::int32_t e = m->h_offsets[i]; e < m->h_offsets[i + 1]; ++e) {
            const std::int64_t j = m->h_columns[e];
            if (j == i || j >= n) continue;
            adj[i].push_back(static_cast<std::int32_t>(j));
            adj[j].push_back(static_cast<std::int32_t>(i));
        }
    std::vector<std::int32_t> colour(n, -1);
    std::vector<std::int64_t> seen;
    for (std::int64_t i = 0; i < n; ++i) {
        seen.assign(adj[i].size() + 2, -1);
        for (std::int32_t j : adj[i])
            if (colour[j] >= 0 && colour[j] < static_cast<std::int32_t>(seen.size())) seen[colour[j]] = i;
        std::int32_t c = 0;
        while (seen[c] == i) ++c;
        colour[i] = c;
    }
    return colour;
}

void dense_ssor_setup(owtk_precond pc)
{
    owtk_matrix m = pc->m;
    if (m->bs > 4 || m->s.layout != Layout::sell) throw unsupported_error("dense-block SSOR supports block sizes up to 4");
    jacobi_setup(pc);  // diagonal block slots + inverse storage
    const std::vector<std::int32_t> colour = greedy_colours(m);
    const std::int32_t colours = colour.empty() ? 0 : *std::max_element(colour.begin(), colour.end()) + 1;
    pc->h_mc_ptr.assign(colours + 1, 0);
    for (std::int32_t c : colour) ++pc->h_mc_ptr[c + 1];
    for (std::int32_t c = 0; c < colours; ++c) pc->h_mc_ptr[c + 1] += pc->h_mc_ptr[c];
    std::vector<std::int32_t> rows(colour.size());
    std::vector<std::int64_t> fill(pc->h_mc_ptr.begin(), pc->h_mc_ptr.end() - 1);
    for (std::int64_t i = 0; i < static_cast<std::int64_t>(colour.size()); ++i) rows[fill[colour[i]]++] = static_cast<std::int32_t>(i);
    // Colour-ordered copies: colour c's rows (ascending) fill copy rows
    // h_mc_seg[c] .. h_mc_seg[c] + count - 1, padded to whole slices.  The
    // forward copy keeps each row's blocks on earlier colours, the backward
    // copy those on later colours, both in the row's slot order (the FMA
    // order of the sweeps); the diagonal copy has one block per copy row.
    pc->h_mc_seg.assign(colours + 1, 0);
    for (std::int32_t c = 0; c < colours; ++c) {
        const std::int64_t cnt = pc->h_mc_ptr[c + 1] - pc->h_mc_ptr[c];
        pc->h_mc_seg[c + 1] = pc->h_mc_seg[c] + (cnt + 63) / 64 * 64;
    }
    const std::int64_t padded = pc->h_mc_seg[colours];
    std::vector<std::int32_t> prow(static_cast<std::size_t>(std::max<std::int64_t>(padded, 1)), -1);
    for (std::int32_t c = 0; c < colours; ++c)
        for (std::int64_t t = 0; t < pc->h_mc_ptr[c + 1] - pc->h_mc_ptr[c]; ++t)
            prow[pc->h_mc_seg[c] + t] = rows[pc->h_mc_ptr[c] + t];
    upload(pc->mc_prow, prow);
    std::vector<std::int64_t> dslot(m->owned);
    OWTK_HIP(hipMemcpy(dslot.data(), pc->tri.dsrc.get(), dslot.size() * sizeof(std::int64_t), hipMemcpyDeviceToHost));
    const int bb = m->bs * m->bs;
    const std::size_t sv = pc->storage == OWTK_F64 ? 8 : (pc->storage == OWTK_F32 ? 4 : 2);
    auto build = [&](McSell& out, int dir) {  // dir -1 forward, +1 backward, 0 diagonal
        std::vector<std::int32_t> len(static_cast<std::size_t>(std::max<std::int64_t>(padded, 1)), 0);
        std::vector<std::vector<std::pair<std::int32_t, std::int64_t>>> ent(static_cast<std::size_t>(padded));
        for (std::int64_t q = 0; q < padded; ++q) {
            const std::int32_t i = prow[q];
            if (i < 0) continue;
            if (dir == 0) {
                ent[q].push_back({i, dslot[i]});
            } else {
                for (std::int32_t e = m->h_offsets[i]; e < m->h_offsets[i + 1]; ++e) {
                    const std::int32_t j = m->h_columns[e];
                    if (j >= m->owned || j == i) continue;
                    if ((dir < 0) == (colour[j] < colour[i])) ent[q].push_back({j, m->s.slot_of_entry[e]});
                }
            }
            len[q] = static_cast<std::int32_t>(ent[q].size());
        }
        const std::int64_t slices = padded / 64;
        std::vector<std::int32_t> sp(static_cast<std::size_t>(slices + 1), 0);
        for (std::int64_t sl = 0; sl < slices; ++sl) {
            int wd = 0;
            for (int l = 0; l < 64; ++l) wd = std::max(wd, len[sl * 64 + l]);
            sp[sl + 1] = sp[sl] + 64 * wd;
        }
        const std::int64_t slots = sp[slices];
        std::vector<std::int32_t> cols(static_cast<std::size_t>(std::max<std::int64_t>(slots, 1)), 0);
        std::vector<std::int64_t> map(static_cast<std::size_t>(std::max<std::int64_t>(slots, 1)), -1);
        for (std::int64_t q = 0; q < padded; ++q)
            for (std::size_t k = 0; k < ent[q].size(); ++k) {
                const std::int64_t slot = sp[q / 64] + 64 * static_cast<std::int64_t>(k) + (q % 64);
                cols[slot] = ent[q][k].first;
                map[slot] = ent[q][k].second;
            }
        if (dir == 0) {  // one block per copy row: slot q
            map.assign(static_cast<std::size_t>(std::max<std::int64_t>(padded, 1)), -1);
            for (std::int64_t q = 0; q < padded; ++q)
                if (prow[q] >= 0) map[q] = dslot[prow[q]];
            out.slots = padded;
        } else {
            upload(out.slice_ptr, sp);
            upload(out.row_len, len);
            upload(out.cols, cols);
            out.slots = slots;
        }
        upload(out.map, map);
        out.vals.allocate(static_cast<std::size_t>(std::max<std::int64_t>(out.slots, 1)) * bb * sv);
    };
    build(pc->mc_fwd, -1);
    build(pc->mc_bwd, 1);
    build(pc->mc_diag, 0);
    const std::size_t nb = static_cast<std::size_t>(m->owned * m->bs);
    if (pc->storage == OWTK_F64) pc->work64.allocate(std::max<std::size_t>(nb, 1));
    else pc->work32.allocate(std::max<std::size_t>(nb, 1));
}

// The copies' values from the matrix, in the preconditioner's storage type.
void dense_ssor_gather(owtk_precond pc)
{
    owtk_matrix m = pc->m;
    const hipStream_t st = m->ctx->stream;
    const int bb = m->bs * m->bs;
    for (McSell* c : {&pc->mc_fwd, &pc->mc_bwd, &pc->mc_diag}) {
        if (c->slots == 0) continue;
        const unsigned int g = grid_for(c->slots * bb);
        switch (pc->storage) {
        case OWTK_F64:
            k_mc_gather<double><<<g, kBlock, 0, st>>>(reinterpret_cast<double*>(c->vals.get()), m->v64.get(),
                                                      c->map.get(), c->slots, bb);
            break;
        case OWTK_F32:
            k_mc_gather<float><<<g, kBlock, 0, st>>>(reinterpret_cast<float*>(c->vals.get()), m->v32.get(),
                                                     c->map.get(), c->slots, bb);
            break;
        default:
            k_mc_gather<std::uint16_t><<<g, kBlock, 0, st>>>(reinterpret_cast<std::uint16_t*>(c->vals.get()),
                                                             m->v16.get(), c->map.get(), c->slots, bb);
            break;
        }
        OWTK_LAUNCH_CHECK();
    }
}

template<class V, class X, class I>
void dense_ssor_apply(owtk_precond pc, const X* in, X* out, const I* inv, X* y, const int* stop)
{
    owtk_matrix m = pc->m;
    const hipStream_t st = m->ctx->stream;
    const double scale = pc->omega * (2.0 - pc->omega);
    const int colours = static_cast<int>(pc->h_mc_ptr.size()) - 1;
    const V* dvals = reinterpret_cast<const V*>(pc->mc_diag.vals.get());
    auto launch = [&](int c, auto fwd) {
        constexpr bool FWD = decltype(fwd)::value;
        const std::int64_t count = pc->h_mc_ptr[c + 1] - pc->h_mc_ptr[c];
        if (count == 0) return;
        const unsigned int g = static_cast<unsigned int>((count + kBlock - 1) / kBlock);
        const McSell& cp = FWD ? pc->mc_fwd : pc->mc_bwd;
        const V* vals = reinterpret_cast<const V*>(cp.vals.get());
        const std::int64_t seg0 = pc->h_mc_seg[c];
        const std::int32_t* prow = pc->mc_prow.get();
        switch (m->bs) {
        case 1: k_mc_ssor<1, V, X, I, FWD><<<g, kBlock, 0, st>>>(prow, seg0, count, cp.slice_ptr.get(), cp.row_len.get(), cp.cols.get(), vals, dvals, pc->omega, scale, in, y, out, inv, stop); break;
        case 2: k_mc_ssor<2, V, X, I, FWD><<<g, kBlock, 0, st>>>(prow, seg0, count, cp.slice_ptr.get(), cp.row_len.get(), cp.cols.get(), vals, dvals, pc->omega, scale, in, y, out, inv, stop); break;
        case 3: k_mc_ssor<3, V, X, I, FWD><<<g, kBlock, 0, st>>>(prow, seg0, count, cp.slice_ptr.get(), cp.row_len.get(), cp.cols.get(), vals, dvals, pc->omega, scale, in, y, out, inv, stop); break;
        default: k_mc_ssor<4, V, X, I, FWD><<<g, kBlock, 0, st>>>(prow, seg0, count, cp.slice_ptr.get(), cp.row_len.get(), cp.cols.get(), vals, dvals, pc->omega, scale, in, y, out, inv, stop); break;
        }
        OWTK_LAUNCH_CHECK();
    };
    const int category = sizeof(X) == 8 ? prof_precond_f64 : prof_precond_low;
    ProfileScope prof(m->ctx, category, precond_apply_bytes(pc));
    for (int c = 0; c < colours; ++c) launch(c, std::true_type{});
    for (int c = colours - 1; c >= 0; --c) launch(c, std::false_type{});
}

void ssor_setup(owtk_precond pc)
{
    owtk_matrix m = pc->m;
    if (!(pc->omega > 0.0 && pc->omega < 2.0)) throw std::invalid_argument("SSOR omega must be in (0,2)");
    if (m->dense()) {
        dense_ssor_setup(pc);
        return;
    }
    const LocalRows L = local_rows(m, pc->block_nodes);
    TriHost t;
    const std::int64_t n = m->owned;
    t.f_off.assign(n + 1, 0);
    t.b_off.assign(n + 1, 0);
    std::vector<std::int64_t> dsrc(n);
    for (std::int64_t row = 0; row < n; ++row) {
        if (L.diag_src[row] == -1) throw std::invalid_argument("SSOR preconditioner row has no diagonal");
        dsrc[row] = L.diag_src[row];
        for (std::int64_t e = L.off[row]; e < L.off[row + 1]; ++e) {
            if (L.col[e] < row) {
                t.f_col.push_back(L.col[e]);
                t.f_src.push_back(L.src[e]);
            } else if (L.col[e] > row) {
                t.b_col.push_back(L.col[e]);
                t.b_src.push_back(L.src[e]);
            }
        }
        t.f_off[row + 1] = static_cast<std::int64_t>(t.f_col.size());
        t.b_off[row + 1] = static_cast<std::int64_t>(t.b_col.size());
    }
    build_schedule(pc, t);
    upload(pc->tri.dsrc, dsrc);
    const int bs = m->bs;
    pc->tri.fval64.allocate(std::max<std::int64_t>(pc->tri.fnnz * bs, 1));
    pc->tri.bval64.allocate(std::max<std::int64_t>(pc->tri.bnnz * bs, 1));
    pc->tri.dval64.allocate(std::max<std::int64_t>(n * bs, 1));
}

void ssor_numeric(owtk_precond pc)
{
    owtk_matrix m = pc->m;
    if (m->dense()) {
        try {
            jacobi_numeric(pc);  // diagonal-block inverses (FP64, and FP32 copy for low storage)
        } catch (const std::invalid_argument&) {
            throw std::invalid_argument("SSOR preconditioner has a singular diagonal block");
        }
        dense_ssor_gather(pc);
        return;
    }
    auto& t = pc->tri;
    const hipStream_t st = m->ctx->stream;
    const int bs = m->bs;
    const std::int64_t stride = comp_stride(m);
    clear_flag(pc);
    if (t.fnnz)
        k_gather<<<grid_for(t.fnnz * bs), kBlock, 0, st>>>(t.fval64.get(), t.fsrc.get(), t.fnnz, bs, stride,
                                                           m->v64.get(), m->d64.get(), pc->omega);
    if (t.bnnz)
        k_gather<<<grid_for(t.bnnz * bs), kBlock, 0, st>>>(t.bval64.get(), t.bsrc.get(), t.bnnz, bs, stride,
                                                           m->v64.get(), m->d64.get(), pc->omega);
    k_gather<<<grid_for(t.rows * bs), kBlock, 0, st>>>(t.dval64.get(), t.dsrc.get(), t.rows, bs, stride,
                                                       m->v64.get(), m->d64.get(), 1.0);
    k_check_diag<<<grid_for(t.rows * bs), kBlock, 0, st>>>(t.dval64.get(), t.rows * bs, kTol, pc->flag.get());
    OWTK_LAUNCH_CHECK();
    int flag = 0;
    read_flag(pc, &flag);
    if (flag != flag_ok) throw std::invalid_argument("SSOR preconditioner has a singular diagonal");
    refresh_storage(pc);
}

// ---------------------------------------------------------------------- ILU --
// Program of k_ilu_factor_chunks (IluChunkProgram) from the factor pattern
// and the update lists.  Left disabled (the level-scheduled k_ilu_factor
// runs) when a row has more than 64 entries or a count does not fit the
// program's byte fields.
void build_ilu_chunks(owtk_precond pc, const std::vector<std::int64_t>& upd_ptr,
                      const std::vector<std::int64_t>& upd_target, const std::vector<std::int64_t>& upd_upper)
{
    auto& f = pc->ilu;
    auto& P = f.chunks;
    const auto& tri = pc->tri;
    P.enabled = false;
    if (f.nnz > 0x7fffffffLL) return;
    int kmax = 1;
    for (std::int64_t row = 0; row < tri.rows; ++row)
        kmax = std::max<int>(kmax, static_cast<int>(f.h_offsets[row + 1] - f.h_offsets[row]));
    if (kmax > 64) return;
    std::vector<std::int32_t> chunk_first(tri.blocks + 1, 0);
    std::vector<std::int64_t> hdr;
    std::vector<std::int32_t> src_a;
    std::vector<std::uint32_t> op_a, op_b;
    std::vector<std::uint16_t> upd_a, upd_b;
    int max_src = 0, max_a = 0, max_nua = 0, max_b = 0, max_nub = 0;
    // a chunk's operations by lane, their updates (target, source) in one pool;
    // kept over the chunks, whose allocations would take half the set-up
    struct Op { int step, es, ps, upd0, count; };
    std::vector<std::vector<std::int32_t>> srcs(64);
    std::vector<std::vector<Op>> as(64), bs_(64);
    std::vector<std::pair<int, int>> upd;
    std::int64_t chunks = 0;
    for (std::int64_t b = 0; b < tri.blocks; ++b) {
        chunk_first[b] = static_cast<std::int32_t>(chunks);
        const std::int64_t r0 = tri.h_row0[b], nb = tri.h_nrows[b];
        for (std::int64_t c0 = 0; c0 < nb; c0 += 64, ++chunks) {
            const int cnt = static_cast<int>(std::min<std::int64_t>(64, nb - c0));
            const std::int64_t first = r0 + c0;
            upd.clear();
            for (int lane = 0; lane < 64; ++lane) {
                srcs[lane].clear();
                as[lane].clear();
                bs_[lane].clear();
            }
            for (int lane = 0; lane < cnt; ++lane) {
                const std::int64_t row = first + lane;
                const std::int64_t rb = f.h_offsets[row];
                for (std::int64_t e = rb; e < f.h_diag[row]; ++e) {
                    const std::int64_t k = f.h_columns[e];
                    const int upd0 = static_cast<int>(upd.size()), count = static_cast<int>(upd_ptr[e + 1] - upd_ptr[e]);
                    if (k < first) {
                        as[lane].push_back({0, static_cast<int>(e - rb), static_cast<int>(srcs[lane].size()), upd0, count});
                        srcs[lane].push_back(static_cast<std::int32_t>(f.h_diag[k]));
                        for (std::int64_t u = upd_ptr[e]; u < upd_ptr[e + 1]; ++u) {
                            upd.push_back({static_cast<int>(upd_target[u] - rb), static_cast<int>(srcs[lane].size())});
                            srcs[lane].push_back(static_cast<std::int32_t>(upd_upper[u]));
                        }
                    } else {
                        const std::int64_t kb = f.h_offsets[k];
                        bs_[lane].push_back({static_cast<int>(k - first), static_cast<int>(e - rb),
                                             static_cast<int>(f.h_diag[k] - kb), upd0, count});
                        for (std::int64_t u = upd_ptr[e]; u < upd_ptr[e + 1]; ++u)
                            upd.push_back({static_cast<int>(upd_target[u] - rb), static_cast<int>(upd_upper[u] - kb)});
                    }
                }
            }
            int nsrc = 0, na = 0, nua = 0, nbo = 0, nub = 0;
            for (int lane = 0; lane < cnt; ++lane) {
                nsrc = std::max<int>(nsrc, static_cast<int>(srcs[lane].size()));
                na = std::max<int>(na, static_cast<int>(as[lane].size()));
                nbo = std::max<int>(nbo, static_cast<int>(bs_[lane].size()));
                for (const auto& o : as[lane]) nua = std::max(nua, o.count);
                for (const auto& o : bs_[lane]) nub = std::max(nub, o.count);
            }
            if (nsrc > 255 || nua > 255 || nub > 255) return;
            hdr.insert(hdr.end(), {first, cnt, static_cast<std::int64_t>(src_a.size()), nsrc,
                                   static_cast<std::int64_t>(op_a.size()), na, static_cast<std::int64_t>(upd_a.size()),
                                   nua, static_cast<std::int64_t>(op_b.size()), nbo,
                                   static_cast<std::int64_t>(upd_b.size()), nub});
            const std::size_t s0 = src_a.size(), a0 = op_a.size(), ua0 = upd_a.size(), b0 = op_b.size(),
                              ub0 = upd_b.size();
            src_a.resize(s0 + static_cast<std::size_t>(nsrc) * 64, -1);
            op_a.resize(a0 + static_cast<std::size_t>(na) * 64, 0xffffffffu);
            upd_a.resize(ua0 + static_cast<std::size_t>(na) * nua * 64, 0);
            op_b.resize(b0 + static_cast<std::size_t>(nbo) * 64, 0xffffffffu);
            upd_b.resize(ub0 + static_cast<std::size_t>(nbo) * nub * 64, 0);
            for (int lane = 0; lane < cnt; ++lane) {
                for (std::size_t t2 = 0; t2 < srcs[lane].size(); ++t2) src_a[s0 + t2 * 64 + lane] = srcs[lane][t2];
                for (std::size_t j = 0; j < as[lane].size(); ++j) {
                    const auto& o = as[lane][j];
                    op_a[a0 + j * 64 + lane] = static_cast<std::uint32_t>(o.es) | (static_cast<std::uint32_t>(o.ps) << 8)
                        | (static_cast<std::uint32_t>(o.count) << 16);
                    for (int u = 0; u < o.count; ++u)
                        upd_a[ua0 + (j * nua + u) * 64 + lane] =
                            static_cast<std::uint16_t>(upd[o.upd0 + u].first | (upd[o.upd0 + u].second << 8));
                }
                for (std::size_t j = 0; j < bs_[lane].size(); ++j) {
                    const auto& o = bs_[lane][j];
                    op_b[b0 + j * 64 + lane] = static_cast<std::uint32_t>(o.step) | (static_cast<std::uint32_t>(o.es) << 8)
                        | (static_cast<std::uint32_t>(o.ps) << 16) | (static_cast<std::uint32_t>(o.count) << 24);
                    for (int u = 0; u < o.count; ++u)
                        upd_b[ub0 + (j * nub + u) * 64 + lane] =
                            static_cast<std::uint16_t>(upd[o.upd0 + u].first | (upd[o.upd0 + u].second << 8));
                }
            }
            max_src = std::max(max_src, nsrc);
            max_a = std::max(max_a, na);
            max_nua = std::max(max_nua, nua);
            max_b = std::max(max_b, nbo);
            max_nub = std::max(max_nub, nub);
        }
    }
    chunk_first[tri.blocks] = static_cast<std::int32_t>(chunks);
    if (std::max({src_a.size(), op_a.size(), upd_a.size(), op_b.size(), upd_b.size()}) > 0x7fffffffULL) return;
    P.kmax = kmax;
    P.max_src = max_src;
    P.max_a = max_a;
    P.max_nua = max_nua;
    P.max_b = max_b;
    P.max_nub = max_nub;
    // Records: at most 3 updates an operation (16 bytes; an ILU(0) factor of
    // a triangulated grid) or 7 (32 bytes), values within 16-bit offsets and
    // the whole within 64 KB of LDS; the general form otherwise.
    const int updates = std::max(max_nua, max_nub);
    P.nu = updates <= 3 ? 3 : updates <= 7 ? 7 : 0;
    if (P.nu && (ilu_rec_fixed(kmax, max_src) > 64 * 1024 || ilu_rec_lds(P) > 64 * 1024)) P.nu = 0;
    if (P.nu) {
        std::vector<std::uint32_t> rec;
        const int nu = P.nu, words = 1 + nu;
        rec.reserve((op_a.size() + op_b.size() + static_cast<std::size_t>(chunks) * 64) * words);
        const std::uint32_t trash = kmax * 512, one = (kmax + 1) * 512, gather = (kmax + 2) * 512;
        for (std::int64_t ch = 0; ch < chunks; ++ch) {
            std::int64_t* h = &hdr[ch * 12];
            const std::int64_t opa = h[4], na = h[5], upa = h[6], nua = h[7], opb = h[8], nb = h[9], upb = h[10],
                               nub = h[11];
            h[4] = static_cast<std::int64_t>(rec.size()) / (64 * words);
            const std::size_t at = rec.size();
            rec.resize(at + static_cast<std::size_t>(na + nb + 1) * 64 * words);
            for (std::int64_t j = 0; j <= na + nb; ++j)
                for (std::uint32_t lane = 0; lane < 64; ++lane) {
                    std::uint32_t* w = &rec[at + (j * 64 + lane) * words];
                    // no operation: trash / one for earlier chunks, row 63 as
                    // the pivot for this chunk's
                    const bool earlier = j < na;
                    const std::uint32_t d = earlier ? op_a[opa + j * 64 + lane]
                                            : j < na + nb ? op_b[opb + (j - na) * 64 + lane] : 0xffffffffu;
                    const std::uint32_t own_trash = trash + 8 * lane;
                    w[0] = own_trash | (earlier ? one : one + 8 * 63) << 16;
                    for (int u = 0; u < nu; ++u) w[1 + u] = one | own_trash << 16;
                    if (d == 0xffffffffu) continue;
                    const std::uint32_t step = d & 255u;
                    const std::uint32_t own = (earlier ? d & 255u : (d >> 8) & 255u) * 512 + 8 * lane;
                    const std::uint32_t pivot = earlier ? gather + ((d >> 8) & 255u) * 512 + 8 * lane
                                                        : ((d >> 16) & 255u) * 512 + 8 * step;
                    const int count = static_cast<int>(earlier ? (d >> 16) & 255u : d >> 24);
                    w[0] = own | pivot << 16;
                    for (int u = 0; u < count; ++u) {
                        const std::uint32_t v = earlier ? upd_a[upa + (j * nua + u) * 64 + lane]
                                                        : upd_b[upb + ((j - na) * nub + u) * 64 + lane];
                        const std::uint32_t target = (v & 255u) * 512 + 8 * lane;
                        const std::uint32_t source = earlier ? gather + (v >> 8) * 512 + 8 * lane
                                                             : (v >> 8) * 512 + 8 * step;
                        w[1 + u] = source | target << 16;
                    }
                }
        }
        upload(P.rec, rec);
    } else {
        if (ilu_chunk_lds(P) > 64 * 1024) return;
        upload(P.op_a, op_a);
        upload(P.op_b, op_b);
        upload(P.upd_a, upd_a);
        upload(P.upd_b, upd_b);
    }
    upload(P.chunk_first, chunk_first);
    upload(P.hdr, hdr);
    upload(P.src_a, src_a);
    P.enabled = true;
}

void ilu_setup(owtk_precond pc)
{
    owtk_matrix m = pc->m;
    if (m->dense()) throw unsupported_error("ILU is defined for component-diagonal matrices");
    const LocalRows L = local_rows(m, pc->block_nodes);
    const std::int64_t n = m->owned;
    const std::size_t fill = static_cast<std::size_t>(std::max(0, pc->fill_level));
    auto& f = pc->ilu;
    f.h_offsets.assign(1, 0);
    f.h_columns.clear();
    f.h_diag.assign(n, 0);
    std::vector<std::int64_t> src;
    std::vector<std::size_t> levels;
    constexpr std::int64_t no_source = -1;
    // build_local_pattern (preconditioner.hpp:373-427), block-restricted
    for (std::int64_t row = 0; row < n; ++row) {
        std::map<std::int64_t, std::pair<std::size_t, std::int64_t>> entries;
        if (m->has_diag_array()) entries.emplace(row, std::pair{std::size_t(0), L.diag_src[row]});
        for (std::int64_t e = L.off[row]; e < L.off[row + 1]; ++e) {
            if (!entries.emplace(L.col[e], std::pair{std::size_t(0), L.src[e]}).second)
                throw std::invalid_argument("ILU requires unique matrix columns");
        }
        for (auto it = entries.begin(); it != entries.end() && it->first < row; ++it) {
            const std::int64_t pivot = it->first;
            const std::size_t lower_level = it->second.first;
            if (lower_level >= fill) continue;
            for (std::int64_t upper = f.h_diag[pivot] + 1; upper < f.h_offsets[pivot + 1]; ++upper) {
                if (levels[upper] > fill - lower_level - 1) continue;
                const std::size_t level = lower_level + levels[upper] + 1;
                auto [target, inserted] = entries.emplace(f.h_columns[upper], std::pair{level, no_source});
                if (!inserted) target->second.first = std::min(target->second.first, level);
            }
        }
        bool diagonal_found = false;
        for (const auto& [column, entry] : entries) {
            const std::int64_t destination = static_cast<std::int64_t>(f.h_columns.size());
            f.h_columns.push_back(column);
            levels.push_back(entry.first);
            src.push_back(entry.second);
            if (column == row) {
                f.h_diag[row] = destination;
                diagonal_found = true;
            }
        }
        if (!diagonal_found) throw std::invalid_argument("ILU(0) row has no diagonal");
        f.h_offsets.push_back(static_cast<std::int64_t>(f.h_columns.size()));
    }
    f.nnz = static_cast<std::int64_t>(f.h_columns.size());
    // update lists: for each lower entry (i,k), targets (i,j) of the pivot row's upper entries (k,j)
    std::vector<std::int64_t> upd_ptr(f.nnz + 1, 0), upd_target, upd_upper;
    for (std::int64_t row = 0; row < n; ++row) {
        for (std::int64_t e = f.h_offsets[row]; e < f.h_offsets[row + 1]; ++e) {
            if (e < f.h_diag[row]) {
                const std::int64_t k = f.h_columns[e];
                for (std::int64_t u = f.h_diag[k] + 1; u < f.h_offsets[k + 1]; ++u) {
                    const std::int64_t j = f.h_columns[u];
                    // find (row, j)
                    const auto begin = f.h_columns.begin() + f.h_offsets[row];
                    const auto end = f.h_columns.begin() + f.h_offsets[row + 1];
                    const auto it = std::lower_bound(begin, end, j);
                    if (it != end && *it == j) {
                        upd_target.push_back(static_cast<std::int64_t>(it - f.h_columns.begin()));
                        upd_upper.push_back(u);
                    }
                }
            }
            upd_ptr[e + 1] = static_cast<std::int64_t>(upd_target.size());
        }
    }
    upload(f.offsets, f.h_offsets);
    upload(f.diag_pos, f.h_diag);
    upload(f.src, src);
    upload(f.upd_ptr, upd_ptr);
    upload(f.upd_target, upd_target);
    upload(f.upd_upper, upd_upper);
    upload(f.columns, f.h_columns);
    f.values.allocate(std::max<std::int64_t>(f.nnz * m->bs, 1));
    // apply schedule: lower entries before the diagonal, upper after, factor order
    TriHost t;
    t.f_off.assign(n + 1, 0);
    t.b_off.assign(n + 1, 0);
    for (std::int64_t row = 0; row < n; ++row) {
        for (std::int64_t e = f.h_offsets[row]; e < f.h_diag[row]; ++e) {
            t.f_col.push_back(f.h_columns[e]);
            t.f_src.push_back(e);
        }
        for (std::int64_t e = f.h_diag[row] + 1; e < f.h_offsets[row + 1]; ++e) {
            t.b_col.push_back(f.h_columns[e]);
            t.b_src.push_back(e);
        }
        t.f_off[row + 1] = static_cast<std::int64_t>(t.f_col.size());
        t.b_off[row + 1] = static_cast<std::int64_t>(t.b_col.size());
    }
    build_schedule(pc, t);
    build_ilu_chunks(pc, upd_ptr, upd_target, upd_upper);
    const int bs = m->bs;
    pc->tri.fval64.allocate(std::max<std::int64_t>(pc->tri.fnnz * bs, 1));
    pc->tri.bval64.allocate(std::max<std::int64_t>(pc->tri.bnnz * bs, 1));
    pc->tri.dval64.allocate(std::max<std::int64_t>(n * bs, 1));
}

void ilu_numeric(owtk_precond pc)
{
    owtk_matrix m = pc->m;
    auto& f = pc->ilu;
    auto& t = pc->tri;
    const hipStream_t st = m->ctx->stream;
    const int bs = m->bs;
    clear_flag(pc);
    k_gather<<<grid_for(f.nnz * bs), kBlock, 0, st>>>(f.values.get(), f.src.get(), f.nnz, bs, comp_stride(m),
                                                      m->v64.get(), m->d64.get(), 1.0);
    OWTK_LAUNCH_CHECK();
    const unsigned int groups = static_cast<unsigned int>(t.blocks * bs);
    if (f.chunks.enabled) {
        const auto& P = f.chunks;
        const IluChunkArgs args{P.chunk_first.get(), P.hdr.get(), P.src_a.get(), P.op_a.get(), P.op_b.get(),
                                P.upd_a.get(), P.upd_b.get(), P.rec.get(), P.kmax, P.max_src, P.max_a, P.max_nua,
                                P.max_b, P.max_nub};
        auto launch = [&](auto kernel) {
            kernel<<<groups, 64, ilu_rec_lds(P), st>>>(args, f.offsets.get(), f.diag_pos.get(), bs, f.values.get(),
                                                       f.nnz, t.rows, t.dval64.get(), pc->flag.get());
        };
        if (P.nu == 3) launch(k_ilu_factor_rec<3>);
        else if (P.nu == 7) launch(k_ilu_factor_rec<7>);
        else
            k_ilu_factor_chunks<<<groups, 64, ilu_chunk_lds(P), st>>>(args, f.offsets.get(), f.diag_pos.get(),
                                                                      t.row0.get(), t.nrows.get(), bs, f.values.get(),
                                                                      f.nnz, t.rows, t.dval64.get(), pc->flag.get());
    } else {
        k_ilu_factor<<<groups, 64, 0, st>>>(tri_args(t), t.frow_lvl.get(), f.offsets.get(), f.diag_pos.get(),
                                            f.upd_ptr.get(), f.upd_target.get(), f.upd_upper.get(), f.columns.get(),
                                            f.values.get(), f.nnz, t.dval64.get(), pc->flag.get());
    }
    OWTK_LAUNCH_CHECK();
    int flag = 0;
    read_flag(pc, &flag);
    if (flag != flag_ok) throw zero_pivot_error("zero pivot in ILU(0)");
    if (t.fnnz)
        k_gather_cm<<<grid_for(t.fnnz * bs), kBlock, 0, st>>>(t.fval64.get(), t.fsrc.get(), t.fnnz, bs,
                                                              f.values.get(), f.nnz);
    if (t.bnnz)
        k_gather_cm<<<grid_for(t.bnnz * bs), kBlock, 0, st>>>(t.bval64.get(), t.bsrc.get(), t.bnnz, bs,
                                                              f.values.get(), f.nnz);
    OWTK_LAUNCH_CHECK();
    refresh_storage(pc);
}

// -------------------------------------------------------------------- apply --
template<TriMode MODE, class X, class V>
void tri_launch(owtk_precond pc, const V* fv, const V* bv, const X* dv, const X* in, X* out, const int* stop)
{
    const auto& t = pc->tri;
    const unsigned int groups = static_cast<unsigned int>(t.blocks * t.bs);
    const std::size_t need = static_cast<std::size_t>(t.max_block_rows) * sizeof(X);
    const int threads = t.max_level_width > 128 ? 256 : (t.max_level_width > 64 ? 128 : 64);
    const X scale = static_cast<X>(pc->omega * (2.0 - pc->omega));
    const hipStream_t st = pc->m->ctx->stream;
    ProfileScope prof(pc->m->ctx, sizeof(X) == 8 ? prof_precond_f64 : prof_precond_low, precond_apply_bytes(pc));
    if (t.chain) {
        const int chains = static_cast<int>(groups);
        const Rows16Args ra{t.row0.get(), t.nrows.get(), t.fnear.get(), t.bnear.get(), t.ftile.get(), t.btile.get(),
                            t.ffar.get(), t.bfar.get(), t.slots16, t.rows, chains, t.block_chunks, t.bs};
        const V* fvals;
        const V* bvals;
        if constexpr (std::is_same_v<V, double>) {
            fvals = t.f16v64.get();
            bvals = t.b16v64.get();
        } else if constexpr (std::is_same_v<V, float>) {
            fvals = t.f16v32.get();
            bvals = t.b16v32.get();
        } else {
            fvals = t.f16v16.get();
            bvals = t.b16v16.get();
        }
        const unsigned int waves = static_cast<unsigned int>((chains + 3) / 4);
        auto launch = [&](auto k) {
            k_tri_rows16<MODE, X, V, decltype(k)::value><<<waves, 128, 0, st>>>(ra, fvals, bvals, dv, in, out, scale, stop);
        };
        if (t.k16 == 4) launch(std::integral_constant<int, 4>{});
        else if (t.k16 == 6) launch(std::integral_constant<int, 6>{});
        else if (t.k16 == 8) launch(std::integral_constant<int, 8>{});
        else launch(std::integral_constant<int, 16>{});
    } else if (need <= lds_limit(pc)) {
        k_tri_apply<MODE, X, V, true><<<groups, threads, need, st>>>(tri_args(t), fv, bv, dv, in, out, scale, stop);
    } else {
        k_tri_apply<MODE, X, V, false><<<groups, threads, 0, st>>>(tri_args(t), fv, bv, dv, in, out, scale, stop);
    }
    OWTK_LAUNCH_CHECK();
}

} // namespace

void precond_apply_f64(owtk_precond pc, const double* in, double* out, const int* stop)
{
    owtk_matrix m = pc->m;
    const hipStream_t st = m->ctx->stream;
    const std::int64_t n = pc->n();
    switch (pc->kind) {
    case OWTK_PC_IDENTITY:
        if (in != out) OWTK_HIP(hipMemcpyAsync(out, in, n * sizeof(double), hipMemcpyDeviceToDevice, st));
        return;
    case OWTK_PC_JACOBI:
        if (m->dense()) {
            const unsigned int g = static_cast<unsigned int>((m->owned + 255) / 256);
            switch (m->bs) {
            case 1: k_block_jacobi_apply<1, double, double><<<g, kBlock, 0, st>>>(pc->inv64.get(), in, out, m->owned, stop); break;
            case 2: k_block_jacobi_apply<2, double, double><<<g, kBlock, 0, st>>>(pc->inv64.get(), in, out, m->owned, stop); break;
            case 3: k_block_jacobi_apply<3, double, double><<<g, kBlock, 0, st>>>(pc->inv64.get(), in, out, m->owned, stop); break;
            default: k_block_jacobi_apply<4, double, double><<<g, kBlock, 0, st>>>(pc->inv64.get(), in, out, m->owned, stop); break;
            }
        } else {
            k_jacobi_apply<double, double><<<grid_for(n), kBlock, 0, st>>>(pc->inv64.get(), in, out, n, stop);
        }
        OWTK_LAUNCH_CHECK();
        return;
    case OWTK_PC_SSOR:
        if (m->dense()) {
            dense_ssor_apply<double, double, double>(pc, in, out, pc->inv64.get(), pc->work64.get(), stop);
            return;
        }
        tri_launch<TriMode::ssor, double, double>(pc, pc->tri.fval64.get(), pc->tri.bval64.get(),
                                                  pc->tri.dval64.get(), in, out, stop);
        return;
    case OWTK_PC_ILU:
        tri_launch<TriMode::ilu, double, double>(pc, pc->tri.fval64.get(), pc->tri.bval64.get(),
                                                 pc->tri.dval64.get(), in, out, stop);
        return;
    case OWTK_PC_LEARNED:
        learned_apply_f64(pc, in, out, stop);
        return;
    default:
        throw unsupported_error("preconditioner kind not available on the FP64 path");
    }
}

void precond_apply_f32(owtk_precond pc, const float* in, float* out, const int* stop)
{
    owtk_matrix m = pc->m;
    const hipStream_t st = m->ctx->stream;
    const std::int64_t n = pc->n();
    if (pc->kind != OWTK_PC_IDENTITY && pc->storage == OWTK_F64)
        throw std::invalid_argument("FP32 apply needs F32 or BF16 preconditioner storage");
    switch (pc->kind) {
    case OWTK_PC_IDENTITY:
        if (in != out) OWTK_HIP(hipMemcpyAsync(out, in, n * sizeof(float), hipMemcpyDeviceToDevice, st));
        return;
    case OWTK_PC_JACOBI:
        if (m->dense()) {
            const unsigned int g = static_cast<unsigned int>((m->owned + 255) / 256);
            switch (m->bs) {
            case 1: k_block_jacobi_apply<1, float, float><<<g, kBlock, 0, st>>>(pc->inv32.get(), in, out, m->owned, stop); break;
            case 2: k_block_jacobi_apply<2, float, float><<<g, kBlock, 0, st>>>(pc->inv32.get(), in, out, m->owned, stop); break;
            case 3: k_block_jacobi_apply<3, float, float><<<g, kBlock, 0, st>>>(pc->inv32.get(), in, out, m->owned, stop); break;
            default: k_block_jacobi_apply<4, float, float><<<g, kBlock, 0, st>>>(pc->inv32.get(), in, out, m->owned, stop); break;
            }
        } else {
            k_jacobi_apply<float, float><<<grid_for(n), kBlock, 0, st>>>(pc->inv32.get(), in, out, n, stop);
        }
        OWTK_LAUNCH_CHECK();
        return;
    case OWTK_PC_SSOR:
    case OWTK_PC_ILU: {
        if (m->dense()) {  // dense-block SSOR (ILU is rejected at creation)
            if (pc->storage == OWTK_F32) {
                if (!m->v32.get()) throw std::invalid_argument("matrix has no FP32 storage");
                dense_ssor_apply<float, float, float>(pc, in, out, pc->inv32.get(), pc->work32.get(), stop);
            } else {
                if (!m->v16.get()) throw std::invalid_argument("matrix has no BF16 storage");
                dense_ssor_apply<std::uint16_t, float, float>(pc, in, out, pc->inv32.get(), pc->work32.get(), stop);
            }
            return;
        }
        const auto& t = pc->tri;
        const bool ilu = pc->kind == OWTK_PC_ILU;
        if (pc->storage == OWTK_F32) {
            if (ilu) tri_launch<TriMode::ilu, float, float>(pc, t.fval32.get(), t.bval32.get(), t.dval32.get(), in, out, stop);
            else tri_launch<TriMode::ssor, float, float>(pc, t.fval32.get(), t.bval32.get(), t.dval32.get(), in, out, stop);
        } else {
            if (ilu) tri_launch<TriMode::ilu, float, std::uint16_t>(pc, t.fval16.get(), t.bval16.get(), t.dval32.get(), in, out, stop);
            else tri_launch<TriMode::ssor, float, std::uint16_t>(pc, t.fval16.get(), t.bval16.get(), t.dval32.get(), in, out, stop);
        }
        return;
    }
    case OWTK_PC_LEARNED:
        learned_apply_f32(pc, in, out, stop);
        return;
    default:
        throw unsupported_error("preconditioner kind not available on the FP32 path");
    }
}

std::int64_t precond_apply_bytes(owtk_precond pc)
{
    const std::int64_t n = pc->n();
    const int sv = pc->storage == OWTK_F64 ? 8 : (pc->storage == OWTK_F32 ? 4 : 2);
    const int sx = pc->storage == OWTK_F64 ? 8 : 4;
    switch (pc->kind) {
    case OWTK_PC_IDENTITY: return 2 * n * sx;
    case OWTK_PC_JACOBI:
        return pc->m->dense() ? n * pc->m->bs * sv + 2 * n * sx : n * sv + 2 * n * sx;
    case OWTK_PC_LEARNED: return learned_apply_bytes(pc);
    case OWTK_PC_SSOR:
        if (pc->m->dense()) {
            // both sweeps read every block once (lower or upper), the diagonal
            // block and inverse once each; in, y, out
            const std::int64_t b2 = std::int64_t(pc->m->bs) * pc->m->bs;
            return pc->m->entries * (b2 * sv + 4) + pc->m->owned * (b2 * sv + b2 * sv + 8) + 4 * n * sx;
        }
        [[fallthrough]];
    default: {
        const auto& t = pc->tri;
        const int bs = pc->m->bs;
        // factor values + block-local columns + row positions/pointers + diagonal + in/out
        return (t.fnnz + t.bnnz) * (bs * sv + 4) + 2 * t.rows * (4 + 8) + n * sx + 2 * n * sx;
    }
    }
}

} // namespace owtk

extern "C" {

void owtk_precond_params_default(owtk_precond_params* p, int32_t kind)
{
    if (!p) return;
    std::memset(p, 0, sizeof(*p));
    p->kind = kind;
    p->storage = OWTK_F64;
    p->omega = 1.0;
    p->minimum_diagonal = 0.0;
    p->block_nodes = 0;
    p->fill_level = 0;
    p->learned_model = nullptr;
}

int owtk_precond_create(owtk_matrix m, const owtk_precond_params* params, owtk_precond* out)
{
    return guarded([&] {
        if (!m || !params || !out) throw std::invalid_argument("null argument");
        *out = nullptr;
        m->ctx->activate();
        auto pc = std::make_unique<owtk_precond_s>();
        pc->m = m;
        pc->ctx = m->ctx;
        pc->kind = params->kind;
        pc->storage = params->storage;
        pc->omega = params->omega;
        pc->minimum_diagonal = params->minimum_diagonal;
        pc->block_nodes = params->block_nodes;
        pc->fill_level = params->fill_level;
        pc->schedule = params->schedule;
        pc->learned = params->learned_model;
        if (pc->schedule < 0 || pc->schedule > 2) throw std::invalid_argument("unknown triangular schedule");
        if (pc->storage < OWTK_F64 || pc->storage > OWTK_BF16) throw std::invalid_argument("unknown storage type");
        if (pc->block_nodes < 0) throw std::invalid_argument("negative block size");
        pc->flag.allocate(4);
        switch (pc->kind) {
        case OWTK_PC_IDENTITY: break;
        case OWTK_PC_JACOBI:
            if (pc->storage == OWTK_BF16) pc->storage = OWTK_F32;
            jacobi_setup(pc.get());
            jacobi_numeric(pc.get());
            break;
        case OWTK_PC_SSOR:
            ssor_setup(pc.get());
            ssor_numeric(pc.get());
            break;
        case OWTK_PC_ILU:
            ilu_setup(pc.get());
            ilu_numeric(pc.get());
            break;
        case OWTK_PC_LEARNED:
            learned_setup(pc.get());
            try {
                learned_numeric(pc.get());
            } catch (...) {
                learned_release(pc.get());
                throw;
            }
            break;
        default: throw unsupported_error("preconditioner kind not available");
        }
        pc->updates = 1;
        m->ctx->sync();
        *out = pc.release();
    });
}

int owtk_precond_update_values(owtk_precond pc)
{
    return guarded([&] {
        if (!pc) throw std::invalid_argument("null preconditioner");
        pc->m->ctx->activate();
        switch (pc->kind) {
        case OWTK_PC_JACOBI: jacobi_numeric(pc); break;
        case OWTK_PC_SSOR: ssor_numeric(pc); break;
        case OWTK_PC_ILU: ilu_numeric(pc); break;
        case OWTK_PC_LEARNED: learned_numeric(pc); break;
        default: break;
        }
        ++pc->updates;
        pc->m->ctx->sync();
    });
}

int owtk_precond_apply(owtk_precond pc, const void* in, void* out)
{
    return guarded([&] {
        if (!pc) throw std::invalid_argument("null preconditioner");
        if (!in || !out) throw std::invalid_argument("null vector");
        pc->m->ctx->activate();
        if (pc->storage == OWTK_F64) precond_apply_f64(pc, static_cast<const double*>(in), static_cast<double*>(out), nullptr);
        else precond_apply_f32(pc, static_cast<const float*>(in), static_cast<float*>(out), nullptr);
    });
}

int owtk_precond_numeric_updates(owtk_precond pc, uint64_t* count)
{
    return guarded([&] {
        if (!pc || !count) throw std::invalid_argument("null argument");
        *count = pc->updates;
    });
}

int owtk_precond_info_get(owtk_precond pc, owtk_precond_info* info)
{
    return guarded([&] {
        if (!pc || !info) throw std::invalid_argument("null argument");
        info->kind = pc->kind;
        info->storage = pc->storage;
        info->blocks = pc->tri.blocks;
        info->forward_levels = pc->tri.max_flevels;
        info->backward_levels = pc->tri.max_blevels;
        info->factor_entries = pc->ilu.nnz;
        info->apply_bytes = precond_apply_bytes(pc);
        info->rows = pc->m->owned;
        info->block_size = pc->m->bs;
    });
}

int owtk_precond_ilu_factors(owtk_precond pc, int64_t* entries, int64_t* row_offsets, int64_t* columns,
                             double* values, double* inverse_diagonal)
{
    return guarded([&] {
        if (!pc || !entries) throw std::invalid_argument("null argument");
        if (pc->kind != OWTK_PC_ILU) throw std::invalid_argument("not an ILU preconditioner");
        pc->m->ctx->activate();
        const auto& f = pc->ilu;
        *entries = f.nnz;
        if (row_offsets) std::copy(f.h_offsets.begin(), f.h_offsets.end(), row_offsets);
        if (columns) std::copy(f.h_columns.begin(), f.h_columns.end(), columns);
        const int bs = pc->m->bs;
        if (values) {
            std::vector<double> cm(static_cast<std::size_t>(f.nnz * bs));
            OWTK_HIP(hipMemcpy(cm.data(), f.values.get(), cm.size() * sizeof(double), hipMemcpyDeviceToHost));
            for (std::int64_t e = 0; e < f.nnz; ++e)
                for (int c = 0; c < bs; ++c) values[e * bs + c] = cm[c * f.nnz + e];
        }
        if (inverse_diagonal) {
            const std::int64_t n = pc->m->owned;
            std::vector<double> cm(static_cast<std::size_t>(n * bs));
            OWTK_HIP(hipMemcpy(cm.data(), pc->tri.dval64.get(), cm.size() * sizeof(double), hipMemcpyDeviceToHost));
            for (std::int64_t r = 0; r < n; ++r)
                for (int c = 0; c < bs; ++c) inverse_diagonal[r * bs + c] = cm[c * n + r];
        }
    });
}

int owtk_precond_destroy(owtk_precond pc)
{
    return guarded([&] {
        if (!pc) return;
        pc->ctx->activate();
        pc->ctx->sync();
        if (pc->kind == OWTK_PC_LEARNED) learned_release(pc);
        delete pc;
    });
}

} // extern "C"
