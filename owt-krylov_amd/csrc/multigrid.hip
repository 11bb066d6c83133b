// Device two-level aggregation multigrid (AggregationMultigrid,
// multigrid.hpp:41-421).  Set-up follows the reference on the host: greedy
// aggregates seeded in row order, the row-averaged coarse matrix (sums in
// fine-row, entry order), inverse diagonals and the greedy red/black
// colourings.  Every operation of a cycle runs on the device:
//   Jacobi / Chebyshev smoothing  SpMV + one update pass
//   red-black Gauss-Seidel (fine) full residual per colour + colour update
//   red-black Gauss-Seidel (coarse, true Gauss-Seidel rows, gauss_seidel_rows
//     multigrid.hpp:365-395) level schedule of each colour's rows: rows of
//     a level touch no earlier row of the same colour, so each level is one
//     parallel pass, one workgroup walks the levels, and the result is the
//     sequential sweep's
//   restriction                   per aggregate, its members in ascending
//                                 order (the reference's summation order)
//   prolongation                  elementwise add
// with the reference's arithmetic in each update.
#include "precond.hpp"
#include "solver_common.hpp"
#include "kernels/blas1.hpp"
#include "kernels/spmv.hpp"

#include <algorithm>
#include <chrono>
#include <cmath>
#include <map>
#include <queue>
#include <vector>

using namespace owtk;

struct owtk_multigrid_s {
    owtk_matrix fine = nullptr;
    owtk_context ctx = nullptr;  // destroy may run after the fine matrix is gone
    owtk_matrix coarse = nullptr;  // owned
    owtk_multigrid_options opt{};
    int bs = 1;
    std::int64_t n = 0, nc = 0;
    std::vector<std::int64_t> h_f2c;
    std::vector<std::int32_t> h_coff, h_ccol;
    std::vector<double> h_cval;
    owtk::DeviceArray<double> fine_inv, coarse_inv, agg_size;
    owtk::DeviceArray<std::int32_t> f2c, agg_ptr, agg_members, fine_red, fine_black;
    std::int64_t n_red = 0, n_black = 0;
    // coarse Gauss-Seidel: the level schedule of each colour
    owtk::DeviceArray<std::int32_t> gs_rows;
    owtk::DeviceArray<std::int64_t> gs_levels;  // device copy of gs_level_ptr
    std::vector<std::int64_t> gs_level_ptr;  // red levels, then black levels
    std::int64_t red_levels = 0;
    // the same rows in sweep (level) order as ELL: position p's k-th
    // off-diagonal entry (CSR order) at k * positions + p, its values at
    // (k * positions + p) * bs + c; padding slots hold the row itself and 0
    owtk::DeviceArray<std::int32_t> gs_len, gs_col;
    owtk::DeviceArray<double> gs_val, gs_diag;
    std::int64_t gs_positions = 0;
    int gs_k = 0;
    // one-wave schedule of the black rows (k_mg_gs_wave); wave_k = 0: not used
    int wave_k = 0;
    std::int64_t wave_chunks = 0, wave_slots = 0;  // chunks run; 64 lanes x (chunks + padding chunks)
    owtk::DeviceArray<std::int32_t> wave_row, wave_near, wave_far;
    owtk::DeviceArray<double> wave_val, wave_diag;
    ~owtk_multigrid_s()
    {
        if (coarse) (void)owtk_matrix_destroy(coarse);
    }
};

namespace owtk {
namespace {

using dev::kBlock;

// x += (w * inv) * (b - work)
__global__ __launch_bounds__(256) void k_mg_jacobi(double* __restrict__ x, const double* __restrict__ b,
                                                   const double* __restrict__ work, const double* __restrict__ inv,
                                                   double w, std::int64_t n)
{
    const std::int64_t step = static_cast<std::int64_t>(gridDim.x) * blockDim.x;
    for (std::int64_t i = static_cast<std::int64_t>(blockIdx.x) * blockDim.x + threadIdx.x; i < n; i += step)
        x[i] = x[i] + (w * inv[i]) * (b[i] - work[i]);
}

// rows of one colour: x += inv * (b - work)
__global__ __launch_bounds__(256) void k_mg_colour(const std::int32_t* __restrict__ rows, std::int64_t count, int bs,
                                                   double* __restrict__ x, const double* __restrict__ b,
                                                   const double* __restrict__ work, const double* __restrict__ inv)
{
    const std::int64_t total = count * bs;
    const std::int64_t step = static_cast<std::int64_t>(gridDim.x) * blockDim.x;
    for (std::int64_t t = static_cast<std::int64_t>(blockIdx.x) * blockDim.x + threadIdx.x; t < total; t += step) {
        const std::int64_t i = static_cast<std::int64_t>(rows[t / bs]) * bs + t % bs;
        x[i] = x[i] + inv[i] * (b[i] - work[i]);
    }
}

// coarse[a] = sum over members m (ascending) of fine[m] / size[a], from zero
__global__ __launch_bounds__(256) void k_mg_restrict(const double* __restrict__ fine, double* __restrict__ coarse,
                                                     const std::int32_t* __restrict__ ptr,
                                                     const std::int32_t* __restrict__ members,
                                                     const double* __restrict__ size, std::int64_t nc, int bs)
{
    const std::int64_t total = nc * bs;
    const std::int64_t step = static_cast<std::int64_t>(gridDim.x) * blockDim.x;
    for (std::int64_t t = static_cast<std::int64_t>(blockIdx.x) * blockDim.x + threadIdx.x; t < total; t += step) {
        const std::int64_t a = t / bs;
        const int k = static_cast<int>(t % bs);
        const double sz = size[a];
        double acc = 0.0;
        for (std::int32_t e = ptr[a]; e < ptr[a + 1]; ++e)
            acc = acc + fine[static_cast<std::int64_t>(members[e]) * bs + k] / sz;
        coarse[t] = acc;
    }
}

// fine[node] += coarse[f2c[node]]
__global__ __launch_bounds__(256) void k_mg_prolong(const double* __restrict__ coarse, double* __restrict__ fine,
                                                    const std::int32_t* __restrict__ f2c, std::int64_t n, int bs)
{
    const std::int64_t total = n * bs;
    const std::int64_t step = static_cast<std::int64_t>(gridDim.x) * blockDim.x;
    for (std::int64_t t = static_cast<std::int64_t>(blockIdx.x) * blockDim.x + threadIdx.x; t < total; t += step)
        fine[t] = fine[t] + coarse[static_cast<std::int64_t>(f2c[t / bs]) * bs + t % bs];
}

struct GsArgs {
    const std::int32_t* rows;
    const std::int32_t* len;
    const std::int32_t* col;
    const double* val;
    const double* diag;
    const double* rhs;
    std::int64_t positions;
    int bs, K;
};

// One colour's Gauss-Seidel sweep, all levels in one workgroup: the rows of
// a level in parallel, a barrier between levels (a level's reads of earlier
// levels' writes stay inside the workgroup).  The rows come from a
// level-ordered ELL copy: a work item's row, row length, diagonal and
// right-hand side, and then eight of its slots at a time, load with no
// dependence on one another (padding slots name the row itself, and their
// products are dropped by a select), so a level costs one round trip for its
// structure and one for the gathered solution values instead of a pointer
// chase through rows, offsets and columns.  The arithmetic and its order are
// the CSR sweep's.  (Loading the next level's structure during the current
// one did not help: vector loads retire in issue order, so the gathers then
// waited for the prefetch as well.)
__device__ inline void gs_row(const GsArgs& g, std::int64_t p, int k, double* x)
{
    constexpr int C = 8;
    const std::int64_t r = g.rows[p];
    const int n = g.len[p];
    const double d = g.diag[p * g.bs + k];
    double rr = g.rhs[r * g.bs + k];
    for (int k0 = 0; k0 < g.K; k0 += C) {
        std::int64_t cj[C];
        double v[C], xv[C];
#pragma unroll
        for (int u = 0; u < C; ++u) {
            const std::int64_t slot = static_cast<std::int64_t>(k0 + u < g.K ? k0 + u : g.K - 1) * g.positions + p;
            cj[u] = g.col[slot];
            v[u] = g.val[slot * g.bs + k];
        }
#pragma unroll
        for (int u = 0; u < C; ++u) xv[u] = x[cj[u] * g.bs + k];
#pragma unroll
        for (int u = 0; u < C; ++u) {
            const double f = rr - v[u] * xv[u];
            rr = k0 + u < n ? f : rr;
        }
    }
    x[r * g.bs + k] = rr / d;
}

__global__ __launch_bounds__(1024) void k_mg_gs_ell(const std::int64_t* __restrict__ level_ptr, std::int64_t first,
                                                    std::int64_t last, GsArgs g, double* x)
{
    for (std::int64_t l = first; l < last; ++l) {
        const std::int64_t a = level_ptr[l];
        const std::int64_t total = (level_ptr[l + 1] - a) * g.bs;
        for (std::int64_t t = threadIdx.x; t < total; t += blockDim.x)
            gs_row(g, a + t / g.bs, static_cast<int>(t % g.bs), x);
        __syncthreads();
    }
}

// A colour of one level: its rows are independent, so the whole grid takes
// them (the red rows of a symmetric pattern).
__global__ __launch_bounds__(256) void k_mg_gs_level(std::int64_t positions, GsArgs g, double* x)
{
    const std::int64_t t = static_cast<std::int64_t>(blockIdx.x) * blockDim.x + threadIdx.x;
    if (t < positions * g.bs) gs_row(g, t / g.bs, static_cast<int>(t % g.bs), x);
}

// The black rows' sweep by one wave per component.  The greedy colouring
// leaves long chains of adjacent black rows (1,026 levels of 27 rows on the
// 512 x 256 grid's coarse level), so a sweep is bound by the latency of one
// level, and a component's levels fit one wave: no workgroup barrier, and no
// component waits for another.  The host packs the rows into chunks of at
// most 64 whose predecessors lie in earlier chunks (longest remaining chain
// first); lane l of a chunk owns one row.  Everything but the newest values
// is loaded ahead: a chunk's slot addresses 2 kWaveAhead chunks before it
// runs, its matrix values, right-hand side, diagonal and older solution
// values kWaveAhead chunks before.  A slot has two addresses, and its
// solution value is the sum of what they hold, one of them always zero (a
// select would take three instructions, and a lone wave is bound by the
// number it issues):
//   far   byte offset into x (component 0) of a row of a later chunk (its
//         previous value), of the other colour, or of a chunk more than
//         kWaveAhead back, stored before the load was issued (accesses of one
//         wave to one address stay in order); the zero behind x otherwise;
//   near  byte address in the LDS ring of the last chunks' results, or of the
//         ring's zero.
// So a level costs one LDS round trip, its products and the division, done
// as reciprocal times value with one FMA correction (Markstein: the correctly
// rounded quotient while its residual is no subnormal, so for dividends above
// 2^-969 and diagonals below 2^1022, and at most a unit in the last place off
// beyond; a result that is not finite is divided for).  Products and their
// order are those of k_mg_gs_ell.  Coarse level of a 512 x 256 grid, block 3
// (about 1,040 chunks): 292 us a sweep, 670 clocks a chunk, most of them issue:
// the wave loads, computes and stores by itself.  One workgroup with a barrier
// per level (k_mg_gs_ell) took 1.6 ms for the two colours.
constexpr int kWaveAhead = 3, kWaveRing = 2 * kWaveAhead;  // chunks
constexpr std::int64_t kWaveLevels = 8;        // chunks per level up to which the wave is used (build_wave)
constexpr int kWaveZero = kWaveRing * 64 * 8;  // byte address of the ring's zero entry
struct GsWaveArgs {
    const std::int32_t* row;   // [slot] byte offset of the row's component 0, -1: idle lane
    const std::int32_t* near;  // [(chunk * K / 2 + pair) * 64 + lane][2]
    const std::int32_t* far;   // likewise
    const double* val;         // [component][(chunk * K / 2 + pair) * 64 + lane][2]
    const double* diag;        // [component][slot][2]: diagonal, reciprocal
    const double* rhs;         // [component][slot]
    std::int64_t chunks, slots;
};

typedef int int2_v __attribute__((ext_vector_type(2)));
typedef double gs_double2 __attribute__((ext_vector_type(2)));

template<int K>
__global__ __launch_bounds__(64, 1) void k_mg_gs_wave(GsWaveArgs g, double* x)
{
    static_assert(K % 2 == 0);
    constexpr int P = kWaveAhead;
    __shared__ double ring[kWaveRing * 64 + 1];
    const unsigned int lane = threadIdx.x;
    const int c = static_cast<int>(blockIdx.x);
    char* xc = reinterpret_cast<char*>(x + c);
    const char* ring_bytes = reinterpret_cast<const char*>(ring);
    for (int t = static_cast<int>(lane); t <= kWaveRing * 64; t += 64) ring[t] = 0.0;
    // wave-uniform bases, the lane added at the load
    const auto* near2 = reinterpret_cast<const int2_v*>(g.near);
    const auto* far2 = reinterpret_cast<const int2_v*>(g.far);
    const auto* val2 = reinterpret_cast<const gs_double2*>(g.val) + c * (g.slots * (K / 2));
    const auto* diag2 = reinterpret_cast<const gs_double2*>(g.diag) + c * g.slots;
    const double* rhs = g.rhs + c * g.slots;
    const std::int32_t* row = g.row;
    int near[2 * P][K], far[P][K];
    double v[P][K], xo[P][K], rr[P];
    gs_double2 dd[P];
    int at[P];
    // chunk q's addresses into stages sn and sf; its values into stage sf
    auto load_codes = [&](std::int64_t q, int sn, int sf) {
#pragma unroll
        for (int j = 0; j < K / 2; ++j) {
            const int2_v w = (near2 + (q * (K / 2) + j) * 64)[lane];
            near[sn][2 * j] = w.x;
            near[sn][2 * j + 1] = w.y;
            const int2_v f = (far2 + (q * (K / 2) + j) * 64)[lane];
            far[sf][2 * j] = f.x;
            far[sf][2 * j + 1] = f.y;
        }
    };
    auto load_values = [&](std::int64_t q, int t) {
#pragma unroll
        for (int k = 0; k < K; ++k) xo[t][k] = *reinterpret_cast<const double*>(xc + static_cast<std::uint32_t>(far[t][k]));
#pragma unroll
        for (int j = 0; j < K / 2; ++j) {
            const gs_double2 w = (val2 + (q * (K / 2) + j) * 64)[lane];
            v[t][2 * j] = w.x;
            v[t][2 * j + 1] = w.y;
        }
        rr[t] = (rhs + q * 64)[lane];
        dd[t] = (diag2 + q * 64)[lane];
        at[t] = (row + q * 64)[lane];
    };
#pragma unroll
    for (int s = 0; s < P; ++s) {
        load_codes(s, s, s);
        load_values(s, s);
    }
#pragma unroll
    for (int s = P; s < 2 * P; ++s) load_codes(s, s, s - P);
    for (std::int64_t q0 = 0; q0 < g.chunks; q0 += 2 * P) {
#pragma unroll
        for (int s = 0; s < 2 * P; ++s) {
            // chunk q = q0 + s (the schedule ends in idle chunks, so no test)
            const int t = s % P;
            double acc = rr[t];
            double xv[K];
#pragma unroll
            for (int k = 0; k < K; ++k)
                xv[k] = *reinterpret_cast<const double*>(ring_bytes + static_cast<std::uint32_t>(near[s][k])) + xo[t][k];
#pragma unroll
            for (int k = 0; k < K; ++k) acc = acc - v[t][k] * xv[k];
            const double d = dd[t].x, ri = dd[t].y;
            const double qt = acc * ri;
            double res = __builtin_fma(__builtin_fma(-qt, d, acc), ri, qt);
            // a wave-uniform branch keeps the division out of the chain
            if (__builtin_amdgcn_ballot_w64(!__builtin_isfinite(res)) != 0) res = __builtin_isfinite(res) ? res : acc / d;
            const int row_at = at[t];
            // chunk q + P's values (its addresses arrived P chunks ago) and
            // chunk q + 2P's addresses, before chunk q's store: a far address
            // names nothing newer than chunk q - 1
            load_values(q0 + s + P, t);
            load_codes(q0 + s + 2 * P, s, t);
            ring[s * 64 + static_cast<int>(lane)] = res;
            if (row_at >= 0) *reinterpret_cast<double*>(xc + static_cast<std::uint32_t>(row_at)) = res;
        }
    }
}

// The right-hand side in the wave schedule's order, [component][slot].
__global__ __launch_bounds__(256) void k_mg_wave_rhs(const double* __restrict__ rhs, double* __restrict__ out,
                                                     const std::int32_t* __restrict__ row, std::int64_t slots, int bs)
{
    const std::int64_t t = static_cast<std::int64_t>(blockIdx.x) * blockDim.x + threadIdx.x;
    if (t >= slots) return;
    const int at = row[t];
    for (int c = 0; c < bs; ++c) out[c * slots + t] = at >= 0 ? rhs[at / 8 + c] : 0.0;
}

template<class T>
void upload(DeviceArray<T>& d, const std::vector<T>& h)
{
    d.allocate(std::max<std::size_t>(h.size(), 1));
    if (!h.empty()) OWTK_HIP(hipMemcpy(d.get(), h.data(), h.size() * sizeof(T), hipMemcpyHostToDevice));
}

// inverse of a CSR-kind matrix's diagonal entries (BlockCsrMatrix::diagonal)
std::vector<double> inverse_diagonal(std::int64_t n, int bs, const std::vector<std::int32_t>& off,
                                     const std::vector<std::int32_t>& col, const std::vector<double>& val)
{
    std::vector<double> d(static_cast<std::size_t>(n) * bs, 0.0);
    for (std::int64_t r = 0; r < n; ++r)
        for (std::int32_t e = off[r]; e < off[r + 1]; ++e)
            if (col[e] == r)
                for (int c = 0; c < bs; ++c) d[r * bs + c] = val[static_cast<std::size_t>(e) * bs + c];
    for (double& v : d) {
        if (v == 0.0) throw std::runtime_error("zero diagonal in multigrid smoother");
        v = 1.0 / v;
    }
    return d;
}

// build_coloring (multigrid.hpp:345-363)
void colouring(std::int64_t n, const std::vector<std::int32_t>& off, const std::vector<std::int32_t>& col,
               std::vector<std::int32_t>& red, std::vector<std::int32_t>& black)
{
    std::vector<int> colours(n, -1);
    for (std::int64_t r = 0; r < n; ++r) {
        bool nred = false;
        for (std::int32_t e = off[r]; e < off[r + 1]; ++e) {
            const std::int64_t c = col[e];
            nred = nred || (c < n && colours[c] == 0);
        }
        colours[r] = nred ? 1 : 0;
        (colours[r] == 0 ? red : black).push_back(static_cast<std::int32_t>(r));
    }
}

// Levels of one colour's sequential sweep: a row waits for every earlier row
// of the list it reads or that reads it (in-place Gauss-Seidel order).
void gs_levels(std::int64_t n, const std::vector<std::int32_t>& off, const std::vector<std::int32_t>& col,
               const std::vector<std::int32_t>& tptr, const std::vector<std::int32_t>& tcol,
               const std::vector<std::int32_t>& list, std::vector<std::int32_t>& rows_out,
               std::vector<std::int64_t>& level_ptr)
{
    std::vector<std::int64_t> pos(n, -1);
    for (std::size_t p = 0; p < list.size(); ++p) pos[list[p]] = static_cast<std::int64_t>(p);
    std::vector<int> level(n, 0);
    int depth = 0;
    for (std::size_t p = 0; p < list.size(); ++p) {
        const std::int32_t r = list[p];
        int lv = 0;
        auto visit = [&](std::int64_t q) {
            if (q != r && q < n && pos[q] >= 0 && pos[q] < static_cast<std::int64_t>(p)) lv = std::max(lv, level[q] + 1);
        };
        for (std::int32_t e = off[r]; e < off[r + 1]; ++e) visit(col[e]);
        for (std::int32_t e = tptr[r]; e < tptr[r + 1]; ++e) visit(tcol[e]);
        level[r] = lv;
        depth = std::max(depth, lv + 1);
    }
    std::vector<std::vector<std::int32_t>> by(depth);
    for (const std::int32_t r : list) by[level[r]].push_back(r);
    for (const auto& l : by) {
        rows_out.insert(rows_out.end(), l.begin(), l.end());
        level_ptr.push_back(static_cast<std::int64_t>(rows_out.size()));
    }
}

// One-wave schedule of a colour's sequential sweep (k_mg_gs_wave): rows in
// chunks of at most 64, every row after the rows of the list before it that
// it reads or that read it, rows with the longest chain behind them first.
// Returns the chunk of each row (-1: not in the list) and the number of
// chunks; rows of chunk q are at order[chunk_ptr[q]...].
void wave_chunks(std::int64_t n, const std::vector<std::int32_t>& off, const std::vector<std::int32_t>& col,
                 const std::vector<std::int32_t>& tptr, const std::vector<std::int32_t>& tcol,
                 const std::vector<std::int32_t>& list, std::vector<std::int64_t>& chunk,
                 std::vector<std::int32_t>& order, std::vector<std::int64_t>& chunk_ptr)
{
    std::vector<std::int64_t> pos(n, -1);
    for (std::size_t p = 0; p < list.size(); ++p) pos[list[p]] = static_cast<std::int64_t>(p);
    // neighbours in the list, each once
    std::vector<std::int64_t> nptr(list.size() + 1, 0);
    std::vector<std::int32_t> nbr, tmp;
    for (std::size_t p = 0; p < list.size(); ++p) {
        const std::int32_t r = list[p];
        tmp.clear();
        auto visit = [&](std::int64_t q) {
            if (q != r && q < n && pos[q] >= 0) tmp.push_back(static_cast<std::int32_t>(pos[q]));
        };
        for (std::int32_t e = off[r]; e < off[r + 1]; ++e) visit(col[e]);
        for (std::int32_t e = tptr[r]; e < tptr[r + 1]; ++e) visit(tcol[e]);
        std::sort(tmp.begin(), tmp.end());
        tmp.erase(std::unique(tmp.begin(), tmp.end()), tmp.end());
        nbr.insert(nbr.end(), tmp.begin(), tmp.end());
        nptr[p + 1] = static_cast<std::int64_t>(nbr.size());
    }
    std::vector<int> height(list.size(), 0), waits(list.size(), 0);
    for (std::size_t p = list.size(); p-- > 0;)
        for (std::int64_t k = nptr[p]; k < nptr[p + 1]; ++k) {
            if (nbr[k] > static_cast<std::int64_t>(p)) height[p] = std::max(height[p], height[nbr[k]] + 1);
            else ++waits[p];
        }
    std::priority_queue<std::pair<int, std::int64_t>> ready;  // height, then later position first: any order is valid
    for (std::size_t p = 0; p < list.size(); ++p)
        if (waits[p] == 0) ready.push({height[p], static_cast<std::int64_t>(p)});
    chunk.assign(n, -1);
    order.clear();
    chunk_ptr.assign(1, 0);
    std::vector<std::int64_t> taken;
    while (!ready.empty()) {
        taken.clear();
        while (!ready.empty() && taken.size() < 64) {
            taken.push_back(ready.top().second);
            ready.pop();
        }
        for (const std::int64_t p : taken) {
            chunk[list[p]] = static_cast<std::int64_t>(chunk_ptr.size()) - 1;
            order.push_back(list[p]);
            for (std::int64_t k = nptr[p]; k < nptr[p + 1]; ++k)
                if (nbr[k] > p && --waits[nbr[k]] == 0) ready.push({height[nbr[k]], nbr[k]});
        }
        chunk_ptr.push_back(static_cast<std::int64_t>(order.size()));
    }
}

// Builds the one-wave schedule of the black rows when it is the faster one.
void build_wave(owtk_multigrid_s* mg, const std::vector<std::int32_t>& tptr, const std::vector<std::int32_t>& tcol,
                const std::vector<std::int32_t>& black)
{
    mg->wave_k = 0;
    const int bs = mg->bs;
    const std::int64_t nc = mg->nc;
    const auto &off = mg->h_coff, &col = mg->h_ccol;
    const std::int64_t levels = static_cast<std::int64_t>(mg->gs_level_ptr.size()) - 1 - mg->red_levels;
    int widest = 0;
    for (const std::int32_t r : black) {
        int w = 0;
        for (std::int32_t e = off[r]; e < off[r + 1]; ++e) w += col[e] != r;
        widest = std::max(widest, w);
    }
    // 32-bit byte offsets into x and the zeros behind it; at most 16 entries
    // per row beside the diagonal
    if (black.empty() || widest > 16 || (nc + 1) * bs * 8 > 0x7fffffff) return;
    std::vector<std::int64_t> chunk, chunk_ptr;
    std::vector<std::int32_t> order;
    wave_chunks(nc, off, col, tptr, tcol, black, chunk, order, chunk_ptr);
    const std::int64_t chunks = static_cast<std::int64_t>(chunk_ptr.size()) - 1;
    if (chunks > kWaveLevels * levels) return;
    const int K = widest <= 4 ? 4 : (widest <= 6 ? 6 : (widest <= 8 ? 8 : (widest <= 10 ? 10 : (widest <= 12 ? 12 : 16))));
    // idle chunks behind the last one: the kernel runs whole groups of
    // 2 kWaveAhead chunks and loads as far ahead
    const std::int64_t total = (chunks + 2 * kWaveAhead - 1) / (2 * kWaveAhead) * (2 * kWaveAhead) + 2 * kWaveAhead;
    const std::int64_t slots = total * 64;
    std::vector<std::int32_t> row(slots, -1), near(static_cast<std::size_t>(slots) * K, kWaveZero);
    std::vector<std::int32_t> far(static_cast<std::size_t>(slots) * K, static_cast<std::int32_t>(nc * bs * 8));
    std::vector<double> val(static_cast<std::size_t>(slots) * K * bs, 0.0), diag(static_cast<std::size_t>(slots) * 2 * bs, 1.0);
    std::vector<int> lane(nc, 0);
    for (std::int64_t q = 0; q < chunks; ++q)
        for (std::int64_t p = chunk_ptr[q]; p < chunk_ptr[q + 1]; ++p) lane[order[p]] = static_cast<int>(p - chunk_ptr[q]);
    for (std::int64_t q = 0; q < chunks; ++q) {
        for (std::int64_t p = chunk_ptr[q]; p < chunk_ptr[q + 1]; ++p) {
            const std::int32_t r = order[p];
            const std::int64_t slot = q * 64 + lane[r];
            row[slot] = static_cast<std::int32_t>(static_cast<std::int64_t>(r) * bs * 8);
            int k = 0;
            for (std::int32_t e = off[r]; e < off[r + 1]; ++e) {
                const std::int32_t j = col[e];
                if (j == r) {
                    for (int c = 0; c < bs; ++c) {
                        const double d = mg->h_cval[static_cast<std::size_t>(e) * bs + c];
                        diag[static_cast<std::size_t>(c * slots + slot) * 2] = d;
                        diag[static_cast<std::size_t>(c * slots + slot) * 2 + 1] = 1.0 / d;
                    }
                    continue;
                }
                const std::int64_t pair = (q * (K / 2) + k / 2) * 64 + lane[r];
                const std::int64_t from = chunk[j];
                const std::size_t at = static_cast<std::size_t>(pair) * 2 + k % 2;
                if (from >= 0 && from < q && q - from <= kWaveAhead)
                    near[at] = static_cast<std::int32_t>(((from % kWaveRing) * 64 + lane[j]) * 8);
                else
                    far[at] = static_cast<std::int32_t>(static_cast<std::int64_t>(j) * bs * 8);
                for (int c = 0; c < bs; ++c)
                    val[static_cast<std::size_t>(c * slots * (K / 2) + pair) * 2 + k % 2] = mg->h_cval[static_cast<std::size_t>(e) * bs + c];
                ++k;
            }
        }
    }
    upload(mg->wave_row, row);
    upload(mg->wave_near, near);
    upload(mg->wave_far, far);
    upload(mg->wave_val, val);
    upload(mg->wave_diag, diag);
    mg->wave_chunks = chunks;
    mg->wave_slots = slots;
    mg->wave_k = K;
}

void mg_setup(owtk_multigrid_s* mg)
{
    owtk_matrix m = mg->fine;
    const auto& o = mg->opt;
    const int bs = m->bs;
    const std::int64_t n = m->owned;
    mg->bs = bs;
    mg->n = n;
    // fine values on the host, [entry][comp] (the reference's BlockCsrMatrix layout)
    std::vector<double> slots(static_cast<std::size_t>(m->value_count));
    OWTK_HIP(hipMemcpy(slots.data(), m->v64.get(), slots.size() * sizeof(double), hipMemcpyDeviceToHost));
    const auto& off = m->h_offsets;
    const auto& col = m->h_columns;
    std::vector<double> val(static_cast<std::size_t>(off[n]) * bs);
    for (std::int64_t e = 0; e < off[n]; ++e)
        for (int c = 0; c < bs; ++c) val[e * bs + c] = slots[m->value_index(m->s.slot_of_entry[e], c)];
    // build_aggregates (multigrid.hpp:237-262)
    constexpr std::int64_t none = -1;
    std::vector<std::int64_t> f2c(n, none), sizes;
    for (std::int64_t seed = 0; seed < n; ++seed) {
        if (f2c[seed] != none) continue;
        const std::int64_t agg = static_cast<std::int64_t>(sizes.size());
        std::int64_t size = 1;
        f2c[seed] = agg;
        for (std::int32_t e = off[seed]; e < off[seed + 1] && static_cast<std::uint64_t>(size) < o.target_aggregate_size;
             ++e) {
            const std::int64_t nb = col[e];
            if (nb < n && f2c[nb] == none) {
                f2c[nb] = agg;
                ++size;
            }
        }
        sizes.push_back(size);
    }
    const std::int64_t nc = static_cast<std::int64_t>(sizes.size());
    mg->nc = nc;
    // build_coarse_matrix (multigrid.hpp:264-305)
    std::vector<std::map<std::int64_t, std::vector<double>>> rows(nc);
    for (std::int64_t r = 0; r < n; ++r) {
        const std::int64_t cr = f2c[r];
        for (std::int32_t e = off[r]; e < off[r + 1]; ++e) {
            const std::int64_t fc = col[e];
            if (fc >= n) continue;
            auto [pos, inserted] = rows[cr].try_emplace(f2c[fc], bs, 0.0);
            for (int c = 0; c < bs; ++c) pos->second[c] += val[static_cast<std::size_t>(e) * bs + c] / static_cast<double>(sizes[cr]);
        }
    }
    mg->h_coff.assign(nc + 1, 0);
    mg->h_ccol.clear();
    mg->h_cval.clear();
    for (std::int64_t r = 0; r < nc; ++r) {
        for (const auto& [c, block] : rows[r]) {
            mg->h_ccol.push_back(static_cast<std::int32_t>(c));
            mg->h_cval.insert(mg->h_cval.end(), block.begin(), block.end());
        }
        mg->h_coff[r + 1] = static_cast<std::int32_t>(mg->h_ccol.size());
    }
    mg->h_f2c = f2c;
    const int rc = owtk_matrix_create_csr(m->ctx, nc, 0, bs, mg->h_coff.data(), mg->h_ccol.data(), mg->h_cval.data(),
                                          &mg->coarse);
    if (rc != OWTK_OK) throw std::runtime_error(std::string("coarse matrix: ") + owtk_last_error());
    upload(mg->fine_inv, inverse_diagonal(n, bs, off, col, val));
    upload(mg->coarse_inv, inverse_diagonal(nc, bs, mg->h_coff, mg->h_ccol, mg->h_cval));
    // aggregate members in ascending order, sizes, fine -> coarse
    std::vector<std::int32_t> aptr(nc + 1, 0), members(n), f2c32(n);
    for (std::int64_t r = 0; r < n; ++r) {
        ++aptr[f2c[r] + 1];
        f2c32[r] = static_cast<std::int32_t>(f2c[r]);
    }
    for (std::int64_t a = 0; a < nc; ++a) aptr[a + 1] += aptr[a];
    {
        std::vector<std::int32_t> next(aptr.begin(), aptr.end() - 1);
        for (std::int64_t r = 0; r < n; ++r) members[next[f2c[r]]++] = static_cast<std::int32_t>(r);
    }
    std::vector<double> sz(sizes.begin(), sizes.end());
    upload(mg->agg_ptr, aptr);
    upload(mg->agg_members, members);
    upload(mg->agg_size, sz);
    upload(mg->f2c, f2c32);
    std::vector<std::int32_t> red, black;
    colouring(n, off, col, red, black);
    mg->n_red = static_cast<std::int64_t>(red.size());
    mg->n_black = static_cast<std::int64_t>(black.size());
    upload(mg->fine_red, red);
    upload(mg->fine_black, black);
    // coarse Gauss-Seidel: level schedules
    std::vector<std::int32_t> cred, cblack;
    colouring(nc, mg->h_coff, mg->h_ccol, cred, cblack);
    std::vector<std::int32_t> tptr(nc + 1, 0), tcol(mg->h_ccol.size());
    for (const std::int32_t c : mg->h_ccol) ++tptr[c + 1];
    for (std::int64_t a = 0; a < nc; ++a) tptr[a + 1] += tptr[a];
    {
        std::vector<std::int32_t> next(tptr.begin(), tptr.end() - 1);
        for (std::int64_t r = 0; r < nc; ++r)
            for (std::int32_t e = mg->h_coff[r]; e < mg->h_coff[r + 1]; ++e)
                tcol[next[mg->h_ccol[e]]++] = static_cast<std::int32_t>(r);
    }
    std::vector<std::int32_t> gs_rows;
    mg->gs_level_ptr.assign(1, 0);
    gs_levels(nc, mg->h_coff, mg->h_ccol, tptr, tcol, cred, gs_rows, mg->gs_level_ptr);
    mg->red_levels = static_cast<std::int64_t>(mg->gs_level_ptr.size()) - 1;
    gs_levels(nc, mg->h_coff, mg->h_ccol, tptr, tcol, cblack, gs_rows, mg->gs_level_ptr);
    upload(mg->gs_rows, gs_rows);
    upload(mg->gs_levels, mg->gs_level_ptr);
    if (mg->opt.smoother == OWTK_MG_RED_BLACK) build_wave(mg, tptr, tcol, cblack);
    // level-ordered ELL copy of the coarse rows for the sweep kernel (the red
    // rows alone where the one-wave sweep takes the black ones)
    if (mg->wave_k) gs_rows.resize(static_cast<std::size_t>(mg->gs_level_ptr[mg->red_levels]));
    const std::int64_t P = static_cast<std::int64_t>(gs_rows.size());
    int K = 0;
    for (const std::int32_t r : gs_rows) {
        int off = 0;
        for (std::int32_t e = mg->h_coff[r]; e < mg->h_coff[r + 1]; ++e) off += mg->h_ccol[e] != r;
        K = std::max(K, off);
    }
    std::vector<std::int32_t> glen(static_cast<std::size_t>(std::max<std::int64_t>(P, 1)), 0);
    std::vector<std::int32_t> gcol(static_cast<std::size_t>(std::max<std::int64_t>(P * K, 1)), 0);
    std::vector<double> gval(static_cast<std::size_t>(std::max<std::int64_t>(P * K * bs, 1)), 0.0);
    std::vector<double> gdiag(static_cast<std::size_t>(std::max<std::int64_t>(P * bs, 1)), 0.0);
    for (std::int64_t p = 0; p < P; ++p) {
        const std::int32_t r = gs_rows[p];
        int k = 0;
        for (int q = 0; q < K; ++q) gcol[static_cast<std::size_t>(q * P + p)] = r;
        for (std::int32_t e = mg->h_coff[r]; e < mg->h_coff[r + 1]; ++e) {
            const std::int32_t c = mg->h_ccol[e];
            if (c == r) {
                for (int j = 0; j < bs; ++j) gdiag[static_cast<std::size_t>(p * bs + j)] = mg->h_cval[static_cast<std::size_t>(e) * bs + j];
                continue;
            }
            gcol[static_cast<std::size_t>(k * P + p)] = c;
            for (int j = 0; j < bs; ++j)
                gval[static_cast<std::size_t>((k * P + p) * bs + j)] = mg->h_cval[static_cast<std::size_t>(e) * bs + j];
            ++k;
        }
        glen[static_cast<std::size_t>(p)] = k;
    }
    mg->gs_positions = P;
    mg->gs_k = K;
    upload(mg->gs_len, glen);
    upload(mg->gs_col, gcol);
    upload(mg->gs_val, gval);
    upload(mg->gs_diag, gdiag);
}

double smoother_weight(const owtk_multigrid_options& o, std::uint64_t step)
{
    if (o.smoother != OWTK_MG_CHEBYSHEV) return o.jacobi_weight;
    const std::uint64_t levels = std::max<std::uint64_t>(1, o.chebyshev_levels);
    const double pi = std::acos(-1.0);
    const double rho = 0.99;
    const double angle = pi * static_cast<double>(2 * (step % levels) + 1) / static_cast<double>(2 * levels);
    const double cs = std::cos(angle);
    return 2.0 / (1.0 + std::sqrt(1.0 - rho * rho * cs * cs));
}

void launch_wave(owtk_multigrid_s* mg, const double* rhs, double* x, hipStream_t st)
{
    const GsWaveArgs a{mg->wave_row.get(), mg->wave_near.get(), mg->wave_far.get(), mg->wave_val.get(), mg->wave_diag.get(), rhs,
                       mg->wave_chunks, mg->wave_slots};
    const unsigned int g = static_cast<unsigned int>(mg->bs);
    switch (mg->wave_k) {
    case 4: k_mg_gs_wave<4><<<g, 64, 0, st>>>(a, x); break;
    case 6: k_mg_gs_wave<6><<<g, 64, 0, st>>>(a, x); break;
    case 8: k_mg_gs_wave<8><<<g, 64, 0, st>>>(a, x); break;
    case 10: k_mg_gs_wave<10><<<g, 64, 0, st>>>(a, x); break;
    case 12: k_mg_gs_wave<12><<<g, 64, 0, st>>>(a, x); break;
    default: k_mg_gs_wave<16><<<g, 64, 0, st>>>(a, x); break;
    }
}

int mg_solve(owtk_multigrid_s* mg, const double* b, double* x, const owtk_solver_options* o, int cycle,
             owtk_solver_result* res)
{
    const auto t0 = std::chrono::steady_clock::now();
    init_result(res);
    if (!valid_options(o)) return OWTK_OK;
    if (cycle < OWTK_MG_V || cycle > OWTK_MG_FULL) throw std::invalid_argument("unknown multigrid cycle");
    owtk_matrix m = mg->fine;
    owtk_context ctx = m->ctx;
    const hipStream_t st = ctx->stream;
    const auto scratch = ctx->scratch();
    const int bs = mg->bs;
    const std::int64_t n = mg->n * bs, nc = mg->nc * bs;
    const std::int64_t L = m->local() * bs;
    DeviceArray<double> vecs;
    const std::int64_t wave_rhs = mg->wave_k ? mg->wave_slots * bs : 0;
    // (bs zeros stay behind the coarse solution: the wave sweep's far zeros)
    vecs.allocate(static_cast<std::size_t>(2 * L + 3 * nc + bs + wave_rhs));
    kern::fill_zero_bytes(st, vecs.get(), vecs.bytes());
    double* residual = vecs.get();
    double* work = residual + L;
    double* crhs = work + L;
    double* csol = crhs + nc;
    double* capplied = csol + nc + bs;
    double* wrhs = capplied + nc;  // the coarse right-hand side in the wave schedule's order
    double* d_norm = ctx->scalars.get();
    std::uint64_t ops = 0, reds = 0;
    const auto& opt = mg->opt;
    auto grid = [](std::int64_t k) { return dev::stream_grid(std::max<std::int64_t>(k, 1), 4); };
    auto read_norm = [&] {
        double v;
        OWTK_HIP(hipMemcpyAsync(&v, d_norm, sizeof(double), hipMemcpyDeviceToHost, st));
        ctx->sync();
        return v;
    };
    auto finish = [&](int status) {
        res->status = status;
        res->operator_applications = ops;
        res->global_reductions = reds;
        if (o->collect_timings)
            res->solve_seconds = std::chrono::duration<double>(std::chrono::steady_clock::now() - t0).count();
        return OWTK_OK;
    };
    auto fine_op = [&](const double* in, double* out) {
        dev::EpiStore<double> e;
        e.y = out;
        spmv_f64(m, in, e);
        ++ops;
    };
    // true_residual (one operator application); with_norm adds detail::norm
    auto true_residual = [&](bool with_norm) {
        dev::EpiResidual e;
        e.y = residual;
        e.b = b;
        e.n = n;
        e.norm_out = with_norm ? d_norm : nullptr;
        spmv_f64(m, x, e);
        ++ops;
        if (!with_norm) return 0.0;
        ++reds;
        return read_norm();
    };
    auto smooth_fine = [&](std::uint64_t steps) {
        for (std::uint64_t s = 0; s < steps; ++s) {
            if (opt.smoother == OWTK_MG_RED_BLACK) {
                fine_op(x, work);
                k_mg_colour<<<grid(mg->n_red * bs), kBlock, 0, st>>>(mg->fine_red.get(), mg->n_red, bs, x, b, work,
                                                                      mg->fine_inv.get());
                fine_op(x, work);
                k_mg_colour<<<grid(mg->n_black * bs), kBlock, 0, st>>>(mg->fine_black.get(), mg->n_black, bs, x, b,
                                                                        work, mg->fine_inv.get());
            } else {
                fine_op(x, work);
                k_mg_jacobi<<<grid(n), kBlock, 0, st>>>(x, b, work, mg->fine_inv.get(), smoother_weight(opt, s), n);
            }
            OWTK_LAUNCH_CHECK();
        }
    };
    // smooth (multigrid.hpp:307-331) on the coarse level; its matrix applies are not counted
    auto smooth_coarse = [&](std::uint64_t steps) {
        for (std::uint64_t s = 0; s < steps; ++s) {
            if (opt.smoother == OWTK_MG_RED_BLACK) {
                // red levels, then black levels (red rows read the previous black values)
                const std::int64_t levels = static_cast<std::int64_t>(mg->gs_level_ptr.size()) - 1;
                const GsArgs ga{mg->gs_rows.get(), mg->gs_len.get(), mg->gs_col.get(), mg->gs_val.get(),
                                mg->gs_diag.get(), crhs, mg->gs_positions, bs, mg->gs_k};
                const std::int64_t n_red = mg->gs_level_ptr[mg->red_levels];
                if (mg->red_levels == 1)
                    k_mg_gs_level<<<static_cast<unsigned int>((n_red * bs + kBlock - 1) / kBlock), kBlock, 0, st>>>(n_red, ga, csol);
                else
                    k_mg_gs_ell<<<1, 1024, 0, st>>>(mg->gs_levels.get(), 0, mg->red_levels, ga, csol);
                if (mg->wave_k)
                    launch_wave(mg, wrhs, csol, st);
                else
                    k_mg_gs_ell<<<1, 1024, 0, st>>>(mg->gs_levels.get(), mg->red_levels, levels, ga, csol);
            } else {
                dev::EpiStore<double> e;
                e.y = capplied;
                spmv_f64(mg->coarse, csol, e);
                const double w = opt.smoother == OWTK_MG_CHEBYSHEV ? smoother_weight(opt, s) : opt.jacobi_weight;
                k_mg_jacobi<<<grid(nc), kBlock, 0, st>>>(csol, crhs, capplied, mg->coarse_inv.get(), w, nc);
            }
            OWTK_LAUNCH_CHECK();
        }
    };
    auto coarse_correction = [&](const double* fine_rhs, bool zero_x) {
        k_mg_restrict<<<grid(nc), kBlock, 0, st>>>(fine_rhs, crhs, mg->agg_ptr.get(), mg->agg_members.get(),
                                                   mg->agg_size.get(), mg->nc, bs);
        kern::fill_zero_bytes(st, csol, nc * sizeof(double));
        if (mg->wave_k)
            k_mg_wave_rhs<<<static_cast<unsigned int>((mg->wave_slots + kBlock - 1) / kBlock), kBlock, 0, st>>>(
                crhs, wrhs, mg->wave_row.get(), mg->wave_slots, bs);
        OWTK_LAUNCH_CHECK();
        smooth_coarse(opt.coarse_smoothing_steps);
        if (zero_x) kern::fill_zero_bytes(st, x, n * sizeof(double));
        k_mg_prolong<<<grid(n), kBlock, 0, st>>>(csol, x, mg->f2c.get(), mg->n, bs);
        OWTK_LAUNCH_CHECK();
    };

    kern::norm_to(st, ctx->fused_scratch(), b, n, d_norm);
    ++reds;
    const double rhs_norm = read_norm();
    if (!std::isfinite(rhs_norm)) {
        res->breakdown_reason = reason_non_finite_scalar;
        return finish(status_breakdown);
    }
    const double thr = threshold_of(rhs_norm, o);
    double nv = true_residual(true);
    res->initial_residual_norm = nv;
    set_residual(res, nv, nv, rhs_norm);
    if (!std::isfinite(nv)) {
        res->breakdown_reason = reason_non_finite_scalar;
        return finish(status_breakdown);
    }
    if (nv <= thr) return finish(status_converged);
    if (cycle == OWTK_MG_FULL) coarse_correction(b, true);
    for (std::uint64_t it = 1; it <= o->maximum_iterations; ++it) {
        res->iterations = it;
        smooth_fine(opt.pre_smoothing_steps);
        const int corrections = cycle == OWTK_MG_W ? 2 : 1;
        for (int k = 0; k < corrections; ++k) {
            true_residual(false);
            coarse_correction(residual, false);
        }
        smooth_fine(opt.post_smoothing_steps);
        nv = true_residual(true);
        set_residual(res, nv, nv, rhs_norm);
        if (!std::isfinite(nv)) {
            res->breakdown_reason = reason_non_finite_scalar;
            return finish(status_breakdown);
        }
        if (nv <= thr) return finish(status_converged);
    }
    return finish(status_maximum_iterations);
}

} // namespace
} // namespace owtk

extern "C" {

void owtk_multigrid_options_default(owtk_multigrid_options* o)
{
    if (!o) return;
    o->pre_smoothing_steps = 2;
    o->post_smoothing_steps = 2;
    o->coarse_smoothing_steps = 24;
    o->target_aggregate_size = 4;
    o->jacobi_weight = 0.8;
    o->smoother = OWTK_MG_JACOBI;
    o->chebyshev_levels = 8;
}

int owtk_multigrid_create(owtk_matrix fine, const owtk_multigrid_options* options, owtk_multigrid* out)
{
    return guarded([&] {
        if (!fine || !options || !out) throw std::invalid_argument("null argument");
        *out = nullptr;
        if (fine->kind != OWTK_MATRIX_CSR)
            throw std::invalid_argument("multigrid needs a component-diagonal BlockCsrMatrix (CSR kind)");
        if (options->target_aggregate_size == 0) throw std::invalid_argument("multigrid aggregate size must be positive");
        if (options->smoother < OWTK_MG_JACOBI || options->smoother > OWTK_MG_CHEBYSHEV)
            throw std::invalid_argument("unknown multigrid smoother");
        fine->ctx->activate();
        auto mg = std::make_unique<owtk_multigrid_s>();
        mg->fine = fine;
        mg->ctx = fine->ctx;
        mg->opt = *options;
        mg_setup(mg.get());
        *out = mg.release();
    });
}

int owtk_multigrid_destroy(owtk_multigrid mg)
{
    return guarded([&] {
        if (!mg) return;
        mg->ctx->activate();
        mg->ctx->sync();
        delete mg;
    });
}

int owtk_multigrid_coarse(owtk_multigrid mg, int64_t* nodes, int64_t* entries, int32_t* row_offsets,
                          int32_t* columns, double* values, int64_t* fine_to_coarse)
{
    return guarded([&] {
        if (!mg || !nodes || !entries) throw std::invalid_argument("null argument");
        *nodes = mg->nc;
        *entries = static_cast<int64_t>(mg->h_ccol.size());
        if (row_offsets) std::copy(mg->h_coff.begin(), mg->h_coff.end(), row_offsets);
        if (columns) std::copy(mg->h_ccol.begin(), mg->h_ccol.end(), columns);
        if (values) std::copy(mg->h_cval.begin(), mg->h_cval.end(), values);
        if (fine_to_coarse) std::copy(mg->h_f2c.begin(), mg->h_f2c.end(), fine_to_coarse);
    });
}

int owtk_multigrid_solve(owtk_multigrid mg, const double* b, double* x, const owtk_solver_options* options,
                         int32_t cycle, owtk_solver_result* result)
{
    return guarded([&] {
        if (!mg || !b || !x || !options || !result) throw std::invalid_argument("null argument");
        require_plain_options(options, "multigrid");
        mg->fine->ctx->activate();
        mg_solve(mg, b, x, options, cycle, result);
    });
}

} // extern "C"
