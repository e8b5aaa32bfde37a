// Batched dense LU factorisation and solve for the implicit radial step.
//
// Implicit_Solve (Linear_Solve.F90:423-457) factors each mode's n x n matrix once per time
// step size (LU_Decompose_full = LAPACK dgetrf, :1034-1045) and every step solves it for
// the right-hand sides of all m of that l (LU_Solve_full = dgetrs 'N', :1087-1107).  Here
// many matrices go in one launch, one workgroup per matrix (factorisation) or per
// matrix and chunk of its right-hand sides (solve).
//
// Factorisation: the right-looking algorithm of dgetf2 -- pivot = first row of largest
// |a_ik|, row swap, subdiagonal scaled by the pivot's reciprocal, rank-1 update of the
// trailing block -- with products and sums rounded separately, in panels.
// Solve: the row interchanges, the unit lower and the upper triangular solves in the
// column order of the reference BLAS dtrsm (column j final, then subtracted from the rows
// below / above it).
#include <algorithm>
#include <cmath>
#include <type_traits>

#include "raysht_internal.h"

namespace raysht {
namespace {

constexpr int kLuThreads = 256;
constexpr int kLuMaxN = 1024;

// Workgroup order of the solves.  Workgroups go to the 8 XCDs round-robin by linear id, so
// XCD k runs ids k, k + 8, k + 16, ...; its r-th workgroup takes column block r % ncb of
// matrix 8 (r / ncb) + k.  Each XCD then works through its own matrices (every eighth)
// one at a time, all column blocks of a matrix together, and the factor they share stays
// in that XCD's L2 instead of every XCD streaming every matrix from the last-level cache.
// The grid is ncb * (nbatch rounded up to 8) workgroups; ids past nbatch leave at once.
// Ungrouped (grouped = 0), matrix b runs as workgroups b, b + nbatch, ...: for small
// factors (dense n <= 256, 0.5 MB) measured faster, as the cache lines the waves read at
// one step spread over many matrices.
struct solve_block {
    int b, cb;
};
__device__ __forceinline__ solve_block solve_block_of(int ncb, int nbatch, int grouped)
{
    if (!grouped) return solve_block{(int)(blockIdx.x % (unsigned)nbatch), (int)(blockIdx.x / (unsigned)nbatch)};
    const int r = (int)(blockIdx.x >> 3);
    return solve_block{8 * (r / ncb) + (int)(blockIdx.x & 7), r % ncb};
}
inline long solve_grid(int ncb, int nbatch, int grouped)
{
    return (long)ncb * (grouped ? (nbatch + 7L) / 8 * 8 : (long)nbatch);
}
// a launch stays below 2^32 threads in all
inline bool solve_grid_fits(int ncb, int nbatch, int grouped, int threads)
{
    return solve_grid(ncb, nbatch, grouped) * threads < (1L << 32);
}

// Factorisation, one workgroup per matrix, panels of kLuNB columns.  A thread owns one row of
// the panel and holds its kLuNB values in registers for all of the panel's column steps.  An
// interchange moves nothing: a thread keeps the position its row stands at, and only these
// change.  Per step each wave finds its candidate (largest |a|, lowest position among equals;
// DPP lane moves) and leaves the whole candidate row in LDS, so after one barrier every
// thread knows the pivot and has its row, scales its own value and updates its own row.  Then
// the rows go back to memory at their positions, the rest of the matrix takes the panel's
// interchanges (a wave per column, at most 32 rows move), U12 is formed by a thread per
// column and the trailing block by register tiles that apply the panel's updates
// k = k0 .. k0 + kLuNB - 1 one after the other.  Products and sums are rounded separately and a
// zero u_kj skipped (dger), so every element sees the operations of dgetf2 in its order and
// the factors are its doubles.
// What it waits for is the column steps (a chain of a reduction, a barrier, LDS reads and a
// reciprocal, about a third of n = 256), then the passes over the trailing block, which the
// caches and FP64 vector arithmetic share (matrix instructions would fuse the product into the
// sum).  256 matrices of n = 64, 128, 256: 0.13, 0.33, 0.87 ms; 128 of n = 512: 3.3 ms, 32 of
// n = 1000: 19 ms.  Steps that go through global memory (the search, the interchange of the
// whole row, the update of the panel) took 0.31, 0.67, 2.39, 9.1 and 45 ms.  Panels of 32 need a
// step code of 137 KB, more than the instruction cache, and were slower at every n.
constexpr int kLuNB = 16;
constexpr int kLuChunk = 256;  // rows of L21 and columns of U12 in LDS at a time

// the largest m of the wave (no NaN), in every lane
__device__ __forceinline__ double lu_wave_max(double m)
{
    auto step = [&](auto ctrl) {
        constexpr int C = decltype(ctrl)::value;
        const long b = __builtin_bit_cast(long, m);
        const int lo = __builtin_amdgcn_update_dpp((int)b, (int)b, C, 0xf, 0xf, false);
        const int hi = __builtin_amdgcn_update_dpp((int)(b >> 32), (int)(b >> 32), C, 0xf, 0xf, false);
        m = fmax(m, __builtin_bit_cast(double, ((long)hi << 32) | (unsigned)lo));
    };
    step(std::integral_constant<int, 0x111>{});  // row_shr 1, 2, 4, 8: lane 15 of a row has its row's
    step(std::integral_constant<int, 0x112>{});
    step(std::integral_constant<int, 0x114>{});
    step(std::integral_constant<int, 0x118>{});
    step(std::integral_constant<int, 0x142>{});  // row_bcast 15, 31: lane 63 has the wave's
    step(std::integral_constant<int, 0x143>{});
    const long b = __builtin_bit_cast(long, m);
    const int lo = __builtin_amdgcn_readlane((int)b, 63), hi = __builtin_amdgcn_readlane((int)(b >> 32), 63);
    return __builtin_bit_cast(double, ((long)hi << 32) | (unsigned)lo);
}

// f(0), f(1), ... with compile-time arguments: register arrays are indexed by constants however
// long the unrolled code is
template <int I, int N, typename F>
__device__ __forceinline__ void static_steps(F &&f)
{
    if constexpr (I < N) {
        f(std::integral_constant<int, I>{});
        static_steps<I + 1, N>(f);
    }
}

// the same until f returns false
template <int I, int N, typename F>
__device__ __forceinline__ void static_while(F &&f)
{
    if constexpr (I < N) {
        if (!f(std::integral_constant<int, I>{})) return;
        static_while<I + 1, N>(f);
    }
}

// LDS of one workgroup: two sets of candidate rows, L11, the moves, U12 and L21 chunks
__host__ __device__ inline int lu_chunk(int n) { return n < kLuChunk ? n : kLuChunk; }
__host__ __device__ inline int lu_ld(int n) { return lu_chunk(n) | 1; }
template <int NT>
size_t lu_lds_bytes(int n)
{
    constexpr int W = NT / 64;
    return sizeof(double) * (2 * W * (kLuNB + 1) + kLuNB * (kLuNB + 2) + 2 * kLuNB * (size_t)lu_ld(n)) +
           sizeof(int) * (2 * W + 2 * 64 + 2);
}

template <int NT>
__global__ __launch_bounds__(NT) void lu_decompose_kernel(int n, double *__restrict__ mats, int *__restrict__ pivots,
                                                          int *__restrict__ infos)
{
#pragma clang fp contract(off)
    constexpr int W = NT / 64, J = NT > 512 ? 4 : 8;
    extern __shared__ double lu_lds[];
    const int ld = lu_ld(n), chunk = lu_chunk(n);
    double *s_row = lu_lds;                              // [2][W][kLuNB] candidate rows
    double *s_val = s_row + 2 * W * kLuNB;               // [2][W] their |a|
    double *s_l11 = s_val + 2 * W;                       // [k][row], rows kLuNB + 2 apart
    double *s_u = s_l11 + kLuNB * (kLuNB + 2);           // [k][column]
    double *s_l = s_u + kLuNB * ld;                      // [k][row]
    int *s_pos = reinterpret_cast<int *>(s_l + kLuNB * ld);  // [2][W] the candidates' positions
    int *s_src = s_pos + 2 * W, *s_dst = s_src + 64, *s_cnt = s_dst + 64, *s_zero = s_cnt + 1;
    double *a = mats + (long)blockIdx.x * n * n;
    int *piv = pivots + (long)blockIdx.x * n;
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    const double sfmin = 2.2250738585072014e-308;
    constexpr int kNone = 1 << 30;
    int info = 0;
    for (int k0 = 0; k0 < n; k0 += kLuNB) {
        const int nb = min(kLuNB, n - k0), kend = k0 + nb, row = k0 + tid;
        // ---- the panel
        double v[kLuNB];
#pragma unroll
        for (int j = 0; j < kLuNB; ++j) v[j] = row < n && j < nb ? a[row + (long)(k0 + j) * n] : 0.0;
        int pos = row < n ? row : -1;
        if (tid == 0) *s_cnt = 0;
        static_steps<0, kLuNB>([&](auto step) {
            constexpr int kk = decltype(step)::value, par = kk & 1;
            if (kk >= nb) return;
            const int k = k0 + kk;
            // idamax: NaNs below the diagonal are passed over, a NaN a_kk is kept (it beats
            // everything, an infinity by its lower key)
            const double x = v[kk];
            const bool in = pos >= k, nan = isnan(x);
            const double m = !in || (nan && pos != k) ? -1.0 : nan ? HUGE_VAL : fabs(x);
            const int key = !in || (nan && pos != k) ? kNone : nan ? -1 : pos;
            const double wm = lu_wave_max(m);
            unsigned long long eq = __ballot(m == wm);
            int bl = __builtin_ctzll(eq);
            if (wm >= 0.0)  // below: no row of this wave is a candidate
                for (eq &= eq - 1; eq != 0; eq &= eq - 1) {  // equal candidates: the lowest position
                    const int l2 = __builtin_ctzll(eq);
                    if (__builtin_amdgcn_readlane(key, l2) < __builtin_amdgcn_readlane(key, bl)) bl = l2;
                }
            if (lane == bl) {
                double *r = s_row + (par * W + wave) * kLuNB;
#pragma unroll
                for (int j = kk; j < kLuNB; ++j) r[j] = v[j];
                s_val[par * W + wave] = m;
                s_pos[par * W + wave] = key;
            }
            __syncthreads();  // the other set of rows was read before the previous step's barrier
            int bw = 0, bk = s_pos[par * W];
            double bv = s_val[par * W];
#pragma unroll
            for (int w = 1; w < W; ++w) {
                const double ov = s_val[par * W + w];
                const int ok = s_pos[par * W + w];
                if (ov > bv || (ov == bv && ok < bk)) {
                    bv = ov;
                    bk = ok;
                    bw = w;
                }
            }
            const int p = bk < 0 || bk == kNone ? k : bk;
            const double *r = s_row + (par * W + __builtin_amdgcn_readfirstlane(bw)) * kLuNB;
            const double pv = r[kk];
            if (tid == 0) piv[k] = p + 1;
            if (pv != 0.0) {
                pos = pos == p ? k : pos == k ? p : pos;
            } else if (info == 0) {
                info = k + 1;
            }
            if (pos > k) {
                double lik = x;
                if (pv != 0.0) lik = fabs(pv) >= sfmin ? x * (1.0 / pv) : x / pv;
                v[kk] = lik;
#pragma unroll
                for (int j = kk + 1; j < kLuNB; ++j) {
                    const double y = r[j], upd = v[j] + lik * -y;
                    v[j] = y != 0.0 ? upd : v[j];
                }
            }
        });
        // ---- back to memory at the rows' positions; L11 and the moves to LDS
        if (row < n) {
#pragma unroll
            for (int j = 0; j < kLuNB; ++j)
                if (j < nb) a[pos + (long)(k0 + j) * n] = v[j];
            if (pos < kend) {
#pragma unroll
                for (int j = 0; j < kLuNB; ++j) s_l11[j * (kLuNB + 2) + pos - k0] = v[j];
            }
            if (pos != row) {
                const int at = atomicAdd(s_cnt, 1);  // a step moves at most two rows: at most 32
                s_src[at] = row;
                s_dst[at] = pos;
            }
        }
        __syncthreads();
        // ---- the interchanges in the other columns, a wave per column, eight in flight
        const int cnt = *s_cnt, others = n - nb;
        if (cnt > 0) {
            const int src = lane < cnt ? s_src[lane] : 0, dst = lane < cnt ? s_dst[lane] : 0;
            constexpr int U = 8;
            for (int q0 = wave; q0 < others; q0 += U * W) {
                double t[U];
#pragma unroll
                for (int u = 0; u < U; ++u) {
                    const int q = q0 + u * W, col = q < k0 ? q : q + nb;
                    t[u] = q < others && lane < cnt ? a[src + (long)col * n] : 0.0;
                }
#pragma unroll
                for (int u = 0; u < U; ++u) {
                    const int q = q0 + u * W, col = q < k0 ? q : q + nb;
                    if (q < others && lane < cnt) a[dst + (long)col * n] = t[u];
                }
            }
        }
        if (kend >= n) break;  // nb = kLuNB from here on
        for (int c0 = kend; c0 < n; c0 += chunk) {
            const int nc = min(chunk, n - c0);
            __syncthreads();
            // ---- U12 of this chunk: rows k0 .. k0 + kLuNB - 1, a thread per column
            for (int e = tid; e < kLuNB * nc; e += NT) {
                const int i = e % kLuNB, c = e / kLuNB;
                s_u[i * ld + c] = a[k0 + i + (long)(c0 + c) * n];
            }
            if (tid == 0) *s_zero = 0;
            __syncthreads();
            for (int c = tid; c < nc; c += NT) {
                double u[kLuNB];
                bool zero = false;
#pragma unroll
                for (int i = 0; i < kLuNB; ++i) u[i] = s_u[i * ld + c];
                static_steps<0, kLuNB>([&](auto step) {
                    constexpr int kk = decltype(step)::value;
                    const double y = u[kk];
                    zero |= y == 0.0;
#pragma unroll
                    for (int i = kk + 1; i < kLuNB; ++i) {
                        const double upd = u[i] + s_l11[kk * (kLuNB + 2) + i] * -y;
                        u[i] = y != 0.0 ? upd : u[i];
                    }
                });
#pragma unroll
                for (int i = 0; i < kLuNB; ++i) s_u[i * ld + c] = u[i];
                if (zero) *s_zero = 1;
            }
            __syncthreads();
            for (int e = tid; e < kLuNB * nc; e += NT) {
                const int i = e % kLuNB, c = e / kLuNB;
                a[k0 + i + (long)(c0 + c) * n] = s_u[i * ld + c];
            }
            // ---- the trailing block: a wave per tile of 64 rows x 4 J columns, lane (li, lg) on rows
            // li + 16 i and columns lg + 4 j (J = 8; 4 where 16 waves leave a thread 128 registers)
            const bool any_zero = *s_zero != 0;
            for (int r0 = kend; r0 < n; r0 += chunk) {
                const int nr = min(chunk, n - r0);
                if (r0 > kend) __syncthreads();
                if (pos >= r0 && pos < r0 + nr) {
#pragma unroll
                    for (int j = 0; j < kLuNB; ++j) s_l[j * ld + pos - r0] = v[j];
                }
                __syncthreads();
                const int nrt = (nr + 63) / 64, nct = (nc + 4 * J - 1) / (4 * J);
                const int li = lane & 15, lg = lane >> 4;
                for (int tile = wave; tile < nrt * nct; tile += W) {
                    const int tr = 64 * (tile % nrt), tc = 4 * J * (tile / nrt);
                    double t[4][J];
#pragma unroll
                    for (int j = 0; j < J; ++j)
#pragma unroll
                        for (int i = 0; i < 4; ++i) {
                            const int rr = tr + li + 16 * i, cc = tc + lg + 4 * j;
                            t[i][j] = rr < nr && cc < nc ? a[r0 + rr + (long)(c0 + cc) * n] : 0.0;
                        }
                    // rows and columns past the chunk take its last one's; their results are not
                    // stored
                    int ol[4], ou[J];
#pragma unroll
                    for (int i = 0; i < 4; ++i) ol[i] = min(tr + li + 16 * i, nr - 1);
#pragma unroll
                    for (int j = 0; j < J; ++j) ou[j] = min(tc + lg + 4 * j, nc - 1);
                    auto sweep = [&](auto skip) {
#pragma unroll 2
                        for (int kk = 0; kk < kLuNB; ++kk) {
                            double l[4], y[J];
#pragma unroll
                            for (int i = 0; i < 4; ++i) l[i] = s_l[kk * ld + ol[i]];
#pragma unroll
                            for (int j = 0; j < J; ++j) y[j] = s_u[kk * ld + ou[j]];
#pragma unroll
                            for (int j = 0; j < J; ++j)
#pragma unroll
                                for (int i = 0; i < 4; ++i) {
                                    const double upd = t[i][j] + l[i] * -y[j];
                                    if constexpr (decltype(skip)::value) t[i][j] = y[j] != 0.0 ? upd : t[i][j];
                                    else t[i][j] = upd;
                                }
                        }
                    };
                    if (any_zero) sweep(std::true_type{});
                    else sweep(std::false_type{});
#pragma unroll
                    for (int j = 0; j < J; ++j)
#pragma unroll
                        for (int i = 0; i < 4; ++i) {
                            const int rr = tr + li + 16 * i, cc = tc + lg + 4 * j;
                            if (rr < nr && cc < nc) a[r0 + rr + (long)(c0 + cc) * n] = t[i][j];
                        }
                }
            }
        }
        __syncthreads();
    }
    if (tid == 0) infos[blockIdx.x] = info;
}

template <int NT>
int launch_lu_decompose(int n, int nbatch, double *mats, int *pivots, int *info, hipStream_t st)
{
    hipLaunchKernelGGL(lu_decompose_kernel<NT>, dim3((unsigned)nbatch), dim3(NT), lu_lds_bytes<NT>(n), st, n, mats,
                       pivots, info);
    RAYSHT_HIP_TRY(hipGetLastError());
    return RAYSHT_OK;
}

// Solve with the right-hand sides in registers: G lanes of a wave own CPL columns, lane
// r holds rows r, r + G, ... (NT of them) of each.  The interchanges are composed into one
// permutation applied when the column is loaded; then each step j takes x_j from its
// owner lane by a lane shuffle and updates the lane's rows in registers.  The factor comes
// through LDS K columns at a time, shared by all the workgroup's right-hand sides, the next K on
// their way in registers meanwhile; one barrier per K columns.  Operation order and rounding are
// those of the reference BLAS order.
// With one column on its way per wave the steps waited for memory (each takes a new cache line from
// every row block) and for the vector cache, which served every wave by itself; rows that a step does not
// touch were loaded and computed too.  256 matrices of n = 64, 128, 256 with 2 (l + 1) columns
// each: 0.15, 0.45, 1.33 ms before, 0.14, 0.32, 0.87 ms now (the arithmetic alone takes 0.25 ms of the
// last); 128 of n = 512 1.64 -> 1.26 ms, 32 of n = 1000 1.48 -> 1.08 ms.  What is left is the chain of a
// step: a shuffle, LDS reads, a product and a difference.
template <int G, int NT, int CPL>
__global__ __launch_bounds__(kLuThreads) void lu_solve_lanes_kernel(int n, int nbatch, int ncb, int grouped,
                                                                    const double *__restrict__ mats,
                                                                    const int *__restrict__ pivots,
                                                                    double *__restrict__ rhs,
                                                                    const long *__restrict__ rhs_off,
                                                                    const int *__restrict__ nrhs)
{
#pragma clang fp contract(off)
    constexpr int R = G * NT, K = R > 256 ? 4 : 8, PT = K * R / kLuThreads;
    __shared__ int perm[R];
    __shared__ double s_col[2 * K * R];
    constexpr int kCols = kLuThreads / G * CPL;
    const solve_block sb = solve_block_of(ncb, nbatch, grouped);
    if (sb.b >= nbatch) return;
    const int b = sb.b, ncol = nrhs[b], col0 = sb.cb * kCols;
    if (col0 >= ncol) return;  // uniform: the whole workgroup leaves
    const double *a = mats + (long)b * n * n;
    const auto piv = (const __attribute__((address_space(4))) int *)(pivots + (long)b * n);  // scalar loads
    const int tid = threadIdx.x;
    // each thread follows its rows through the interchanges
    for (int i = tid; i < n; i += kLuThreads) {
        int pos = i;
#pragma unroll 8
        for (int k = 0; k < n; ++k) {
            const int p = piv[k] - 1;
            if (p >= 0 && p < n) pos = pos == k ? p : pos == p ? k : pos;
        }
        perm[pos] = i;
    }
    __syncthreads();
    const int lane = tid % G, cg = col0 + (tid / G) * CPL;
    double x[CPL][NT];
#pragma unroll
    for (int q = 0; q < CPL; ++q) {
        const bool live = cg + q < ncol;
        const double *xg = rhs + rhs_off[b] + (long)(live ? cg + q : col0) * n;
#pragma unroll
        for (int t = 0; t < NT; ++t) {
            const int i = G * t + lane;
            x[q][t] = live && i < n ? xg[perm[i]] : 0.0;
        }
    }
    // Groups of K columns, 0 .. ng - 1 for the lower sweep and back for the upper one.  A buffer of
    // the matrix's size keeps the reads inside it; rows past the matrix reach no result.
    const int ng = (n + K - 1) / K;
    const __amdgpu_buffer_rsrc_t ra =
        __builtin_amdgcn_make_buffer_rsrc(const_cast<double *>(a), (short)0, 8 * n * n, 0x00020000);
    double pf[PT];
    auto fetch = [&](int s) {
        const int j0 = K * (s < ng ? s : 2 * ng - 1 - s);
#pragma unroll
        for (int q = 0; q < PT; ++q) {
            const int e = tid + q * kLuThreads, off = 8 * ((j0 + e / R) * n + e % R);
            pf[q] = __builtin_bit_cast(double, __builtin_amdgcn_raw_buffer_load_b64(ra, off, 0, 0));
        }
    };
    auto stage = [&](int s) {
#pragma unroll
        for (int q = 0; q < PT; ++q) s_col[(s & 1) * K * R + tid + q * kLuThreads] = pf[q];
    };
    // f(kq) for the columns of a group, the next group on its way meanwhile
    auto group = [&](int s, auto &&steps) {
        __syncthreads();
        if (s + 1 < 2 * ng) fetch(s + 1);
        steps(s_col + (s & 1) * K * R);
        if (s + 1 < 2 * ng) stage(s + 1);
    };
    fetch(0);
    stage(0);
    // unit lower: x_i -= x_j l_ij for i > j
    static_steps<0, NT>([&](auto block) {
        constexpr int tb = decltype(block)::value;
        for (int h = 0; h < G / K; ++h) {
            const int j0 = G * tb + K * h;
            if (j0 >= n) break;
            group(j0 / K, [&](const double *col) {
#pragma unroll 1
                for (int kq = 0; kq < K; ++kq) {
                    const int r = K * h + kq;
                    double l[NT];
#pragma unroll
                    for (int t = tb; t < NT; ++t) l[t] = col[kq * R + G * t + lane];
#pragma unroll
                    for (int q = 0; q < CPL; ++q) {
                        const double xj = __shfl(x[q][tb], r, G);
                        if (xj != 0.0) {
                            if (lane > r) x[q][tb] = x[q][tb] - xj * l[tb];
#pragma unroll
                            for (int t = tb + 1; t < NT; ++t) x[q][t] = x[q][t] - xj * l[t];
                        }
                    }
                }
            });
        }
    });
    // upper: x_j /= u_jj, then x_i -= x_j u_ij for i < j; x_j is final
    static_steps<0, NT>([&](auto block) {
        constexpr int tb = NT - 1 - decltype(block)::value;
        for (int h = G / K - 1; h >= 0; --h) {
            const int j0 = G * tb + K * h;
            if (j0 >= n) continue;
            group(2 * ng - 1 - j0 / K, [&](const double *col) {
#pragma unroll 1
                for (int kq = min(K, n - j0) - 1; kq >= 0; --kq) {
                    const int r = K * h + kq;
                    double u[NT];
#pragma unroll
                    for (int t = 0; t <= tb; ++t) u[t] = col[kq * R + G * t + lane];
                    const double ujj = col[kq * R + j0 + kq];
#pragma unroll
                    for (int q = 0; q < CPL; ++q) {
                        double xj = __shfl(x[q][tb], r, G);
                        if (xj != 0.0) {
                            xj = xj / ujj;
                            if (lane < r) x[q][tb] = x[q][tb] - xj * u[tb];
#pragma unroll
                            for (int t = 0; t < tb; ++t) x[q][t] = x[q][t] - xj * u[t];
                        }
                        if (lane == r) x[q][tb] = xj;
                    }
                }
            });
        }
    });
#pragma unroll
    for (int q = 0; q < CPL; ++q)
        if (cg + q < ncol) {
            double *xg = rhs + rhs_off[b] + (long)(cg + q) * n;
#pragma unroll
            for (int t = 0; t < NT; ++t) {
                const int i = G * t + lane;
                if (i < n) xg[i] = x[q][t];
            }
        }
}

// Two right-hand sides per lane group for n <= 512: three waves per SIMD.  One costs 1.03 ms instead
// of 0.87 at n = 256 (twice the LDS reads), three 1.07 and four 1.01 (fewer waves).  For n > 512 the
// staged columns (68 KB of LDS) leave a CU two workgroups whatever their registers are, and a
// column's reads, which two lane groups of a wave shared below, serve one: every right-hand side
// more costs a workgroup less than the last.  What counts is how many rounds of two workgroups on
// 256 CUs a launch takes.  At n = 1000 (ms for 2 / 3 / 4 per group): one round with two, 64 matrices of 64
// columns 1.40 / 1.69 / 1.55, 16 of 200 1.35 / 1.66 / 1.56; more, 64 of 2 (l + 1) (half of the groups
// empty) 2.22 / 1.70 / 2.01, 64 of 200 4.60 / 4.16 / 3.89, 64 of 512 9.97 / 8.54 / 7.38; n = 513, 256 of 2 (l + 1)
// 10.6 / 8.9 / 8.3.  So two as long as they fit one round, four from two rounds of fours on, three in between.
constexpr long kSolveSlots = 512;

// workgroups of a solve with cpl right-hand sides per group of G lanes
template <int G>
long lanes_workgroups(int cpl, int nbatch, int max_nrhs)
{
    const int cols = kLuThreads / G * cpl;
    return (long)nbatch * ((max_nrhs + (long)cols - 1) / cols);
}

template <int G, int NT, int CPL>
int launch_lanes(int n, int nbatch, const double *mats, const int *pivots, double *rhs, const long *rhs_off,
                 const int *nrhs, int max_nrhs, hipStream_t st)
{
    constexpr int kCols = kLuThreads / G * CPL;
    const int ncb = (max_nrhs + kCols - 1) / kCols, grouped = n > 256;
    if (!solve_grid_fits(ncb, nbatch, grouped, kLuThreads)) return RAYSHT_EUNSUPPORTED;
    hipLaunchKernelGGL((lu_solve_lanes_kernel<G, NT, CPL>), dim3((unsigned)solve_grid(ncb, nbatch, grouped)),
                       dim3(kLuThreads), 0, st, n, nbatch, ncb, grouped, mats, pivots, rhs, rhs_off, nrhs);
    return RAYSHT_OK;
}

}  // namespace
}  // namespace raysht

using namespace raysht;

// Banded factorisation: LU_Decompose_band (Linear_Solve.F90:1041-1055, dgbtrf with
// kl = ku = (ldab - 1) / 3) in the unblocked order of dgbtf2, one workgroup per matrix in
// LAPACK band storage ab(ldab, n) (1-based AB(i, j) below; full element (r, c) at row
// kv + 1 + r - c of column c, kv = kl + ku).  Per column: the fill-in rows LAPACK clears, the
// pivot (first largest |a| of the kl + 1 candidates, idamax's rules for NaN), the interchange
// over columns j..ju, the multipliers scaled by the pivot's reciprocal, and the rank-1 update
// of the km x (ju - j) block, a column skipped where the pivot row's entry is 0 (dger);
// products and sums rounded separately, so the factors are the oracle's doubles.
constexpr int kBandMaxKv = 1024;
__global__ __launch_bounds__(kLuThreads) void band_lu_decompose_kernel(int n, int kl, int ku, int ldab,
                                                                       double *__restrict__ mats,
                                                                       int *__restrict__ pivots,
                                                                       int *__restrict__ infos)
{
#pragma clang fp contract(off)
    __shared__ double s_val[kLuThreads];
    __shared__ int s_idx[kLuThreads];
    __shared__ double s_y[kBandMaxKv + 1];  // the pivot row, columns j + 1 .. ju
    const int tid = threadIdx.x;
    double *ab = mats + (long)blockIdx.x * ldab * n;
    int *piv = pivots + (long)blockIdx.x * n;
    const int kv = ku + kl;
#define AB(i, j) ab[(long)((j) - 1) * ldab + ((i) - 1)]
    // dgbtf2's zeroed fill-in: rows max(1, kv - c + 2) .. kl of columns c = ku + 2 .. n
    for (long e = tid; e < (long)kl * n; e += kLuThreads) {
        const int i = 1 + (int)(e % kl), c = 1 + (int)(e / kl);
        if (c >= ku + 2 && i >= kv - c + 2) AB(i, c) = 0.0;
    }
    __syncthreads();
    int info = 0, ju = 1;
    for (int j = 1; j <= n; ++j) {
        const int km = min(kl, n - j);
        double best = -1.0;
        int bi = 1 << 30;
        for (int i = 1 + tid; i <= km + 1; i += kLuThreads) {
            const double v = fabs(AB(kv + i, j));
            if (v > best) {
                best = v;
                bi = i;
            }
        }
        s_val[tid] = best;
        s_idx[tid] = bi;
        __syncthreads();
        for (int sh = kLuThreads / 2; sh > 0; sh >>= 1) {
            if (tid < sh) {
                const double v = s_val[tid + sh];
                const int q = s_idx[tid + sh];
                if (v > s_val[tid] || (v == s_val[tid] && q < s_idx[tid])) {
                    s_val[tid] = v;
                    s_idx[tid] = q;
                }
            }
            __syncthreads();
        }
        // idamax: a NaN first entry is kept (nothing compares larger); later NaNs are passed over
        const int jp = (s_idx[0] > km + 1 || isnan(AB(kv + 1, j))) ? 1 : s_idx[0];
        const double pv = AB(kv + jp, j);
        __syncthreads();  // every thread has the pivot before the interchange moves it
        if (tid == 0) piv[j - 1] = jp + j - 1;
        if (pv != 0.0) {
            ju = max(ju, min(j + ku + jp - 1, n));
            if (jp != 1)
                for (int c = tid; c <= ju - j; c += kLuThreads) {
                    const double t = AB(kv + jp - c, j + c);
                    AB(kv + jp - c, j + c) = AB(kv + 1 - c, j + c);
                    AB(kv + 1 - c, j + c) = t;
                }
            __syncthreads();
            if (km > 0) {
                const double r = 1.0 / AB(kv + 1, j);
                for (int i = 1 + tid; i <= km; i += kLuThreads) AB(kv + 1 + i, j) = r * AB(kv + 1 + i, j);
                for (int c = 1 + tid; c <= ju - j; c += kLuThreads) s_y[c] = AB(kv + 1 - c, j + c);
                __syncthreads();
                // element e = (i - 1) + km (c - 1), e = tid, tid + kLuThreads, ...: i and c stepped
                // without divisions, four elements per thread at a time with their operands (row
                // j and column j, which the update does not write) read before any is written
                const int w = ju - j, tot = km * w, di = kLuThreads % km, dc = kLuThreads / km;
                int i = 1 + tid % km, c = 1 + tid / km;
                constexpr int U = 4;
                for (int e = tid; e < tot; e += U * kLuThreads) {
                    int iu[U], cu[U];
                    bool on[U];
#pragma unroll
                    for (int u = 0; u < U; ++u) {
                        on[u] = e + u * kLuThreads < tot;
                        iu[u] = on[u] ? i : 1;
                        cu[u] = on[u] ? c : 1;
                        i += di;
                        c += dc;
                        if (i > km) {
                            i -= km;
                            ++c;
                        }
                    }
                    double y[U], a[U], x[U];
#pragma unroll
                    for (int u = 0; u < U; ++u) {
                        y[u] = s_y[cu[u]];
                        a[u] = AB(kv + 1 + iu[u] - cu[u], j + cu[u]);
                        x[u] = AB(kv + 1 + iu[u], j);
                    }
#pragma unroll
                    for (int u = 0; u < U; ++u)
                        if (on[u] && y[u] != 0.0) AB(kv + 1 + iu[u] - cu[u], j + cu[u]) = a[u] + x[u] * (-y[u]);
                }
                __syncthreads();
            }
        } else if (info == 0) {
            info = j;
        }
    }
    if (tid == 0) infos[blockIdx.x] = info;
#undef AB
}

// The same factorisation with its active window in LDS.  Step j of dgbtf2 reads and writes
// only matrix rows j .. j + kl and columns j .. j + kv (the pivot search, the interchange
// over columns j .. ju <= j + kv, the multipliers and the rank-1 update), so that window
// lives in an LDS ring (matrix row % (kl + 2), column % (kv + 2), column-major, ld apart)
// while the factorisation walks down the band.  The ring has one row and one column more
// than the step uses: row j + kl + 1 (plain band entries, loaded before the pivot search) and
// column j + kv + 1 (rows j + 1 .. j + kl: dgbtf2's zeroed fill-in, so zeros are written, not
// read) come in for step j + 1 while step j works.  A step has three barriers: every wave
// finds the pivot by itself; then the interchange writes row j (U, final) and the scaling
// column j (L, final) to LDS and the band storage in one pass; then the rank-1 update, in
// which a thread stays on one ring row and keeps its multiplier in a register.  The arithmetic,
// its order and the pivot choice are the global-memory kernel's, so the factors and pivots
// are the same doubles.  Used where the window fits one workgroup's LDS.  Where only the step's own
// rows and columns do (SPARE = false), the next ones come in after the update, into the slots
// that the step has done with, at the price of a fourth barrier and a load that is waited for:
// n = 640, kl = 30, ku = 612 (32 matrices) 1.99 ms instead of 5.22 in global memory, 400, 63, 255 1.31
// instead of 3.97.
// What bounds it is the chain of a column's phases (LDS latency, the barriers), then the LDS
// rate of the update (three accesses per element).  With seven barriers a step, four LDS accesses per element
// and 256 threads at every size it took, ms, against now: 170 matrices of n = 192, kl = 72 .813, .420;
// 128, 40 .377, .186; 64, 20 .167, .080; 256 of n = 256, kl = 96 1.37, .704; n = 512, kl = 8 1.38, .637.
template <int NT, bool SPARE>
__global__ __launch_bounds__(NT) void band_lu_decompose_lds_kernel(int n, int kl, int ku, int ldab, int ld,
                                                                   double *__restrict__ mats,
                                                                   int *__restrict__ pivots, int *__restrict__ infos)
{
#pragma clang fp contract(off)
    extern __shared__ double win[];
    const int tid = threadIdx.x, lane = tid & 63;
    double *ab = mats + (long)blockIdx.x * ldab * n;
    int *piv = pivots + (long)blockIdx.x * n;
    const int kv = ku + kl, R = kl + (SPARE ? 2 : 1), C = kv + (SPARE ? 2 : 1);  // ring rows and columns
#define AB(i, j) ab[(long)((j) - 1) * ldab + ((i) - 1)]
    // the first window, rows 1 .. min(kl + 1, n) x columns 1 .. min(kv + 1, n); entries more than
    // ku above the diagonal are fill-in, zero at the start
    {
        const int nrw = min(kl + 1, n), ncl = min(kv + 1, n);
        for (int e = tid; e < nrw * ncl; e += NT) {
            const int row = 1 + e % nrw, col = 1 + e / nrw;
            win[col % C * ld + row % R] = col - row > ku ? 0.0 : AB(kv + 1 + row - col, col);
        }
    }
    __syncthreads();
    const int rs = tid % ld, g = tid / ld, G = NT / ld;  // the update's ring row and its columns g, g + G, ...
    int info = 0, ju = 1, jr = 1 % R, jc = 1 % C;        // jr, jc: the ring row and column of j
    for (int j = 1; j <= n; ++j) {
        // ring rows / columns at an offset below R / C from j
        auto ring_row = [&](int i) { return jr + i >= R ? jr + i - R : jr + i; };
        auto ring_col = [&](int c) { return jc + c >= C ? jc + c - C : jc + c; };
        const int km = min(kl, n - j), rn = j + kl + 1, cn = j + kv + 1;
        const double in = SPARE && rn <= n && j + 1 + tid <= min(cn, n) ? AB(kv + rn - j - tid, j + 1 + tid) : 0.0;
        double *colj = win + jc * ld;
        // the largest |a| with the lowest index among equals; NaNs never enter
        double best = -1.0;
        int bi = 1 << 30;
        for (int i = lane; i <= km; i += 64) {
            const double v = fabs(colj[ring_row(i)]);
            if (v > best) {
                best = v;
                bi = i;
            }
        }
        const double wm = lu_wave_max(best);
        unsigned long long eq = __ballot(best == wm);
        int p = __builtin_amdgcn_readlane(bi, __builtin_ctzll(eq));
        for (eq &= eq - 1; eq != 0; eq &= eq - 1)
            p = min(p, (int)__builtin_amdgcn_readlane(bi, __builtin_ctzll(eq)));
        // idamax: a NaN first entry is kept (nothing compares larger); later NaNs are passed over
        const double d0 = colj[jr];
        if (p > km || isnan(d0)) p = 0;
        const int pr = ring_row(p);
        const double pv = colj[pr];
        __syncthreads();  // every wave has the pivot before the interchange moves it
        if (tid == 0) piv[j - 1] = j + p;
        const bool work = pv != 0.0;
        if (work)
            ju = max(ju, min(j + ku + p, n));
        else if (info == 0)
            info = j;
        // row j of columns j + 1 .. (the first half of the threads), column j (the second half)
        const int w = ju - j, ncr = min(kv, n - j);
        if (tid < NT / 2) {
            for (int c = 1 + tid; c <= ncr; c += NT / 2) {
                double *col = win + ring_col(c) * ld;
                const double old = col[jr];
                double u = old;
                if (work && p != 0 && c <= w) {
                    u = col[pr];
                    col[pr] = old;
                    col[jr] = u;
                }
                AB(kv + 1 - c, j + c) = u;
            }
        } else {
            const double r = 1.0 / pv;
            for (int i = tid - NT / 2; i <= km; i += NT / 2) {
                double l = i == 0 ? pv : i == p ? d0 : colj[ring_row(i)];  // without a pivot p = 0
                if (work && i > 0) l = r * l;
                if (i > 0) colj[ring_row(i)] = l;
                AB(kv + 1 + i, j) = l;
            }
        }
        // row j + kl + 1 and column j + kv + 1 into the ring slots nr and ncol
        auto bring_in = [&](int nr, int ncol) {
            if (rn <= n)
                for (int c = tid; c <= min(kv, n - j - 1); c += NT)
                    win[ring_col(c + 1) * ld + nr] = SPARE && c == tid ? in : AB(kv + rn - j - c, j + 1 + c);
            if (cn <= n)
                for (int i = 1 + tid; i <= min(kl, n - j); i += NT) win[ncol * ld + ring_row(i)] = 0.0;
        };
        if (SPARE) bring_in(jr > 0 ? jr - 1 : R - 1, jc > 0 ? jc - 1 : C - 1);  // those of row and column j - 1
        __syncthreads();
        int i = rs - jr;
        if (i < 0) i += R;
        if (work && rs < R && g < G && i >= 1 && i <= km) {
            const double x = colj[rs];
            constexpr int U = 4;
            int cs = jc + 1 + g;
            for (int c = 1 + g; c <= w; c += U * G) {
                double y[U], a[U];
                int at[U];
#pragma unroll
                for (int u = 0; u < U; ++u) {
                    const bool on = c + u * G <= w;
                    if (cs >= C) cs -= C;
                    at[u] = on ? cs * ld : jc * ld;
                    cs += G;
                    y[u] = win[at[u] + jr];
                    a[u] = win[at[u] + rs];
                    if (!on) y[u] = 0.0;
                }
#pragma unroll
                for (int u = 0; u < U; ++u)
                    if (y[u] != 0.0) win[at[u] + rs] = a[u] + x * (-y[u]);
            }
        }
        __syncthreads();
        if (!SPARE) {  // those of row and column j
            bring_in(jr, jc);
            __syncthreads();
        }
        if (++jr == R) jr = 0;
        if (++jc == C) jc = 0;
    }
    if (tid == 0) infos[blockIdx.x] = info;
#undef AB
}

template <int NT, bool SPARE>
void launch_band_lds(int n, int kl, int ku, int nbatch, double *mats, int ldab, int ld, int *pivots, int *info,
                     hipStream_t st)
{
    const size_t columns = kl + ku + (SPARE ? 2 : 1);
    hipLaunchKernelGGL((band_lu_decompose_lds_kernel<NT, SPARE>), dim3((unsigned)nbatch), dim3(NT),
                       sizeof(double) * columns * ld, st, n, kl, ku, ldab, ld, mats, pivots, info);
}

// Banded solve: LU_Solve_Band (Linear_Solve.F90:1056-1086, dgbtrs 'N').  One wave solves CPL
// right-hand-side columns of matrix blockIdx.y, held in registers across its lanes (row
// 64 s + lane in slot s, NS slots).  Per step j the wave reads x_j from its owner lane and
// updates only the slots the band reaches, with one coalesced load of the factor column shared
// by its CPL columns: the L solve (interchange, then dger's x(r) + l (-x(j)), skipped where
// x(j) = 0) and dtbsv's upper solve (x(j) / u(j, j), then x(r) - x(j) u(r, j) for the kl + ku
// rows above, skipped where x(j) = 0).  Factor entry (r, j) of both is band row kv + r - j.
// The slots rotate: while step j runs over the 64 rows of segment S = j / 64, slot k of a
// lane holds absolute slot (S + k) mod NS, so row j is always in slot 0 and every slot index
// in the loop bodies is a compile-time register index (a select over NS slots per access
// was most of the kernel's instructions).  Segments advance by one rotation of the NS
// slots, and NS rotations restore the natural order.
// What bounds it is the chain of a step: the factor column's load (asked for before anything
// else of the step), x_j, the division.  x_j and the interchange's rows are read with v_readlane, a
// segment's pivots are held one per lane, and one division serves the CPL columns, lane c
// dividing for column c.  With LDS-path shuffles, a pivot load per step and a division per column it took, ms,
// against now: 256 matrices of n = 256, kl = 96 2.18, 1.75; 170 of n = 192, kl = 72 .734, .632; 64, 20
// .222, .203; 64 of n = 300, kl = 98 .759, .711; 64 of n = 600, kl = 40 1.79, 1.69; 256 of n = 512, kl = 8 is
// even at 4.4.  The next step's column loaded one to four steps ahead costs registers and so
// waves: 2.54 instead of 1.75 ms at n = 256.  NS = 8 is held to four waves per SIMD (4.4 against 5.0 ms at
// n = 512, kl = 8).
// For NS >= 4 a pass over the slots leaves where the band ends, so a step costs what its band
// reaches: the slots of a step are neighbours (downwards from row j's in the L solve, upwards in the
// U solve).  A branch around each of the 16 or 32 slots outside the band, in the load and again in the
// update, was most of a narrow band's step; ms with those branches, now, 170 matrices with 2 (l + 1)
// columns: n = 192, kl = 72 .626, .585; 256, 96 .877, .843; 300, 98 1.76, 1.19; 512, 8 2.21, 1.40;
// 600, 40 7.79, 5.31; 1000, 4 11.8, 6.5.  NS = 1 and 2 are even (one branch, at most two slots).
template <int NS>
__device__ __forceinline__ void slots_rotate_down(double (&x)[NS])  // slot k takes slot k + 1
{
    const double x0 = x[0];
#pragma unroll
    for (int k = 0; k + 1 < NS; ++k) x[k] = x[k + 1];
    x[NS - 1] = x0;
}

template <int NS>
__device__ __forceinline__ void slots_rotate_up(double (&x)[NS])  // slot k takes slot k - 1
{
    const double xl = x[NS - 1];
#pragma unroll
    for (int k = NS - 1; k > 0; --k) x[k] = x[k - 1];
    x[0] = xl;
}

// f(k) for slots k = 0 .. NS - 1: with STOP until f returns false, else all of them
template <int NS, bool STOP, typename F>
__device__ __forceinline__ void each_slot(F &&f)
{
    if constexpr (STOP) {
        static_while<0, NS>(f);
    } else {
#pragma unroll
        for (int k = 0; k < NS; ++k) (void)f(k);
    }
}

// the value of lane `l` (the same in every lane)
__device__ __forceinline__ double lane_value(double v, int l)
{
    const long b = __builtin_bit_cast(long, v);
    const int lo = __builtin_amdgcn_readlane((int)b, l), hi = __builtin_amdgcn_readlane((int)(b >> 32), l);
    return __builtin_bit_cast(double, ((long)hi << 32) | (unsigned)lo);
}

template <int NS, int CPL>
__global__ __launch_bounds__(64, NS == 8 ? 4 : 1) void band_lu_solve_kernel(int n, int kl, int ku, int ldab, int nbatch, int ncb,
                                                           const double *__restrict__ mats,
                                                           const int *__restrict__ pivots, double *__restrict__ rhs,
                                                           const long *__restrict__ rhs_off,
                                                           const int *__restrict__ nrhs)
{
#pragma clang fp contract(off)
    const solve_block sb = solve_block_of(ncb, nbatch, 1);
    if (sb.b >= nbatch) return;
    const int b = sb.b, lane = threadIdx.x, c0 = sb.cb * CPL;
    const int nc = min(CPL, nrhs[b] - c0);
    if (nc <= 0) return;
    const double *ab = mats + (long)b * ldab * n;
    const int *piv = pivots + (long)b * n;
    double *x0 = rhs + rhs_off[b] + (long)c0 * n;
    const int kv = kl + ku;
    double x[CPL][NS];
#pragma unroll
    for (int c = 0; c < CPL; ++c)
#pragma unroll
        for (int s = 0; s < NS; ++s) {
            const int r = s * 64 + lane;
            x[c][s] = (c < nc && r < n) ? x0[(long)c * n + r] : 0.0;
        }
    constexpr int D = NS == 1 ? 2 : 1;  // steps whose factor columns are loaded together
    constexpr bool kStop = NS >= 4;     // leave a pass over the slots where the band ends
    // L solve with the interchanges, segment by segment (row j in slot 0)
#pragma unroll 1
    for (int S = 0; S < NS; ++S) {
        const int jend = kl > 0 ? min(64 * (S + 1), n - 1) : 0;
        const int pj = 64 * S + lane < n ? piv[64 * S + lane] : 0;
        double a[D][NS];
        auto fetch = [&](int j0) {
#pragma unroll
            for (int d = 0; d < D; ++d) {
                const int j = j0 + d, lm = min(kl, n - 1 - j);
                const double *col = ab + (long)j * ldab + kv - j;  // col[r] = factor entry (r, j)
                auto load = [&](int k) {
                    const int r = (S + k) * 64 + lane;
                    a[d][k] = j < jend && r > j && r <= j + lm ? col[r] : 0.0;
                };
                if constexpr (NS == 1) load(0);
                else
                    static_while<0, NS>([&](auto k) {
                        if (kStop && (S + k) * 64 > j + lm) return false;
                        load(k);
                        return true;
                    });
            }
        };
#pragma unroll 1
        for (int j0 = 64 * S; j0 < jend; j0 += D) {
            fetch(j0);
            static_steps<0, D>([&](auto step) {
#pragma clang fp contract(off)
                constexpr int d = decltype(step)::value;
                const int j = j0 + d;
                if (j >= jend) return;
                const int jj = j & 63, lm = min(kl, n - 1 - j);
                const int l = __builtin_amdgcn_readlane(pj, jj) - 1, lrel = (l >> 6) - S;
                double y[CPL];
#pragma unroll
                for (int c = 0; c < CPL; ++c) y[c] = lane_value(x[c][0], jj);
                if (l != j)
                    static_while<0, NS>([&](auto slot) {
                        constexpr int k = decltype(slot)::value;
                        if (k != lrel) return true;
                        asm volatile("" ::"n"(k));  // keeps the slots' branches apart: x[lrel] would put x into memory
#pragma unroll
                        for (int c = 0; c < CPL; ++c) {
                            const double xl = lane_value(x[c][k], l & 63);
                            if (lane == jj) x[c][0] = xl;
                            if (lane == (l & 63)) x[c][k] = y[c];
                            y[c] = xl;
                        }
                        return false;
                    });
                const int klo = ((j + 1) >> 6) - S, khi = ((j + lm) >> 6) - S;
                each_slot<NS, kStop>([&](auto slot) {
#pragma clang fp contract(off)
                    const int k = slot, r = (S + k) * 64 + lane;
                    if (kStop && k > khi) return false;
                    if (!kStop && (k < klo || k > khi)) return true;
                    if (r > j && r <= j + lm) {
#pragma unroll
                        for (int c = 0; c < CPL; ++c)
                            if (y[c] != 0.0) x[c][k] = x[c][k] + a[d][k] * (-y[c]);
                    }
                    return true;
                });
            });
        }
#pragma unroll
        for (int c = 0; c < CPL; ++c) slots_rotate_down(x[c]);
    }
    // U solve, segments from the last down (row j in slot 0, rows above in slots NS - 1, ...)
#pragma unroll 1
    for (int S = NS - 1; S >= 0; --S) {
#pragma unroll
        for (int c = 0; c < CPL; ++c) slots_rotate_up(x[c]);
        double a[D][NS], dg[D];
        auto fetch = [&](int j0) {
#pragma unroll
            for (int d = 0; d < D; ++d) {
                const int j = j0 - d, lo = max(0, j - kv);
                const bool on = j >= 64 * S;
                const double *col = ab + (long)j * ldab + kv - j;
                dg[d] = on ? col[j] : 1.0;
                each_slot<NS, kStop>([&](auto slot) {  // upwards from row j's
                    const int i = slot, k = i == 0 ? 0 : NS - i, sa = S - i, r = sa * 64 + lane;
                    if (kStop && sa * 64 + 63 < lo) return false;
                    a[d][k] = on && r >= lo && r < j ? col[r] : 0.0;
                    return true;
                });
            }
        };
        const int jtop = min(64 * S + 63, n - 1);
#pragma unroll 1
        for (int j0 = jtop; j0 >= 64 * S; j0 -= D) {
            fetch(j0);
            static_steps<0, D>([&](auto step) {
#pragma clang fp contract(off)
                constexpr int d = decltype(step)::value;
                const int j = j0 - d;
                if (j < 64 * S) return;
                const int jj = j & 63;
                // lane c divides for column c; dtbsv skips a column where x(j) is 0 before the division
                double t[CPL], q = 0.0;
                bool nz[CPL];
#pragma unroll
                for (int c = 0; c < CPL; ++c) {
                    t[c] = lane_value(x[c][0], jj);
                    nz[c] = t[c] != 0.0;
                    if (lane == c) q = t[c];
                }
                q = q / dg[d];
#pragma unroll
                for (int c = 0; c < CPL; ++c)
                    if (nz[c]) {
                        t[c] = lane_value(q, c);
                        if (lane == jj) x[c][0] = t[c];
                    }
                if (j == 0) return;
                const int lo = max(0, j - kv), slo = lo >> 6, shi = (j - 1) >> 6;
                each_slot<NS, kStop>([&](auto slot) {
#pragma clang fp contract(off)
                    const int i = slot, k = i == 0 ? 0 : NS - i, sa = S - i, r = sa * 64 + lane;
                    if (kStop && sa < slo) return false;
                    if (!kStop && (sa < slo || sa > shi)) return true;
                    if (r >= lo && r < j) {
#pragma unroll
                        for (int c = 0; c < CPL; ++c)
                            if (nz[c]) x[c][k] = x[c][k] - t[c] * a[d][k];
                    }
                    return true;
                });
            });
        }
    }
#pragma unroll
    for (int c = 0; c < CPL; ++c)
#pragma unroll
        for (int s = 0; s < NS; ++s) {
            const int r = s * 64 + lane;
            if (c < nc && r < n) x0[(long)c * n + r] = x[c][s];
        }
}

template <int NS, int CPL>
int launch_band_solve(int n, int kl, int ku, int nbatch, const double *mats, int ldab, const int *pivots,
                      double *rhs, const long *rhs_off, const int *nrhs, int max_nrhs, hipStream_t st)
{
    const int ncb = (max_nrhs + CPL - 1) / CPL;
    if (!solve_grid_fits(ncb, nbatch, 1, 64)) return RAYSHT_EUNSUPPORTED;
    hipLaunchKernelGGL((band_lu_solve_kernel<NS, CPL>), dim3((unsigned)solve_grid(ncb, nbatch, 1)), dim3(64), 0, st, n,
                       kl, ku, ldab, nbatch, ncb, mats, pivots, rhs, rhs_off, nrhs);
    return RAYSHT_OK;
}

extern "C" {

int raysht_lu_decompose_full(int n, int nbatch, double *mats, int *pivots, int *info, void *stream)
{
    if (n < 1 || nbatch < 0 || (nbatch > 0 && (!mats || !pivots || !info))) return RAYSHT_EINVAL;
    if (n > kLuMaxN) return RAYSHT_EUNSUPPORTED;
    if (nbatch == 0) return RAYSHT_OK;
    hipStream_t st = reinterpret_cast<hipStream_t>(stream);
    // a thread per row; up to 256 rows 512 threads, whose other waves only take trailing tiles, beat
    // 256 at n = 256 (0.87 against 0.93 ms) and are even at 192
    if (n <= 64) return launch_lu_decompose<64>(n, nbatch, mats, pivots, info, st);
    if (n <= 128) return launch_lu_decompose<128>(n, nbatch, mats, pivots, info, st);
    if (n <= 512) return launch_lu_decompose<512>(n, nbatch, mats, pivots, info, st);
    return launch_lu_decompose<1024>(n, nbatch, mats, pivots, info, st);
}

int raysht_lu_solve_full(int n, int nbatch, const double *mats, const int *pivots, double *rhs, const long *rhs_off,
                         const int *nrhs, int max_nrhs, void *stream)
{
    if (n < 1 || nbatch < 0 || max_nrhs < 0) return RAYSHT_EINVAL;
    if (nbatch > 0 && (!mats || !pivots || !rhs || !rhs_off || !nrhs)) return RAYSHT_EINVAL;
    if (n > kLuMaxN) return RAYSHT_EUNSUPPORTED;
    if (nbatch == 0 || max_nrhs == 0) return RAYSHT_OK;
    hipStream_t st = reinterpret_cast<hipStream_t>(stream);
    int rc;
    if (n <= 64)
        rc = launch_lanes<16, 4, 2>(n, nbatch, mats, pivots, rhs, rhs_off, nrhs, max_nrhs, st);
    else if (n <= 128)
        rc = launch_lanes<16, 8, 2>(n, nbatch, mats, pivots, rhs, rhs_off, nrhs, max_nrhs, st);
    else if (n <= 256)
        rc = launch_lanes<16, 16, 2>(n, nbatch, mats, pivots, rhs, rhs_off, nrhs, max_nrhs, st);
    else if (n <= 512)
        rc = launch_lanes<32, 16, 2>(n, nbatch, mats, pivots, rhs, rhs_off, nrhs, max_nrhs, st);
    else if (lanes_workgroups<64>(2, nbatch, max_nrhs) <= kSolveSlots)
        rc = launch_lanes<64, 16, 2>(n, nbatch, mats, pivots, rhs, rhs_off, nrhs, max_nrhs, st);
    else if (lanes_workgroups<64>(4, nbatch, max_nrhs) < 2 * kSolveSlots)
        rc = launch_lanes<64, 16, 3>(n, nbatch, mats, pivots, rhs, rhs_off, nrhs, max_nrhs, st);
    else
        rc = launch_lanes<64, 16, 4>(n, nbatch, mats, pivots, rhs, rhs_off, nrhs, max_nrhs, st);
    // a grid beyond the launch limit: fewer workgroups with three columns each
    if (rc == RAYSHT_EUNSUPPORTED && n > 256 && n <= 512)
        rc = launch_lanes<32, 16, 3>(n, nbatch, mats, pivots, rhs, rhs_off, nrhs, max_nrhs, st);
    if (rc != RAYSHT_OK) return rc;
    RAYSHT_HIP_TRY(hipGetLastError());
    return RAYSHT_OK;
}


int raysht_lu_decompose_band(int n, int kl, int ku, int nbatch, double *mats, int ldab, int *pivots, int *info,
                             void *stream)
{
    if (n < 1 || kl < 0 || ku < 0 || nbatch < 0 || ldab < 2 * kl + ku + 1) return RAYSHT_EINVAL;
    if (nbatch > 0 && (!mats || !pivots || !info)) return RAYSHT_EINVAL;
    if (kl + ku > kBandMaxKv) return RAYSHT_EUNSUPPORTED;
    if (nbatch == 0) return RAYSHT_OK;
    // the LDS-window kernel where its window fits one workgroup's LDS, with a row and a column
    // to spare if it can; an odd distance between columns keeps the interchange of a row off the
    // same banks
    int dev = 0, lds_max = 0;
    RAYSHT_HIP_TRY(hipGetDevice(&dev));
    RAYSHT_HIP_TRY(hipDeviceGetAttribute(&lds_max, hipDeviceAttributeMaxSharedMemoryPerBlock, dev));
    auto window = [&](int spare, int *ld) {
        const long rows = kl + 1 + spare, room = lds_max / (8L * (kl + ku + 1 + spare));
        *ld = (int)((rows | 1) <= room ? rows | 1 : rows);
        return rows <= room;
    };
    int ld = 0;
    const bool spare = window(1, &ld), tight = !spare && window(0, &ld);
    hipStream_t st = reinterpret_cast<hipStream_t>(stream);
    // threads by the size of the rank-1 update: 256 / 512 / 1024 take .080 / .089 / .100 ms at n = 64,
    // kl = 20 (170 matrices), .208 / .186 / .225 at 128, 40, .552 / .420 / .433 at 192, 72 and
    // 1.196 / .726 / .704 at 256, 96 (256 matrices), and without the spare row and column 3.09 / 2.18 /
    // 1.99 at 640, 30, ku = 612 (32 matrices); a launch stays below 2^32 threads in all
    auto fits = [&](int threads) { return (long)nbatch * threads < (1L << 32); };
    if (spare && kl > 80 && fits(1024))
        launch_band_lds<1024, true>(n, kl, ku, nbatch, mats, ldab, ld, pivots, info, st);
    else if (spare && kl > 24 && fits(512))
        launch_band_lds<512, true>(n, kl, ku, nbatch, mats, ldab, ld, pivots, info, st);
    else if (spare)
        launch_band_lds<256, true>(n, kl, ku, nbatch, mats, ldab, ld, pivots, info, st);
    else if (tight && fits(1024))
        launch_band_lds<1024, false>(n, kl, ku, nbatch, mats, ldab, ld, pivots, info, st);
    else if (tight)
        launch_band_lds<256, false>(n, kl, ku, nbatch, mats, ldab, ld, pivots, info, st);
    else
        hipLaunchKernelGGL(band_lu_decompose_kernel, dim3((unsigned)nbatch), dim3(kLuThreads), 0, st, n, kl,
                           ku, ldab, mats, pivots, info);
    RAYSHT_HIP_TRY(hipGetLastError());
    return RAYSHT_OK;
}

int raysht_lu_solve_band(int n, int kl, int ku, int nbatch, const double *mats, int ldab, const int *pivots,
                         double *rhs, const long *rhs_off, const int *nrhs, int max_nrhs, void *stream)
{
    if (n < 1 || kl < 0 || ku < 0 || nbatch < 0 || max_nrhs < 0 || ldab < 2 * kl + ku + 1) return RAYSHT_EINVAL;
    if (nbatch > 0 && (!mats || !pivots || !rhs || !rhs_off || !nrhs)) return RAYSHT_EINVAL;
    if (n > kLuMaxN) return RAYSHT_EUNSUPPORTED;
    if (nbatch == 0 || max_nrhs == 0) return RAYSHT_OK;
    hipStream_t st = reinterpret_cast<hipStream_t>(stream);
    int rc;
    if (n <= 64)
        rc = launch_band_solve<1, 8>(n, kl, ku, nbatch, mats, ldab, pivots, rhs, rhs_off, nrhs, max_nrhs, st);
    else if (n <= 128)
        rc = launch_band_solve<2, 8>(n, kl, ku, nbatch, mats, ldab, pivots, rhs, rhs_off, nrhs, max_nrhs, st);
    else if (n <= 256)
        rc = launch_band_solve<4, 4>(n, kl, ku, nbatch, mats, ldab, pivots, rhs, rhs_off, nrhs, max_nrhs, st);
    else if (n <= 512)
        rc = launch_band_solve<8, 4>(n, kl, ku, nbatch, mats, ldab, pivots, rhs, rhs_off, nrhs, max_nrhs, st);
    else
        rc = launch_band_solve<16, 2>(n, kl, ku, nbatch, mats, ldab, pivots, rhs, rhs_off, nrhs, max_nrhs, st);
    if (rc != RAYSHT_OK) return rc;
    RAYSHT_HIP_TRY(hipGetLastError());
    return RAYSHT_OK;
}

}  // extern "C"
