// FP64-MFMA Legendre contractions: every m-block of uneven length in one grouped launch.
//
// StP (Legendre_Transforms.F90:968-1074): for each m the reference forms
//   E = p_lm_even^T . s_even   and   O = p_lm_odd^T . s_odd       (nt/2 x nrhs each)
// with one DGEMM per parity and writes out(j) = E + O, out(nt+1-j) = E - O.
// PtS (:1077-1175): folds f(j) +/- f(nt+1-j), contracts with the integration-weighted
// tables and scatters even/odd l back into the interleaved l column.
//
// Here one workgroup owns an output tile of one m-block and computes BOTH parities
// for it, so the fold / reflection and the l gather / scatter happen in registers
// and LDS instead of separate passes through HBM.  Work items for all m-blocks are
// listed on the host (largest contraction first) and launched as one grid.
//
// MFMA used: v_mfma_f64_16x16x4_f64 (wave64).  Per lane: A = A[i][k] with
// i = lane%16, k = lane/16; B = B[k][j] with j = lane%16, k = lane/16; the 16x16
// result holds D[i][j] at i = lane/16 + 4*v, j = lane%16 (v = 0..3) -- the rows
// of the FP64 result are interleaved by 4, unlike the FP32 MFMA result layout.
// Both kernels compute the transposed product (columns of the right-hand side on
// the i axis) so that the 16 consecutive lanes of a store walk the unit-stride
// axis of the output (theta for StP, l for PtS).
#include "raysht_internal.h"
#include "uniform.h"

namespace raysht {
namespace {

typedef double double4_t __attribute__((ext_vector_type(4)));

__device__ __forceinline__ double4_t mfma_f64(double a, double b, double4_t c)
{
    return __builtin_amdgcn_mfma_f64_16x16x4f64(a, b, c, 0, 0, 0);
}

// Both kernels run two 8-wave workgroups per CU (128 VGPRs).  A wave alone keeps its SIMD's
// matrix pipe busy for 64 cycles per MFMA, so what counts is that some wave always has an
// MFMA to issue: one barrier per chunk, no staging of the data operand (two barriers and
// twelve loads and LDS writes per wave and chunk before), 16-byte loads, and the loads of
// the next chunk issued among this chunk's MFMAs.  On one long contraction (K = 512) StP
// went from 58 to 71 TFLOP/s (a register-only MFMA loop reaches 74) and PtS from 58 to 66.
// l_max = 511, N_theta = 768, N_r = 192, 8 fields: StP 6.60 -> 5.64 ms, PtS 6.60 -> 5.80 ms
// (55 / 53 TFLOP/s; 5.5 - 5.9 and 5.6 - 6.1 over several machines); without their stores and data
// loads the same kernels take 4.4 / 4.8 ms, so what is left above the matrix time is mostly the
// 14.0 and 18.3 GB that they move (13.3 GB at least).
// Measured and not kept: 4-wave workgroups with 32 columns per wave (half the LDS reads,
// same rate at K = 512, 3-7 % slower on the whole path), wave priorities per workgroup,
// scheduling barriers after every StP step.
constexpr int kFp64MinWaves = 4;

// Raw buffer access: each dword of a load whose byte offset falls outside [0, bytes) reads 0
// without touching memory (a 16-byte load may straddle the end), so tile edges need no
// branches.  The whole offset goes in the VGPR operand: the SGPR offset of a buffer load is not
// range-checked.  A negative offset reads as a huge unsigned one, so it is out of range too.
__device__ __forceinline__ __amdgpu_buffer_rsrc_t make_rsrc(const double *base, long bytes)
{
    return __builtin_amdgcn_make_buffer_rsrc(const_cast<double *>(base), (short)0, (int)bytes, 0x00020000);
}

__device__ __forceinline__ double2 load_f64x2(__amdgpu_buffer_rsrc_t r, int voff)
{
    return __builtin_bit_cast(double2, __builtin_amdgcn_raw_buffer_load_b128(r, voff, 0, 0));
}

// stores past the range are dropped
__device__ __forceinline__ void store_f64(__amdgpu_buffer_rsrc_t r, int voff, double v)
{
    typedef unsigned int uint2_t __attribute__((ext_vector_type(2)));
    __builtin_amdgcn_raw_buffer_store_b64(__builtin_bit_cast(uint2_t, v), r, voff, 0, 0);
}

__device__ __forceinline__ void store_f64x2(__amdgpu_buffer_rsrc_t r, int voff, double2 v)
{
    typedef unsigned int uint4_t __attribute__((ext_vector_type(4)));
    __builtin_amdgcn_raw_buffer_store_b128(__builtin_bit_cast(uint4_t, v), r, voff, 0, 0);
}

// the same with the nt bit (2) of the cache policy
__device__ __forceinline__ void store_f64_nt(__amdgpu_buffer_rsrc_t r, int voff, double v)
{
    typedef unsigned int uint2_t __attribute__((ext_vector_type(2)));
    __builtin_amdgcn_raw_buffer_store_b64(__builtin_bit_cast(uint2_t, v), r, voff, 0, 2);
}

// ---------------------------------------------------------------- StP
// Workgroup tile: (waves x 16) columns (c) x 64 southern nodes (j), both parities; wave w
// owns 16 columns: NB node blocks x 2 parities of 16x16 accumulators.  K runs over chunks of
// 16 parity-l values, four MFMA steps each.  A wave's data columns are its own and the MFMA
// operand of lane (li, lg) at step s is the pair s(2k), s(2k + 1) of column li, k = k0 + 4 s +
// lg, so each lane loads its pairs straight into the operand registers with one 16-byte
// load, and reloads the registers of two steps for the next chunk as soon as their MFMAs have
// been issued.  Only the table chunk is shared by the waves: double-buffered in LDS, one
// barrier per chunk, its global loads issued at the chunk's start and written to the other
// buffer between the MFMA steps, so no wave stands between two barriers without matrix work.
constexpr int STP_THREADS = 512;
constexpr int STP_TC = (STP_THREADS / 64) * 16;
constexpr int STP_TJ = 64;
constexpr int STP_KC = 16;
constexpr int STP_A_LD = STP_TJ + 16;            // table row stride in LDS (doubles): lane groups 0 / 1 on disjoint banks
constexpr int STP_ABUF = STP_KC * STP_A_LD;      // one parity's table chunk
static_assert(STP_KC * STP_TJ == 2 * STP_THREADS, "one 16-byte table piece per thread and parity");

// One workgroup per work item; the hardware dispatcher balances the uneven items
// (a persistent variant that prefetched across items measured slower).
struct stp_item {
    int j0, c0, nl, ne, no, nt_stores;
    __amdgpu_buffer_rsrc_t rs, rpe, rpo, ro;
};

// The tile with NB 16-node blocks: 4, or fewer for the last nodes of a hemisphere.
template <int NB>
__device__ __forceinline__ void stp_tile(const stp_item &cur, int nt, int nt2, int nrhs, double *__restrict__ Tb)
{
    const int tid = threadIdx.x, wave = tid >> 6, lane = tid & 63;
    const int li = lane & 15, lg = lane >> 4;
    // a wave whose columns all lie past nrhs only helps with the table
    const int wc = cur.c0 + 16 * wave;
    const bool active = uniform((int)(wc < nrhs)) != 0;
    // table pieces: row tk, nodes j0 + 2 tp, + 1 of each parity
    const int tk = tid >> 5, tp = tid & 31;
    const int t_at = tk * STP_A_LD + 2 * tp;
    const int tv = (tk * nt2 + cur.j0 + 2 * tp) * 8;
    double2 te, to;
    auto fetch_t = [&](int k0) {
        if (tp < 8 * NB) {
            te = load_f64x2(cur.rpe, tv + k0 * nt2 * 8);
            to = load_f64x2(cur.rpo, tv + k0 * nt2 * 8);
        }
    };
    auto settle_t = [&](int buf) {
        if (tp < 8 * NB) {
            double *T = Tb + buf * (2 * STP_ABUF) + t_at;
            *reinterpret_cast<double2 *>(T) = te;
            *reinterpret_cast<double2 *>(T + STP_ABUF) = to;
        }
    };
    // the lane's data pair of step s of the chunk at k0.  In the last chunk a pair may reach past
    // the column's last l (into the next column; what lies past the buffer reads 0): those
    // values are zeroed before they are used.
    const int dv = ((wc + li) * cur.nl + 2 * lg) * 8;
    double2 d[4];
    auto fetch_d = [&](int k0, int s) { d[s] = load_f64x2(cur.rs, dv + k0 * 16 + s * 64); };

    double4_t acc_e[NB], acc_o[NB];
#pragma unroll
    for (int b = 0; b < NB; ++b) {
        acc_e[b] = double4_t{0.0, 0.0, 0.0, 0.0};
        acc_o[b] = double4_t{0.0, 0.0, 0.0, 0.0};
    }
    const int klast = (cur.ne - 1) & ~(STP_KC - 1);  // the last chunk
    fetch_t(0);
    if (!active) {
        settle_t(0);
        for (int k0 = 0, buf = 1; k0 < klast; k0 += STP_KC, buf ^= 1) {
            __syncthreads();
            fetch_t(k0 + STP_KC);
            settle_t(buf);
        }
        __syncthreads();
        return;
    }
#pragma unroll
    for (int s = 0; s < 4; ++s) fetch_d(0, s);
    settle_t(0);
    int buf = 0;
    auto step = [&](const double *T, int s, double de, double dd) {
        const double *Te = T + (4 * s + lg) * STP_A_LD + li, *To = Te + STP_ABUF;
        double be[NB], bo[NB];
#pragma unroll
        for (int b = 0; b < NB; ++b) {
            be[b] = Te[16 * b];
            bo[b] = To[16 * b];
        }
#pragma unroll
        for (int b = 0; b < NB; ++b) {
            acc_e[b] = mfma_f64(de, be[b], acc_e[b]);
            acc_o[b] = mfma_f64(dd, bo[b], acc_o[b]);
        }
    };
    for (int k0 = 0; k0 < klast; k0 += STP_KC) {
        __syncthreads();
        // the other buffer was last read before this barrier
        fetch_t(k0 + STP_KC);
        const double *T = Tb + buf * (2 * STP_ABUF);
        buf ^= 1;
#pragma unroll
        for (int s = 0; s < 4; ++s) {
            step(T, s, d[s].x, d[s].y);
            if (s & 1) {  // the two loads of a 128-byte line together
                fetch_d(k0 + STP_KC, s - 1);
                fetch_d(k0 + STP_KC, s);
            }
            if (s == 2) settle_t(buf);
        }
    }
    // the last chunk: only the steps that hold a parity-l row
    __syncthreads();
    {
        const double *T = Tb + buf * (2 * STP_ABUF);
        const int ns = (cur.ne - klast + 3) >> 2, l = 2 * (klast + lg);
#pragma unroll
        for (int s = 0; s < 4; ++s)
            if (s < ns)
                step(T, s, l + 8 * s < cur.nl ? d[s].x : 0.0, l + 8 * s + 1 < cur.nl ? d[s].y : 0.0);
    }
    // Rows past nrhs lie past the buffer and are dropped; nodes past the equator (the last
    // block only) are skipped.
    const int vn = ((wc + lg) * nt + cur.j0 + li) * 8;                            // + 128 b
    const int vs = ((wc + lg) * nt + nt - 1 - cur.j0 - li - 16 * (NB - 1)) * 8;  // + 128 (NB - 1 - b)
    auto store = [&](auto put) {
#pragma unroll
        for (int v = 0; v < 4; ++v)
#pragma unroll
            for (int b = 0; b < NB; ++b)
                if (b < NB - 1 || cur.j0 + 16 * b + li < nt2) {
                    const double e = acc_e[b][v], o = acc_o[b][v];
                    put(cur.ro, vn + v * nt * 32 + 128 * b, e + o);
                    put(cur.ro, vs + v * nt * 32 + 128 * (NB - 1 - b), e - o);
                }
    };
    if (cur.nt_stores) store(store_f64_nt);
    else store(store_f64);
}

__global__ __launch_bounds__(STP_THREADS, kFp64MinWaves) void stp_fp64_kernel(
    const batch_io io, const fp64_item *__restrict__ work)
{
    __shared__ __align__(16) double Tb[2 * 2 * STP_ABUF];  // [buffer][parity] table chunks

    const fp64_item it = work[blockIdx.x];
    stp_item cur;
    cur.nl = uniform(it.nl);
    if (cur.nl == 0) return;  // padding item of the XCD-balanced schedule
    const int nt2 = uniform(it.nt2), nrhs = uniform(it.nrhs), pi = uniform(it.prob), nb = uniform(it.blocks);
    cur.j0 = uniform(it.r0);
    cur.c0 = uniform(it.c0);
    cur.nt_stores = uniform(it.nt_stores);
    cur.ne = (cur.nl + 1) >> 1;
    cur.no = cur.nl >> 1;
    cur.rs = make_rsrc(uniform(io.in[pi]) + uniform(it.s_off), (long)cur.nl * nrhs * 8);
    // one double more than the table: a 16-byte piece may start at its last value
    cur.rpe = make_rsrc(uniform(it.te), (long)cur.ne * nt2 * 8 + 8);
    cur.rpo = make_rsrc(uniform(it.to), (long)cur.no * nt2 * 8 + 8);
    cur.ro = make_rsrc(uniform(io.out[pi]) + uniform(it.p_off), (long)nrhs * 2 * nt2 * 8);
    switch (nb) {
    case 4: stp_tile<4>(cur, 2 * nt2, nt2, nrhs, Tb); break;
    case 3: stp_tile<3>(cur, 2 * nt2, nt2, nrhs, Tb); break;
    case 2: stp_tile<2>(cur, 2 * nt2, nt2, nrhs, Tb); break;
    default: stp_tile<1>(cur, 2 * nt2, nt2, nrhs, Tb); break;
    }
}

// ---------------------------------------------------------------- PtS
// Workgroup tile: (waves x 16) columns (c) x 64 parity-l values of each parity (128 l).
// Wave w owns 16 columns: NB l blocks x 2 parities of 16x16 accumulators.  K runs over
// chunks of 16 southern nodes.  As in StP a wave's data columns are its own and only the
// table chunk is shared: double-buffered in LDS, one barrier per chunk.  The order of the
// nodes inside a chunk is free as long as both operands follow it: step 2 h + q takes node
// j0 + 8 h + 2 lg + q on lane group lg, so one 16-byte load of a column and one of its mirror
// give a lane two steps of f(j) and f(nt+1-j); the fold f(j) +/- f(nt+1-j) forms the operands in
// registers, and the pair of loads for the next chunk goes out as soon as it has.
constexpr int PTS_THREADS = 512;
constexpr int PTS_TC = (PTS_THREADS / 64) * 16;
constexpr int PTS_TK = 64;             // parity-l rows of a full tile, per parity
constexpr int PTS_KJ = 16;             // nodes per K chunk: 4 MFMA steps of 4
constexpr int PTS_I_LD = PTS_TK + 4;   // table chunk row stride (doubles): lane groups 0 / 1 on disjoint banks
constexpr int PTS_IBUF = PTS_KJ * PTS_I_LD;  // one parity's table chunk in LDS
static_assert(PTS_KJ * PTS_TK == 2 * PTS_THREADS, "one 16-byte table piece per thread and parity");

struct pts_item {
    int k0, c0, nl, ne, no;
    __amdgpu_buffer_rsrc_t rp, rie, rio, ro;
};

// One PtS tile of NB 16-row blocks of each parity: 4, or fewer for the last rows of an
// m-block, which would leave part of a full tile idle.  Column pieces past nrhs read 0.
template <int NB>
__device__ __forceinline__ void pts_tile(const pts_item &cur, int nt, int nt2, int nrhs, double *__restrict__ Ib)
{
    const int tid = threadIdx.x, wave = tid >> 6, lane = tid & 63;
    const int li = lane & 15, lg = lane >> 4;
    // a wave whose columns all lie past nrhs only helps with the table
    const bool active = uniform((int)(cur.c0 + 16 * wave < nrhs)) != 0;
    const int c = cur.c0 + 16 * wave + li;
    const int va = (c * nt + 2 * lg) * 8;           // + 8 j0 + 64 h: nodes j, j + 1
    const int vb = (c * nt + nt - 2 - 2 * lg) * 8;  // - 8 j0 - 64 h: mirrors of j + 1, j
    double2 fa[2], fb[2];
    auto fetch_f = [&](int j0, int h) {
        fa[h] = load_f64x2(cur.rp, va + 8 * j0 + 64 * h);
        fb[h] = load_f64x2(cur.rp, vb - 8 * j0 - 64 * h);
    };
    // table pieces: parity-l row tk, nodes j0 + 2 tj, + 1, left at the chunk rows 4 lg + s of the
    // steps that use them
    const int tj = tid & 7, tk = tid >> 3;
    const int vt = ((cur.k0 + tk) * nt2 + 2 * tj) * 8;
    const int t_at = (4 * (tj & 3) + 2 * (tj >> 2)) * PTS_I_LD + tk;
    double2 te, to;
    auto fetch_t = [&](int j0) {
        if (NB == 4 || tk < 16 * NB) {
            te = load_f64x2(cur.rie, vt + 8 * j0);
            to = load_f64x2(cur.rio, vt + 8 * j0);
        }
    };
    auto settle_t = [&](int buf) {
        if (NB == 4 || tk < 16 * NB) {
            double *T = Ib + buf * (2 * PTS_IBUF) + t_at;
            T[0] = te.x;
            T[PTS_I_LD] = te.y;
            T[PTS_IBUF] = to.x;
            T[PTS_IBUF + PTS_I_LD] = to.y;
        }
    };

    double4_t acc_e[NB], acc_o[NB];
#pragma unroll
    for (int b = 0; b < NB; ++b) {
        acc_e[b] = double4_t{0.0, 0.0, 0.0, 0.0};
        acc_o[b] = double4_t{0.0, 0.0, 0.0, 0.0};
    }
    const int jlast = (nt2 - 1) & ~(PTS_KJ - 1);  // the last chunk
    fetch_t(0);
    if (!active) {
        settle_t(0);
        for (int j0 = 0, buf = 1; j0 < jlast; j0 += PTS_KJ, buf ^= 1) {
            __syncthreads();
            fetch_t(j0 + PTS_KJ);
            settle_t(buf);
        }
        __syncthreads();
        return;
    }
    fetch_f(0, 0);
    fetch_f(0, 1);
    settle_t(0);
    auto step = [&](const double *T, int s, double fe, double fo) {
        const double *Te = T + (4 * lg + s) * PTS_I_LD + li, *To = Te + PTS_IBUF;
        double be[NB], bo[NB];
#pragma unroll
        for (int b = 0; b < NB; ++b) {
            be[b] = Te[16 * b];
            bo[b] = To[16 * b];
        }
#pragma unroll
        for (int b = 0; b < NB; ++b) {
            acc_e[b] = mfma_f64(fe, be[b], acc_e[b]);
            acc_o[b] = mfma_f64(fo, bo[b], acc_o[b]);
        }
    };
    int buf = 0;
    for (int j0 = 0; j0 < jlast; j0 += PTS_KJ) {
        __syncthreads();
        // the other buffer was last read before this barrier
        fetch_t(j0 + PTS_KJ);
        // keep the loads where they are: the scheduler would sink them next to their uses
        __builtin_amdgcn_sched_barrier(0);
        const double *T = Ib + buf * (2 * PTS_IBUF);
        buf ^= 1;
#pragma unroll
        for (int h = 0; h < 2; ++h) {
            const double e0 = fa[h].x + fb[h].y, o0 = fa[h].x - fb[h].y;
            const double e1 = fa[h].y + fb[h].x, o1 = fa[h].y - fb[h].x;
            fetch_f(j0 + PTS_KJ, h);
            __builtin_amdgcn_sched_barrier(0);
            step(T, 2 * h, e0, o0);
            if (h == 1) settle_t(buf);
            step(T, 2 * h + 1, e1, o1);
        }
    }
    // the last chunk: nodes past the equator count as zeros
    __syncthreads();
    {
        const double *T = Ib + buf * (2 * PTS_IBUF);
#pragma unroll
        for (int h = 0; h < 2; ++h) {
            if (jlast + 8 * h >= nt2) break;
            const int j = jlast + 8 * h + 2 * lg;
            const bool in0 = j < nt2, in1 = j + 1 < nt2;
            step(T, 2 * h, in0 ? fa[h].x + fb[h].y : 0.0, in0 ? fa[h].x - fb[h].y : 0.0);
            step(T, 2 * h + 1, in1 ? fa[h].y + fb[h].x : 0.0, in1 ? fa[h].y - fb[h].x : 0.0);
        }
    }

    // l = m + 2 k and m + 2 k + 1 are neighbours: one 16-byte store; columns past nrhs lie past
    // the buffer and are dropped
    const int vo = ((cur.c0 + 16 * wave + lg) * cur.nl + 2 * (cur.k0 + li)) * 8;
#pragma unroll
    for (int v = 0; v < 4; ++v)
#pragma unroll
        for (int b = 0; b < NB; ++b) {
            const int k = cur.k0 + 16 * b + li, at = vo + v * cur.nl * 32 + 256 * b;
            if (k < cur.no) store_f64x2(cur.ro, at, make_double2(acc_e[b][v], acc_o[b][v]));
            else if (k < cur.ne) store_f64(cur.ro, at, acc_e[b][v]);
        }
}

__global__ __launch_bounds__(PTS_THREADS, kFp64MinWaves) void pts_fp64_kernel(
    const batch_io io, const fp64_item *__restrict__ work)
{
    __shared__ double Ib[2 * 2 * PTS_IBUF];  // [buffer][parity] table chunks

    const fp64_item it = work[blockIdx.x];
    pts_item cur;
    cur.nl = uniform(it.nl);
    if (cur.nl == 0) return;  // padding item of the XCD-balanced schedule
    const int nt2 = uniform(it.nt2), nrhs = uniform(it.nrhs), pi = uniform(it.prob), nb = uniform(it.blocks);
    const int nt = 2 * nt2;
    cur.k0 = uniform(it.r0);
    cur.c0 = uniform(it.c0);
    cur.ne = (cur.nl + 1) >> 1;
    cur.no = cur.nl >> 1;
    cur.rp = make_rsrc(uniform(io.in[pi]) + uniform(it.p_off), (long)nrhs * nt * 8);
    cur.ro = make_rsrc(uniform(io.out[pi]) + uniform(it.s_off), (long)nrhs * cur.nl * 8);
    // one double more than the table: a 16-byte piece may start at its last value
    cur.rie = make_rsrc(uniform(it.te), (long)cur.ne * nt2 * 8 + 8);
    cur.rio = make_rsrc(uniform(it.to), (long)cur.no * nt2 * 8 + 8);
    switch (nb) {
    case 4: pts_tile<4>(cur, nt, nt2, nrhs, Ib); break;
    case 3: pts_tile<3>(cur, nt, nt2, nrhs, Ib); break;
    case 2: pts_tile<2>(cur, nt, nt2, nrhs, Ib); break;
    default: pts_tile<1>(cur, nt, nt2, nrhs, Ib); break;
    }
}

}  // namespace

int launch_stp_fp64_batch(const batch_io &io, const fp64_item *work, int n_work, hipStream_t st)
{
    if (n_work == 0) return RAYSHT_OK;
    hipLaunchKernelGGL(stp_fp64_kernel, dim3(n_work), dim3(STP_THREADS), 0, st, io, work);
    RAYSHT_HIP_TRY(hipGetLastError());
    return RAYSHT_OK;
}

int launch_pts_fp64_batch(const batch_io &io, const fp64_item *work, int n_work, hipStream_t st)
{
    if (n_work == 0) return RAYSHT_OK;
    hipLaunchKernelGGL(pts_fp64_kernel, dim3(n_work), dim3(PTS_THREADS), 0, st, io, work);
    RAYSHT_HIP_TRY(hipGetLastError());
    return RAYSHT_OK;
}

int launch_stp_fp64(raysht_plan *p, const double *s, double *p2, hipStream_t st)
{
    batch_io io{};
    io.in[0] = s;
    io.out[0] = p2;
    return launch_stp_fp64_batch(io, p->d_work_stp, p->n_work_stp, st);
}

int launch_pts_fp64(raysht_plan *p, const double *p2, double *s, hipStream_t st)
{
    batch_io io{};
    io.in[0] = p2;
    io.out[0] = s;
    return launch_pts_fp64_batch(io, p->d_work_pts, p->n_work_pts, st);
}

// Tile geometry the host work lists are built with.
int stp_tile_rows() { return STP_TJ; }
int stp_tile_cols() { return STP_TC; }
int pts_tile_rows() { return PTS_TK; }
int pts_tile_cols() { return PTS_TC; }

}  // namespace raysht
