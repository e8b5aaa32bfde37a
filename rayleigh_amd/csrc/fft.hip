// Batched in-place real FFTs along phi and the one-rank row permutes around them.
//
// FFT_To_Physical / FFT_To_Spectral (Fourier_Transform.F90:56-183) run FFTW's
// unnormalised c2r (e^{+i}) / r2c (e^{-i}) in place on lines of nphi+2 doubles
// holding Re/Im of m = 0..nphi/2.  A length-nphi real transform is done as a
// length-nphi/2 complex transform plus the usual even/odd split pass.  All are bound by HBM
// and hold the line in registers, exchanging through LDS: nphi/2 = 3 * 2^k (Rayleigh's
// nphi = 3 (l_max + 1)) and 2^k with everything known at compile time, other even lengths
// 2^a 3^b 5^c 7^d with a run-time schedule of radices 2 to 16.
//
// Transpose_2a3a / 3b2b (Spherical_Buffer.F90:196-703) reduce on one rank to
// pure index maps between the hybrid layout p2[mp][c][theta] and the physical
// layout p3[f][theta][r][nphi+2]; the m > l_max part of every line is zero after
// 2a->3a, which is Rayleigh's implicit de-aliasing in phi.
#include <algorithm>
#include <map>
#include <mutex>
#include <type_traits>
#include <utility>

#include "raysht_internal.h"

// The hybrid intermediate of raysht_spectral_to_physical_scratch: a file-scope device array,
// one copy per GPU, held until the process ends.  Host code never passes this name to a
// kernel or a copy (on the host it is only a stand-in for the symbol): it uses the device
// address that hipGetSymbolAddress gives for the current device (scratch_address below).
static __device__ __align__(256) double scratch[RAYSHT_SCRATCH_BYTES / sizeof(double)];

namespace raysht {
namespace {

// Every product that is fused into a sum is written as one (fma): left to the compiler, which
// products it fuses depends on the code around an inlined transform, and the fused reform
// kernels must give the doubles of the separate calls.
#pragma clang fp contract(off)

struct cplx {
    double re, im;
};

__host__ __device__ __forceinline__ double fm(double a, double b, double c) { return __builtin_fma(a, b, c); }
__host__ __device__ __forceinline__ cplx cmul(cplx a, cplx b)
{
    return {fm(a.re, b.re, -(a.im * b.im)), fm(a.re, b.im, a.im * b.re)};
}
__host__ __device__ __forceinline__ cplx cadd(cplx a, cplx b) { return {a.re + b.re, a.im + b.im}; }
__host__ __device__ __forceinline__ cplx csub(cplx a, cplx b) { return {a.re - b.re, a.im - b.im}; }
__host__ __device__ __forceinline__ cplx cconj(cplx a) { return {a.re, -a.im}; }

constexpr int kMaxHalf = 4096;  // largest complex length (nphi/2)

// cos / sin of 2 pi k / 5 and 2 pi k / 7 (k = 1, 2 / 1, 2, 3), the constants of the radix-5
// and radix-7 butterflies
constexpr double kC51 = 0.3090169943749474241022934171828190588602, kS51 = 0.9510565162951535721164393333793821434783;
constexpr double kC52 = -0.8090169943749474241022934171828190588602, kS52 = 0.5877852522924731291687059546390727685978;
constexpr double kC71 = 0.6234898018587335305250048840042398106324, kS71 = 0.7818314824680298087084445266740577502325;
constexpr double kC72 = -0.2225209339563144042889025644967947594664, kS72 = 0.9749279121818236070181316829939312172327;
constexpr double kC73 = -0.9009688679024191262361023195074450511660, kS73 = 0.4338837391175581204757683328483587546099;

// y_k = sum_r v_r e^{sign 2 pi i r k / 5}: with t = v1 + v4, v2 + v3 and u = v1 - v4, v2 - v3,
// y_1,4 = v0 + c1 t1 + c2 t2 +- i sign (s1 u1 + s2 u2), y_2,3 = v0 + c2 t1 + c1 t2 +- i sign (s2 u1 - s1 u2)
__host__ __device__ __forceinline__ void dft5(const cplx (&v)[5], cplx (&y)[5], int sign)
{
    const cplx t1 = cadd(v[1], v[4]), t2 = cadd(v[2], v[3]), u1 = csub(v[1], v[4]), u2 = csub(v[2], v[3]);
    y[0] = cadd(v[0], cadd(t1, t2));
    const cplx a1 = {fm(kC52, t2.re, fm(kC51, t1.re, v[0].re)), fm(kC52, t2.im, fm(kC51, t1.im, v[0].im))};
    const cplx a2 = {fm(kC51, t2.re, fm(kC52, t1.re, v[0].re)), fm(kC51, t2.im, fm(kC52, t1.im, v[0].im))};
    const cplx b1 = {fm(kS51, u1.re, kS52 * u2.re), fm(kS51, u1.im, kS52 * u2.im)};
    const cplx b2 = {fm(kS52, u1.re, -(kS51 * u2.re)), fm(kS52, u1.im, -(kS51 * u2.im))};
    const cplx ib1 = {-sign * b1.im, sign * b1.re}, ib2 = {-sign * b2.im, sign * b2.re};
    y[1] = cadd(a1, ib1);
    y[4] = csub(a1, ib1);
    y[2] = cadd(a2, ib2);
    y[3] = csub(a2, ib2);
}

// the same for 7: t_k = v_k + v_{7-k}, u_k = v_k - v_{7-k} (k = 1, 2, 3),
// y_j, y_{7-j} = v0 + sum_k cos(2 pi j k / 7) t_k +- i sign sum_k sin(2 pi j k / 7) u_k
__host__ __device__ __forceinline__ void dft7(const cplx (&v)[7], cplx (&y)[7], int sign)
{
    const cplx t1 = cadd(v[1], v[6]), t2 = cadd(v[2], v[5]), t3 = cadd(v[3], v[4]);
    const cplx u1 = csub(v[1], v[6]), u2 = csub(v[2], v[5]), u3 = csub(v[3], v[4]);
    y[0] = cadd(v[0], cadd(t1, cadd(t2, t3)));
    // cos / sin of 2 pi j k / 7 for j = 1, 2, 3 and k = 1, 2, 3 (jk mod 7 folded into 1..3 with signs)
    const double C[3][3] = {{kC71, kC72, kC73}, {kC72, kC73, kC71}, {kC73, kC71, kC72}};
    const double S[3][3] = {{kS71, kS72, kS73}, {kS72, -kS73, -kS71}, {kS73, -kS71, kS72}};
#pragma unroll
    for (int j = 0; j < 3; ++j) {
        const cplx a = {fm(C[j][2], t3.re, fm(C[j][1], t2.re, fm(C[j][0], t1.re, v[0].re))),
                        fm(C[j][2], t3.im, fm(C[j][1], t2.im, fm(C[j][0], t1.im, v[0].im)))};
        const cplx b = {fm(S[j][2], u3.re, fm(S[j][1], u2.re, S[j][0] * u1.re)),
                        fm(S[j][2], u3.im, fm(S[j][1], u2.im, S[j][0] * u1.im))};
        const cplx ib = {-sign * b.im, sign * b.re};
        y[j + 1] = cadd(a, ib);
        y[6 - j] = csub(a, ib);
    }
}

// ---------------------------------------------------------------------------
// Register-resident real FFTs for the line lengths with n2 = nphi / 2 = 3 * 2^k (24 .. 3072,
// Rayleigh's nphi = 3 (l_max + 1)) and n2 = 2^k (16 .. 4096).  The complex length-n2 transform
// runs as radix-8 Stockham passes followed by one pass of the radix that is left (3, 6 or 12;
// 4, 8 or 16), all sizes and strides compile-time: every thread holds P points of one line in
// registers (24 or 16), n2 / P threads share a line, and the passes exchange through LDS.
// The exchange moves the real parts and then the imaginary parts through the same buffer:
// with 8 bytes per point instead of 16 the LDS of a wave is 13 KB (3 * 2^k) or 9 KB (2^k), so
// 12 or 16 waves fit a CU's LDS where 6 did, and these kernels wait for memory most of the time.
// On 1.6 GB of lines (read and written once): c2r 3.5 - 4.5 TB/s, r2c 4.3 - 5.2 TB/s; before, 3 * 2^k
// ran at 2.7 - 3.9 and 4.1 - 5.1, and 2^k, in the LDS kernel for any length, at 1.0 - 2.0.
// The buffer is padded by one double in 8, 16 or 32 (the best of the three for a length's
// strides; at most 1.75 passes of 32 lanes per access instead of 1).  Lines of up to 64
// threads lie in one wave, so their exchanges need no workgroup barrier.  The
// real-to-complex packing rides on the first pass (c2r) or a final exchange (r2c), so each
// line is read and written in HBM exactly once.

__host__ __device__ constexpr int fft_points(int n) { return n % 3 == 0 ? 24 : 16; }

__host__ __device__ constexpr int fft_n8(int n)  // radix-8 passes before the last
{
    int a = 0;
    if (n % 3 == 0) {
        while (n % 8 == 0 && n / 8 >= 3 && (n / 8 == 3 || n / 8 == 6 || n / 8 == 12 || n / 8 >= 24)) {
            n /= 8;
            ++a;
        }
    } else {
        while (n > 16) {  // leaves 16, 8 or 4
            n /= 8;
            ++a;
        }
    }
    return a;
}
__host__ __device__ constexpr int pow8(int a) { return a == 0 ? 1 : 8 * pow8(a - 1); }
__host__ __device__ constexpr int fft_last(int n) { return n / pow8(fft_n8(n)); }
__host__ __device__ constexpr bool fft_reg_ok(int n)
{
    return n >= fft_points(n) && n % fft_points(n) == 0 && fft_points(n) % fft_last(n) == 0 && fft_last(n) >= 3 &&
           pow8(fft_n8(n)) * fft_last(n) == n;
}

// everything compile-time about one length: P points per thread, T threads per line, A
// radix-8 passes and one of radix F, R0 the first pass's radix, LDS padding and line stride
template <int N>
struct fft_geom {
    static constexpr int P = fft_points(N), T = N / P, A = fft_n8(N), F = fft_last(N), R0 = A > 0 ? 8 : F;
    static constexpr int SH = T == 16 ? 4 : T >= 64 ? 5 : 3;
    static constexpr int WANT = T <= 16 ? T : 0;  // line stride mod 32: the lines of a wave on other banks
    static constexpr int RAW = (N - 1) + ((N - 1) >> SH) + 1;
    static constexpr int STRIDE = RAW + ((WANT - RAW) % 32 + 32) % 32;
    static constexpr int THREADS = T > 64 ? T : 64;  // a workgroup of the in-place kernels
    static constexpr int WAVES = P == 24 ? 2 : 3;    // per SIMD: at most 256 or 168 VGPRs
    static_assert(fft_reg_ok(N), "length without a register-resident schedule");
    static_assert((T & (T - 1)) == 0, "index splitting below");
    __device__ static __forceinline__ int pad(int i) { return i + (i >> SH); }
    // pad(i + c) for a constant c >= 0 or c < 0 (after unrolling): one address per i and an
    // immediate where c is a multiple of the padding's period, instead of an address per c
    __device__ static __forceinline__ int pad(int i, int c)
    {
        return c % (1 << SH) == 0 ? pad(i) + c + (c / (1 << SH)) : pad(i + c);
    }
    // (b / NS) NS R + b % NS for b = t + T u, t < T, in a part of t and a constant part
    template <int R, int NS>
    __device__ static __forceinline__ int out_t(int t)
    {
        return T % NS == 0 ? (t / NS) * NS * R + (t & (NS - 1)) : t;
    }
    template <int R, int NS>
    __device__ static __forceinline__ constexpr int out_u(int u)
    {
        return T % NS == 0 ? T * R * u : (T * u / NS) * NS * R + (T * u) % NS;
    }
    // b % NS for the same b
    template <int NS>
    __device__ static __forceinline__ int low(int t, int u)
    {
        return T % NS == 0 ? t & (NS - 1) : t + (T * u) % NS;
    }
};

// LDS written by a line's threads before this is visible to them after it
template <int N>
__device__ __forceinline__ void line_sync()
{
    if constexpr (fft_geom<N>::T <= 64) {
        // one wave: its LDS instructions run in order, only the compiler must keep the order
        __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
        __builtin_amdgcn_wave_barrier();
        __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
    } else {
        __syncthreads();
    }
}

// in-place small DFTs, y_k = sum_n v_n e^{sign 2 pi i n k / R}
__host__ __device__ __forceinline__ cplx mul_i(cplx a, int sign) { return {-sign * a.im, sign * a.re}; }

__host__ __device__ __forceinline__ void dft3(cplx &a0, cplx &a1, cplx &a2, int sign)
{
    const double h = 0.8660254037844386467637231707529361834714;  // sqrt(3)/2
    const cplx t1 = cadd(a1, a2);
    const cplx t2 = {fm(-0.5, t1.re, a0.re), fm(-0.5, t1.im, a0.im)};
    const cplx d0 = csub(a1, a2);
    const cplx t3 = {-sign * h * d0.im, sign * h * d0.re};
    a0 = cadd(a0, t1);
    a1 = cadd(t2, t3);
    a2 = csub(t2, t3);
}

__host__ __device__ __forceinline__ void dft4(cplx &a0, cplx &a1, cplx &a2, cplx &a3, int sign)
{
    const cplx a = cadd(a0, a2), b = csub(a0, a2);
    const cplx c = cadd(a1, a3), d = mul_i(csub(a1, a3), sign);
    a0 = cadd(a, c);
    a1 = cadd(b, d);
    a2 = csub(a, c);
    a3 = csub(b, d);
}

__host__ __device__ __forceinline__ void dft8(cplx (&v)[8], int sign)
{
    cplx e0 = v[0], e1 = v[2], e2 = v[4], e3 = v[6], o0 = v[1], o1 = v[3], o2 = v[5], o3 = v[7];
    dft4(e0, e1, e2, e3, sign);
    dft4(o0, o1, o2, o3, sign);
    const double r2 = 0.7071067811865475244008443621048490392848;  // 1/sqrt(2)
    const cplx t1 = cmul(o1, cplx{r2, sign * r2});
    const cplx t2 = mul_i(o2, sign);
    const cplx t3 = cmul(o3, cplx{-r2, sign * r2});
    v[0] = cadd(e0, o0), v[4] = csub(e0, o0);
    v[1] = cadd(e1, t1), v[5] = csub(e1, t1);
    v[2] = cadd(e2, t2), v[6] = csub(e2, t2);
    v[3] = cadd(e3, t3), v[7] = csub(e3, t3);
}

__host__ __device__ __forceinline__ void dft6(cplx (&v)[6], int sign)
{
    cplx e0 = v[0], e1 = v[2], e2 = v[4], o0 = v[1], o1 = v[3], o2 = v[5];
    dft3(e0, e1, e2, sign);
    dft3(o0, o1, o2, sign);
    const double h = 0.8660254037844386467637231707529361834714;
    const cplx t1 = cmul(o1, cplx{0.5, sign * h});   // e^{sign 2 pi i / 6}
    const cplx t2 = cmul(o2, cplx{-0.5, sign * h});  // e^{sign 4 pi i / 6}
    v[0] = cadd(e0, o0), v[3] = csub(e0, o0);
    v[1] = cadd(e1, t1), v[4] = csub(e1, t1);
    v[2] = cadd(e2, t2), v[5] = csub(e2, t2);
}

__host__ __device__ __forceinline__ void dft12(cplx (&v)[12], int sign)
{
    cplx e[6] = {v[0], v[2], v[4], v[6], v[8], v[10]}, o[6] = {v[1], v[3], v[5], v[7], v[9], v[11]};
    dft6(e, sign);
    dft6(o, sign);
    const double h = 0.8660254037844386467637231707529361834714;
    const cplx w[6] = {{1.0, 0.0},  {h, sign * 0.5},  {0.5, sign * h},
                       {0.0, 1.0 * sign}, {-0.5, sign * h}, {-h, sign * 0.5}};  // e^{sign 2 pi i k / 12}
#pragma unroll
    for (int k = 0; k < 6; ++k) {
        const cplx t = k == 0 ? o[0] : cmul(o[k], w[k]);
        v[k] = cadd(e[k], t);
        v[k + 6] = csub(e[k], t);
    }
}

__host__ __device__ __forceinline__ void dft16(cplx (&v)[16], int sign)
{
    cplx e[8] = {v[0], v[2], v[4], v[6], v[8], v[10], v[12], v[14]};
    cplx o[8] = {v[1], v[3], v[5], v[7], v[9], v[11], v[13], v[15]};
    dft8(e, sign);
    dft8(o, sign);
    const double c1 = 0.9238795325112867561281831893967882868224;  // cos(pi/8)
    const double s1 = 0.3826834323650897717284599840303988667613;  // sin(pi/8)
    const double r2 = 0.7071067811865475244008443621048490392848;  // 1/sqrt(2)
    // e^{sign 2 pi i k / 16}
    const cplx w[8] = {{1.0, 0.0}, {c1, sign * s1}, {r2, sign * r2}, {s1, sign * c1},
                       {0.0, 1.0 * sign}, {-s1, sign * c1}, {-r2, sign * r2}, {-c1, sign * s1}};
#pragma unroll
    for (int k = 0; k < 8; ++k) {
        const cplx t = k == 0 ? o[0] : k == 4 ? mul_i(o[4], sign) : cmul(o[k], w[k]);
        v[k] = cadd(e[k], t);
        v[k + 8] = csub(e[k], t);
    }
}

__host__ __device__ __forceinline__ void dft9(cplx (&v)[9], int sign)
{
    // 3 x 3: columns n1 = 0, 1, 2 of elements n1 + 3 n2, twiddles e^{sign 2 pi i n1 k2 / 9}, then rows
    const double c1 = 0.7660444431189780352023926505554166739358, s1 = 0.6427876096865393263226434099072632329083;
    const double c2 = 0.1736481776669303488517166267693147215837, s2 = 0.9848077530122080593667430245895230136705;
    const double c4 = -0.9396926207859083840541092773247314699361, s4 = 0.3420201433256687330440996146822595807630;
    dft3(v[0], v[3], v[6], sign);
    dft3(v[1], v[4], v[7], sign);
    dft3(v[2], v[5], v[8], sign);
    v[4] = cmul(v[4], cplx{c1, sign * s1});
    v[7] = cmul(v[7], cplx{c2, sign * s2});
    v[5] = cmul(v[5], cplx{c2, sign * s2});
    v[8] = cmul(v[8], cplx{c4, sign * s4});
    dft3(v[0], v[1], v[2], sign);  // k = 3 k1 + k2 with k2 = 0, in v[k1]
    dft3(v[3], v[4], v[5], sign);
    dft3(v[6], v[7], v[8], sign);
    cplx y[9];
#pragma unroll
    for (int k1 = 0; k1 < 3; ++k1)
#pragma unroll
        for (int k2 = 0; k2 < 3; ++k2) y[3 * k1 + k2] = v[3 * k2 + k1];
#pragma unroll
    for (int k = 0; k < 9; ++k) v[k] = y[k];
}

template <int R>
__host__ __device__ __forceinline__ void dft_r(cplx (&v)[R], int sign);

// R = A B with A and B coprime (Good-Thomas): element (B n1 + A n2) mod R, a DFT of length B over
// n2 and one of length A over n1, result (k1, k2) at the k with k mod A = k1, k mod B = k2; no
// twiddles, since e^{2 pi i (B n1 + A n2) k / R} = e^{2 pi i n1 k / A} e^{2 pi i n2 k / B}
template <int A, int B>
__host__ __device__ __forceinline__ void dft_coprime(cplx (&v)[A * B], int sign)
{
    constexpr int R = A * B;
    cplx y[A][B];
#pragma unroll
    for (int n1 = 0; n1 < A; ++n1) {
#pragma unroll
        for (int n2 = 0; n2 < B; ++n2) y[n1][n2] = v[(B * n1 + A * n2) % R];
        dft_r<B>(y[n1], sign);
    }
#pragma unroll
    for (int k2 = 0; k2 < B; ++k2) {
        cplx z[A];
#pragma unroll
        for (int n1 = 0; n1 < A; ++n1) z[n1] = y[n1][k2];
        dft_r<A>(z, sign);
#pragma unroll
        for (int n1 = 0; n1 < A; ++n1) y[n1][k2] = z[n1];
    }
#pragma unroll
    for (int k = 0; k < R; ++k) v[k] = y[k % A][k % B];
}

template <int R>
__host__ __device__ __forceinline__ void dft_r(cplx (&v)[R], int sign)
{
    if constexpr (R == 16) dft16(v, sign);
    else if constexpr (R == 15) dft_coprime<3, 5>(v, sign);
    else if constexpr (R == 14) dft_coprime<2, 7>(v, sign);
    else if constexpr (R == 12) dft12(v, sign);
    else if constexpr (R == 10) dft_coprime<2, 5>(v, sign);
    else if constexpr (R == 9) dft9(v, sign);
    else if constexpr (R == 8) dft8(v, sign);
    else if constexpr (R == 6) dft6(v, sign);
    else if constexpr (R == 4) dft4(v[0], v[1], v[2], v[3], sign);
    else if constexpr (R == 3) dft3(v[0], v[1], v[2], sign);
    else if constexpr (R == 5 || R == 7) {
        cplx y[R];
        if constexpr (R == 5) dft5(v, y, sign);
        else dft7(v, y, sign);
#pragma unroll
        for (int k = 0; k < R; ++k) v[k] = y[k];
    } else {
        static_assert(R == 2, "no butterfly of this radix");
        const cplx a = v[0];
        v[0] = cadd(a, v[1]);
        v[1] = csub(a, v[1]);
    }
}

// Keeps the scheduler from hoisting the loads (twiddles, rows, buffer) of all of a thread's
// P points to the front, which takes 200 to 330 VGPRs and leaves one wave per SIMD: group u of R
// points starts after about eight points before it are done.
template <int R>
__device__ __forceinline__ void group_barrier(int u)
{
    if (u > 0 && (u * R) % 8 < R) __builtin_amdgcn_sched_barrier(0);
}

// One Stockham pass of radix R with input stride NS over the thread's P points:
// butterfly u (b = t + T u) takes in[u*R + r] = element b + r N/R, twiddles input r by
// e^{sign 2 pi i r (b mod NS) / (NS R)} (table of e^{2 pi i v / 2N}), and leaves
// out element (b / NS) NS R + b mod NS + r NS in v[u*R + r].
template <int N, int R, int NS>
__device__ __forceinline__ void fft_pass(cplx (&v)[fft_geom<N>::P], int t, const double2 *__restrict__ tw, int sign)
{
    constexpr int P = fft_geom<N>::P;
#pragma unroll
    for (int u = 0; u < P / R; ++u) {
        group_barrier<R>(u);
        const int k = fft_geom<N>::template low<NS>(t, u);  // (t + T u) mod NS
        cplx y[R];
#pragma unroll
        for (int r = 0; r < R; ++r) {
            y[r] = v[u * R + r];
            if (NS > 1 && r > 0) {
                const double2 w = tw[2 * r * k * (N / (NS * R))];
                y[r] = cmul(y[r], cplx{w.x, sign * w.y});
            }
        }
        dft_r<R>(y, sign);
#pragma unroll
        for (int r = 0; r < R; ++r) v[u * R + r] = y[r];
    }
}

// the points of the pass (R, NS) in v to the order the next pass, of radix R2, takes them in,
// one part (0 real, 1 imaginary) at a time through the line's buffer
template <int N, int R, int NS, int R2>
__device__ __forceinline__ void fft_exchange(double *__restrict__ buf, cplx (&v)[fft_geom<N>::P], int t)
{
    using G = fft_geom<N>;
    constexpr int T = G::T, P = G::P;
    const int o = G::template out_t<R, NS>(t);
#pragma unroll
    for (int part = 0; part < 2; ++part) {
#pragma unroll
        for (int u = 0; u < P / R; ++u)
#pragma unroll
            for (int r = 0; r < R; ++r)
                buf[G::pad(o, G::template out_u<R, NS>(u) + r * NS)] = part ? v[u * R + r].im : v[u * R + r].re;
        line_sync<N>();
#pragma unroll
        for (int u = 0; u < P / R2; ++u)
#pragma unroll
            for (int r = 0; r < R2; ++r) {
                const double x = buf[G::pad(t, T * u + r * (N / R2))];
                if (part) v[u * R2 + r].im = x;
                else v[u * R2 + r].re = x;
            }
        line_sync<N>();
    }
}

// the radix-8 passes P8 .. A-1 and the last pass, each after its exchange; pass 0 is done by
// the caller
template <int N, int P8>
__device__ __forceinline__ void fft_middle(double *__restrict__ buf, cplx (&v)[fft_geom<N>::P], int t,
                                           const double2 *__restrict__ tw, int sign)
{
    constexpr int A = fft_geom<N>::A, F = fft_geom<N>::F;
    if constexpr (P8 < A) {
        constexpr int NS = pow8(P8);
        fft_exchange<N, 8, NS / 8, 8>(buf, v, t);
        fft_pass<N, 8, NS>(v, t, tw, sign);
        fft_middle<N, P8 + 1>(buf, v, t, tw, sign);
    } else if constexpr (A > 0) {
        constexpr int NS = pow8(A);
        fft_exchange<N, 8, NS / 8, F>(buf, v, t);
        fft_pass<N, F, NS>(v, t, tw, sign);
    }
}

// z_k = A_k + i B_k of a c2r, A = X_k + conj X_{N-k}, B = (X_k - conj X_{N-k}) e^{2 pi i k / 2N},
// from a = X_k and bc = conj X_{N-k}
__device__ __forceinline__ cplx c2r_pack(cplx a, cplx bc, double2 w)
{
    const cplx Ak = cadd(a, bc);
    const cplx Bk = cmul(csub(a, bc), cplx{w.x, w.y});
    return {Ak.re - Bk.im, Ak.im + Bk.re};
}

// X_k = (Z_k + conj Z_{N-k}) / 2 - i e^{-2 pi i k / 2N} (Z_k - conj Z_{N-k}) / 2 of an r2c, from zk = Z_k
// and zn = Z_{N-k}, w = e^{2 pi i k / 2N}
__device__ __forceinline__ cplx r2c_unpack(cplx zk, cplx zn, double2 w)
{
    const cplx zc = cconj(zn);
    const cplx E = {0.5 * (zk.re + zc.re), 0.5 * (zk.im + zc.im)};
    const cplx D = csub(zk, zc);
    const cplx O = {0.5 * D.im, -0.5 * D.re};
    return cadd(E, cmul(O, cplx{w.x, -w.y}));
}

// c2r: z_k from the line's modes, inverse length-N FFT, x_{2n} + i x_{2n+1} = z_n.
template <int N>
__global__ __launch_bounds__(fft_geom<N>::THREADS, fft_geom<N>::WAVES) void fft_reg_c2r_kernel(
    long howmany, double *__restrict__ x, const double2 *__restrict__ tw)
{
    using G = fft_geom<N>;
    constexpr int T = G::T, LPB = G::THREADS / T;
    __shared__ double lds[LPB * G::STRIDE];
    const int t = threadIdx.x % T, li = threadIdx.x / T;
    const long line = (long)blockIdx.x * LPB + li;
    if (line >= howmany) return;  // whole lines: the synchronisations below see only complete lines
    double *xl = x + line * (2L * N + 2);
    double *buf = lds + li * G::STRIDE;
    cplx v[G::P];
#pragma unroll
    for (int u = 0; u < G::P / G::R0; ++u) {
        group_barrier<G::R0>(u);
#pragma unroll
        for (int r = 0; r < G::R0; ++r) {
            const int k = t + T * u + r * (N / G::R0);
            const double2 xa = reinterpret_cast<const double2 *>(xl)[k];
            const double2 xb = reinterpret_cast<const double2 *>(xl)[N - k];
            // Im X_0 and Im X_N do not enter
            v[u * G::R0 + r] = c2r_pack(cplx{xa.x, k == 0 ? 0.0 : xa.y}, cplx{xb.x, k == 0 ? 0.0 : -xb.y}, tw[k]);
        }
    }
    fft_pass<N, G::R0, 1>(v, t, tw, +1);
    fft_middle<N, 1>(buf, v, t, tw, +1);
    constexpr int NSL = N / G::F;
#pragma unroll
    for (int u = 0; u < G::P / G::F; ++u)
#pragma unroll
        for (int r = 0; r < G::F; ++r)
            reinterpret_cast<double2 *>(xl)[t + T * u + r * NSL] =
                make_double2(v[u * G::F + r].re, v[u * G::F + r].im);
    if (t == 0) reinterpret_cast<double2 *>(xl)[N] = make_double2(0.0, 0.0);
}

// After the last pass of an r2c: zk[u] = Z_k and zn[u] = Z_{(N-k) % N} for k = t + T u <= N / 2 (the
// last u holds k = N / 2, thread 0's alone), through the line's buffer: real parts, then
// imaginary parts.
template <int N>
__device__ __forceinline__ void r2c_pairs(double *__restrict__ buf, const cplx (&v)[fft_geom<N>::P],
                                          cplx (&zk)[fft_geom<N>::P / 2 + 1], cplx (&zn)[fft_geom<N>::P / 2 + 1], int t)
{
    using G = fft_geom<N>;
    constexpr int NSL = N / G::F;
#pragma unroll
    for (int part = 0; part < 2; ++part) {
#pragma unroll
        for (int u = 0; u < G::P / G::F; ++u)
#pragma unroll
            for (int r = 0; r < G::F; ++r)
                buf[G::pad(t, G::T * u + r * NSL)] = part ? v[u * G::F + r].im : v[u * G::F + r].re;
        line_sync<N>();
#pragma unroll
        for (int u = 0; u <= G::P / 2; ++u) {
            // the last u: k = N / 2 for every thread; u = 0: Z_N is Z_0
            const double a = u < G::P / 2 ? buf[G::pad(t, G::T * u)] : buf[G::pad(N / 2)];
            const double b = u == 0          ? buf[G::pad(t == 0 ? 0 : N - t)]
                             : u < G::P / 2 ? buf[G::pad(N - t, -G::T * u)]
                                            : buf[G::pad(N / 2)];
            if (part) {
                zk[u].im = a;
                zn[u].im = b;
            } else {
                zk[u].re = a;
                zn[u].re = b;
            }
        }
        line_sync<N>();
    }
}

// r2c: z_n = x_{2n} + i x_{2n+1}, forward length-N FFT, then X_k of r2c_unpack, k = 0..N.
template <int N>
__global__ __launch_bounds__(fft_geom<N>::THREADS, fft_geom<N>::WAVES) void fft_reg_r2c_kernel(
    long howmany, double *__restrict__ x, const double2 *__restrict__ tw, int rescale)
{
    using G = fft_geom<N>;
    constexpr int T = G::T, LPB = G::THREADS / T;
    __shared__ double lds[LPB * G::STRIDE];
    const int t = threadIdx.x % T, li = threadIdx.x / T;
    const long line = (long)blockIdx.x * LPB + li;
    if (line >= howmany) return;
    double *xl = x + line * (2L * N + 2);
    double *buf = lds + li * G::STRIDE;
    cplx v[G::P], zk[G::P / 2 + 1], zn[G::P / 2 + 1];
#pragma unroll
    for (int u = 0; u < G::P / G::R0; ++u)
#pragma unroll
        for (int r = 0; r < G::R0; ++r) {
            const double2 z = reinterpret_cast<const double2 *>(xl)[t + T * u + r * (N / G::R0)];
            v[u * G::R0 + r] = {z.x, z.y};
        }
    fft_pass<N, G::R0, 1>(v, t, tw, -1);
    fft_middle<N, 1>(buf, v, t, tw, -1);
    r2c_pairs<N>(buf, v, zk, zn, t);
    auto put = [&](int k, cplx X) {
        double re = X.re, im = X.im;
        if (rescale) {
            // r2c_ip4D_fftw_rsc: X(k > 0) / nphi, Re X_0 / (2 nphi), Im X_0 untouched
            re = k == 0 ? re / (4.0 * N) : re / (2.0 * N);
            if (k > 0) im = im / (2.0 * N);
        }
        reinterpret_cast<double2 *>(xl)[k] = make_double2(re, im);
    };
    if constexpr (G::P == 24 && T <= 4) {
        // each lane has its line nearly to itself: from one end to the other its stores fill one
        // cache line after the next, in pairs from both ends they come back to each later (192 MB
        // of lines, N = 24, 48, 96: 78, 73, 68 us in pairs, 75, 67, 62 in order; for P = 16 pairs are as
        // fast or faster)
        cplx xk[G::P / 2 + 1], xn[G::P / 2 + 1];
#pragma unroll
        for (int u = 0; u <= G::P / 2; ++u) {
            group_barrier<2>(u);
            const int k = u < G::P / 2 ? t + T * u : N / 2;
            xk[u] = r2c_unpack(zk[u], zn[u], tw[k]);
            xn[u] = r2c_unpack(zn[u], zk[u], tw[N - k]);
        }
#pragma unroll
        for (int u = 0; u < G::P / 2; ++u) put(t + T * u, xk[u]);
        if (t == 0) put(N / 2, xk[G::P / 2]);
#pragma unroll
        for (int u = G::P / 2 - 1; u >= 0; --u) put(N - t - T * u, xn[u]);
        return;
    }
#pragma unroll
    for (int u = 0; u <= G::P / 2; ++u) {
        group_barrier<2>(u);
        const int k = u < G::P / 2 ? t + T * u : N / 2;
        if (u == G::P / 2 && t > 0) continue;
        put(k, r2c_unpack(zk[u], zn[u], tw[k]));
        if (k != N / 2) put(N - k, r2c_unpack(zn[u], zk[u], tw[N - k]));  // k = 0: X_N, Z_N = Z_0
    }
}

// ---------------------------------------------------------------------------
// Every other length, n2 = 2^a 3^b 5^c 7^d <= 4096 (N_theta = 240, 288, 360, ... and odd ones).  The
// schedule is a run-time one, but the shape is the same: T = n2 / (smallest radix) threads
// share a line, each holds one butterfly of up to 16 points per stage in registers, and the
// stages (two for most lengths up to 240, three up to 2400) exchange through a padded LDS buffer of 8 bytes
// per point, real parts and then imaginary parts.  The first stage reads the line from HBM,
// the last stage of a c2r writes it there.  Lines of more than 256 threads take the instance (MR, threads)
// whose registers let most waves share a CU: radices up to 10 fit the 128 VGPRs of four waves per
// SIMD and so of workgroups up to 1024 threads; up to 6 (n2 = 1875, 3125, 3750) 72 VGPRs, and two or
// three lines of 625 or 750 threads share a CU instead of one (1.6 GB of lines, c2r / r2c: n2 = 1875 2.60 /
// 2.65 -> 1.58 / 1.54 ms, 3750 1.72 / 1.81 -> 1.06 / 1.08); n2 = 3675 alone needs a radix of 15 and 735 threads, and
// gets 168 VGPRs and three waves per SIMD (at 128 its spills took 4.96 / 3.77 ms, now 1.92 / 2.09).
// (A Stockham in LDS with radices up to 8, two buffers of 16 bytes per point and the first and
// last pass over LDS on their own ran at 0.8 - 1.7 TB/s; this runs c2r at 1.9 - 4.0 and r2c at 2.2 - 4.9
// where a line takes at most 256 threads, 1.2 - 3.0 above.)
constexpr int kMaxRadix = 16, kMaxRadixLong = 10, kMaxRadixLow = 6, kMaxStages = 6;

// Division of 0 <= x < 2^16 by a d that every thread shares, 1 <= d <= 2^13, as one high
// multiplication by m = ceil(2^32 / d): exact, since m d - 2^32 < d and x d < 2^32.
struct fast_div {
    unsigned m;
    int d;
    __host__ __device__ explicit fast_div(int dd = 1) : m(dd > 1 ? 0xffffffffu / (unsigned)dd + 1u : 0u), d(dd) {}
    __device__ __forceinline__ int operator()(int x) const { return d > 1 ? (int)__umulhi((unsigned)x, m) : x; }
};

struct any_sched {
    int n2, threads_line, lines, nst;  // complex length, threads per line (T), lines per workgroup, stages
    int radix[kMaxStages];
    fast_div by_t;
    fast_div by_ns[kMaxStages];  // by the product of the radices before a stage
};

__host__ __device__ inline int any_pad(int i) { return i + (i >> 4); }
__host__ __device__ inline int any_stride(int n2) { return any_pad(n2) | 1; }

template <int MR>
__device__ __forceinline__ void any_dft(cplx (&v)[MR], int R, int sign)
{
    auto run = [&](auto r) {
        constexpr int RR = decltype(r)::value;
        if constexpr (RR <= MR) {
            cplx y[RR];
#pragma unroll
            for (int i = 0; i < RR; ++i) y[i] = v[i];
            dft_r<RR>(y, sign);
#pragma unroll
            for (int i = 0; i < RR; ++i) v[i] = y[i];
        }
    };
    switch (R) {
    case 2: run(std::integral_constant<int, 2>{}); break;
    case 3: run(std::integral_constant<int, 3>{}); break;
    case 4: run(std::integral_constant<int, 4>{}); break;
    case 5: run(std::integral_constant<int, 5>{}); break;
    case 6: run(std::integral_constant<int, 6>{}); break;
    case 7: run(std::integral_constant<int, 7>{}); break;
    case 8: run(std::integral_constant<int, 8>{}); break;
    case 9: run(std::integral_constant<int, 9>{}); break;
    case 10: run(std::integral_constant<int, 10>{}); break;
    case 12: run(std::integral_constant<int, 12>{}); break;
    case 14: run(std::integral_constant<int, 14>{}); break;
    case 15: run(std::integral_constant<int, 15>{}); break;
    case 16: run(std::integral_constant<int, 16>{}); break;
    default: break;  // 1: a line of two values
    }
}

// One line's FFT from the points of its first stage in v (zeros where a thread has no butterfly)
// to those of the last: on return output base + r ns of the line is v[r], r < R, where busy.
// `on`: the thread's line exists; every thread of the workgroup takes part.
struct any_state {
    int R, m, ns, base;
    bool busy;
};

__device__ __forceinline__ void any_first(const any_sched &a, any_state &q, int t, bool on)
{
    q.R = a.radix[0];
    q.m = a.n2 / q.R;
    q.ns = 1;
    q.busy = on && t < q.m;
}

// A thread's points in groups of GROUP: load(r, i) of each point r = g + i < R of a group, then
// use(r, i).  A group's loads go out together; with its use behind each load a thread waits for
// them one by one, which a launch of few lines has nothing to hide behind.  With CLAMP (c2r, three
// loads a point) a group is loaded whole and without a branch, point 0 again for those at and above
// R, whose results mean nothing.  Groups of four in the workgroups of 256 threads: c2r / r2c of one
// line of N_phi = 480 8.8 / 10.6 -> 7.3 / 9.2 us (7.2 is what the host takes for a launch), 192 MB of
// them 100 / 84 -> 75 / 82, N_phi = 30 248 / 161 -> 191 / 156 (c2r 369 with CLAMP off); of one, as it was,
// where a line takes more threads (N_phi/2 = 2625, 192 MB, c2r 268 -> 290 with four).
template <int MR, int GROUP, bool CLAMP, typename L, typename U>
__device__ __forceinline__ void any_points(int R, L &&load, U &&use)
{
    constexpr bool whole = CLAMP && GROUP > 1;
#pragma unroll
    for (int g = 0; g < MR; g += GROUP)
        if (g < R) {
#pragma unroll
            for (int i = 0; i < GROUP; ++i)
                if (g + i < MR && (whole || g + i < R)) load(whole && g + i >= R ? 0 : g + i, i);
#pragma unroll
            for (int i = 0; i < GROUP; ++i)
                if (g + i < MR && (whole || g + i < R)) use(g + i, i);
        }
}

template <int MR, int GROUP, bool CLAMP>
__device__ __forceinline__ void any_stages(const any_sched &a, cplx (&v)[MR], any_state &q, int t, bool on,
                                           double *__restrict__ buf, const double2 *__restrict__ tw, int sign)
{
    for (int s = 0;; ++s) {
        const int jq = a.by_ns[s](t), jm = t - jq * q.ns;
        if (s > 0 && q.busy) {
            const int step = 2 * (q.m / q.ns) * jm;  // jm nphi / (ns R); times r below nphi
            double2 w[GROUP];
            any_points<MR, GROUP, CLAMP>(
                q.R, [&](int r, int i) { w[i] = tw[step * r]; },
                [&](int r, int i) {
                    if (r > 0) v[r] = cmul(v[r], cplx{w[i].x, sign * w[i].y});
                });
        }
        any_dft(v, q.R, sign);
        q.base = jq * q.ns * q.R + jm;
        if (s + 1 == a.nst) return;
        const int Rn = a.radix[s + 1], mn = a.n2 / Rn;
        const bool next = on && t < mn;
        double re[MR];
#pragma unroll
        for (int r = 0; r < MR; ++r)
            if (r < q.R && q.busy) buf[any_pad(q.base + r * q.ns)] = v[r].re;
        __syncthreads();
#pragma unroll
        for (int r = 0; r < MR; ++r) re[r] = r < Rn && next ? buf[any_pad(t + r * mn)] : 0.0;
        __syncthreads();
#pragma unroll
        for (int r = 0; r < MR; ++r)
            if (r < q.R && q.busy) buf[any_pad(q.base + r * q.ns)] = v[r].im;
        __syncthreads();
#pragma unroll
        for (int r = 0; r < MR; ++r) v[r] = {re[r], r < Rn && next ? buf[any_pad(t + r * mn)] : 0.0};
        __syncthreads();
        q.ns *= q.R;
        q.R = Rn;
        q.m = mn;
        q.busy = next;
    }
}

template <bool C2R, int THREADS, int MR>
__global__ __launch_bounds__(THREADS, (MR == kMaxRadixLow ? 7 : MR == kMaxRadixLong ? 4 : 3)) void fft_any_kernel(
    any_sched a, long howmany, double *__restrict__ x, const double2 *__restrict__ tw, int rescale)
{
    extern __shared__ double any_lds[];
    const int n2 = a.n2, T = a.threads_line, tid = threadIdx.x;
    const int li = a.by_t(tid), t = tid - li * T;
    const long line = (long)blockIdx.x * a.lines + li;
    const bool on = line < howmany;
    double2 *xl = reinterpret_cast<double2 *>(x + (on ? line : 0) * (2L * n2 + 2));
    double *buf = any_lds + li * any_stride(n2);
    cplx v[MR];
    any_state q;
    any_first(a, q, t, on);
    constexpr int GROUP = THREADS == 256 ? 4 : 1;
#pragma unroll
    for (int r = 0; r < MR; ++r) v[r] = {0.0, 0.0};
    if (q.busy) {
        double2 xa[GROUP], xb[GROUP], w[GROUP];
        any_points<MR, GROUP, C2R>(
            q.R,
            [&](int r, int i) {
                const int k = t + r * q.m;
                xa[i] = xl[k];
                if constexpr (C2R) {
                    xb[i] = xl[n2 - k];
                    w[i] = tw[k];
                }
            },
            [&](int r, int i) {
                // Im X_0 and Im X_{n2} do not enter
                const bool k0 = t + r * q.m == 0;
                if constexpr (C2R) v[r] = c2r_pack(cplx{xa[i].x, k0 ? 0.0 : xa[i].y}, cplx{xb[i].x, k0 ? 0.0 : -xb[i].y}, w[i]);
                else v[r] = {xa[i].x, xa[i].y};
            });
    }
    any_stages<MR, GROUP, C2R>(a, v, q, t, on, buf, tw, C2R ? +1 : -1);
    if constexpr (C2R) {
#pragma unroll
        for (int r = 0; r < MR; ++r)
            if (r < q.R && q.busy) xl[q.base + r * q.ns] = make_double2(v[r].re, v[r].im);
        if (on && t == 0) xl[n2] = make_double2(0.0, 0.0);
    } else {
        // X_k and X_{n2-k} for k = t + i T <= n2 / 2; T >= n2 / MR
        constexpr int kPairs = MR / 2 + 1;
        constexpr int kTogether = GROUP > 1 ? 3 : 1;  // pairs whose twiddles are loaded together, as in any_points
        double kr[kPairs], nr[kPairs];
        double2 wk[kTogether], wn[kTogether];
#pragma unroll
        for (int part = 0; part < 2; ++part) {
#pragma unroll
            for (int r = 0; r < MR; ++r)
                if (r < q.R && q.busy) buf[any_pad(q.base + r * q.ns)] = part ? v[r].im : v[r].re;
            __syncthreads();
#pragma unroll
            for (int i = 0; i < kPairs; ++i) {
                if (kTogether > 1 && part == 1 && i % kTogether == 0 && 2 * (t + i * T) <= n2)
#pragma unroll
                    for (int j = 0; j < kTogether; ++j) {
                        const int k = min(t + (i + j) * T, n2);
                        wk[j] = tw[k];
                        wn[j] = tw[n2 - k];
                    }
                const int k = t + i * T;
                if (2 * k <= n2 && on) {
                    const double zk = buf[any_pad(k)], zn = buf[any_pad(k == 0 ? 0 : n2 - k)];
                    if (part == 0) {
                        kr[i] = zk;
                        nr[i] = zn;
                    } else {
                        auto put = [&](int i2, cplx X) {
                            double re = X.re, im = X.im;
                            if (rescale) {
                                // r2c_ip4D_fftw_rsc: X(k > 0) / nphi, Re X_0 / (2 nphi), Im X_0 untouched
                                re = i2 == 0 ? re / (4.0 * n2) : re / (2.0 * n2);
                                if (i2 > 0) im = im / (2.0 * n2);
                            }
                            xl[i2] = make_double2(re, im);
                        };
                        const cplx a0 = {kr[i], zk}, a1 = {nr[i], zn};
                        put(k, r2c_unpack(a0, a1, kTogether > 1 ? wk[i % kTogether] : tw[k]));
                        if (2 * k != n2) put(n2 - k, r2c_unpack(a1, a0, kTogether > 1 ? wn[i % kTogether] : tw[n2 - k]));
                    }
                }
            }
            __syncthreads();
        }
    }
}

// ---------------------------------------------------------------------------
// The row transposes fused into the register-resident transforms (the reform_* and
// spectral_to_physical / physical_to_spectral entry points): a workgroup transforms TB lines
// of one (r, f) at TB consecutive theta and moves the modes m <= l_max between its lines and the
// hybrid rows p2[mp][c][theta] itself, so the padded grid is written (c2r) or read (r2c)
// once and no pass over it only reorders.  A thread moves two theta of a row (16 bytes); the
// rows of one part (all real, then all imaginary) go through the lines' LDS buffers.  The
// arithmetic is the separate kernels' own, so the results are identical.  Bytes of rows plus
// grid over the time, c2r / r2c: 3.3 / 4.0 TB/s at N = 384, 3.1 / 3.7 at 1536 (a 2a -> 3a pass and
// the c2r: 1.9; the r2c fused over 16-byte points: 3.6 and 3.0).  Work unit
// w = (f, r, theta block), theta block fastest; workgroup b takes unit (b % 8) per + b / 8, so
// consecutive theta blocks of one (r, f) run on one XCD and share the cache lines of the
// hybrid rows in its L2.
// Lines per workgroup, in waves of 64 threads (even, at most 32 lines).  Measured over 1, 2, 4 and
// 8 waves on 1.6 GB grids (GB/s of rows plus grid, c2r / r2c): T = 4: 1 (4376 / 4874; two 4240 /
// 4588); T = 8: 2 (4316 / 4513; four 3672 / 3697); T = 16: c2r 2, r2c 4 (3487 / 3998; the other
// way 3420 / 3759); T = 32: 4 (3706 / 4306; two 3386 / 2877); T = 64: 8 (3065 / 3663;
// four 3007 / 2637); T >= 128: 4 (c2r 2722; eight 2415).  More lines make longer pieces of the
// hybrid rows (8 bytes a line), fewer leave more workgroups to overlap their phases.
// Where rows and grid stay in the last-level cache the r2c of T = 16 and 64 is faster with half the
// lines: the pieces merge there, and a small grid has workgroups for more CUs.  N = 384, us with 4 / 2
// waves by MB of grid: 2.4 10.8 / 9.0, 38 21.0 / 18.9, 151 61 / 57, 302 133 / 143, 605 252 / 273; N = 1536 with
// 8 / 4: 9.4 18.1 / 13.0, 38 23.4 / 22.5, 75 46 / 33, 151 76 / 63, 302 175 / 236, 604 310 / 470.  T = 32 is not (9.4
// 11.4 / 9.7, 38 20.6 / 20.2, 151 61 / 63, 302 147 / 207), and T = 128 is as fast or faster with 4 waves
// at any size (19 22 / 16, 75 53 / 36, 302 185 / 162, 1208 743 / 743).
// The c2r keeps its lines at every size: with half of them grids below 10 MB take less (N = 384, 2.4 MB
// 10.0 / 8.9 us, N = 1536, 9.4 MB 17.9 / 13.8), from 40 MB on they are even or slower (384, 302 MB 154 / 162,
// 1536, 1208 MB 677 / 692).
constexpr double kCachedGridBytes = 200e6;
template <int N, bool C2R>
__host__ __device__ constexpr int hyb_lines(bool cached = false)
{
    constexpr int T = fft_geom<N>::T;
    constexpr int W = T <= 4 ? 1 : T == 8 ? 2 : T == 16 ? (C2R ? 2 : 4) : T == 32 || T >= 128 ? 4 : 8;
    const int w = cached && !C2R && (T == 16 || T == 64) ? W / 2 : W;
    return w * 64 / T > 32 ? 32 : w * 64 / T < 2 ? 2 : w * 64 / T;
}

struct hyb_args {
    int nt, nr, nf, lmax, ntb, units;
    const int *mp_of_m;
};

__device__ __forceinline__ bool hyb_unit(const hyb_args &a, int &r, int &f, int &t0, int TB)
{
    const int per = gridDim.x >> 3, b = blockIdx.x;
    const int w = (b & 7) * per + (b >> 3);
    if (w >= a.units) return false;
    const int tb = w % a.ntb, rf = w / a.ntb;
    r = rf % a.nr;
    f = rf / a.nr;
    t0 = tb * TB;
    return true;
}

// 2a -> 3a and c2r.  U = row pieces per thread: at most P / 3 (rounded up) where l_max + 1 <= 2 N / 3,
// Rayleigh's dealiased grids, else P / 2.
template <int N, int U>
__global__ __launch_bounds__((hyb_lines<N, true>() * fft_geom<N>::T),
                                  fft_geom<N>::WAVES) void fft_reg_c2r_hyb_kernel(hyb_args a,
                                    const double *__restrict__ p2, double *__restrict__ p3,
                                    const double2 *__restrict__ tw)
{
    using G = fft_geom<N>;
    constexpr int T = G::T, TB = hyb_lines<N, true>(), NTH = TB * T, PPR = TB / 2;
    extern __shared__ double hyb_lds[];
    int r, f, t0;
    if (!hyb_unit(a, r, f, t0, TB)) return;
    const int tid = threadIdx.x, t = tid % T, li = tid / T;
    const long nrhs = 2L * a.nr * a.nf, part_step = (long)a.nr * a.nt;
    double2 re[U], im[U];
    {
        // branch-free: a piece past l_max, past N_theta or of an m the plan has not reads the
        // array's first values and becomes zeros
        int mp[U];
#pragma unroll
        for (int u = 0; u < U; ++u) {
            const int m = (tid + u * NTH) / PPR;
            mp[u] = m <= a.lmax ? a.mp_of_m[m] : -1;
        }
#pragma unroll
        for (int u = 0; u < U; ++u) {
            const int th = t0 + 2 * ((tid + u * NTH) % PPR);
            const bool on = mp[u] >= 0 && th < a.nt;
            const double *row = p2 + (on ? ((long)mp[u] * nrhs + r + 2L * a.nr * f) * a.nt + th : 0);
            re[u] = *reinterpret_cast<const double2 *>(row);
            im[u] = *reinterpret_cast<const double2 *>(row + (on ? part_step : 0));
        }
#pragma unroll
        for (int u = 0; u < U; ++u) {
            const bool on = mp[u] >= 0 && t0 + 2 * ((tid + u * NTH) % PPR) < a.nt;
            re[u] = on ? re[u] : make_double2(0.0, 0.0);
            im[u] = on ? im[u] : make_double2(0.0, 0.0);
        }
    }
    auto spread = [&](const double2(&x)[U]) {
#pragma unroll
        for (int u = 0; u < U; ++u) {
            const int m = (tid + u * NTH) / PPR, l0 = 2 * ((tid + u * NTH) % PPR);  // m < N
            hyb_lds[l0 * G::STRIDE + G::pad(m)] = x[u].x;
            hyb_lds[(l0 + 1) * G::STRIDE + G::pad(m)] = x[u].y;
        }
    };
    double *buf = hyb_lds + li * G::STRIDE;
    // element k of the line's buffer, zero above l_max (what is there has not been written)
    auto mode = [&](int i, int c) {  // k = i + c
        const double x = buf[i + c < N ? G::pad(i, c) : 0];
        return i + c <= a.lmax ? x : 0.0;
    };
    cplx v[G::P];
    double nre[G::P];  // Re X_{N-k}
    spread(re);
    __syncthreads();
#pragma unroll
    for (int u = 0; u < G::P / G::R0; ++u) {
        group_barrier<G::R0>(u);
#pragma unroll
        for (int q = 0; q < G::R0; ++q) {
            const int c = T * u + q * (N / G::R0);
            v[u * G::R0 + q].re = mode(t, c);
            nre[u * G::R0 + q] = mode(N - t, -c);
        }
    }
    __syncthreads();
    spread(im);
    __syncthreads();
#pragma unroll
    for (int u = 0; u < G::P / G::R0; ++u) {
        group_barrier<G::R0>(u);
#pragma unroll
        for (int q = 0; q < G::R0; ++q) {
            const int c = T * u + q * (N / G::R0), k = t + c, i = u * G::R0 + q;
            const double ia = mode(t, c), ib = mode(N - t, -c);
            v[i] = c2r_pack(cplx{v[i].re, k == 0 ? 0.0 : ia}, cplx{nre[i], k == 0 ? 0.0 : -ib}, tw[k]);
        }
    }
    line_sync<N>();
    fft_pass<N, G::R0, 1>(v, t, tw, +1);
    fft_middle<N, 1>(buf, v, t, tw, +1);
    if (t0 + li >= a.nt) return;
    double *xl = p3 + (((long)f * a.nt + t0 + li) * a.nr + r) * (2L * N + 2);
    constexpr int NSL = N / G::F;
#pragma unroll
    for (int u = 0; u < G::P / G::F; ++u)
#pragma unroll
        for (int q = 0; q < G::F; ++q)
            reinterpret_cast<double2 *>(xl)[t + T * u + q * NSL] =
                make_double2(v[u * G::F + q].re, v[u * G::F + q].im);
    if (t == 0) reinterpret_cast<double2 *>(xl)[N] = make_double2(0.0, 0.0);
}

// r2c and 3b -> 2b; the grid is left unchanged.  TB lines to a workgroup.
template <int N, int TB>
__global__ __launch_bounds__((TB * fft_geom<N>::T),
                                  fft_geom<N>::WAVES) void fft_reg_r2c_hyb_kernel(hyb_args a,
                                    const double *__restrict__ p3, double *__restrict__ p2,
                                    const double2 *__restrict__ tw)
{
    using G = fft_geom<N>;
    constexpr int T = G::T, NTH = TB * T, PPR = TB / 2;
    extern __shared__ double hyb_lds[];
    int r, f, t0;
    if (!hyb_unit(a, r, f, t0, TB)) return;
    const int tid = threadIdx.x, t = tid % T, li = tid / T, th = t0 + li;
    const bool line_in = th < a.nt;
    const double *xl = p3 + (((long)f * a.nt + (line_in ? th : 0)) * a.nr + r) * (2L * N + 2);
    double *buf = hyb_lds + li * G::STRIDE;
    cplx v[G::P], zk[G::P / 2 + 1], zn[G::P / 2 + 1];
#pragma unroll
    for (int u = 0; u < G::P / G::R0; ++u)
#pragma unroll
        for (int q = 0; q < G::R0; ++q) {
            const double2 z = reinterpret_cast<const double2 *>(xl)[t + T * u + q * (N / G::R0)];
            v[u * G::R0 + q] = {z.x, z.y};
        }
    fft_pass<N, G::R0, 1>(v, t, tw, -1);
    fft_middle<N, 1>(buf, v, t, tw, -1);
    r2c_pairs<N>(buf, v, zk, zn, t);
    // the modes m <= l_max of the TB lines to the hybrid rows, one part at a time, two theta per
    // thread; the block indices of eight pieces are loaded together
    const long nrhs = 2L * a.nr * a.nf;
    constexpr int U = 8;
    const int npieces = (a.lmax + 1) * PPR;
    // unconditional (modes above l_max are left in the buffer): straight-line code keeps the
    // registers within bounds
    auto keep = [&](int u, double k, double n) {
        if (u < G::P / 2) buf[G::pad(t, T * u)] = k;
        else if (t == 0) buf[G::pad(N / 2)] = k;
        if (u < G::P / 2 && (u > 0 || t > 0)) buf[G::pad(N - t, -T * u)] = n;  // not X_N, above l_max
    };
    double ik[G::P / 2 + 1], in[G::P / 2 + 1];  // Im X_k, Im X_{N-k}
#pragma unroll
    for (int u = 0; u <= G::P / 2; ++u) {
        group_barrier<2>(u);
        const int k = u < G::P / 2 ? t + T * u : N / 2;
        const cplx xk = r2c_unpack(zk[u], zn[u], tw[k]), xn = r2c_unpack(zn[u], zk[u], tw[N - k]);
        ik[u] = xk.im;
        in[u] = xn.im;
        // computed here: sunk to their use behind the first part's stores they would keep all of
        // Z_k, Z_{N-k} and the twiddles alive
        asm volatile("" : "+v"(ik[u]), "+v"(in[u]));
        keep(u, xk.re, xn.re);
    }
#pragma unroll
    for (int part = 0; part < 2; ++part) {
        if (part) {
            __syncthreads();
#pragma unroll
            for (int u = 0; u <= G::P / 2; ++u) keep(u, ik[u], in[u]);
        }
        __syncthreads();
        for (int base = tid; base < npieces; base += U * NTH) {
            int mp[U];
#pragma unroll
            for (int u = 0; u < U; ++u) {
                const int i = base + u * NTH;
                mp[u] = i < npieces ? a.mp_of_m[i / PPR] : -1;
            }
#pragma unroll
            for (int u = 0; u < U; ++u) {
                const int i = base + u * NTH, m = i / PPR, l0 = 2 * (i - m * PPR), th2 = t0 + l0;
                if (mp[u] >= 0 && th2 < a.nt) {
                    const double *b = hyb_lds + l0 * G::STRIDE + G::pad(m);
                    double *row = p2 + ((long)mp[u] * nrhs + r + (long)part * a.nr + 2L * a.nr * f) * a.nt;
                    *reinterpret_cast<double2 *>(row + th2) = make_double2(b[0], b[G::STRIDE]);
                }
            }
        }
    }
}

// 2a -> 3a and c2r of any length: the lines of a workgroup are consecutive theta of one (r, f), and
// their modes come from the hybrid rows as in fft_reg_c2r_hyb_kernel, at most eight pieces of
// two theta per thread (a line has T >= n2 / 16 threads).  Lines of at most 128 threads (an even
// number of lines in 256 threads); longer ones run the separate kernels.
__global__ __launch_bounds__(256, 3) void fft_any_c2r_hyb_kernel(any_sched a, hyb_args h, fast_div by_ppr,
                                                                 const double *__restrict__ p2, double *__restrict__ p3,
                                                                 const double2 *__restrict__ tw)
{
    extern __shared__ double any_lds[];
    int r0, f, t0;
    if (!hyb_unit(h, r0, f, t0, a.lines)) return;
    const int n2 = a.n2, T = a.threads_line, tid = threadIdx.x, nth = blockDim.x, stride = any_stride(n2);
    const int li = a.by_t(tid), t = tid - li * T;
    const bool on = t0 + li < h.nt;
    const long nrhs = 2L * h.nr * h.nf, part_step = (long)h.nr * h.nt;
    double *buf = any_lds + li * stride;
    constexpr int U = kMaxRadix / 2;
    const int pieces = (h.lmax + 1) * by_ppr.d;
    double2 re[U], im[U];
    {
        int mp[U];
#pragma unroll
        for (int u = 0; u < U; ++u) {
            const int i = tid + u * nth;
            mp[u] = i < pieces ? h.mp_of_m[by_ppr(i)] : -1;
        }
        // branch-free, as in fft_reg_c2r_hyb_kernel
#pragma unroll
        for (int u = 0; u < U; ++u) {
            const int i = tid + u * nth, m = by_ppr(i), th = t0 + 2 * (i - m * by_ppr.d);
            const bool in = mp[u] >= 0 && th < h.nt;
            const double *row = p2 + (in ? ((long)mp[u] * nrhs + r0 + 2L * h.nr * f) * h.nt + th : 0);
            re[u] = *reinterpret_cast<const double2 *>(row);
            im[u] = *reinterpret_cast<const double2 *>(row + (in ? part_step : 0));
            re[u] = in ? re[u] : make_double2(0.0, 0.0);
            im[u] = in ? im[u] : make_double2(0.0, 0.0);
        }
    }
    auto spread = [&](const double2(&x)[U]) {
#pragma unroll
        for (int u = 0; u < U; ++u) {
            const int i = tid + u * nth, m = by_ppr(i);
            if (i < pieces) {
                double *b = any_lds + 2 * (i - m * by_ppr.d) * stride + any_pad(m);
                b[0] = x[u].x;
                b[stride] = x[u].y;
            }
        }
    };
    auto mode = [&](int k) { return k <= h.lmax ? buf[any_pad(k)] : 0.0; };
    cplx v[kMaxRadix];
    double nre[kMaxRadix];  // Re X_{n2-k}
    any_state q;
    any_first(a, q, t, on);
    spread(re);
    __syncthreads();
#pragma unroll
    for (int r = 0; r < kMaxRadix; ++r) {
        v[r] = {0.0, 0.0};
        nre[r] = 0.0;
        if (r < q.R && q.busy) {
            const int k = t + r * q.m;
            v[r].re = mode(k);
            nre[r] = mode(n2 - k);
        }
    }
    __syncthreads();
    spread(im);
    __syncthreads();
#pragma unroll
    for (int r = 0; r < kMaxRadix; ++r)
        if (r < q.R && q.busy) {
            const int k = t + r * q.m;
            const double ia = mode(k), ib = mode(n2 - k);
            v[r] = c2r_pack(cplx{v[r].re, k == 0 ? 0.0 : ia}, cplx{nre[r], k == 0 ? 0.0 : -ib}, tw[k]);
        }
    __syncthreads();
    any_stages<kMaxRadix, 4, true>(a, v, q, t, on, buf, tw, +1);
    if (!on) return;
    double2 *xl = reinterpret_cast<double2 *>(p3 + (((long)f * h.nt + t0 + li) * h.nr + r0) * (2L * n2 + 2));
#pragma unroll
    for (int r = 0; r < kMaxRadix; ++r)
        if (r < q.R && q.busy) xl[q.base + r * q.ns] = make_double2(v[r].re, v[r].im);
    if (t == 0) xl[n2] = make_double2(0.0, 0.0);
}

// The one-rank row transposes are 2-D transposes per (r, f): the hybrid side is
// (mode q = 2m+imi) x theta with theta contiguous, the physical side theta x q with q
// contiguous.  A Q (q) x 64 (theta) tile goes through LDS; both sides move 16-byte
// pairs (theta pairs on the hybrid side, (Re, Im) of one m on the physical side), so a
// hybrid row is read or written as 512 contiguous bytes and a physical row as Q * 8.
// Rows are 16-byte aligned: N_theta and N_phi + 2 are even.
constexpr int kPT = 64, kPQ = 32;

// 2a -> 3a: p3 line (f, theta, r) gets Re/Im of m at 2m, 2m+1 and zeros elsewhere.
// Tiles of Q modes (q) x 64 theta: a physical row is written as Q * 8 contiguous bytes.
template <int Q>
__global__ __launch_bounds__(256) void permute_2a3a_kernel(int nt, int nr, int nf, int nphi, int lmax,
                                                           const int *__restrict__ mp_of_m,
                                                           const double *__restrict__ p2, double *__restrict__ p3)
{
    __shared__ double tile[Q][kPT + 2];  // [q][theta]
    const int t0 = blockIdx.x * kPT, q0 = blockIdx.y * Q;
    const int rf = blockIdx.z, r = rf % nr, f = rf / nr;
    const long ld = nphi + 2, nrhs = 2L * nr * nf;
    const int tid = threadIdx.x;
    const bool any_m = (q0 >> 1) <= lmax;  // uniform: the tile holds modes of the plan
    if (any_m) {
        const int pr = tid & 31;  // theta pair of a hybrid row
#pragma unroll
        for (int i = 0; i < Q / 8; ++i) {
            const int qq = (tid >> 5) + 8 * i, q = q0 + qq, m = q >> 1, t = t0 + 2 * pr;
            double2 v = make_double2(0.0, 0.0);
            if (m <= lmax && t < nt) {
                const int mp = mp_of_m[m];
                if (mp >= 0)
                    v = *reinterpret_cast<const double2 *>(
                        p2 + ((long)mp * nrhs + r + (long)(q & 1) * nr + 2L * nr * f) * nt + t);
            }
            tile[qq][2 * pr] = v.x;
            tile[qq][2 * pr + 1] = v.y;
        }
        __syncthreads();
    }
    constexpr int QP = Q / 2, TR = 256 / QP;  // (Re, Im) pairs of a physical row, rows per pass
    const int qp = tid % QP;
#pragma unroll
    for (int i = 0; i < kPT / TR; ++i) {
        const int tt = tid / QP + TR * i, t = t0 + tt, q = q0 + 2 * qp;
        if (t < nt && q < nphi + 2) {
            const double2 v = any_m ? make_double2(tile[2 * qp][tt], tile[2 * qp + 1][tt]) : make_double2(0.0, 0.0);
            *reinterpret_cast<double2 *>(p3 + (((long)f * nt + t) * nr + r) * ld + q) = v;
        }
    }
}

// 64 modes per 2a -> 3a tile: 512-byte physical row segments; measured faster than 32 at
// l_max = 255 and level with it at l_max = 1023.
constexpr int kPQ2a3a = 64;

// 3b -> 2b: the inverse map, reading back only the m of the plan (m <= lmax).
__global__ __launch_bounds__(256) void permute_3b2b_kernel(int nt, int nr, int nf, int nphi, int lmax,
                                                           const int *__restrict__ mp_of_m,
                                                           const double *__restrict__ p3, double *__restrict__ p2)
{
    __shared__ double tile[kPQ][kPT + 2];  // [q][theta]
    const int t0 = blockIdx.x * kPT, q0 = blockIdx.y * kPQ;
    const int rf = blockIdx.z, r = rf % nr, f = rf / nr;
    const long ld = nphi + 2, nrhs = 2L * nr * nf;
    const int tid = threadIdx.x, qmax = 2 * (lmax + 1);
    const int qp = tid & 15;
#pragma unroll
    for (int i = 0; i < 4; ++i) {
        const int tt = (tid >> 4) + 16 * i, t = t0 + tt, q = q0 + 2 * qp;
        double2 v = make_double2(0.0, 0.0);
        if (t < nt && q < qmax) v = *reinterpret_cast<const double2 *>(p3 + (((long)f * nt + t) * nr + r) * ld + q);
        tile[2 * qp][tt] = v.x;
        tile[2 * qp + 1][tt] = v.y;
    }
    __syncthreads();
    const int pr = tid & 31;
#pragma unroll
    for (int i = 0; i < 4; ++i) {
        const int qq = (tid >> 5) + 8 * i, q = q0 + qq, m = q >> 1, t = t0 + 2 * pr;
        if (q < qmax && t < nt) {
            const int mp = mp_of_m[m];
            if (mp >= 0)
                *reinterpret_cast<double2 *>(p2 + ((long)mp * nrhs + r + (long)(q & 1) * nr + 2L * nr * f) * nt + t) =
                    make_double2(tile[qq][2 * pr], tile[qq][2 * pr + 1]);
        }
    }
}

struct twiddle_cache {
    std::mutex mu;
    std::map<std::pair<int, int>, double2 *> tables;
} g_tw;

// The device table of e^{+2 pi i u / nphi} of the current device, made on first use.  With
// create = false the table must exist already (RAYSHT_ENOTREADY otherwise): nothing is
// allocated or copied.
int get_twiddles(int nphi, const double2 **out, bool create = true)
{
    int dev = 0;
    RAYSHT_HIP_TRY(hipGetDevice(&dev));
    std::lock_guard<std::mutex> lock(g_tw.mu);
    auto key = std::make_pair(dev, nphi);
    auto it = g_tw.tables.find(key);
    if (it != g_tw.tables.end()) {
        *out = it->second;
        return RAYSHT_OK;
    }
    if (!create) return RAYSHT_ENOTREADY;
    std::vector<double> c(nphi), s(nphi);
    fft_twiddles(nphi, c.data(), s.data());
    std::vector<double2> h(nphi);
    for (int i = 0; i < nphi; ++i) h[i] = make_double2(c[i], s[i]);
    double2 *d = nullptr;
    if (hipMalloc(&d, sizeof(double2) * nphi) != hipSuccess) return RAYSHT_ENOMEM;
    RAYSHT_HIP_TRY(hipMemcpy(d, h.data(), sizeof(double2) * nphi, hipMemcpyHostToDevice));
    g_tw.tables[key] = d;
    *out = d;
    return RAYSHT_OK;
}

// calls f(std::integral_constant<int, N>) for a length n2 = N with register-resident kernels
// (3 * 2^k, 24 .. 3072, and 2^k, 16 .. 4096); false for other lengths, which fft_any_kernel and
// fft_any_c2r_hyb_kernel take
template <typename F>
bool with_reg_length(int n2, F &&f)
{
#define RAYSHT_LENGTH(N) \
    case N: f(std::integral_constant<int, N>{}); return true;
    switch (n2) {
        RAYSHT_LENGTH(24) RAYSHT_LENGTH(48) RAYSHT_LENGTH(96) RAYSHT_LENGTH(192) RAYSHT_LENGTH(384)
        RAYSHT_LENGTH(768) RAYSHT_LENGTH(1536) RAYSHT_LENGTH(3072)
        RAYSHT_LENGTH(16) RAYSHT_LENGTH(32) RAYSHT_LENGTH(64) RAYSHT_LENGTH(128) RAYSHT_LENGTH(256)
        RAYSHT_LENGTH(512) RAYSHT_LENGTH(1024) RAYSHT_LENGTH(2048) RAYSHT_LENGTH(4096)
    default: return false;
    }
#undef RAYSHT_LENGTH
}

// f(first line, lines) for pieces of `howmany` lines whose launches stay below 2^32 threads in
// all (`block` threads take `per_block` lines); the pieces start at a workgroup's first line
template <typename F>
int in_pieces(long howmany, int per_block, int block, F &&f)
{
    const long most = ((1L << 32) - 1) / block * per_block;
    for (long at = 0; at < howmany; at += most) {
        f(at, std::min(most, howmany - at));
        RAYSHT_HIP_TRY(hipGetLastError());
    }
    return RAYSHT_OK;
}

// LDS asked for and not used: where one to four threads take a line, a lane walks its own cache
// lines, and the 16 or more lines of a wave fill half of the 32 KB of a CU's vector cache.  Five
// waves on a CU instead of nine or twelve keep what they walk in it.  192 MB of lines, c2r / r2c
// without it -> with it, us: N = 16 82 / 80 -> 78 / 70, 24 102 / 82 -> 88 / 75, 32 89 / 65 -> 75 / 62, 48 131 / 68
// -> 100 / 67, 64 90 / 63 -> 62 / 60, 96 106 / 66 -> 88 / 62; 6 KB are too few, 26 KB too many for some.
template <int N>
constexpr size_t reg_spare_lds()
{
    return fft_geom<N>::T <= 4 ? 14000 : 0;
}

template <int N>
int launch_reg(bool c2r, long howmany, double *x, const double2 *tw, int rescale, hipStream_t st)
{
    constexpr size_t spare = reg_spare_lds<N>();
    constexpr int threads = fft_geom<N>::THREADS, lpb = threads / fft_geom<N>::T;
    return in_pieces(howmany, lpb, threads, [&](long at, long lines) {
        const dim3 grid((unsigned)((lines + lpb - 1) / lpb));
        double *xa = x + at * (2L * N + 2);
        if (c2r) hipLaunchKernelGGL(fft_reg_c2r_kernel<N>, grid, dim3(threads), spare, st, lines, xa, tw);
        else hipLaunchKernelGGL(fft_reg_r2c_kernel<N>, grid, dim3(threads), spare, st, lines, xa, tw, rescale);
    });
}

bool reg_dispatch(int n2, bool c2r, long howmany, double *x, const double2 *tw, int rescale, hipStream_t st, int *rc)
{
    return with_reg_length(
        n2, [&](auto n) { *rc = launch_reg<decltype(n)::value>(c2r, howmany, x, tw, rescale, st); });
}

// the fused kernels of one register-resident length (arguments checked): c2r from the hybrid
// rows in `src` to the grid, or r2c from the grid to the hybrid rows
template <int N, bool C2R, int TB>
int launch_hyb_lines(const raysht_plan *p, const double *src, double *dst, const double2 *tw, hipStream_t st)
{
    constexpr int NTH = TB * fft_geom<N>::T, P = fft_geom<N>::P;
    constexpr int US = (P + 2) / 3, UL = P / 2;
    static_assert(TB % 2 == 0 && 2 * US * fft_geom<N>::T <= N && 2 * UL * fft_geom<N>::T <= N,
                  "a thread moves two theta of a row, pieces stay within a line's modes");
    hyb_args a;
    a.nt = p->nt;
    a.nr = p->nr;
    a.nf = p->nf;
    a.lmax = p->lmax;
    a.ntb = (p->nt + TB - 1) / TB;
    a.mp_of_m = p->d_mp_of_m;
    const long units = (long)a.ntb * p->nr * p->nf;
    if (units > 0x7fffffffL / 16) return RAYSHT_EUNSUPPORTED;
    a.units = (int)units;
    const size_t lds = (size_t)TB * fft_geom<N>::STRIDE * sizeof(double);
    const dim3 grid((unsigned)(8 * ((units + 7) / 8))), block(NTH);
    if constexpr (!C2R)
        hipLaunchKernelGGL((fft_reg_r2c_hyb_kernel<N, TB>), grid, block, lds, st, a, src, dst, tw);
    else if ((p->lmax + 1) * (TB / 2) <= US * NTH)
        hipLaunchKernelGGL((fft_reg_c2r_hyb_kernel<N, US>), grid, block, lds, st, a, src, dst, tw);
    else
        hipLaunchKernelGGL((fft_reg_c2r_hyb_kernel<N, UL>), grid, block, lds, st, a, src, dst, tw);
    RAYSHT_HIP_TRY(hipGetLastError());
    return RAYSHT_OK;
}

template <int N, bool C2R>
int launch_hyb(const raysht_plan *p, const double *src, double *dst, const double2 *tw, hipStream_t st)
{
    constexpr int TB = hyb_lines<N, C2R>(), TBC = hyb_lines<N, C2R>(true);
    if (TBC != TB && 8.0 * (2 * N + 2) * p->nt * p->nr * p->nf <= kCachedGridBytes)
        return launch_hyb_lines<N, C2R, TBC>(p, src, dst, tw, st);
    return launch_hyb_lines<N, C2R, TB>(p, src, dst, tw, st);
}

// The schedule of fft_any_kernel for n2 = 2^a 3^b 5^c 7^d: the fewest stages of radix 2 .. 16, and
// among those the one whose smallest radix is largest (fewest threads per line, all with a
// full butterfly); where that takes more than 256 threads, the same with radices up to 10 if
// 1024 threads suffice (they do for all but n2 = 3675, whose 735 threads have radices up to 15).
// False for other lengths.
bool any_schedule(int n2, bool c2r, any_sched *out)
{
    static const int radices[] = {16, 15, 14, 12, 10, 9, 8, 7, 6, 5, 4, 3, 2};
    int best[kMaxStages], cur[kMaxStages], nbest = 0, smallest = 0;
    // radices in descending order, each at most the one before
    auto search = [&](auto &&self, int n, int depth, int from) -> void {
        if (n == 1) {
            const int least = depth > 0 ? cur[depth - 1] : 1;
            if (depth < nbest || (depth == nbest && least > smallest)) {
                nbest = depth;
                smallest = least;
                std::copy(cur, cur + depth, best);
            }
            return;
        }
        if (depth >= kMaxStages || depth >= nbest) return;
        int reach = 1;  // what the stages left can make of radices up to radices[from]
        for (int d = depth; d < std::min(nbest, kMaxStages) && reach < n; ++d) reach *= radices[from];
        if (reach < n) return;
        for (int i = from; i < 13; ++i)
            if (n % radices[i] == 0) {
                cur[depth] = radices[i];
                self(self, n / radices[i], depth + 1, i);
            }
    };
    auto schedule = [&](int from) {  // from radices[from] down
        nbest = kMaxStages + 1;
        smallest = 0;
        search(search, n2, 0, from);
        return nbest <= kMaxStages;
    };
    if (!schedule(0)) return false;
    if (n2 > 256 * std::max(smallest, 1) && (!schedule(4) || n2 > 1024 * smallest)) schedule(0);
    // n2 / radix threads have a butterfly of a stage, so the stages that move the line to and from
    // HBM get the two smallest radices: a c2r, which reads two values per point, starts with the
    // smallest (4 to 14 % faster), an r2c with the second smallest (2 to 4 % faster).
    if (nbest > 2) std::rotate(best, best + nbest - (c2r ? 1 : 2), best + nbest - (c2r ? 0 : 1));
    if (nbest == 0) {  // n2 = 1
        nbest = 1;
        best[0] = 1;
    }
    out->n2 = n2;
    out->nst = nbest;
    out->threads_line = n2 / std::max(smallest, 1);
    out->lines = std::max(1, 256 / out->threads_line);
    out->by_t = fast_div(out->threads_line);
    int ns = 1;
    for (int i = 0; i < kMaxStages; ++i) {
        out->radix[i] = i < nbest ? best[i] : 1;
        out->by_ns[i] = fast_div(ns);
        ns *= out->radix[i];
    }
    return true;
}

template <bool C2R>
int launch_any(int nphi, long howmany, double *x, const double2 *tw, int rescale, hipStream_t st)
{
    any_sched a;
    if (!any_schedule(nphi / 2, C2R, &a)) return RAYSHT_EUNSUPPORTED;
    const size_t lds = sizeof(double) * (size_t)a.lines * any_stride(a.n2);
    const int threads = a.lines * a.threads_line, most = *std::max_element(a.radix, a.radix + kMaxStages);
    auto launch = [&](auto kernel) {
        return in_pieces(howmany, a.lines, threads, [&](long at, long lines) {
            hipLaunchKernelGGL(kernel, dim3((unsigned)((lines + a.lines - 1) / a.lines)), dim3(threads), lds, st, a, lines,
                               x + at * (nphi + 2L), tw, rescale);
        });
    };
    if (threads <= 256) return launch(fft_any_kernel<C2R, 256, kMaxRadix>);
    if (most <= kMaxRadixLow && threads <= 768) return launch(fft_any_kernel<C2R, 768, kMaxRadixLow>);
    if (most <= kMaxRadixLong && threads <= 1024) return launch(fft_any_kernel<C2R, 1024, kMaxRadixLong>);
    if (threads <= 768) return launch(fft_any_kernel<C2R, 768, kMaxRadix>);
    return RAYSHT_EUNSUPPORTED;  // no length's schedule
}

// the fused 2a -> 3a and c2r of any length; false where a line takes more than 128 threads
bool launch_any_hyb(const raysht_plan *p, int nphi, const double *p2, double *p3, const double2 *tw, hipStream_t st,
                    int *rc)
{
    any_sched a;
    if (!any_schedule(nphi / 2, true, &a) || a.threads_line > 128) return false;
    a.lines = std::min(32, 256 / a.threads_line) & ~1;
    hyb_args h;
    h.nt = p->nt;
    h.nr = p->nr;
    h.nf = p->nf;
    h.lmax = p->lmax;
    h.ntb = (p->nt + a.lines - 1) / a.lines;
    h.mp_of_m = p->d_mp_of_m;
    const long units = (long)h.ntb * p->nr * p->nf;
    if (units > 0x7fffffffL / 16) return false;
    h.units = (int)units;
    const size_t lds = sizeof(double) * (size_t)a.lines * any_stride(a.n2);
    hipLaunchKernelGGL(fft_any_c2r_hyb_kernel, dim3((unsigned)(8 * ((units + 7) / 8))), dim3(a.lines * a.threads_line),
                       lds, st, a, h, fast_div(a.lines / 2), p2, p3, tw);
    const hipError_t e = hipGetLastError();
    if (e != hipSuccess) set_last_hip_error(e, "fft_any_c2r_hyb_kernel");
    *rc = e == hipSuccess ? RAYSHT_OK : RAYSHT_EHIP;
    return true;
}

int check_fft_args(int nphi, long howmany, const double *x)
{
    if (nphi < 2 || (nphi & 1) || howmany < 0 || (!x && howmany > 0)) return RAYSHT_EINVAL;
    int n2 = nphi / 2;
    if (n2 > kMaxHalf) return RAYSHT_EUNSUPPORTED;
    for (int p : {2, 3, 5, 7})  // every such length up to kMaxHalf has a schedule
        while (n2 % p == 0) n2 /= p;
    return n2 == 1 ? RAYSHT_OK : RAYSHT_EUNSUPPORTED;
}

// the c2r of `howmany` lines with the twiddle table tw of nphi (arguments checked)
int launch_c2r(int nphi, long howmany, double *x, const double2 *tw, hipStream_t st)
{
    int rc = RAYSHT_OK;
    if (reg_dispatch(nphi / 2, true, howmany, x, tw, 0, st, &rc)) return rc;
    return launch_any<true>(nphi, howmany, x, tw, 0, st);
}

}  // namespace

// 2a -> 3a then c2r for a plan (arguments checked), in one kernel where a line takes at most
// 128 threads or its length is a register-resident one
int permute_c2r(raysht_plan *p, int nphi, const double *p2, double *p3, const double2 *tw, hipStream_t st)
{
    int rc = RAYSHT_OK;
    if (with_reg_length(nphi / 2,
                        [&](auto n) { rc = launch_hyb<decltype(n)::value, true>(p, p2, p3, tw, st); }))
        return rc;
    if (launch_any_hyb(p, nphi, p2, p3, tw, st, &rc)) return rc;
    dim3 grid((p->nt + kPT - 1) / kPT, (nphi + 2 + kPQ2a3a - 1) / kPQ2a3a, p->nr * p->nf);
    hipLaunchKernelGGL(permute_2a3a_kernel<kPQ2a3a>, grid, dim3(256), 0, st, p->nt, p->nr, p->nf, nphi, p->lmax,
                       p->d_mp_of_m, p2, p3);
    RAYSHT_HIP_TRY(hipGetLastError());
    return launch_c2r(nphi, (long)p->nr * p->nt * p->nf, p3, tw, st);
}

int fft_prepare(int nphi)
{
    const double2 *tw = nullptr;
    return get_twiddles(nphi, &tw);
}

}  // namespace raysht

using namespace raysht;

extern "C" {

int raysht_fft_to_physical(int nphi, long howmany, double *x, void *stream)
{
    int rc = check_fft_args(nphi, howmany, x);
    if (rc != RAYSHT_OK || howmany == 0) return rc;
    const double2 *tw = nullptr;
    if ((rc = get_twiddles(nphi, &tw)) != RAYSHT_OK) return rc;
    return launch_c2r(nphi, howmany, x, tw, reinterpret_cast<hipStream_t>(stream));
}

int raysht_fft_to_spectral(int nphi, long howmany, double *x, int rescale, void *stream)
{
    int rc = check_fft_args(nphi, howmany, x);
    if (rc != RAYSHT_OK || howmany == 0) return rc;
    const double2 *tw = nullptr;
    if ((rc = get_twiddles(nphi, &tw)) != RAYSHT_OK) return rc;
    if (reg_dispatch(nphi / 2, false, howmany, x, tw, rescale ? 1 : 0, reinterpret_cast<hipStream_t>(stream), &rc))
        return rc;
    return launch_any<false>(nphi, howmany, x, tw, rescale ? 1 : 0, reinterpret_cast<hipStream_t>(stream));
}

namespace {
// the device address of `scratch` on the current device, looked up once per device
struct scratch_table {
    std::mutex mu;
    std::map<int, double *> addr;
} g_scratch;

int scratch_address(double **out)
{
    int dev = 0;
    RAYSHT_HIP_TRY(hipGetDevice(&dev));
    std::lock_guard<std::mutex> lock(g_scratch.mu);
    auto it = g_scratch.addr.find(dev);
    if (it == g_scratch.addr.end()) {
        void *ptr = nullptr;
        RAYSHT_HIP_TRY(hipGetSymbolAddress(&ptr, HIP_SYMBOL(scratch)));
        if (!ptr) return RAYSHT_EHIP;
        it = g_scratch.addr.emplace(dev, static_cast<double *>(ptr)).first;
    }
    *out = it->second;
    return RAYSHT_OK;
}
}  // namespace

int raysht_spectral_to_physical_scratch(raysht_plan *p, int nphi, const double *s, double *p3, void *stream)
{
    if (!p || !s || !p3) return RAYSHT_EINVAL;
    int rc = check_fft_args(nphi, 1, p3);
    if (rc != RAYSHT_OK) return rc;
    if (raysht_hybrid_size(p) > RAYSHT_SCRATCH_BYTES / sizeof(double)) return RAYSHT_EINVAL;
    if (p->nr < 1 || nphi < 2 * (p->lmax + 1) || (long)p->nr * p->nf > 65535) return RAYSHT_EINVAL;
    const double2 *tw = nullptr;
    if ((rc = get_twiddles(nphi, &tw, false)) != RAYSHT_OK) return rc;
    double *work = nullptr;
    if ((rc = scratch_address(&work)) != RAYSHT_OK) return rc;
    const hipStream_t st = reinterpret_cast<hipStream_t>(stream);
    if ((rc = raysht_legendre_stp(p, s, work, stream)) != RAYSHT_OK) return rc;
    return permute_c2r(p, nphi, work, p3, tw, st);
}

int raysht_permute_2a3a(raysht_plan *p, int nphi, const double *p2, double *p3, void *stream)
{
    if (!p || !p2 || !p3 || p->nr < 1 || nphi < 2 * (p->lmax + 1) || (nphi & 1)) return RAYSHT_EINVAL;
    if ((long)p->nr * p->nf > 65535) return RAYSHT_EUNSUPPORTED;
    dim3 grid((p->nt + kPT - 1) / kPT, (nphi + 2 + kPQ2a3a - 1) / kPQ2a3a, p->nr * p->nf);
    hipLaunchKernelGGL(permute_2a3a_kernel<kPQ2a3a>, grid, dim3(256), 0, reinterpret_cast<hipStream_t>(stream), p->nt,
                       p->nr, p->nf, nphi, p->lmax, p->d_mp_of_m, p2, p3);
    RAYSHT_HIP_TRY(hipGetLastError());
    return RAYSHT_OK;
}

int raysht_permute_3b2b(raysht_plan *p, int nphi, const double *p3, double *p2, void *stream)
{
    if (!p || !p2 || !p3 || p->nr < 1 || nphi < 2 * (p->lmax + 1) || (nphi & 1)) return RAYSHT_EINVAL;
    if ((long)p->nr * p->nf > 65535) return RAYSHT_EUNSUPPORTED;
    dim3 grid((p->nt + kPT - 1) / kPT, (2 * (p->lmax + 1) + kPQ - 1) / kPQ, p->nr * p->nf);
    hipLaunchKernelGGL(permute_3b2b_kernel, grid, dim3(256), 0, reinterpret_cast<hipStream_t>(stream), p->nt, p->nr,
                       p->nf, nphi, p->lmax, p->d_mp_of_m, p3, p2);
    RAYSHT_HIP_TRY(hipGetLastError());
    return RAYSHT_OK;
}

int raysht_reform_to_physical(raysht_plan *p, int nphi, const double *p2, double *p3, void *stream)
{
    if (!p || !p2 || !p3) return RAYSHT_EINVAL;
    int rc = check_fft_args(nphi, 1, p3);
    if (rc != RAYSHT_OK) return rc;
    if (p->nr < 1 || nphi < 2 * (p->lmax + 1) || (long)p->nr * p->nf > 65535) return RAYSHT_EINVAL;
    const double2 *tw = nullptr;
    if ((rc = get_twiddles(nphi, &tw)) != RAYSHT_OK) return rc;
    return permute_c2r(p, nphi, p2, p3, tw, reinterpret_cast<hipStream_t>(stream));
}

int raysht_reform_to_spectral(raysht_plan *p, int nphi, double *p3, double *p2, void *stream)
{
    if (!p || !p2 || !p3) return RAYSHT_EINVAL;
    int rc = check_fft_args(nphi, 1, p3);
    if (rc != RAYSHT_OK) return rc;
    if (p->nr < 1 || nphi < 2 * (p->lmax + 1) || (long)p->nr * p->nf > 65535) return RAYSHT_EINVAL;
    const double2 *tw = nullptr;
    if ((rc = get_twiddles(nphi, &tw)) != RAYSHT_OK) return rc;
    // the 3 * 2^k lengths: one kernel, p3 left unchanged; all others transform p3 in place
    if (nphi % 3 == 0 && with_reg_length(nphi / 2, [&](auto n) {
            if constexpr (decltype(n)::value % 3 == 0)
                rc = launch_hyb<decltype(n)::value, false>(p, p3, p2, tw, reinterpret_cast<hipStream_t>(stream));
        }))
        return rc;
    if ((rc = raysht_fft_to_spectral(nphi, (long)p->nr * p->nt * p->nf, p3, 0, stream)) != RAYSHT_OK) return rc;
    return raysht_permute_3b2b(p, nphi, p3, p2, stream);
}

int raysht_spectral_to_physical(raysht_plan *p, int nphi, const double *s, double *work, double *p3, void *stream)
{
    if (!p || !s || !work || !p3) return RAYSHT_EINVAL;
    int rc = check_fft_args(nphi, 1, p3);
    if (rc != RAYSHT_OK) return rc;
    if (p->nr < 1 || nphi < 2 * (p->lmax + 1) || (long)p->nr * p->nf > 65535) return RAYSHT_EINVAL;
    if ((rc = raysht_legendre_stp(p, s, work, stream)) != RAYSHT_OK) return rc;
    return raysht_reform_to_physical(p, nphi, work, p3, stream);
}

int raysht_physical_to_spectral(raysht_plan *p, int nphi, double *p3, double *work, double *s, void *stream)
{
    if (!p || !s || !work || !p3) return RAYSHT_EINVAL;
    int rc = raysht_reform_to_spectral(p, nphi, p3, work, stream);
    if (rc != RAYSHT_OK) return rc;
    return raysht_legendre_pts(p, work, s, stream);
}

}  // extern "C"
