// tpsc_pencil.hpp -- register-resident tau-pencil transforms and splines for gfx950 (FP64).
//
// A pencil of L = 8 NT samples (L = 512 .. 4096) belongs to NT threads with eight values each, W = NT/64
// wavefronts.  A length-L FFT is an eight-point DFT in registers and eight sub-transforms of length NT,
// each inside one wavefront (8 x 8 x W points), so only the hand-over between the two crosses
// wavefronts: a transform takes one or two workgroup barriers and never keeps its data in LDS.
//   pen_fft_dif: thread c holds x[c + NT r]; it ends with X[pen_beta + NT m] in thread order
//   pen_fft_dit: thread t holds the chunk x[8 t + c]; it ends with X[t + NT m]
// The clamped spline works on the chunks: first-order recursions in registers, carries by DPP shifts
// between lanes, one barrier for the wavefront edges.
#pragma once
#include "tpsc_device.hpp"

#define TPSC_CASE_L(X, ...) case X: { constexpr int LL = X; __VA_ARGS__; } break;
#define TPSC_LS_256(...)                                                                               \
    TPSC_CASE_L(16, __VA_ARGS__) TPSC_CASE_L(32, __VA_ARGS__) TPSC_CASE_L(64, __VA_ARGS__)             \
    TPSC_CASE_L(128, __VA_ARGS__) TPSC_CASE_L(256, __VA_ARGS__)
#define TPSC_LS_1024(...)                                                                              \
    TPSC_CASE_L(1024, __VA_ARGS__) TPSC_CASE_L(2048, __VA_ARGS__) TPSC_CASE_L(4096, __VA_ARGS__)
#define DISPATCH_L_SHORT(Lv, ...) \
    switch (Lv) { TPSC_LS_256(__VA_ARGS__) default: return hipErrorInvalidValue; }
#define DISPATCH_L_TO512(Lv, ...) \
    switch (Lv) { TPSC_LS_256(__VA_ARGS__) TPSC_CASE_L(512, __VA_ARGS__) default: return hipErrorInvalidValue; }
#define DISPATCH_L_LONG(Lv, ...) \
    switch (Lv) { TPSC_CASE_L(512, __VA_ARGS__) TPSC_LS_1024(__VA_ARGS__) default: return hipErrorInvalidValue; }
#define DISPATCH_L_FROM1024(Lv, ...) \
    switch (Lv) { TPSC_LS_1024(__VA_ARGS__) default: return hipErrorInvalidValue; }

// SS: storage / slab type of the tau and iqn arrays; ST: stored form of Sigma(k,iwn)
#define DISPATCH_S(prec, ...)     \
    if (prec) {                   \
        using SS [[maybe_unused]] = float;         \
        using ST [[maybe_unused]] = cf;            \
        __VA_ARGS__;              \
    } else {                      \
        using SS [[maybe_unused]] = double;        \
        using ST [[maybe_unused]] = cd;            \
        __VA_ARGS__;              \
    }

namespace tpsc {

template <int L>
struct Pen {
    static constexpr int NT = L / 8, W = NT / 64, G1 = 8 * W;
    static constexpr int PS = NT + 1;            // LDS row stride (complex values): odd, rows spread over the banks
    static constexpr int ZD = 2 * (9 * NT + 2);  // doubles of the LDS buffer: 8 rows, or two padded sample arrays
    static constexpr int YS = 9 * NT + 2;        // stride of the sample arrays: sample j at j + j/8
    static_assert(L % 512 == 0 && 2 * 8 * PS <= ZD, "L = 512 .. 4096");
};

// v[k] *= w^k, k = 1 .. 7, from w, w^2, w^4
__device__ __forceinline__ void twiddle8(cd* v, cd w1, cd w2, cd w4)
{
    const cd w3 = w1 * w2;
    v[1] = v[1] * w1;
    v[2] = v[2] * w2;
    v[3] = v[3] * w3;
    v[4] = v[4] * w4;
    v[5] = v[5] * (w4 * w1);
    v[6] = v[6] * (w4 * w2);
    v[7] = v[7] * (w4 * w3);
}

// The thread index t is a parameter throughout: a caller with a loop over pencils passes it through an
// empty asm first, so that table values and LDS offsets are not hoisted out of the loop into registers.

// row of thread t of the eight (one wavefront holds 8/W of them)
template <int L>
__device__ __forceinline__ int pen_row(int t)
{
    return (t >> 6) * (8 / Pen<L>::W) + (t & 63) / Pen<L>::G1;
}
// offset of the thread's outputs in a row of length NT: row[o + (NT/8) m], m < 8
template <int L>
__device__ __forceinline__ int pen_o(int t)
{
    constexpr int W = Pen<L>::W;
    return ((t & 63) / W) % 8 + 8 * ((t & 63) % W);
}
// column of the thread's outputs after pen_fft_dif
template <int L>
__device__ __forceinline__ int pen_beta(int t)
{
    return pen_row<L>(t) + 8 * pen_o<L>(t);
}

// Forward DFTs of length NT of the rows of Z, in place of registers: on exit v[m] is output
// pen_o + (NT/8) m of the thread's row.  The rows must be complete (barrier); every exchange stays in the
// wavefront's own rows.  tw[TS t] = exp(-2 pi i t / L).  Stage B: eight points over r of row[l + G1 r];
// stage C: eight over r of l = lam + W r; stage D: W over lam.
template <int L, int TS = 1>
__device__ __forceinline__ void pen_rows(cd* v, cd* Z, const cd* __restrict__ tw, int t)
{
    constexpr int W = Pen<L>::W, G1 = Pen<L>::G1, PS = Pen<L>::PS, M = 8 / W - 1;
    const int lane = t & 63;
    const int l = lane % G1, lam = lane % W, k2 = (lane / W) % 8, xm = k2 & M;
    const cd b1 = tw[8 * TS * l], b2 = tw[16 * TS * l], b4 = tw[32 * TS * l];
    cd* const row = Z + pen_row<L>(t) * PS;
#pragma unroll
    for (int r = 0; r < 8; r++) v[r] = row[l + G1 * r];
    reg_dft<8>(v);
    twiddle8(v, b1, b2, b4);
    wave_lds_order();
#pragma unroll
    for (int k = 0; k < 8; k++) row[k * G1 + (l ^ ((k & M) * W))] = v[k];
    wave_lds_order();
    cd* const rc = row + k2 * G1;
#pragma unroll
    for (int r = 0; r < 8; r++) v[r] = rc[lam + W * (r ^ xm)];
    reg_dft<8>(v);
    if constexpr (W > 1) {
        twiddle8(v, tw[64 * TS * lam], tw[128 * TS * lam], tw[256 * TS * lam]);
        wave_lds_order();
#pragma unroll
        for (int k = 0; k < 8; k++) rc[((lam + k) & (W - 1)) + W * (k ^ xm)] = v[k];
        wave_lds_order();
        cd u[8 / W][W];
#pragma unroll
        for (int i = 0; i < 8 / W; i++)
#pragma unroll
            for (int s = 0; s < W; s++) u[i][s] = rc[((s + lam) & (W - 1)) + W * ((lam + W * i) ^ xm)];
#pragma unroll
        for (int i = 0; i < 8 / W; i++) {
            reg_dft<W>(u[i]);
#pragma unroll
            for (int k = 0; k < W; k++) v[i + (8 / W) * k] = u[i][k];
        }
    }
}

// Forward DFT, v[r] = x[t + NT r] on entry, v[m] = X[pen_beta + NT m] on exit.  Z must be free on entry; no
// thread's rows are read by others afterwards.
template <int L, int TS = 1>
__device__ __forceinline__ void pen_fft_dif(cd* v, cd* Z, const cd* __restrict__ tw, int t)
{
    constexpr int PS = Pen<L>::PS;
    const cd a1 = tw[TS * t], a2 = tw[2 * TS * t], a4 = tw[4 * TS * t];
    reg_dft<8>(v);
    twiddle8(v, a1, a2, a4);
#pragma unroll
    for (int k = 0; k < 8; k++) Z[k * PS + t] = v[k];
    __syncthreads();
    pen_rows<L, TS>(v, Z, tw, t);
}

// Forward DFT of x, whose element 8 p + c lies at Z[c PS + p] (written before, no barrier yet); on exit v[m] = X[t +
// NT m], t = the thread.  w1, w2, w4: the factors exp(-2 pi i (t + s)/L) and its powers (s = 0; s = 1/2 for
// frequencies shifted by one half, x[8 p + c] then carries exp(-8 pi i p/L)).  The last reads of Z are of
// columns Z[k PS + .] of the thread's own wavefront.
template <int L, int TS = 1>
__device__ __forceinline__ void pen_fft_placed(cd* v, cd* Z, const cd* __restrict__ tw, cd w1, cd w2, cd w4, int t)
{
    constexpr int PS = Pen<L>::PS, NT = Pen<L>::NT;
    __syncthreads();
    pen_rows<L, TS>(v, Z, tw, t);
    wave_lds_order();
    // position p of a row is stored at p ^ (8/W (p/8) mod 8): both sides then spread over the banks
    constexpr int X = 8 / Pen<L>::W;
    const int o = pen_o<L>(t);
    cd* const row = Z + pen_row<L>(t) * PS + (o ^ ((X * (o >> 3)) & 7));
#pragma unroll
    for (int m = 0; m < 8; m++) row[(NT / 8) * m] = v[m];
    __syncthreads();
    const int ts = t ^ ((X * (t >> 3)) & 7);
#pragma unroll
    for (int c = 0; c < 8; c++) v[c] = Z[c * PS + ts];
    twiddle8(v, w1, w2, w4);
    reg_dft<8>(v);
}
// the same for v[c] = x[8 t + c]; Z must be free on entry
template <int L>
__device__ __forceinline__ void pen_fft_dit(cd* v, cd* Z, const cd* __restrict__ tw, cd w1, cd w2, cd w4, int t)
{
    constexpr int PS = Pen<L>::PS;
#pragma unroll
    for (int c = 0; c < 8; c++) Z[c * PS + t] = v[c];
    pen_fft_placed<L>(v, Z, tw, w1, w2, w4, t);
}

// x of the lane before (after) in the wavefront, 0 in lane 0 (63)
__device__ __forceinline__ double lane_shr1(double x)
{
    const long long b = __double_as_longlong(x);
    const int lo = __builtin_amdgcn_update_dpp(0, (int)(b & 0xffffffffLL), 0x138, 0xF, 0xF, false);
    const int hi = __builtin_amdgcn_update_dpp(0, (int)(b >> 32), 0x138, 0xF, 0xF, false);
    return __longlong_as_double(((long long)hi << 32) | (unsigned int)lo);
}
__device__ __forceinline__ double lane_shl1(double x)
{
    const long long b = __double_as_longlong(x);
    const int lo = __builtin_amdgcn_update_dpp(0, (int)(b & 0xffffffffLL), 0x130, 0xF, 0xF, false);
    const int hi = __builtin_amdgcn_update_dpp(0, (int)(b >> 32), 0x130, 0xF, 0xF, false);
    return __longlong_as_double(((long long)hi << 32) | (unsigned int)lo);
}
__device__ __forceinline__ double lane_get(double x, int lane)
{
    const long long b = __double_as_longlong(x);
    const int lo = __builtin_amdgcn_readlane((int)(b & 0xffffffffLL), lane);
    const int hi = __builtin_amdgcn_readlane((int)(b >> 32), lane);
    return __longlong_as_double(((long long)hi << 32) | (unsigned int)lo);
}

// sum over the wavefront, in lane 63: shifts by 1, 2, 4, 8 within the rows of 16 lanes, then two row broadcasts
template <int CTRL, int ROWS>
__device__ __forceinline__ double dpp_add(double x)
{
    const long long b = __double_as_longlong(x);
    const int lo = __builtin_amdgcn_update_dpp(0, (int)(b & 0xffffffffLL), CTRL, ROWS, 0xF, false);
    const int hi = __builtin_amdgcn_update_dpp(0, (int)(b >> 32), CTRL, ROWS, 0xF, false);
    return x + __longlong_as_double(((long long)hi << 32) | (unsigned int)lo);
}
__device__ __forceinline__ double wave_total63(double x)
{
    x = dpp_add<0x111, 0xF>(x);
    x = dpp_add<0x112, 0xF>(x);
    x = dpp_add<0x114, 0xF>(x);
    x = dpp_add<0x118, 0xF>(x);
    x = dpp_add<0x142, 0xA>(x);
    return dpp_add<0x143, 0xC>(x);
}
// sums over the rows of 16 lanes, in lanes 15, 31, 47, 63
__device__ __forceinline__ double row_total15(double x)
{
    x = dpp_add<0x111, 0xF>(x);
    x = dpp_add<0x112, 0xF>(x);
    x = dpp_add<0x114, 0xF>(x);
    return dpp_add<0x118, 0xF>(x);
}

// Step of a pencil's spline: h, 1/h, 6/h, 6/h^2 (formed on the host: uniform values stay out of the vector registers)
struct PenStep {
    double h, ih, r1, r2;
};
inline PenStep pen_step(double h)
{
    const double ih = 1.0 / h;
    return PenStep{h, ih, 6.0 * ih, 6.0 * ih * ih};
}

// LDS table of zc^i, zc = z^C, i <= 48/C, and a zero (|z|^48 < 1e-27): carries and boundary modes by lane.  The
// first 48/C + 2 threads fill it; a barrier must follow.
template <int C>
struct SplineTab {
    static constexpr int I = 48 / C;
    double v[I + 2];
    __device__ __forceinline__ void fill(int t)
    {
        if (t > I + 1) return;
        double p = 1.0;
        for (int i = 0; i < t; i++) p *= spline_zpow(C);
        v[t] = (t > I) ? 0.0 : p;
    }
    __device__ __forceinline__ double operator[](int i) const { return v[i < I + 1 ? i : I + 1]; }
};

// The clamped spline of block_spline_fixed (tpsc_device.hpp) on chunks, K sequences at once: thread t holds
// y[k][1 + c] = sample C t + c and its two neighbours (y[k][0] of the first thread is not used), N = C NT
// intervals, and gets the moments M[k][c] = S''(C t + c), c = 0 .. C (M[k][C] is the next thread's first).
// Both recursions start from zero in each chunk; the state S that enters a chunk adds z^(c+1) S, a
// chunk's own carries come from the lanes before by D Horner steps, and those of the wavefront before
// through sx (3 K W doubles) over the one barrier.  M[k][C] is the next thread's M[k][0] to the last bit (from
// the next lane, or formed from the same numbers by the same operations at the wavefront's end): the Fourier sums
// of (M_(j+1) - M_j)/h telescope, and two roundings of one moment would leave L/(2 pi n) times as much noise in them.
// The second differences are formed from first differences, exact for neighbouring samples (6/h^2 multiplies their
// rounding); yl (may be null) holds low-order parts of the samples.  The boundary modes come from lane 0 of the first and lane 63 of the last wavefront;
// their mutual term z^(N-1) is below 1e-290 here.  trap[k] (may be null): the thread's part of the integral.
template <int N, int NT, int K>
__device__ __forceinline__ void pen_spline(const double (*y)[N / NT + 2], const PenStep& g, const double* d0, const double* dN,
                                           double (*M)[N / NT + 1], double* sx, const SplineTab<N / NT>& zt,
                                           double* trap, int tid, const float (*yl)[N / NT + 2] = nullptr)
{
    constexpr int C = N / NT, W = NT / 64;
    static_assert(N >= 512 && N % NT == 0, "long pencils");
    constexpr double z = kSplineZ, A = 0.28867513459481288225, zc = spline_zpow(C);
    constexpr int D = spline_carry_terms(zc, 48);
    constexpr auto zp = spline_ztable<0, 1, C>();
    const int lane = tid & 63, wave = tid >> 6;
    double uE[K], Su[K], Sw[K];
#pragma unroll
    for (int k = 0; k < K; k++) {
        double* const T = M[k];
        double r[C];
#pragma unroll
        for (int c = 0; c < C; c++) {
            r[c] = (y[k][c + 2] - y[k][c + 1]) - (y[k][c + 1] - y[k][c]);
            if (yl) r[c] += (double)((yl[k][c + 2] - yl[k][c + 1]) - (yl[k][c + 1] - yl[k][c]));
            r[c] *= g.r2;
        }
        r[0] = (tid == 0) ? 0.0 : r[0];
        double s = 0.0;
#pragma unroll
        for (int c = 0; c < C; c++) {
            s = r[c] + z * s;
            T[c] = s - r[c];
        }
        uE[k] = s;
        s = 0.0;
#pragma unroll
        for (int c = C - 1; c >= 0; c--) {
            s = r[c] + z * s;
            T[c] += s;
        }
        double a = 0.0, b = 0.0;
#pragma unroll
        for (int d = 0; d < D; d++) {
            a = lane_shr1(uE[k] + zc * a);
            b = lane_shl1(s + zc * b);
        }
        Su[k] = a;
        Sw[k] = b;
        if constexpr (W > 1) {
            if (lane == 63) sx[(3 * k) * W + wave] = fma(zc, a, uE[k]);
            if (lane == 0) {
                sx[(3 * k + 1) * W + wave] = s;
                sx[(3 * k + 2) * W + wave] = b;
            }
        }
        __builtin_amdgcn_sched_barrier(0);  // one sequence after the other: fewer registers
    }
    __syncthreads();
#pragma unroll
    for (int k = 0; k < K; k++) {
        double sn = 0.0, bn = 0.0;  // of the next wavefront's first lane
        const double X = fma(zc, Su[k], uE[k]);
        if constexpr (W > 1) {
            if (wave > 0) Su[k] += zt[lane] * sx[(3 * k) * W + wave - 1];
            if (wave < W - 1) {
                sn = sx[(3 * k + 1) * W + wave + 1];
                bn = sx[(3 * k + 2) * W + wave + 1];
                Sw[k] += zt[63 - lane] * fma(zc, bn, sn);
            }
        }
        double* const m = M[k];
#pragma unroll
        for (int c = 0; c < C; c++) m[c] = A * fma(zp.v[C - c], Sw[k], fma(zp.v[c + 1], Su[k], m[c]));
        m[C] = A * fma(zp.v[C], bn, fma(zp.v[1], X, sn));  // lane 63; the others' follows
        constexpr double idg = 1.0 / (2.0 + z);
        if (wave == 0) {
            const double r0 = g.r1 * ((y[k][2] - y[k][1]) * g.ih - d0[k]);
            const double al = lane_get((r0 - 2.0 * m[0] - m[1]) * idg, 0) * zt[lane];
#pragma unroll
            for (int c = 0; c < C; c++) m[c] += al * zp.v[c];
        }
        if (wave == W - 1) {
            const double rN = g.r1 * (dN[k] - (y[k][C + 1] - y[k][C]) * g.ih);
            const double be = lane_get((rN - m[C - 1] - 2.0 * m[C]) * idg, 63);
            const double bz = be * (z * zt[63 - lane]);
#pragma unroll
            for (int c = 0; c < C; c++) m[c] += bz * zp.v[C - 1 - c];
            m[C] += be;  // lane 63: j = N
        }
        const double mn = lane_shl1(m[0]);
        m[C] = (lane == 63) ? m[C] : mn;
        if (trap) {
            double sy = 0.0, sm = 0.0;
#pragma unroll
            for (int c = 0; c < C; c++) {
                sy += y[k][c + 1] + y[k][c + 2];
                sm += m[c] + m[c + 1];
            }
            trap[k] = 0.5 * g.h * sy - g.h * g.h * g.h * sm * (1.0 / 24.0);
        }
    }
}

}  // namespace tpsc
