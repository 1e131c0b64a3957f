// tpsc_device.hpp -- device building blocks of the TPSC hot path on gfx950 (CDNA4).
//
//  * cd            : complex double; division by the plain formula with one reciprocal of
//                    (c^2+d^2)
//  * wave_r2r_lines: FFTW REDFT00 / RODFT00 of LDS-resident lines, two real lines packed into
//                    one complex sequence of period N = A B: A-point and B-point DFTs in
//                    registers, one exchange through the lines' own LDS, only the lanes that
//                    the even (odd) symmetry leaves independent
//  * block_fft     : workgroup Stockham radix-4/2 complex FFT of a tau-pencil in LDS
//  * block_spline  : clamped cubic spline moments on a uniform grid, solved as a
//                    causal + anti-causal first-order recursion (pole sqrt(3)-2) over
//                    chunks with a 32-sample warm-up, plus the two boundary modes
//  * block reductions in FP64
#pragma once
#include <hip/hip_runtime.h>
#include <stdint.h>

namespace tpsc {

constexpr double kPi = 3.14159265358979323846;

struct cd {
    double x, y;
};
__host__ __device__ inline cd operator+(cd a, cd b) { return cd{a.x + b.x, a.y + b.y}; }
__host__ __device__ inline cd operator-(cd a, cd b) { return cd{a.x - b.x, a.y - b.y}; }
__host__ __device__ inline cd operator-(cd a) { return cd{-a.x, -a.y}; }
__host__ __device__ inline cd operator*(cd a, cd b) { return cd{a.x * b.x - a.y * b.y, a.x * b.y + a.y * b.x}; }
__host__ __device__ inline cd operator*(double s, cd a) { return cd{s * a.x, s * a.y}; }
__host__ __device__ inline cd operator*(cd a, double s) { return cd{a.x * s, a.y * s}; }
__host__ __device__ inline cd operator/(cd a, double s) { return cd{a.x / s, a.y / s}; }
__host__ __device__ inline cd operator/(cd a, cd b)
{
    const double r = 1.0 / (b.x * b.x + b.y * b.y);
    return cd{(a.x * b.x + a.y * b.y) * r, (a.y * b.x - a.x * b.y) * r};
}
__host__ __device__ inline cd operator/(double s, cd b) { return cd{s, 0.0} / b; }
__host__ __device__ inline cd conjg(cd a) { return cd{a.x, -a.y}; }
__host__ __device__ inline double cabs2(cd a) { return sqrt(a.x * a.x + a.y * a.y); }
__device__ inline cd cexpd(cd z)
{
    if (z.y == 0.0) return cd{exp(z.x), z.y};  // the two-pole asymptotes' poles are real as a rule
    double s, c;
    sincos(z.y, &s, &c);
    const double e = exp(z.x);
    return cd{e * c, e * s};
}
__device__ inline cd cis(double ang)
{
    double s, c;
    sincos(ang, &s, &c);
    return cd{c, s};
}
__device__ inline cd csqrtd(cd z)
{
    // principal branch, cut along the negative real axis
    const double r = hypot(z.x, z.y);
    if (r == 0.0) return cd{0.0, z.y};
    if (z.x >= 0.0) {
        const double t = sqrt(0.5 * (r + z.x));
        return cd{t, z.y / (2.0 * t)};
    }
    const double t = sqrt(0.5 * (r - z.x));
    return cd{fabs(z.y) / (2.0 * t), copysign(t, z.y)};
}

__device__ inline long widx(long l, long m) { return m + (l * (l + 1)) / 2; }
// weight of wedge point (l, m), m <= l, in sums over the full zone: 8 images, halved on each
// of the edges l, m in {0, nk - 1} and on the diagonal m = l (green0.cpp:192-195)
__device__ inline double wedge_weight(int l, int m, int nk)
{
    double ww = 8;
    if (l == 0 || l == nk - 1) ww /= 2;
    if (m == 0 || m == nk - 1) ww /= 2;
    if (m == l) ww /= 2;
    return ww;
}
__device__ inline long fold_idx(long x, long y, long N)
{
    if (x > N / 2) x = N - x;
    if (y > N / 2) y = N - y;
    if (y > x) {
        const long t = x;
        x = y;
        y = t;
    }
    return widx(x, y);
}

// blockIdx -> logical block so that consecutive logical blocks run on the same XCD
// (the hardware deals workgroups round-robin over 8 XCDs); neighbouring pencils then
// share L2 lines of the tau-major arrays.
__device__ inline int xcd_remap(int b, int nb)
{
    const int nx = 8;
    const int per = (nb + nx - 1) / nx;
    const int x = b % nx, i = b / nx;
    const int full = nb - (per - 1) * nx;  // XCDs that get `per` blocks
    int base = (x < full) ? x * per : full * per + (x - full) * (per - 1);
    int lb = base + i;
    return lb;
}

// single-precision complex for the FP32 slab transforms of the mixed-precision path
struct cf {
    float x, y;
};
__host__ __device__ inline cf operator+(cf a, cf b) { return cf{a.x + b.x, a.y + b.y}; }
__host__ __device__ inline cf operator-(cf a, cf b) { return cf{a.x - b.x, a.y - b.y}; }
__host__ __device__ inline cf operator*(cf a, cf b) { return cf{a.x * b.x - a.y * b.y, a.x * b.y + a.y * b.x}; }

template <typename Real>
struct cplx_of;
template <>
struct cplx_of<double> {
    using type = cd;
};
template <>
struct cplx_of<float> {
    using type = cf;
};

// ---------------------------------------------------------------------------------
// in-register DFT of length R (R = 1, 2, 3, 4, 6, 8, 12, 16), forward sign, natural order output
// ---------------------------------------------------------------------------------
template <typename C>
__device__ inline C mul_mi(C a) { return C{a.y, -a.x}; }  // a * (-i)

template <int R, typename C>
__device__ __forceinline__ void reg_dft(C* v)
{
    if constexpr (R == 2) {
        const C a = v[0], b = v[1];
        v[0] = a + b;
        v[1] = a - b;
    } else if constexpr (R == 3) {
        // w = exp(-2 pi i/3) = -1/2 - i sqrt(3)/2: X1,2 = a - (b + c)/2 -/+ i (sqrt(3)/2) (b - c)
        using F = decltype(C{}.x);
        const F h = (F)0.86602540378443864676;
        const C a = v[0], s = v[1] + v[2], d = v[1] - v[2];
        const C m = C{a.x - (F)0.5 * s.x, a.y - (F)0.5 * s.y};
        v[0] = a + s;
        v[1] = m + mul_mi(C{h * d.x, h * d.y});
        v[2] = m - mul_mi(C{h * d.x, h * d.y});
    } else if constexpr (R == 4) {
        const C a0 = v[0], a1 = v[1], a2 = v[2], a3 = v[3];
        const C s02 = a0 + a2, d02 = a0 - a2, s13 = a1 + a3, d13 = a1 - a3;
        v[0] = s02 + s13;
        v[2] = s02 - s13;
        v[1] = d02 + mul_mi(d13);
        v[3] = d02 - mul_mi(d13);
    } else if constexpr (R == 8) {
        using F = decltype(C{}.x);
        const F h = (F)0.70710678118654752440;
        C e[4] = {v[0], v[2], v[4], v[6]}, o[4] = {v[1], v[3], v[5], v[7]};
        reg_dft<4>(e);
        reg_dft<4>(o);
        const C w1 = C{h, -h}, w3 = C{-h, -h};
        o[1] = o[1] * w1;
        o[2] = mul_mi(o[2]);
        o[3] = o[3] * w3;
#pragma unroll
        for (int k = 0; k < 4; k++) {
            v[k] = e[k] + o[k];
            v[k + 4] = e[k] - o[k];
        }
    } else if constexpr (R == 6) {
        // 2 x 3: two-point DFTs over n = n2 + 3 n1, w6^(n2 k1), three-point DFTs over n2
        using F = decltype(C{}.x);
        const F h = (F)0.86602540378443864676;
        C e[3], o[3];
#pragma unroll
        for (int i = 0; i < 3; i++) {
            e[i] = v[i] + v[i + 3];
            o[i] = v[i] - v[i + 3];
        }
        o[1] = o[1] * C{(F)0.5, -h};
        o[2] = o[2] * C{(F)-0.5, -h};
        reg_dft<3>(e);
        reg_dft<3>(o);
#pragma unroll
        for (int i = 0; i < 3; i++) {
            v[2 * i] = e[i];
            v[2 * i + 1] = o[i];
        }
    } else if constexpr (R == 12) {
        // 3 x 4: three-point DFTs over n = n2 + 4 n1, w12^(n2 k1), four-point DFTs over n2
        using F = decltype(C{}.x);
        const F h = (F)0.86602540378443864676, q = (F)0.5;
        C a[3][4];
#pragma unroll
        for (int n2 = 0; n2 < 4; n2++) {
            C t[3] = {v[n2], v[n2 + 4], v[n2 + 8]};
            reg_dft<3>(t);
            a[0][n2] = t[0];
            a[1][n2] = t[1];
            a[2][n2] = t[2];
        }
        a[1][1] = a[1][1] * C{h, -q};
        a[1][2] = a[1][2] * C{q, -h};
        a[1][3] = mul_mi(a[1][3]);
        a[2][1] = a[2][1] * C{q, -h};
        a[2][2] = a[2][2] * C{-q, -h};
        a[2][3] = C{-a[2][3].x, -a[2][3].y};
#pragma unroll
        for (int k1 = 0; k1 < 3; k1++) {
            reg_dft<4>(a[k1]);
#pragma unroll
            for (int k2 = 0; k2 < 4; k2++) v[k1 + 3 * k2] = a[k1][k2];
        }
    } else if constexpr (R == 16) {
        // 4 x 4: four-point DFTs over n = n2 + 4 n1, w16^(n2 k1), four-point DFTs over n2
        using F = decltype(C{}.x);
        const F h = (F)0.70710678118654752440, c1 = (F)0.92387953251128675613, s1 = (F)0.38268343236508977173;
        C a[4][4];
#pragma unroll
        for (int n2 = 0; n2 < 4; n2++) {
            C t[4] = {v[n2], v[n2 + 4], v[n2 + 8], v[n2 + 12]};
            reg_dft<4>(t);
#pragma unroll
            for (int k1 = 0; k1 < 4; k1++) a[k1][n2] = t[k1];
        }
        auto w2 = [&](C z) { return C{h * (z.x + z.y), h * (z.y - z.x)}; };   // z w16^2
        auto w6 = [&](C z) { return C{h * (z.y - z.x), -h * (z.x + z.y)}; };  // z w16^6
        a[1][1] = a[1][1] * C{c1, -s1};
        a[1][2] = w2(a[1][2]);
        a[1][3] = a[1][3] * C{s1, -c1};
        a[2][1] = w2(a[2][1]);
        a[2][2] = mul_mi(a[2][2]);
        a[2][3] = w6(a[2][3]);
        a[3][1] = a[3][1] * C{s1, -c1};
        a[3][2] = w6(a[3][2]);
        a[3][3] = a[3][3] * C{-c1, s1};
#pragma unroll
        for (int k1 = 0; k1 < 4; k1++) {
            reg_dft<4>(a[k1]);
#pragma unroll
            for (int k2 = 0; k2 < 4; k2++) v[k1 + 4 * k2] = a[k1][k2];
        }
    }
}

// ---------------------------------------------------------------------------------
// Slab transforms: REDFT00 (kind 0) and RODFT00 (kind 1) along both axes of an LDS slab.
//
// A slab holds element (i, j), 0 <= i, j < nk = N/2+1, at base[j + i * LD].  A kind-1 axis keeps the
// natural index too: its elements are 1 .. nk-2, and lines 0 and nk-1 hold nothing.  The even
// (odd) extension of a line has period N, and its DFT is real (imaginary), so two lines packed as real
// and imaginary parts give both transforms from one complex FFT of length N = A B:
//   z[p + B k] -> A-point DFTs over k (lane p) -> w_N^(p k1) -> B-point DFTs over p (lane k1)
//   -> Z[k1 + A k2].
// The packed sequence is itself even (odd), so z[N - j] = +-z[j] fixes the DFTs of p > B/2 from
// those of B - p, and the outputs of k1 > A/2 from those of A - k1: max(A, B)/2 + 1 lanes carry a
// whole FFT (9 of 16 for N = 256) and a wavefront takes 2F lines, line f with line f + F.  The
// intermediate values are exchanged inside the wavefront through the LDS of the two lines themselves
// (real parts in the first, imaginary parts in the second), so an axis takes one workgroup barrier.
//
// What bounds it: FP64 (FP32) VALU issue and LDS bandwidth, in about equal parts: at N = 256 a lane
// issues two 16-point DFTs, 16 complex products and ~140 LDS accesses per line pair.  LD = lanes per
// FFT (mod 16) spreads the lanes of a wavefront over the LDS banks in both axes; the exchange slots
// are rotated within their blocks of B for the same reason, and every address is a lane register and
// an immediate, with one select where the rotation wraps (1024 slabs of N = 256 alone on the chip:
// 41.5 us per 2D transform in FP64, 25.2 in FP32; 48.5 and 27.1 with slots permuted by an exclusive or
// and offsets computed per access).
// Kernel times at 256^2 x 2048 (kernel trace; three streams overlap), against cross-lane radix-2 stages (one
// FFT per wavefront, shuffles between lanes, a full-period FFT for a line pair): FP64 chi0 1004 -> 248 us,
// vertex 298 -> 94, Sigma 1092 -> 281, h and f0 with hV and f0V 3011 -> 2 x 445; FP32 384 -> 184,
// 115 -> 57, 440 -> 197, 1417 -> 2 x 290.
// ---------------------------------------------------------------------------------
constexpr int slab_A(int N)
{
    return N == 4 ? 2 : (N == 8 || N == 16) ? 4 : (N == 12 || N == 24 || N == 48) ? 6
         : (N == 32 || N == 64 || N == 128) ? 8 : (N == 96 || N == 192) ? 12 : 16;
}
struct SlabDims {
    int nk, A, B, lanes, F, slots, LD, rows, waves, threads;
    long elems;
};
constexpr SlabDims slab_dims(int N)
{
    SlabDims d{};
    d.nk = N / 2 + 1;
    d.A = slab_A(N);
    d.B = N / d.A;
    d.lanes = (d.A > d.B ? d.A : d.B) / 2 + 1;  // lanes per FFT
    const int most = 64 / d.lanes;
    d.waves = (d.nk + 2 * most - 1) / (2 * most);
    d.F = (d.nk + 2 * d.waves - 1) / (2 * d.waves);  // FFTs per wavefront
    d.slots = d.B * (d.A / 2 + 1) - (d.B - 1) / 2;   // exchanged values per FFT
    // the place of a lone line's partner lies beyond the lines: nk lines from 0, or nk - 2 from 1
    int least = d.slots;
    for (int kind = 0; kind < 2; kind++) {
        const int n = d.nk - 2 * kind, w = (n + 2 * d.F - 1) / (2 * d.F), rest = n - 2 * d.F * (w - 1);
        const int end = kind + 2 * d.F * (w - 1) + (rest < d.F ? rest : d.F) + d.F;
        if (end > least) least = end;
    }
    d.LD = least;
    while (d.LD % 16 != d.lanes % 16) d.LD++;
    d.rows = least;
    // one round of FFTs per axis, and at least four wavefronts for the pointwise phases
    d.threads = 64 * (d.waves > 4 ? d.waves : 4);
    d.elems = (long)d.rows * d.LD;
    return d;
}
template <int N>
struct SlabShape {
    static constexpr SlabDims D = slab_dims(N);
    static constexpr int A = D.A, B = D.B, F = D.F, LD = D.LD, NT = D.threads;
};
// LDS bytes of a slab and its twiddle table
constexpr size_t slab_bytes(int N, size_t elem)
{
    return (((size_t)slab_dims(N).elems * elem + 15) & ~(size_t)15) +
           2 * elem * (size_t)((slab_dims(N).B / 2 + 1) * (slab_dims(N).A / 2));
}
// the twiddle table behind the slab, 16-byte aligned
template <int N, typename Real>
__device__ __forceinline__ typename cplx_of<Real>::type* slab_tw(Real* slab)
{
    constexpr size_t off = ((size_t)slab_dims(N).elems * sizeof(Real) + 15) & ~(size_t)15;
    return (typename cplx_of<Real>::type*)((char*)slab + off);
}
// tw[(k1 - 1)(B/2 + 1) + p] = exp(-2 pi i p k1 / N), 1 <= k1 <= A/2, p <= B/2: the lanes p of a product
// read neighbours (block-cooperative; caller syncs); the angle is evaluated in FP64 and rounded to
// the table precision
template <int N, typename C>
__device__ __forceinline__ void fill_twiddles(C* tw)
{
    using F = decltype(C{}.x);
    constexpr int W = SlabShape<N>::B / 2 + 1;
    for (int t = threadIdx.x; t < W * (SlabShape<N>::A / 2); t += blockDim.x) {
        double s, c;
        sincospi(2.0 * (double)((t / W + 1) * (t % W)) / (double)N, &s, &c);
        tw[t] = C{(F)c, (F)(-s)};
    }
}

// LDS accesses of one wavefront complete in order; this keeps the compiler's order
__device__ __forceinline__ void wave_lds_order()
{
    __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
    __builtin_amdgcn_wave_barrier();
}

// A lane's LDS byte offset plus a compile-time constant c: the DS instructions add an immediate below
// 64 KB, so a column (137 x 1096 bytes at N = 256 in FP64) takes up to three bases, kept apart from the
// constants by an empty asm; a row takes one.
template <int MAXC>
struct LdsAddr {
    static constexpr int H = 57344, NB = MAXC / H + 1;
    int b[NB];
    __device__ __forceinline__ explicit LdsAddr(int o)
    {
        b[0] = o;
#pragma unroll
        for (int i = 1; i < NB; i++) {
            b[i] = o + i * H;
            asm("" : "+v"(b[i]));
        }
    }
    __device__ __forceinline__ int operator()(int c) const { return b[c / H] + c % H; }
};
template <int MAXC>
__device__ __forceinline__ int lds_pick(bool t, const LdsAddr<MAXC>& x, const LdsAddr<MAXC>& y, int c)
{
    constexpr int H = LdsAddr<MAXC>::H;
    return (t ? x.b[c / H] : y.b[c / H]) + c % H;
}

// transforms of the lines base + i * LS, i < nlines; element e of a line at e * ES
template <typename Real, int N, int KIND, int LS, int ES>
__device__ __forceinline__ void wave_r2r_lines(Real* base, int nlines, const typename cplx_of<Real>::type* tw)
{
    using C = typename cplx_of<Real>::type;
    constexpr SlabDims D = SlabShape<N>::D;
    constexpr int A = D.A, B = D.B, F = D.F, MIR = (B - 1) / 2;
    constexpr int E = ES * (int)sizeof(Real);          // bytes from one element to the next
    constexpr int PAIR = F * LS * (int)sizeof(Real);   // bytes from a line to its partner
    constexpr int MAXC = (N / 2 + B) * E;
    // the lane index through an empty asm: otherwise the compiler computes the lane's LDS offsets
    // once for all the transforms of a kernel and keeps them in registers across them
    int lane = threadIdx.x & 63;
    asm volatile("" : "+v"(lane));
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int sub = lane / D.lanes, p = lane % D.lanes;
    const int f = 2 * F * wave + sub;  // the first line
    if (2 * F * wave >= nlines) return;
    const bool ok = sub < F && f < nlines;
    const bool has2 = f + F < nlines;
    // element at byte offset o of the first (a) or the second (b) line
    const int lb0 = f * LS * (int)sizeof(Real);
    auto la = [&](int o) -> Real& { return *(Real*)((char*)base + o); };
    auto lb = [&](int o) -> Real& { return *(Real*)((char*)base + o + PAIR); };
    if (ok && p <= B / 2) {
        const LdsAddr<MAXC> up(lb0 + p * E), down(lb0 - p * E), upw(lb0 + p * E - B * E);
        // a lone last line is packed with itself; its partner's place only holds the exchange
        const int pair = has2 ? PAIR : 0;
        C v[A];
#pragma unroll
        for (int k = 0; k < A; k++) {
            const int o = (k < A / 2) ? up(B * k * E) : down(B * (A - k) * E);
            Real a = la(o), b = *(Real*)((char*)base + o + pair);
            if constexpr (KIND == 1) {
                if (k == 0 || k == A / 2) {
                    a = (p == 0) ? (Real)0 : a;
                    b = (p == 0) ? (Real)0 : b;
                }
                if (k >= A / 2) {
                    a = -a;
                    b = -b;
                }
            }
            v[k] = C{a, b};
        }
        reg_dft<A>(v);
        la(up(0)) = v[0].x;
        lb(up(0)) = v[0].y;
        // slot of (p, k1 > 0): B k1 - MIR + (p + k1 + MIR) mod B, of (p, 0): p
        const bool mirror = p != 0 && 2 * p != B;
#pragma unroll
        for (int k1 = 1; k1 <= A / 2; k1++) {
            constexpr int W = B / 2 + 1;
            const int kk = (k1 + MIR) % B;
            const C w = tw[(k1 - 1) * W + p];
            const C e = v[k1] * w;
            const int o = lds_pick(p >= B - kk, upw, up, (B * k1 - MIR + kk) * E);
            la(o) = e.x;
            lb(o) = e.y;
            if constexpr (B > 2) {
                if (mirror) {
                    C m = v[A - k1] * C{w.x, -w.y};
                    if constexpr (KIND == 1) m = C{-m.x, -m.y};
                    const int om = down((B * k1 - MIR + kk) * E) + ((kk >= MIR || p <= kk) ? 0 : B * E);
                    la(om) = m.x;
                    lb(om) = m.y;
                }
            }
        }
    }
    wave_lds_order();
    if (ok && p <= A / 2) {
        int q = p;
        asm volatile("" : "+v"(q));
        C v[B];
        if constexpr (B == 16) {
            // q > 0: (r + q + 7) mod 16 wraps at r + q >= 9, always for r > 8; q = 0 reads r, and the
            // value of 16 - r for r > 8
            const int at0 = lb0 + 17 * q * E, atw = at0 - B * E;
            const unsigned q17 = 17u * q * E;
#pragma unroll
            for (int r = 0; r < B; r++) {
                int o;
                if (r <= 8) {
                    o = ((q >= 9 - r) ? atw : at0) + r * E;
                } else {
                    const unsigned c = (16 - r) * E;
                    o = (int)((q17 > c ? q17 : c) - (q17 < c ? q17 : c)) + lb0;
                }
                Real a = la(o), b = lb(o);
                if constexpr (KIND == 1) {
                    if (r > 8) {
                        a = (q == 0) ? -a : a;
                        b = (q == 0) ? -b : b;
                    }
                }
                v[r] = C{a, b};
            }
        } else {
            const int qm = (q == 0) ? 0 : (q + MIR) & (B - 1);
            const int at0 = lb0 + ((q == 0) ? 0 : B * q - MIR + qm) * E, atw = at0 - B * E;
#pragma unroll
            for (int r = 0; r < B; r++) {
                int o = ((qm >= B - r) ? atw : at0) + r * E;
                if (r > B / 2) o = (q == 0) ? lb0 + (B - r) * E : o;
                Real a = la(o), b = lb(o);
                if constexpr (KIND == 1) {
                    if (r > B / 2) {
                        a = (q == 0) ? -a : a;
                        b = (q == 0) ? -b : b;
                    }
                }
                v[r] = C{a, b};
            }
        }
        reg_dft<B>(v);
        wave_lds_order();
        // Z[q + A k2]: the direct index up to N/2, the mirrored one beyond (equal up to the
        // parity; lanes 0 and A/2 write some values twice)
        const LdsAddr<MAXC> up(lb0 + q * E), down(lb0 - q * E);
#pragma unroll
        for (int k2 = 0; k2 < B; k2++) {
            const bool direct = k2 < (B + 1) / 2;
            const int o = direct ? up(A * k2 * E) : down(A * (B - k2) * E);
            if constexpr (KIND == 0) {
                la(o) = v[k2].x;
                if (has2) lb(o) = v[k2].y;
            } else {
                la(o) = direct ? -v[k2].y : v[k2].y;
                if (has2) lb(o) = direct ? v[k2].x : -v[k2].x;
            }
        }
    }
}

// 2D transform of a slab, axis 1 (the contiguous one) then axis 0: KIND0 along axis 0, KIND1 = 0
// along axis 1
template <typename Real, int N, int KIND0>
__device__ __forceinline__ void slab_r2r_2d(Real* slab, const typename cplx_of<Real>::type* tw)
{
    constexpr int LD = SlabShape<N>::LD, nk = N / 2 + 1;
    wave_r2r_lines<Real, N, 0, LD, 1>(slab + KIND0 * LD, nk - 2 * KIND0, tw);
    __syncthreads();
    wave_r2r_lines<Real, N, KIND0, 1, LD>(slab, nk, tw);
    __syncthreads();
}

// ---------------------------------------------------------------------------------
// Workgroup Stockham FFT in place in LDS: radix-8 passes, then one radix-4 or radix-2 pass
// for the remaining factor of L.  sign = -1: exp(-2 pi i jk/L) (FFTW_FORWARD); sign = +1:
// FFTW_BACKWARD.  twg: global table exp(-2 pi i t / L), t < L.
// Pass with butterfly span Ns: butterfly b (k = b mod Ns) reads x[b + r L/RAD], multiplies
// by w^(r k L/(Ns RAD)), takes an RAD-point DFT and writes y[(b/Ns) Ns RAD + k + m Ns].
// The twiddles w^r come from three table reads (w, w^2, w^4) and products, issued before
// the LDS reads and the barrier so their latency overlaps them.
// ---------------------------------------------------------------------------------
// PP (ping-pong): the pass reads src and writes a different buffer dst, so the barrier
// between its reads and its writes is not needed; in place (src == dst) it is.
template <int RAD, int L, int NT, bool PP = false>
__device__ __forceinline__ void fft_pass(const cd* src, cd* dst, int sign, const cd* __restrict__ twg, int Ns)
{
    constexpr int NB = L / RAD;
    constexpr int PER = (NB + NT - 1) / NT;
    const int tid = threadIdx.x;
    const int stride = L / (Ns * RAD);
    cd w1[PER], w2[PER], w4[PER];
#pragma unroll
    for (int i = 0; i < PER; i++) {
        const int b = tid + i * NT;
        const int k = b % Ns;
        cd a = cd{1.0, 0.0}, c2 = cd{1.0, 0.0}, c4 = cd{1.0, 0.0};
        if (Ns > 1 && b < NB) {
            a = twg[(k * stride) & (L - 1)];
            if (RAD >= 4) c2 = twg[(2 * k * stride) & (L - 1)];
            if (RAD >= 8) c4 = twg[(4 * k * stride) & (L - 1)];
        }
        if (sign > 0) {
            a.y = -a.y;
            c2.y = -c2.y;
            c4.y = -c4.y;
        }
        w1[i] = a;
        w2[i] = c2;
        w4[i] = c4;
    }
    cd v[PER][RAD];
#pragma unroll
    for (int i = 0; i < PER; i++) {
        const int b = tid + i * NT;
        if (b < NB) {
#pragma unroll
            for (int r = 0; r < RAD; r++) v[i][r] = src[b + r * NB];
        }
    }
    if constexpr (!PP) __syncthreads();
#pragma unroll
    for (int i = 0; i < PER; i++) {
        const int b = tid + i * NT;
        if (b < NB) {
            const int k = b % Ns;
            if (Ns > 1) {
                v[i][1] = v[i][1] * w1[i];
                if (RAD >= 4) {
                    v[i][2] = v[i][2] * w2[i];
                    v[i][3] = v[i][3] * (w1[i] * w2[i]);
                }
                if (RAD >= 8) {
                    const cd w3 = w1[i] * w2[i];
                    v[i][4] = v[i][4] * w4[i];
                    v[i][5] = v[i][5] * (w4[i] * w1[i]);
                    v[i][6] = v[i][6] * (w4[i] * w2[i]);
                    v[i][7] = v[i][7] * (w4[i] * w3);
                }
            }
            if (sign > 0) {
#pragma unroll
                for (int r = 0; r < RAD; r++) v[i][r].y = -v[i][r].y;
            }
            reg_dft<RAD>(v[i]);
            if (sign > 0) {
#pragma unroll
                for (int r = 0; r < RAD; r++) v[i][r].y = -v[i][r].y;
            }
            const int o = (b / Ns) * Ns * RAD + k;
#pragma unroll
            for (int r = 0; r < RAD; r++) dst[o + r * Ns] = v[i][r];
        }
    }
    __syncthreads();
}

template <int L, int NT>
__device__ __forceinline__ void block_fft(cd* buf, int sign, const cd* __restrict__ twg)
{
    constexpr int LOG2 = __builtin_ctz(L);
    constexpr int P8 = LOG2 / 3;
    constexpr int REM = LOG2 - 3 * P8;
    int Ns = 1;
#pragma unroll
    for (int pass = 0; pass < P8; pass++) {
        fft_pass<8, L, NT>(buf, buf, sign, twg, Ns);
        Ns *= 8;
    }
    if constexpr (REM == 2) fft_pass<4, L, NT>(buf, buf, sign, twg, Ns);
    if constexpr (REM == 1) fft_pass<2, L, NT>(buf, buf, sign, twg, Ns);
}

// The same transform with a second LDS buffer tmp of L values: the passes alternate between
// buf and tmp and take one barrier each instead of two.  buf must be complete on entry (the
// caller's barrier); the result is in buf (after an odd number of passes it is copied back).
template <int L, int NT>
__device__ __forceinline__ void block_fft_pp(cd* buf, cd* tmp, int sign, const cd* __restrict__ twg)
{
    constexpr int LOG2 = __builtin_ctz(L);
    constexpr int P8 = LOG2 / 3;
    constexpr int REM = LOG2 - 3 * P8;
    constexpr int NP = P8 + (REM > 0 ? 1 : 0);
    cd* a = buf;
    cd* b = tmp;
    int Ns = 1;
#pragma unroll
    for (int pass = 0; pass < P8; pass++) {
        fft_pass<8, L, NT, true>(a, b, sign, twg, Ns);
        cd* t = a;
        a = b;
        b = t;
        Ns *= 8;
    }
    if constexpr (REM == 2) fft_pass<4, L, NT, true>(a, b, sign, twg, Ns);
    if constexpr (REM == 1) fft_pass<2, L, NT, true>(a, b, sign, twg, Ns);
    if constexpr (NP % 2 == 1) {
        for (int j = threadIdx.x; j < L; j += NT) buf[j] = tmp[j];
        __syncthreads();
    }
}

// ---------------------------------------------------------------------------------
// Clamped cubic spline on a uniform grid x_j = j h, j = 0..N (N intervals).
// Moments M_j = S''(x_j) solve
//   2 M_0 + M_1 = r_0,  M_{j-1} + 4 M_j + M_{j+1} = r_j,  M_{N-1} + 2 M_N = r_N
// with r_0 = 6/h ((y_1-y_0)/h - d0), r_j = 6/h^2 (y_{j+1} - 2 y_j + y_{j-1}),
// r_N = 6/h (dN - (y_N-y_{N-1})/h).  The interior operator has Green's function
// A z^{|j|}, z = sqrt(3)-2, A = 1/(2 sqrt 3); P_j = A sum_{i=1}^{N-1} z^{|j-i|} r_i
// = A (u_j + w_j - r_j) with u (w) the causal (anti-causal) recursion s <- r + z s.
// M_j = P_j + alpha z^j + beta z^{N-j}; alpha, beta from the two boundary rows.
// The boundary modes reach 2 KW samples into the sequence (|z|^66 < 1e-37, below FP64
// rounding of the moments).
// ---------------------------------------------------------------------------------
constexpr int KW = 33;

// z^e of the spline pole z = sqrt(3) - 2 by repeated multiplication, z^(N-1) by repeated
// squaring, and the number of neighbouring chunks whose carries count (|z^(C (d-1))| > 1e-19,
// at most maxd)
constexpr double kSplineZ = 1.7320508075688772935 - 2.0;
constexpr double spline_zpow(int e)
{
    double p = 1.0;
    for (int i = 0; i < e; i++) p *= kSplineZ;
    return p;
}
constexpr double spline_zpow_sq(int e)
{
    double r = 1.0, zz = kSplineZ;
    while (e > 0) {
        if (e & 1) r *= zz;
        zz *= zz;
        e >>= 1;
    }
    return r;
}
// z^(S0 + C i), i = 0..I, as compile-time constants: v[i] is the product of S0 + C i factors z
// taken in turn from 1, as a run-time loop p *= z forms it (the same roundings)
template <int I>
struct SplineZTable {
    double v[I + 1];
};
template <int S0, int C, int I>
constexpr SplineZTable<I> spline_ztable()
{
    SplineZTable<I> t{};
    for (int i = 0; i <= I; i++) t.v[i] = spline_zpow(S0 + C * i);
    return t;
}
constexpr int kZSelMax = 16;  // longest table picked by selects instead of a multiply loop
constexpr int spline_carry_terms(double zc, int maxd)
{
    int d = 0;
    double zd = 1.0;
    while (d < maxd && (zd > 1.0e-19 || zd < -1.0e-19)) {
        d++;
        zd *= zc;
    }
    return d;
}

// The clamped spline above, in place, for K sequences of length N (known at compile time) at
// once, their latencies overlapping: yM[k] holds y_0..y_N on entry and the
// moments M_0..M_N on exit.  Each thread keeps its chunk of the right-hand side in registers, so
// no scratch array is needed.  The two first-order recursions run once from a zero state to get
// the chunk-end states, and again after the exchange, seeded with the carries of the
// neighbouring chunks, S_{t-1} = sum_{d>=1} z^{C(d-1)} E_{t-d}, truncated once z^{C(d-1)} <
// 1e-19.  The chunk layout is fixed at compile time, with almost no divergent branches: the
// sequences are padded with zeros past N (the anti-causal recursion then reaches N in the zero
// state it starts from, so the moments do not change), the carries take their compile-time
// number of terms with out-of-range neighbours read as zero, full chunks store without
// per-element tests, and only the chunks within 2 KW of an end take the boundary modes.
// trap (optional): trap[k] receives this thread's part of sum_j h (y_j + y_{j+1})/2
// - h^3 (M_j + M_{j+1})/24, the integral of spline k over [0, N h]; the caller adds the parts.
// ES: LDS scratch of K*(2*NT + 8) doubles.
template <int N, int NT, int K>
__device__ __forceinline__ void block_spline_fixed(double* const* yM, double h, const double* d0, const double* dN,
                                                   double* ES, double* trap)
{
    constexpr int C = (N + 1 + NT - 1) / NT;
    constexpr double z = kSplineZ;
    constexpr double A = 0.28867513459481288225;
    constexpr double zc = spline_zpow(C);
    constexpr int D = spline_carry_terms(zc, NT - 1);
    constexpr int tN = N / C, cN = N % C;                  // thread and slot of j = N
    constexpr int t1 = 1 / C, c1 = 1 % C;                  // of j = 1
    constexpr int tM = (N - 1) / C, cM = (N - 1) % C;      // of j = N - 1
    constexpr double zN1 = spline_zpow_sq(N - 1);
    constexpr double dg = 2.0 + z, off = zN1 * (1.0 + 2.0 * z);
    constexpr double idet = 1.0 / (dg * dg - off * off);
    constexpr int TL = 2 * KW / C;                                     // last thread with j0 <= 2 KW
    constexpr int MH = (2 * KW >= cN + 1) ? (2 * KW - cN - 1) / C + 1 : 0;  // last m with N - jl <= 2 KW
    const int tid = threadIdx.x;
    const int j0 = tid * C;
    const bool full = j0 + C - 1 <= N;
    const double ih = 1.0 / h;
    double* bnd = ES + 2 * K * NT;  // per sequence: r_0, r_N, M_0, M_1, M_{N-1}, M_N (8 slots)
    double ri[K][C], u[K][C];
    double tr[K];
#pragma unroll
    for (int k = 0; k < K; k++) {
        const double* y = yM[k];
        double yv[C + 2];  // y[j0 - 1 .. j0 + C], indices clamped to [0, N]
#pragma unroll
        for (int i = 0; i < C + 2; i++) yv[i] = y[min(max(j0 - 1 + i, 0), N)];
        tr[k] = 0.0;
#pragma unroll
        for (int c = 0; c < C; c++) {
            const int j = j0 + c;
            // from first differences, exact for neighbouring samples: 6/h^2 multiplies their rounding
            const double r = 6.0 * ih * ih * ((yv[c + 2] - yv[c + 1]) - (yv[c + 1] - yv[c]));
            ri[k][c] = (j >= 1 && j <= N - 1) ? r : 0.0;
            if (trap && j < N) tr[k] += h * (yv[c + 1] + yv[c + 2]) * 0.5;
        }
        if (tid == 0) bnd[8 * k + 0] = 6.0 * ih * ((yv[2] - yv[1]) * ih - d0[k]);
        if (tid == tN) bnd[8 * k + 1] = 6.0 * ih * (dN[k] - (yv[cN + 1] - yv[cN]) * ih);
    }
    // chunk-end states of the two recursions from a zero start
#pragma unroll
    for (int k = 0; k < K; k++) {
        double sa = 0.0;
#pragma unroll
        for (int c = 0; c < C; c++) sa = ri[k][c] + z * sa;
        ES[2 * k * NT + tid] = sa;
        sa = 0.0;
#pragma unroll
        for (int c = C - 1; c >= 0; c--) sa = ri[k][c] + z * sa;
        ES[2 * k * NT + NT + tid] = sa;
    }
    __syncthreads();  // all reads of y are done
#pragma unroll
    for (int k = 0; k < K; k++) {
        double Su = 0.0, Sw = 0.0, zd = 1.0;
#pragma unroll
        for (int d = 1; d <= D; d++) {
            const double el = ES[2 * k * NT + max(tid - d, 0)];
            const double er = ES[2 * k * NT + NT + min(tid + d, NT - 1)];
            Su += zd * (tid - d >= 0 ? el : 0.0);
            Sw += zd * (tid + d < NT ? er : 0.0);
            zd *= zc;
        }
        // the recursions again, seeded with the carries from the neighbouring chunks
        double sa = Su;
#pragma unroll
        for (int c = 0; c < C; c++) {
            sa = ri[k][c] + z * sa;
            u[k][c] = sa;
        }
        sa = Sw;
#pragma unroll
        for (int c = C - 1; c >= 0; c--) {
            sa = ri[k][c] + z * sa;
            u[k][c] = A * (u[k][c] + sa - ri[k][c]);
        }
        double* y = yM[k];
        if (full) {
#pragma unroll
            for (int c = 0; c < C; c++) y[j0 + c] = u[k][c];
        } else if (j0 <= N) {
#pragma unroll
            for (int c = 0; c < C; c++)
                if (j0 + c <= N) y[j0 + c] = u[k][c];
        }
        // end moments for the boundary modes (read after the barrier, never rewritten)
        if (tid == 0) bnd[8 * k + 2] = u[k][0];
        if (tid == t1) bnd[8 * k + 3] = u[k][c1];
        if (tid == tM) bnd[8 * k + 4] = u[k][cM];
        if (tid == tN) bnd[8 * k + 5] = u[k][cN];
    }
    __syncthreads();
    const bool edge = j0 <= N && (j0 <= 2 * KW || j0 + C - 1 >= N - 2 * KW);
#pragma unroll
    for (int k = 0; k < K; k++) {
        if (edge) {
            const double R0 = bnd[8 * k + 0] - 2.0 * bnd[8 * k + 2] - bnd[8 * k + 3];
            const double RN = bnd[8 * k + 1] - bnd[8 * k + 4] - 2.0 * bnd[8 * k + 5];
            const double alpha = (dg * R0 - off * RN) * idet;
            const double beta = (dg * RN - off * R0) * idet;
            // z^j and z^(N-j) of this chunk by repeated multiplication from the chunk's first
            // power: z^j0 (thread tid <= TL) and z^(N-jl) (thread tN - m, m <= MH: exponent
            // cN + 1 + (m - 1) C) picked from compile-time tables, no serial loop
            double zlo[C], zhi[C];
            // the thread index through an empty asm, so the picks stay here instead of being
            // hoisted out of a caller's loop into registers held across it
            int ts = tid;
            asm volatile("" : "+v"(ts));
            double zp = 1.0;
            if constexpr (TL <= kZSelMax) {
                constexpr auto tlo = spline_ztable<0, C, TL>();
#pragma unroll
                for (int t = 1; t <= TL; t++) zp = (ts == t) ? tlo.v[t] : zp;
            } else if (j0 <= 2 * KW) {
                for (int e = 0; e < j0; e++) zp *= z;
            }
#pragma unroll
            for (int c = 0; c < C; c++) {
                zlo[c] = zp;
                zp *= z;
            }
            const int jl = min(j0 + C - 1, N);
            zp = 1.0;
            if constexpr (MH <= kZSelMax) {
                if constexpr (MH >= 1) {
                    constexpr auto thi = spline_ztable<cN + 1, C, MH - 1>();
#pragma unroll
                    for (int m = 1; m <= MH; m++) zp = (ts == tN - m) ? thi.v[m - 1] : zp;
                }
            } else if (N - jl <= 2 * KW) {
                for (int e = 0; e < N - jl; e++) zp *= z;
            }
#pragma unroll
            for (int c = C - 1; c >= 0; c--) {
                zhi[c] = zp;
                if (j0 + c <= jl) zp *= z;
            }
            double* y = yM[k];
#pragma unroll
            for (int c = 0; c < C; c++) {
                const int j = j0 + c;
                double add = 0.0;
                if (j <= 2 * KW) add += alpha * zlo[c];
                if (N - j <= 2 * KW) add += beta * zhi[c];
                if (add != 0.0 && j <= N) {
                    const double m = u[k][c] + add;
                    y[j] = m;
                    u[k][c] = m;
                }
            }
        }
        if (trap) {
            double tm = 0.0;
#pragma unroll
            for (int c = 0; c < C; c++) {
                const int j = j0 + c;
                tm += (j > N) ? 0.0 : (j == 0 || j == N) ? u[k][c] : 2.0 * u[k][c];
            }
            trap[k] = tr[k] - h * h * h * tm * (1.0 / 24.0);
        }
    }
    __syncthreads();
}


// ---------------------------------------------------------------------------------
// reductions
// ---------------------------------------------------------------------------------
__device__ inline double wave_sum(double v)
{
#pragma unroll
    for (int o = 32; o >= 1; o >>= 1) v += __shfl_xor(v, o, 64);
    return v;
}
// 1/x for finite, nonzero x of normal range: the hardware reciprocal (v_rcp_f64, relative
// error below 2^-22) refined by two Newton steps, which leave it within an ulp of the quotient;
// five instructions against about ten of an IEEE division.  x = 0 gives NaN, not inf.
__device__ __forceinline__ double rcp_nr(double x)
{
    double r = __builtin_amdgcn_rcp(x);
    r = fma(fma(-x, r, 1.0), r, r);
    return fma(fma(-x, r, 1.0), r, r);
}

// s / b (real s, complex b != 0) with one rcp_nr of |b|^2
__device__ __forceinline__ cd sdiv_rcp(double s, cd b)
{
    const double r = s * rcp_nr(b.x * b.x + b.y * b.y);
    return cd{b.x * r, -b.y * r};
}

// block-wide sums of K values at once; every thread gets the results.
// scratch: LDS double[>= K * nwaves]
template <int K>
__device__ __forceinline__ void block_sum_k(double* v, double* scratch)
{
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6, nw = blockDim.x >> 6;
#pragma unroll
    for (int k = 0; k < K; k++) v[k] = wave_sum(v[k]);
    __syncthreads();
    if (lane == 0)
#pragma unroll
        for (int k = 0; k < K; k++) scratch[k * nw + wave] = v[k];
    __syncthreads();
#pragma unroll
    for (int k = 0; k < K; k++) {
        double s = 0.0;
        for (int i = 0; i < nw; i++) s += scratch[k * nw + i];
        v[k] = s;
    }
    __syncthreads();
}

// block-wide sum; every thread gets the result. scratch: LDS double[>= nwaves]
__device__ inline double block_sum(double v, double* scratch)
{
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6, nw = blockDim.x >> 6;
    v = wave_sum(v);
    __syncthreads();
    if (lane == 0) scratch[wave] = v;
    __syncthreads();
    double s = 0.0;
    for (int i = 0; i < nw; i++) s += scratch[i];
    __syncthreads();
    return s;
}


// ---------------------------------------------------------------------------------
// pointwise loops over a slab, the tau dependence of G0 and the Sigma(k,iwn) storage forms (shared by
// the slab and pencil kernels of all files)
// ---------------------------------------------------------------------------------
// f(a, b, i) for every wedge point i (packed index) of the workgroup's share, a and b the slab offsets
// of (l, m) and (m, l), from the table wt (k_model): a pointwise phase then reads its wedge arrays in
// order and does no index arithmetic.  The loop is unrolled in at most two batches, so that the loads of
// a batch are in flight together.
template <int N>
constexpr int wedge_per_thread() { return ((N / 2 + 1) * (N / 2 + 2) / 2 + SlabShape<N>::NT - 1) / SlabShape<N>::NT; }
template <int N, typename Fn>
__device__ __forceinline__ void each_wedge(const unsigned* __restrict__ wt, Fn&& f)
{
    constexpr int nk8 = (N / 2 + 1) * (N / 2 + 2) / 2;
    constexpr int PER = wedge_per_thread<N>(), U = (PER <= 8) ? PER : (PER + 1) / 2;
#pragma unroll 1
    for (int c0 = 0; c0 < PER; c0 += U) {
#pragma unroll
        for (int u = 0; u < U; u++) {
            const int i = threadIdx.x + (c0 + u) * SlabShape<N>::NT;
            if (i < nk8) {
                const unsigned w = wt[i];
                f((int)(w & 0xffffu), (int)(w >> 16), i);
            }
        }
    }
}
// the same with the slot c of the point among the thread's own, fully unrolled: f may index registers by c
template <int N, typename Fn>
__device__ __forceinline__ void each_wedge_slot(const unsigned* __restrict__ wt, Fn&& f)
{
    constexpr int nk8 = (N / 2 + 1) * (N / 2 + 2) / 2;
    int tid = threadIdx.x;
    asm volatile("" : "+v"(tid));  // indices and offsets are read again in each phase, not kept
#pragma unroll
    for (int c = 0; c < wedge_per_thread<N>(); c++) {
        const int i = tid + c * SlabShape<N>::NT;
        if (i < nk8) {
            const unsigned w = wt[i];
            f((int)(w & 0xffffu), (int)(w >> 16), i, c);
        }
    }
}
// the thread's wedge values of a global array, ahead of a transform that hides their latency
template <int N, typename S>
__device__ __forceinline__ void load_wedge(const S* __restrict__ a, S* v)
{
    constexpr int nk8 = (N / 2 + 1) * (N / 2 + 2) / 2;
#pragma unroll
    for (int c = 0; c < wedge_per_thread<N>(); c++) {
        const int i = threadIdx.x + c * SlabShape<N>::NT;
        v[c] = (i < nk8) ? a[i] : (S)0;
    }
}
// f(l, m, s) for every point of the Lambda grid: kx index l + 1 (slab line l + 1), s = m + l nk
template <int N, typename Fn>
__device__ __forceinline__ void each_lambda(Fn&& f)
{
    constexpr int nk = N / 2 + 1, nq = nk * (nk - 2);
#pragma unroll 2
    for (int s = threadIdx.x; s < nq; s += SlabShape<N>::NT) {
        const int l = s / nk;
        f(l, s - l * nk, s);
    }
}
// slab offset of element (l, m)
template <int N>
__device__ __forceinline__ int at(int l, int m)
{
    return m + l * SlabShape<N>::LD;
}
// G0(k,tau) without its weight, e^{-x t} (x = eps - mu0 >= 0) or e^{x (beta - t)}: times
// fw = f / N^2, f = 1/(e^{-|x|/T} + 1) (k_mu0_root), it is -G0(k,t)/N^2 and, with t -> beta - t,
// G0(k,-t)/N^2 (chi0.cpp:468-471, 486-489)
__device__ __forceinline__ double g0_exp(double x, double t, double bt) { return exp(x >= 0.0 ? -t * x : bt * x); }

// Sinf/z + s2/z^2 + s3/z^3 + R/z^4, z = i wn (green.cpp:3039), iw = 1/wn
__device__ __forceinline__ cd sigma_mom_i(double Sinf, double s2, double s3, cd R, double iw)
{
    const double iw2 = iw * iw;
    return cd{(-s2 + R.x * iw2) * iw2, (-Sinf + (s3 + R.y * iw) * iw2) * iw};
}
__device__ __forceinline__ cd sigma_mom(double Sinf, double s2, double s3, cd R, double wn)
{
    return sigma_mom_i(Sinf, s2, s3, R, rcp_nr(wn));
}

// Sigma(k, i w_n), w_n > 0, at offset o of the stored form: the remainder R (FP64 path,
// assembled with the moments) or the assembled value itself (mixed path)
__device__ __forceinline__ cd sigma_kw(const cd* __restrict__ Self, long o, double Sinf, double s2, double s3,
                                       double wn)
{
    return sigma_mom(Sinf, s2, s3, Self[o], wn);
}
__device__ __forceinline__ cd sigma_kw(const cf* __restrict__ Self, long o, double, double, double, double)
{
    const cf v = Self[o];
    return cd{(double)v.x, (double)v.y};
}

// Point scalars formed on the device by the queued solve (tpsc_capi.cpp) where the host passes
// them by value otherwise, with the host's rounding (no contraction into fused multiply-adds):
// U (3 Usp + Uch) / div, and the charge sum rule's constant part
// A0 - (nsr + Usp nsr^2 / (2U) - nsr^2), A0 = n - n^2/2 (chi.cpp:830-843).
__device__ __forceinline__ double vfact(double U, double Usp, double Uch, double div)
{
#pragma clang fp contract(off)
    return U * (3.0 * Usp + Uch) / div;
}
__device__ __forceinline__ double uch_a0(double A0, double nsr, double U, double Usp)
{
#pragma clang fp contract(off)
    return A0 - (nsr + Usp * nsr * nsr / (2.0 * U) - nsr * nsr);
}

}  // namespace tpsc
