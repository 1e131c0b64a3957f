// tpsc_tau.hip -- the tau <-> Matsubara pencils of chi0, V and Sigma (chi0.cpp:566-698, chi.cpp:123-170,
// green.cpp:1925-2018).  Compiled like tpsc_jj.hip, without machine-level loop-invariant code motion.
#include "tpsc_launch.hpp"
#include "tpsc_pencil.hpp"

namespace tpsc {

#define PEN_THREADS 256

// A workgroup takes two adjacent pencils as real and imaginary parts of one transform: a row of the tau-major arrays
// is one access of both values (their only alignment is the element's).  Of an odd count's last pair the missing
// pencil is read as zero; the read itself may pass the array's end by one element, for which every device array has
// room (dalloc).  Four pencils (two pairs in turn, one access a row) measured 0-30% slower: more registers, fewer
// workgroups.  The split of a pair is exact to the rounding of the larger of the two, and a NaN in one pencil
// spreads to its partner.
template <typename S, int Q>
struct __attribute__((packed, aligned(sizeof(S)))) Row {
    S v[Q];
};
template <typename S, int Q>
__device__ __forceinline__ void load_row(const S* a, int nq, S* v)
{
    const Row<S, Q> r = *(const Row<S, Q>*)a;
#pragma unroll
    for (int i = 0; i < Q; i++) v[i] = (i < nq) ? r.v[i] : S(0);
}
template <typename S, int Q>
__device__ __forceinline__ void store_row(S* a, int nq, const S* v)
{
    if (nq == Q) {
        Row<S, Q> r;
#pragma unroll
        for (int i = 0; i < Q; i++) r.v[i] = v[i];
        *(Row<S, Q>*)a = r;
    } else {
#pragma unroll
        for (int i = 0; i < Q; i++)
            if (i < nq) a[i] = v[i];
    }
}
// The samples 8 t .. 8 t + 7 of Q pencils from tau-major rows of nk8 values, and of the lanes at the wavefront's ends
// the neighbour beyond it (sample 8 t - 1 of lane 0, 8 t + 8 of lane 63)
template <typename S, int Q>
struct Chunks {
    S v[8][Q], e[Q];
    __device__ __forceinline__ void load(const S* a, long nk8, int nq, int t)
    {
        const S* const p = a + 8 * t * nk8;
#pragma unroll
        for (int c = 0; c < 8; c++) load_row<S, Q>(p + c * nk8, nq, v[c]);
        const int lane = t & 63;
#pragma unroll
        for (int i = 0; i < Q; i++) e[i] = S(0);
        if (lane == 63 || (lane == 0 && t > 0)) load_row<S, Q>(p + (lane == 0 ? -nk8 : 8 * nk8), nq, e);
    }
    // as pen_spline takes them
    __device__ __forceinline__ void chunk(int t, double (*y)[10]) const
    {
        const int lane = t & 63;
#pragma unroll
        for (int k = 0; k < 2; k++) {
#pragma unroll
            for (int c = 0; c < 8; c++) y[k][1 + c] = (double)v[c][k];
            const double x = (double)e[k], l = lane_shr1(y[k][8]), h = lane_shl1(y[k][1]);
            y[k][0] = (lane == 0) ? x : l;
            y[k][9] = (lane == 63) ? x : h;
        }
    }
};

// ================================================================== chi0
// chi0.cpp:586-698 (L <= 512): per wedge q, clamped spline of chi0(q,tau_j), j=0..Nw/2, slopes
// (dchiqt0[q], 0); F = BACKWARD DFT_Nw of the antisymmetrised 6a_j; tails.
// Reads chi0(q,tau) from chit, writes chi0(q,iqn) to chiw in FP64 (chiw may alias chit in
// the FP64 path: each block reads its column completely before writing it).
template <int L, typename S>
__global__ void __launch_bounds__(PEN_THREADS)
    k_chi0_pencil_short(const S* chit, double* chiw, const double* __restrict__ dchiqt0, double* chi0inf,
                  double* chi0inf2, long nk8, double T, const cd* __restrict__ tw)
{
    constexpr int NS = L / 2;  // intervals
    constexpr int PJ = (NS + PEN_THREADS - 1) / PEN_THREADS;  // intervals per thread
    // The spline samples, then in place their moments (NS + 1 doubles), live in the FFT buffer
    // until the transform input is formed: 36 KB of LDS per workgroup, four per CU.
    static_assert(NS + 1 <= 2 * L, "the spline array fits in the transform buffer");
    __shared__ cd X[L];
    __shared__ double ES[2 * PEN_THREADS + 8];
    __shared__ double sc[16];
    const long q = xcd_remap(blockIdx.x, gridDim.x);
    if (q >= nk8) return;
    const int tid = threadIdx.x, nt = blockDim.x;
    double* y = (double*)X;
    for (int j = tid; j <= NS; j += nt) y[j] = (double)chit[q + (long)j * nk8];
    const double d0 = dchiqt0[q], dN = 0.0;
    const double h = 1.0 / (L * T);
    __syncthreads();
    // y -> moments M in place; integ: this thread's part of the spline's integral
    double integ = 0.0, a6v[PJ];
    {
        double* const ys[1] = {y};
        block_spline_fixed<NS, PEN_THREADS, 1>(ys, h, &d0, &dN, ES, &integ);
    }
    const double* M = y;
#pragma unroll
    for (int c = 0; c < PJ; c++) {
        const int j = tid + c * nt;
        a6v[c] = (j < NS) ? (M[j + 1] - M[j]) / h : 0.0;
    }
    __syncthreads();  // every read of y and M is done: X may be written
#pragma unroll
    for (int c = 0; c < PJ; c++) {
        const int j = tid + c * nt;
        if (j < NS) {
            X[j] = cd{a6v[c], 0.0};
            X[L - 1 - j] = cd{-a6v[c], 0.0};
        }
    }
    integ = block_sum(integ, sc);
    block_fft<L, PEN_THREADS>(X, +1, tw);
    if (tid == 0) chiw[q] = 2 * integ;
    if (q != 0) {
        const double inf = -2.0 * d0;
        for (int j = 1 + tid; j <= NS; j += nt) {
            const double wn = 2 * j * kPi * T;
            // cos, sin of 2 pi j / L from the twiddle table tw[j] = exp(-2 pi i j / L)
            const cd e = tw[j];
            chiw[q + (long)j * nk8] =
                inf / (wn * wn) + ((1.0 - e.x) * X[j].x - e.y * X[j].y) / (wn * wn * wn * wn);
        }
        if (tid == 0) {
            chi0inf[q] = inf;
            chi0inf2[q] = 2.0 * X[NS].x;
        }
    } else {
        for (int j = 1 + tid; j <= NS; j += nt) chiw[(long)j * nk8] = 0.0;
        if (tid == 0) {
            chi0inf[0] = 0.0;
            chi0inf2[0] = 0.0;
        }
    }
}

// The same for L >= 1024, two adjacent pencils per workgroup as real and imaginary parts.  With w = 2 pi n T, phi =
// 2 pi n/L, NS = L/2 intervals of step h, the antisymmetrised transform is, summed by parts,
//   chi0(iq_n) = inf/w^2 - (8 sin^2(phi/2)/h) D_n/w^4,  D_n = M_0/2 + sum_{0<j<NS} M_j cos(phi j) + (-1)^n M_NS/2,
// whose explicit small factor keeps the rounding of D out of the low frequencies (differences 6a_j transformed two to an
// FFT leave L/(2 pi n) times more).  The means m_j = (M_j + M_{j+1})/2 give D_n cos(phi/2) = sum_j m_j cos(phi (j + 1/2)):
// a cosine transform C_n = (e^{-i phi/2} V_n + e^{i phi/2} V_{NS-n})/2 from the length-NS DFT V of the even samples
// followed by the odd ones backwards, a quarter of the work of one length-L FFT per pencil.  n = NS, where cos(phi/2) = 0,
// and chi0inf2 take the alternating sum of 6a_j.
// What bounds it: the columns of the tau-major arrays (a line request per row and workgroup), then latency.  256^2 x 2048
// in FP64 takes 66 us (one length-L LDS FFT per pencil: 141), x 4096 146 (328).
template <int L, typename S>
__global__ void __launch_bounds__(L / 16, 3)
    k_chi0_pencil(const S* chit, double* chiw, const double* __restrict__ dchiqt0, double* chi0inf, double* chi0inf2,
                  int nk8, PenStep g, double w1, const cd* __restrict__ tw, const cd* __restrict__ twX)
{
    constexpr int NS = L / 2, NT = Pen<NS>::NT, W = Pen<NS>::W, PS = Pen<NS>::PS, Q = 2;
    __shared__ __align__(16) cd Z[Pen<NS>::ZD / 2];
    __shared__ double sx[6 * W], sc[4 * W];
    __shared__ SplineTab<8> zt;
    const int t = threadIdx.x;
    zt.fill(t);  // ordered by the barrier of the spline
    const int q0 = Q * xcd_remap(blockIdx.x, gridDim.x), nq = min(Q, nk8 - q0);
    const long ld = nk8;
    Chunks<S, Q> ch;
    ch.load(chit + q0, ld, nq, t);
    double d[Q];
    load_row<double, Q>(dchiqt0 + q0, nq, d);
    const double dN[2] = {0.0, 0.0};
    double out[8][Q];
    cd v[8];
    {
        double y[2][10], M[2][9], integ[2];
        ch.chunk(t, y);
        pen_spline<NS, NT, 2>(y, g, d, dN, M, sx, zt, integ, t);
        // alternating sums of 6a_j (8 t is even)
        double alt[2];
#pragma unroll
        for (int k = 0; k < 2; k++) {
            alt[k] = 0.0;
#pragma unroll
            for (int c = 0; c < 8; c++) alt[k] += (c & 1) ? M[k][c] - M[k][c + 1] : M[k][c + 1] - M[k][c];
            integ[k] = wave_total63(integ[k]);
            alt[k] = wave_total63(alt[k]);
        }
        if ((t & 63) == 63) {
            sc[t >> 6] = integ[0];
            sc[W + (t >> 6)] = integ[1];
            sc[2 * W + (t >> 6)] = alt[0];
            sc[3 * W + (t >> 6)] = alt[1];
        }
        // element i of the transform's input at Z[(i mod 8) PS + i/8]: even samples 2i, then the odd ones backwards
        cd* const lo = Z + 4 * (t & 1) * PS + (t >> 1);
        cd* const hi = Z + (7 - 4 * (t & 1)) * PS + NT - 1 - (t >> 1);
#pragma unroll
        for (int c = 0; c < 8; c += 2) {
            lo[(c / 2) * PS] = cd{M[0][c] + M[0][c + 1], M[1][c] + M[1][c + 1]};
            hi[-(c / 2) * PS] = cd{M[0][c + 1] + M[0][c + 2], M[1][c + 1] + M[1][c + 2]};
        }
    }
    pen_fft_placed<NS, 2>(v, Z, tw, tw[2 * t], tw[4 * t], tw[8 * t], t);
    wave_lds_order();
#pragma unroll
    for (int m = 0; m < 8; m++) Z[m * PS + t] = v[m];
    __syncthreads();
    // V_{NS-k}, k = t + NT m: thread NT - t, row 7 - m; for t = 0 the next row's first column
    const cd* const zq = Z + NT - t + (t == 0 ? 1 : 0);
    const double i0 = -2.0 * d[0], i1 = -2.0 * d[1];
#pragma unroll
    for (int m = 0; m < 8; m++) {
        const int n = t + NT * m;
        const cd x = twX[n];  // cos, sin of phi/2 = pi n/L
        const cd E = (n == 0) ? v[0] : zq[(7 - m) * PS];
        const cd P = conjg(x) * v[m] + x * E;  // 4 C_n (the means' halves left out)
        const double w = n * w1, i2 = rcp_nr(w * w), f = -2.0 * g.ih * x.y * x.y * rcp_nr(x.x) * i2;
        out[m][0] = (i0 + f * P.x) * i2;
        out[m][1] = (i1 + f * P.y) * i2;
    }
    if (t == 0) {  // n = 0: the integral
        out[0][0] = out[0][1] = 0.0;
        for (int i = 0; i < W; i++) {
            out[0][0] += 2.0 * sc[i];
            out[0][1] += 2.0 * sc[W + i];
        }
    }
    if (q0 == 0) {  // chi0(q = 0, iq_n) = 0 for n > 0
#pragma unroll
        for (int m = 0; m < 8; m++)
            if (m > 0 || t > 0) out[m][0] = 0.0;
    }
#pragma unroll
    for (int m = 0; m < 8; m++) store_row<double, Q>(chiw + (t + NT * m) * ld + q0, nq, out[m]);
    if (t == 0) {
        double s[2] = {0.0, 0.0}, o[2], a[2] = {i0, i1};
        for (int i = 0; i < W; i++) {
            s[0] += sc[2 * W + i];
            s[1] += sc[3 * W + i];
        }
        const double w = NS * w1, i2 = rcp_nr(w * w);
#pragma unroll
        for (int k = 0; k < 2; k++) {
            s[k] *= 4.0 * g.ih;
            o[k] = (a[k] + s[k] * i2) * i2;
        }
        if (q0 == 0) s[0] = o[0] = a[0] = 0.0;
        store_row<double, Q>(chiw + NS * ld + q0, nq, o);
        store_row<double, Q>(chi0inf + q0, nq, a);
        store_row<double, Q>(chi0inf2 + q0, nq, s);
    }
}

// ================================================================== V(r,tau)
// chi.cpp:123-170 (L <= 256): REDFT00 over n (length Nw/2+1) for two wedge points per block, as one
// complex FFT of length Nw of the even extensions; then V += fact * chi0(r,tau)
template <int L, typename S>
__global__ void __launch_bounds__(PEN_THREADS)
    k_vertex_pencil_short(S* V, const S* __restrict__ chirt, const double* __restrict__ chirt0, double* V0, long nk8,
                    double fact, const cd* __restrict__ tw, double U, const double* __restrict__ dsc)
{
    if (dsc) fact = vfact(U, dsc[kPscUsp + 1], dsc[kPscUch + 1], 8.0);
    constexpr int H = L / 2;
    __shared__ cd X[L];
    const long q = 2 * (long)xcd_remap(blockIdx.x, gridDim.x);
    if (q >= nk8) return;
    const bool two = (q + 1) < nk8;
    const int tid = threadIdx.x, nt = blockDim.x;
    for (int j = tid; j <= H; j += nt) {
        const double a = (double)V[q + (long)j * nk8];
        const double b = two ? (double)V[q + 1 + (long)j * nk8] : 0.0;
        X[j] = cd{a, b};
        if (j > 0 && j < H) X[L - j] = cd{a, b};
    }
    __syncthreads();
    block_fft<L, PEN_THREADS>(X, -1, tw);
    for (int j = tid; j <= H; j += nt) {
        const long o = q + (long)j * nk8;
        V[o] = (S)(X[j].x + fact * (double)chirt[o]);
        if (two) V[o + 1] = (S)(X[j].y + fact * (double)chirt[o + 1]);
    }
    if (tid == 0) {  // tau = 0 in FP64 for the boundary kernels
        V0[q] = X[0].x + fact * chirt0[q];
        if (two) V0[q + 1] = X[0].y + fact * chirt0[q + 1];
    }
}

// The same for L >= 512 in registers.  What bounds it: as k_chi0_pencil.  256^2 x 2048 mixed takes 66 us (LDS
// passes: 102), FP64 96 (107); x 4096 mixed 142 (246).
template <int L, typename S>
__global__ void __launch_bounds__(Pen<L>::NT, 4)
    k_vertex_pencil(S* V, const S* __restrict__ chirt, const double* __restrict__ chirt0, double* V0, int nk8,
                    double fact, const cd* __restrict__ tw, double U, const double* __restrict__ dsc)
{
    if (dsc) fact = vfact(U, dsc[kPscUsp + 1], dsc[kPscUch + 1], 8.0);
    constexpr int H = L / 2, NT = Pen<L>::NT, PS = Pen<L>::PS, Q = 2;
    __shared__ __align__(16) cd Z[Pen<L>::ZD / 2];
    const int t = threadIdx.x;
    const int q0 = Q * xcd_remap(blockIdx.x, gridDim.x), nq = min(Q, nk8 - q0);
    const long ld = nk8;
    const int j0 = pen_beta<L>(t);
    S in[5][Q], cr[5][Q];  // slots t + NT m; chi0(r,tau) at the outputs' tau = beta + NT m
#pragma unroll
    for (int m = 0; m < 4; m++) load_row<S, Q>(V + (t + NT * m) * ld + q0, nq, in[m]);
#pragma unroll
    for (int m = 0; m < 4; m++) load_row<S, Q>(chirt + (j0 + NT * m) * ld + q0, nq, cr[m]);
#pragma unroll
    for (int i = 0; i < Q; i++) in[4][i] = cr[4][i] = S(0);
    if (t == 0) {
        load_row<S, Q>(V + H * ld + q0, nq, in[4]);
        load_row<S, Q>(chirt + H * ld + q0, nq, cr[4]);
    }
    double v0[Q];
    cd v[8];
#pragma unroll
    for (int m = 0; m < 5; m++) v[m] = cd{(double)in[m][0], (double)in[m][1]};
#pragma unroll
    for (int m = 0; m < 4; m++) Z[m * PS + t] = v[m];
    __syncthreads();
    // element L - n, n = t + NT m: of thread NT - t, row 7 - m; for t = 0 the next row's first column
    const cd* const zq = Z + NT - t + (t == 0 ? 1 : 0);
#pragma unroll
    for (int m = 4; m < 8; m++)
        if (m > 4 || t > 0) v[m] = zq[(7 - m) * PS];
    __syncthreads();
    pen_fft_dif<L>(v, Z, tw, t);
    v0[0] = v[0].x;
    v0[1] = v[0].y;
#pragma unroll
    for (int m = 0; m < 5; m++) {
        in[m][0] = (S)(v[m].x + fact * (double)cr[m][0]);
        in[m][1] = (S)(v[m].y + fact * (double)cr[m][1]);
    }
#pragma unroll
    for (int m = 0; m < 4; m++) store_row<S, Q>(V + (j0 + NT * m) * ld + q0, nq, in[m]);
    if (t == 0) {
        store_row<S, Q>(V + H * ld + q0, nq, in[4]);
        double c0[Q];  // tau = 0 in FP64 for the boundary kernels
        load_row<double, Q>(chirt0 + q0, nq, c0);
#pragma unroll
        for (int i = 0; i < Q; i++) v0[i] += fact * c0[i];
        store_row<double, Q>(V0 + q0, nq, v0);
    }
}

// ================================================================== Sigma(k,iwn)
__device__ __forceinline__ void store_self(cd* Self, long o, cd R, double, double, double, double) { Self[o] = R; }
__device__ __forceinline__ void store_self(cf* Self, long o, cd R, double Sinf, double s2, double s3, double wn)
{
    const cd v = sigma_mom(Sinf, s2, s3, R, wn);
    Self[o] = cf{(float)v.x, (float)v.y};
}

// green.cpp:1925-2018 (L <= 256): per wedge k, spline of Sigma(k,tau_j) (j=0..Nw) with slopes dSig,
// F = BACKWARD DFT[exp(i pi j/Nw) 6a_j], R(k,n) = (1 - exp(i pi (2n+1)/Nw)) F_n
template <int L, typename S, typename SelfT>
__global__ void __launch_bounds__(PEN_THREADS)
    k_sigma_pencil_short(const S* __restrict__ Stau, const double* __restrict__ Sb, const double* __restrict__ dSig,
                   long nk8, double T, SelfT* Self,
                   double* Sinf2, double* Sinf3, double* Sinf4, double* Sinfp,
                   const cd* __restrict__ tw, const cd* __restrict__ twX, const cd* __restrict__ twS)
{
    constexpr int NT = PEN_THREADS;
    __shared__ double y[L + 1];  // the samples, then in place their spline moments
    __shared__ cd X[L];
    __shared__ double ES[2 * NT + 8];
    const long k = xcd_remap(blockIdx.x, gridDim.x);
    if (k >= nk8) return;
    const int tid = threadIdx.x, nt = blockDim.x;
    for (int j = tid; j <= L; j += nt)
        y[j] = (j == 0) ? Sb[k] : (j == L) ? Sb[nk8 + k] : (double)Stau[k + (long)j * nk8];
    const double d0 = dSig[k], dN = dSig[k + nk8];
    const double h = 1.0 / (L * T);
    __syncthreads();
    {
        double* const ys[1] = {y};
        block_spline_fixed<L, NT, 1>(ys, h, &d0, &dN, ES, nullptr);
    }
    const double* M = y;
    for (int j = tid; j < L; j += nt) {
        const double a6 = (M[j + 1] - M[j]) / h;
        X[j] = twX[j] * a6;
    }
    __syncthreads();
    block_fft<L, NT>(X, +1, tw);
    // Sigma_inf = -(Sigma(k=0, 0+) + Sigma(k=0, beta-)) from the boundary values; stored by k = 0
    const double s2 = d0 + dN, s3 = -(M[0] + M[L]), Si = -(Sb[0] + Sb[nk8]);
    if (k == 0 && tid == 0) Sinfp[0] = Si;
    for (int n = tid; n < L / 2; n += nt) {
        const cd R = twS[n] * X[n];
        store_self(Self, k * (L / 2) + n, R, Si, s2, s3, (2 * n + 1) * kPi * T);
        if (n == L / 2 - 1) Sinf4[k] = R.x;
    }
    if (tid == 0) {
        Sinf2[k] = s2;
        Sinf3[k] = s3;
    }
}

// R = (1 - e^{i th}) F, th = (2n+1) pi/L, F = sum_j 6a_j e^{i th j}, 6a_j = (M_{j+1} - M_j)/h, from the transform C = sum_{j<L} M_j
// e^{i th j} of the moments.  Summed by parts, R = -(4 sin^2(th/2)/h) C' + i (sin th/h) (M_0 + M_L), C' with half weights
// at both ends: the small factor keeps the rounding of C, shared by two pencils, out of the low frequencies.  x = 1 -
// e^{i th} in the reference's rounding, whose error of up to an ulp of 1 multiplies F (Sigma by ~1e-8 at T = 0.02, Nw =
// 4096): that part is added.
__device__ __forceinline__ cd sigma_tail(cd C, cd x, double u, double M0, double ML, double ih)
{
    const double c1x = C.x - M0, d = x.x - 0.5 * u, s = -x.y;
    const double fx = s * C.y - x.x * c1x - ML * (1.0 - x.x) - M0, fy = ML * s - x.x * C.y - s * c1x;
    return cd{ih * (d * fx - u * (C.x - 0.5 * (M0 + ML))), ih * (d * fy - u * C.y + s * (M0 + ML))};
}

// The same for L >= 512, two adjacent pencils per workgroup: for real M_j the half-integer frequencies obey A(L-1-n) =
// conj A(n), so one transform D of a + i b (with the other sign) gives conj A(n) = (D_n + conj D_{L-1-n})/2 and conj
// B(n) = (D_n - conj D_{L-1-n})/(2i).  What bounds it: as k_chi0_pencil.  256^2 x 2048 mixed takes 106 us (one LDS FFT per
// pencil: 339), FP64 180 (287); x 4096 mixed 233 (1539).
template <int L, typename S, typename SelfT>
__global__ void __launch_bounds__(Pen<L>::NT, 4)
    k_sigma_pencil(const S* __restrict__ Stau, const double* __restrict__ Sb, const double* __restrict__ dSig, int nk8,
                   PenStep g, double piT, SelfT* Self, double* Sinf2, double* Sinf3, double* Sinf4, double* Sinfp,
                   const cd* __restrict__ tw, const cd* __restrict__ twX, const cd* __restrict__ twS, const double* __restrict__ tw4)
{
    constexpr int H = L / 2, NT = Pen<L>::NT, W = Pen<L>::W, PS = Pen<L>::PS, Q = 2;
    __shared__ __align__(16) cd Z[Pen<L>::ZD / 2];
    __shared__ double sx[6 * W], ends[4];
    __shared__ SplineTab<8> zt;
    const int t = threadIdx.x;
    zt.fill(t);  // ordered by the barrier of the spline
    const int k0 = Q * xcd_remap(blockIdx.x, gridDim.x), nq = min(Q, nk8 - k0);
    Chunks<S, Q> ch;
    ch.load(Stau + k0, nk8, nq, t);
    double d0[Q], dN[Q], b0[Q], bL[Q];
    load_row<double, Q>(dSig + k0, nq, d0);
    load_row<double, Q>(dSig + nk8 + k0, nq, dN);
    load_row<double, Q>(Sb + k0, nq, b0);
    load_row<double, Q>(Sb + nk8 + k0, nq, bL);
    const double Si = -(Sb[0] + Sb[nk8]);  // Sigma_inf = -(Sigma(k=0, 0+) + Sigma(k=0, beta-)); stored by k = 0
    if (k0 == 0 && t == 0) Sinfp[0] = Si;
    cd v[8];
    {
        double y[2][10], M[2][9];
        ch.chunk(t, y);
#pragma unroll
        for (int k = 0; k < 2; k++) {
            y[k][1] = (t == 0) ? b0[k] : y[k][1];
            y[k][9] = (t == NT - 1) ? bL[k] : y[k][9];
        }
        pen_spline<L, NT, 2>(y, g, d0, dN, M, sx, zt, nullptr, t);
        if (t == 0) {
            ends[0] = M[0][0];
            ends[1] = M[1][0];
        }
        if (t == NT - 1) {
            ends[2] = M[0][8];
            ends[3] = M[1][8];
        }
        const cd h = tw[4 * t];  // exp(-8 pi i t / L)
#pragma unroll
        for (int i = 0; i < 8; i++) v[i] = h * cd{M[0][i], M[1][i]};
    }
    pen_fft_dit<L>(v, Z, tw, conjg(twX[2 * t + 1]), tw[2 * t + 1], tw[4 * t + 2], t);
    wave_lds_order();
#pragma unroll
    for (int m = 0; m < 4; m++) Z[m * PS + t] = v[4 + m];
    __syncthreads();
    const int ka = k0;
    const bool two = nq > 1;
    const double s20 = d0[0] + dN[0], s21 = d0[1] + dN[1];
    const double s30 = -(ends[0] + ends[2]), s31 = -(ends[1] + ends[3]);
#pragma unroll
    for (int m = 0; m < 4; m++) {
        const int n = t + NT * m;
        const cd D = v[m], E = Z[(3 - m) * PS + NT - 1 - t], x = twS[n];
        const double u = tw4[n];
        const cd A = sigma_tail(cd{0.5 * (D.x + E.x), -0.5 * (D.y - E.y)}, x, u, ends[0], ends[2], g.ih);
        const cd B = sigma_tail(cd{0.5 * (D.y + E.y), 0.5 * (D.x - E.x)}, x, u, ends[1], ends[3], g.ih);
        const double wn = (2 * n + 1) * piT;
        store_self(Self, (long)ka * H + n, A, Si, s20, s30, wn);
        if (two) store_self(Self, (long)(ka + 1) * H + n, B, Si, s21, s31, wn);
        if (n == H - 1) {
            Sinf4[ka] = A.x;
            if (two) Sinf4[ka + 1] = B.x;
        }
    }
    if (t == 0) {
        Sinf2[ka] = s20;
        Sinf3[ka] = s30;
    }
    if (t == 0 && two) {
        Sinf2[ka + 1] = s21;
        Sinf3[ka + 1] = s31;
    }
}

// ================================================================== launchers
hipError_t launch_chi0_pencil(const Grid& g, const DevArrays& d, hipStream_t s)
{
    const PenStep step = pen_step(1.0 / (g.Nw * g.T));
    const dim3 gr((unsigned)((g.nk8 + 1) / 2));
    DISPATCH_S(g.prec, {
        if (g.Nw <= 512) {
            DISPATCH_L_TO512(g.Nw, hipLaunchKernelGGL((k_chi0_pencil_short<LL, SS>), dim3((unsigned)g.nk8),
                             dim3(PEN_THREADS), 0, s, (const SS*)d.chi, d.chiw, d.dchiqt0, d.chi0inf, d.chi0inf2, g.nk8,
                             g.T, d.twN));
        } else {
            DISPATCH_L_FROM1024(g.Nw, hipLaunchKernelGGL((k_chi0_pencil<LL, SS>), gr, dim3(LL / 16), 0, s,
                                (const SS*)d.chi, d.chiw, d.dchiqt0, d.chi0inf, d.chi0inf2, (int)g.nk8, step,
                                2 * kPi * g.T, d.twN, d.twX));
        }
    });
    return hipGetLastError();
}

hipError_t launch_vertex_pencil(const Grid& g, const DevArrays& d, double U, double Usp, double Uch, hipStream_t s,
                                const double* dsc)
{
    const double fact = U * (3.0 * Usp + Uch) / 8.0;
    const dim3 gr((unsigned)((g.nk8 + 1) / 2));
    DISPATCH_S(g.prec, {
        if (g.Nw <= 256) {
            DISPATCH_L_SHORT(g.Nw, hipLaunchKernelGGL((k_vertex_pencil_short<LL, SS>), gr, dim3(PEN_THREADS), 0, s,
                             (SS*)d.V, (const SS*)d.chirt, d.chirt0, d.V0, g.nk8, fact, d.twN, U, dsc));
        } else {
            DISPATCH_L_LONG(g.Nw, hipLaunchKernelGGL((k_vertex_pencil<LL, SS>), gr, dim3(Pen<LL>::NT), 0, s,
                            (SS*)d.V, (const SS*)d.chirt, d.chirt0, d.V0, (int)g.nk8, fact,
                            d.twN, U, dsc));
        }
    });
    return hipGetLastError();
}

hipError_t launch_sigma_pencil(const Grid& g, const DevArrays& d, hipStream_t s)
{
    const PenStep step = pen_step(1.0 / (g.Nw * g.T));
    const dim3 gr((unsigned)((g.nk8 + 1) / 2));
    DISPATCH_S(g.prec, {
        if (g.Nw <= 256) {
            DISPATCH_L_SHORT(g.Nw, hipLaunchKernelGGL((k_sigma_pencil_short<LL, SS, ST>), dim3((unsigned)g.nk8),
                             dim3(PEN_THREADS), 0, s, (const SS*)d.Stau, d.Sb, d.dSig, g.nk8, g.T, (ST*)d.Self, d.Sinf2,
                             d.Sinf3, d.Sinf4, d.Sinf, d.twN, d.twX, d.twS));
        } else {
            DISPATCH_L_LONG(g.Nw, hipLaunchKernelGGL((k_sigma_pencil<LL, SS, ST>), gr, dim3(Pen<LL>::NT), 0, s,
                            (const SS*)d.Stau, d.Sb, d.dSig, (int)g.nk8, step, kPi * g.T,
                            (ST*)d.Self, d.Sinf2, d.Sinf3, d.Sinf4, d.Sinf, d.twN, d.twX, d.twS, d.tw4));
        }
    });
    return hipGetLastError();
}

}  // namespace tpsc
