// tpsc_jj.hip -- Lambda_jj along the tau pencils: two-pole asymptotes, per-point splines and transforms, the
// kx = 0, pi rows of the diamagnetic term.
//
// Compiled without machine-level loop-invariant code motion (Makefile): it lifts every FP64 constant and table
// address out of the loop over the points, and the registers of the transforms then spill.
#include "tpsc_launch.hpp"
#include "tpsc_pencil.hpp"

namespace tpsc {

struct Poles {
    cd r1, r2, a1, a2, b1, b2, den1, den2;
};

// roots of z^2 + (mu - e) z - Sigma_inf with Newton polish (generique.cpp:1666-1726)
__device__ __forceinline__ void roots2(cd A, cd B, cd Cc, cd* roots)
{
    if (!(cabs2(A) > 1.0e-15)) return;
    const cd Rr = csqrtd(B * B - 4.0 * A * Cc);
    roots[0] = (-B - Rr) / (2.0 * A);
    roots[1] = (-B + Rr) / (2.0 * A);
    for (int j = 0; j < 2; j++) {
        cd x = roots[j];
        cd yv = A * x * x + B * x + Cc;
        cd p = 2.0 * A * x + B;
        const cd y0 = yv;
        int it = 0;
        while (cabs2(p) != 0.0 && it < 10 && cabs2(yv) > 1.0e-16) {
            const cd x2 = x, y2 = yv;
            const cd cc = yv - p * x;
            x = (-cc) / p;
            yv = A * x * x + B * x + Cc;
            p = 2.0 * A * x + B;
            if (cabs2(y2) < cabs2(yv)) {
                x = 0.5 * (x + x2);
                yv = A * x * x + B * x + Cc;
                p = 2.0 * A * x + B;
            }
            it++;
        }
        if (cabs2(yv) < cabs2(y0)) roots[j] = x;
    }
}

// the same for real roots (B^2 - 4 Cc >= 0, A = 1) in real arithmetic: a chain of dependent operations on few threads,
// so its latency counts (complex roots for every point: k_jj_poles 10.4 us at 16 x 16, 19.2 at 256 x 256; now 7.6, 12.9)
__device__ __forceinline__ void roots2_real(double B, double Cc, double* roots)
{
    const double Rr = sqrt(B * B - 4.0 * Cc);
    roots[0] = 0.5 * (-B - Rr);
    roots[1] = 0.5 * (-B + Rr);
    for (int j = 0; j < 2; j++) {
        double x = roots[j], yv = x * x + B * x + Cc, p = 2.0 * x + B;
        const double y0 = yv;
        for (int it = 0; p != 0.0 && it < 10 && fabs(yv) > 1.0e-16; it++) {
            const double x2 = x, y2 = yv;
            x = (p * x - yv) / p;
            yv = x * x + B * x + Cc;
            p = 2.0 * x + B;
            if (fabs(y2) < fabs(yv)) {
                x = 0.5 * (x + x2);
                yv = x * x + B * x + Cc;
                p = 2.0 * x + B;
            }
            if (x == x2) break;  // the remaining steps would repeat this one
        }
        if (fabs(yv) < fabs(y0)) roots[j] = x;
    }
}

__device__ __forceinline__ Poles make_poles(double e, double mu, double Sinf, double CJ1, double T)
{
    Poles P;
    cd roots[2] = {cd{0, 0}, cd{0, 0}};
    if ((mu - e) * (mu - e) + 4.0 * Sinf >= 0.0) {
        double r[2];
        roots2_real(mu - e, -Sinf, r);
        roots[0].x = r[0];
        roots[1].x = r[1];
    } else {
        roots2(cd{1.0, 0.0}, cd{-e + mu, 0.0}, cd{-Sinf, 0.0}, roots);
    }
    P.r1 = roots[0];
    P.r2 = roots[1];
    P.a1 = P.r1 / (P.r1 - P.r2);
    P.a2 = P.r2 / (P.r2 - P.r1);
    P.b1 = CJ1 / (P.r1 - P.r2);
    P.b2 = -P.b1;
    P.den1 = (P.r1.x > 0 ? cexpd(-(P.r1 / T)) : cexpd(P.r1 / T)) + cd{1.0, 0.0};
    P.den2 = (P.r2.x > 0 ? cexpd(-(P.r2 / T)) : cexpd(P.r2 / T)) + cd{1.0, 0.0};
    return P;
}

// Two-pole asymptote data of every Lambda-grid point (cond_opt.cpp:3409-3467): the roots of
// z^2 + (mu - e) z - Sigma_inf, the residues over the denominators, and the pole parts of the tau = 0+ / beta-
// slopes and of k0.  One thread per point.
struct JJPoles {
    cd r1, r2;
    cd a1d, a2d, b1d, b2d;  // a1/den1, a2/den2, b1/den1, b2/den2
    double s1, s2;          // exp(-|r| dt) of real poles, dt = the pencil threads' stride in tau
    double Jinf_beta;       // the two-pole part of J at tau = beta
    double dGp, dGm, dJ0, dJb, k0r;
};
static_assert(sizeof(JJPoles) <= 64 * sizeof(double), "DevArrays::poles holds 64 doubles per point");

__global__ void k_jj_poles(const double* __restrict__ ek, const double* __restrict__ hVb,
                           const double* __restrict__ Sinfp, int N, double T, double mu, double dt, JJPoles* out,
                           const double* __restrict__ dsc)
{
    if (dsc) mu = dsc[kPscMu + 1];
    const int nk = N / 2 + 1;
    const long nq = (long)nk * (nk - 2);
    const long q = blockIdx.x * (long)blockDim.x + threadIdx.x;
    if (q >= nq) return;
    const int l = (int)(q / nk), m = (int)(q % nk);
    const double e = ek[m + (l + 1) * nk];
    const double CJ1 = -hVb[q] - hVb[nq + q];
    JJPoles o;
    const Poles P = make_poles(e, mu, Sinfp[0], CJ1, T);
    o.r1 = P.r1;
    o.r2 = P.r2;
    o.a1d = P.a1 / P.den1;
    o.a2d = P.a2 / P.den2;
    o.b1d = P.b1 / P.den1;
    o.b2d = P.b2 / P.den2;
    o.s1 = exp(-dt * fabs(P.r1.x));
    o.s2 = exp(-dt * fabs(P.r2.x));
    // factor at tau = beta of a pole with Re r > 0 (at 0 otherwise); the other end's is 1
    const double beta = 1.0 / T;
    const bool p1 = P.r1.x > 0, p2 = P.r2.x > 0;
    const cd x1 = p1 ? cexpd(-(beta * P.r1)) : cexpd(beta * P.r1), x2 = p2 ? cexpd(-(beta * P.r2)) : cexpd(beta * P.r2);
    o.Jinf_beta = ((p1 ? o.b1d : o.b1d * x1) + (p2 ? o.b2d : o.b2d * x2)).x;
    const cd f1p = p1 ? o.a1d : o.a1d * x1, f1m = p1 ? o.a1d * x1 : o.a1d;
    const cd f2p = p2 ? o.a2d : o.a2d * x2, f2m = p2 ? o.a2d * x2 : o.a2d;
    const cd g1 = P.r1 * o.b1d, g2 = P.r2 * o.b2d;
    o.dGp = (P.r1 * f1p + P.r2 * f2p).x;
    o.dGm = (P.r1 * f1m + P.r2 * f2m).x;
    o.dJ0 = ((p1 ? g1 * x1 : g1) + (p2 ? g2 * x2 : g2)).x;
    o.dJb = ((p1 ? g1 : g1 * x1) + (p2 ? g2 : g2 * x2)).x;
    o.k0r = (f1m + f2m).x;
    out[q] = o;
}

// Per-k Lambda_jj contributions (cond_opt.cpp:3179-3822).  Workgroup blk handles the points
// q = blk + kk*nblk, kk < kp, one at a time, or, by angle of k (cond_opt.cpp:3792-3793), the points
// order[i], first[blk] <= i < first[blk+1], all of one bin (JJGroups), and writes one pair of rows:
// part[blk*2*nwb + n] (bubble) and part[blk*2*nwb + nwb + n] (Maki-Thompson).
//
// Per point, two complex FFTs of pairs of sequences whose transforms have a known symmetry:
//   (1) the f0V and hV spline moments 6a_j (real) at half-integer frequencies: for real a,
//       A(n) = sum_j a_j e^{2 pi i j (n + 1/2)/L} obeys A(L-1-n) = conj A(n), so the transform D of
//       a + i b with the other sign splits into conj A(n) = (D_n + conj D_{L-1-n})/2 and
//       conj B(n) = (D_n - conj D_{L-1-n})/(2i);
//   (2) G(ikn) - G2 and conj(J(ikn)) (both Hermitian in n -> -n-1): the transform of
//       Gn + i conj Jn at tau_j is real for each, G(tau_j) + i J(tau_j) before the two-pole terms.
// Everything after the products -G(tau) G(-tau) and G(tau) J(-tau) is linear in them: the spline
// over [0, beta], its integral and the third transform.  The weighted products and end slopes
// are therefore summed over the points of a workgroup, and the spline and the transform follow once
// per workgroup instead of once per point.  The sums of up to 16 points carry their
// rounding along (add_lo), since the spline divides second differences by h^2; up to L = 256 that
// factor is small and plain sums do.
// The bubble samples are symmetric about beta/2 (the product is the same in both orders), so
// the clamped spline over [0, beta] with end slopes (dchi, -dchi) is, on [0, beta/2], the
// reference's spline with slopes (dchi, 0), and its integral is twice that of the half.
// Imaginary parts of G(tau), J(tau) are zero in exact arithmetic and are not formed.
// hT, f0T are the hV, f0V pencils in point-major layout [q][j] (k_transpose); the pole data come
// from k_jj_poles.
//
// L = 512 .. 4096: L/8 threads per point, the transforms of tpsc_pencil.hpp, eight barriers a point.  LDS holds
// one exchange buffer and the Maki-Thompson sums, 53 KB at L = 2048: three workgroups per CU at 160 registers.
// What bounds it: FP64 VALU issue, then LDS.  With the last spline and transform once per workgroup, half
// the slots (n >= 0), real poles by two exponentials and no LDS-resident passes, 256^2 x 2048 takes 0.44 ms in FP64
// and 0.42 mixed (before: 1.55 and 1.48), 256^2 x 4096 mixed 0.94 (3.50), 128^2 x 1024 0.070 (0.40).

// Scales of the Lambda pencils, formed on the host: T, pi T, beta, 1/N^2 and the threads' stride in tau
struct JJScale {
    double T, piT, beta, nf, dt;
};

// Matsubara data of slot n >= 0 (k_n = (2n+1) pi T, ik = 1/k_n): from the split transforms A, B of
// f0V, hV and Sigma sg, Gn = G - G2 and Jn = G J - G2 (-CJ1/(i k)) (cond_opt.cpp:3302-3407).
struct JJPoint {
    double e0, Sinf, C2, C3;              // mu - e, the moments of Sigma
    double cj01, cj02, cj03, cj1, cj2, cj3;  // tails of the f0V and hV transforms
};
__device__ __forceinline__ cd sigma_ik(cd R, double Sinf, double s2, double s3, double iw)
{
    return sigma_mom_i(Sinf, s2, s3, R, iw);
}
__device__ __forceinline__ cd sigma_ik(cf v, double, double, double, double) { return cd{(double)v.x, (double)v.y}; }
template <typename SelfT>
__device__ __forceinline__ void jj_slot(const JJPoint& c, cd A, cd B, cd ts, SelfT raw, double kn, double T, cd& Gn,
                                        cd& Jn, double& qn0)
{
    const double ik = rcp_nr(kn), ik2 = ik * ik;
    // -i c1/k - c2/k^2 + i c3/k^3 + a/k^4 (cond_opt.cpp:3302-3311)
    const cd af = ts * A, ah = ts * B;
    const cd J0 = cd{(-c.cj02 + af.x * ik2) * ik2, (-c.cj01 + (c.cj03 + af.y * ik) * ik2) * ik};
    const cd Jv = cd{(-c.cj2 + ah.x * ik2) * ik2, (-c.cj1 + (c.cj3 + ah.y * ik) * ik2) * ik};
    const cd sg = sigma_ik(raw, c.Sinf, c.C2, c.C3, ik);
    const cd G = sdiv_rcp(T, cd{c.e0 - sg.x, kn - sg.y});
    const cd G2 = sdiv_rcp(T, cd{c.e0, kn + c.Sinf * ik});
    const cd GG = G * G;
    qn0 = GG.x * J0.x - GG.y * J0.y;
    const double cg = c.cj1 * ik;
    Gn = G - G2;
    Jn = cd{G.x * Jv.x - G.y * Jv.y - G2.y * cg, G.x * Jv.y + G.y * Jv.x + G2.x * cg};
}

// Two-pole parts of G(tau_j) and J(tau_j), added to v[m] = G + i J at tau_j = t0 + m dt, m < M = beta/dt.  Poles
// on the real axis (Sigma_inf > 0 puts both there): with rho = |r|, s = exp(-rho dt), the two factors of
// a pole are exp(-rho t0) s^m and exp(-rho (dt - t0)) s^(M-1-m), both walked in the direction in which they
// fall, so that an underflow is the right value.  Others: each factor directly.
template <int M>
__device__ __forceinline__ void jj_real_pole(cd* v, double r, double s, double ca, double cb, double t0, double dt)
{
    const double rho = fabs(r);
    double d = exp(-rho * t0);
    double u = (rho * dt < 300.0) ? s * rcp_nr(d) : exp(-rho * (dt - t0));
    // the empty asm keeps the compiler from merging the branches' last stores into one through a pointer, which
    // would put v into scratch memory
    if (r > 0) {
#pragma unroll
        for (int m = 0; m < M; m++) {
            v[m].x += ca * d;
            v[M - 1 - m].y += cb * u;
            d *= s;
            u *= s;
        }
        asm volatile("; falling G" ::);
    } else {
#pragma unroll
        for (int m = 0; m < M; m++) {
            v[M - 1 - m].x += ca * u;
            v[m].y += cb * d;
            d *= s;
            u *= s;
        }
        asm volatile("; rising G" ::);
    }
}
// cell[m stride]: LDS of this thread, M values (free on entry), through which the general case goes: it then
// needs no registers beside the caller's
template <int M>
__device__ __forceinline__ void jj_poles_add(cd* v, const JJPoles& pp, double t0, double dt, double beta, cd* cell,
                                             int stride)
{
    if (pp.r1.y == 0.0 && pp.r2.y == 0.0) {
        jj_real_pole<M>(v, pp.r1.x, pp.s1, -pp.a1d.x, pp.b1d.x, t0, dt);
        jj_real_pole<M>(v, pp.r2.x, pp.s2, -pp.a2d.x, pp.b2d.x, t0, dt);
        return;
    }
#pragma unroll
    for (int m = 0; m < M; m++) cell[m * stride] = v[m];
    // e(t) = exp(-t r) or exp((beta - t) r), ej(t) = exp(r (t - beta)) or exp(r t): modulus <= 1 on [0, beta]
#pragma unroll 1
    for (int i = 0; i < 4 * M; i++) {
        const int m = i >> 2;
        const double tm = t0 + m * dt;
        const cd r = (i & 1) ? pp.r2 : pp.r1;
        const bool isj = i & 2;
        const cd ca = isj ? ((i & 1) ? pp.b2d : pp.b1d) : -((i & 1) ? pp.a2d : pp.a1d);
        const double x = (r.x > 0) == isj ? tm - beta : tm, xs = isj ? x : -x;
        double sn, cs;
        sincospi(xs * r.y * (1.0 / kPi), &sn, &cs);
        double* const o = isj ? &cell[m * stride].y : &cell[m * stride].x;
        *o += exp(xs * r.x) * (ca.x * cs - ca.y * sn);
    }
#pragma unroll
    for (int m = 0; m < M; m++) v[m] = cell[m * stride];
}

// Lambda rows at i w_n, n >= 1, from the packed transform of the two splines' moments (Fn at n, Fq at L - n).  Summed by
// parts, with phi = 2 pi n/L and C'_n the transform with half weights at both ends,
//   (1 - e^{-i phi}) sum_j 6a_j e^{-i phi j} = -(4 sin^2(phi/2)/h) C'_n + i (sin phi/h) (M_L - M_0),
// whose explicit small factor keeps the rounding of the transform out of the low frequencies.  x = exp(i phi/2), w1 =
// 2 pi T, ih = 1/h.
__device__ __forceinline__ void jj_rows(double* c1, double* c2, int n, cd Fn, cd Fq, cd x, double MJ1, double MJ3,
                                        double dchi, double w1, double ih)
{
    const double iw = rcp_nr(n * w1), iw2 = iw * iw;
    const double s2 = 2.0 * x.y * ih, u = s2 * x.y;  // 4 sin^2(phi/2)/(2h): the halves of the split of F
    const double ay = -u * (Fn.y - Fq.y) - s2 * x.x * MJ3, bx = -u * (Fn.y + Fq.y);
    // -2 MJ1/wn + 2 MJ3/wn^3 + 2 a/wn^4, then / wn
    c2[n] = -((-2.0 * MJ1 + (2.0 * MJ3 + 2.0 * ay * iw) * iw2) * iw) * iw;
    c1[n] = -((-2.0 * dchi + bx * iw2) * iw2);
}

// hi += p, the rounding of the sum added to lo
__device__ __forceinline__ void add_lo(double& hi, float& lo, double p)
{
    const double s = hi + p, b = s - hi;
    lo += (float)((hi - (s - b)) + (p - b));
    hi = s;
}

template <int L, typename S, typename SelfT>
__global__ void __launch_bounds__(Pen<L>::NT, (L > 2048 ? 2 : 3))
    k_jj_pencil(const double* __restrict__ ek, const double* __restrict__ dek, const double* __restrict__ d2ek,
                const S* __restrict__ hT, const S* __restrict__ f0T, const double* __restrict__ dhV,
                const double* __restrict__ df0V, const double* __restrict__ hVb, const double* __restrict__ f0Vb,
                const JJPoles* __restrict__ poles, const SelfT* __restrict__ Self, const double* __restrict__ Sinf2,
                const double* __restrict__ Sinf3, const double* __restrict__ Sinfp, int N, PenStep g, JJScale u, double mu,
                const cd* __restrict__ tw, const cd* __restrict__ twX, const cd* __restrict__ twS, double* part, double* scal,
                JJGroups gr, int kp, const double* __restrict__ dsc)
{
    if (dsc) mu = dsc[kPscMu + 1];
    using P8 = Pen<L>;
    constexpr int NT = P8::NT, W = P8::W, PS = P8::PS, H = L / 2, NWB = H + 1;
    __shared__ __align__(16) cd Z[P8::ZD / 2];
    __shared__ double aM[L];
    __shared__ double sx[6 * W];   // spline carries
    __shared__ double ends[4];     // end moments of the two splines
    __shared__ double sc[4 * W];   // wavefront sums
    __shared__ double tot[4];      // thread 0's sums over the points: end slopes and sample L of the Maki-Thompson
                                   // spline, end slope of the bubble's
    const int nk = N / 2 + 1;
    const int nq = nk * (nk - 2);
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    const int blk = xcd_remap(blockIdx.x, gridDim.x);
    const int nblk = gridDim.x;
    __shared__ SplineTab<8> zt;
    zt.fill(tid);
    __syncthreads();
    JJPoint c;
    c.Sinf = Sinfp[0];
    double k0acc = 0.0, inf1 = 0.0, inf2 = 0.0, inf4 = 0.0;
    const int i0 = gr.order ? gr.first[blk] : 0, ni = gr.order ? gr.first[blk + 1] - i0 : kp;
    // sums of the products at j = beta + NT m: bubble (j <= L/2) in registers, Maki-Thompson in the thread's
    // own LDS cells
    double aB[4], aH = 0.0, aq = 0.0;
    float lM[8], lB[4];
#pragma unroll
    for (int m = 0; m < 8; m++) {
        aM[m * NT + tid] = 0.0;
        lM[m] = 0.0f;
    }
#pragma unroll
    for (int m = 0; m < 4; m++) {
        aB[m] = 0.0;
        lB[m] = 0.0f;
    }
    if (tid == 0) tot[0] = tot[1] = tot[2] = tot[3] = 0.0;
    // the workgroups resident on one XCD (consecutive blk) work on consecutive q at the same time and
    // share the cache lines of Sigma and of the pole data
#pragma unroll 1
    for (int kk = 0; kk < ni; kk++) {
        const int q = gr.order ? gr.order[i0 + kk] : blk + kk * nblk;
        if (q >= nq) break;
        int t = tid;
        asm volatile("" : "+v"(t));
        const int l = q / nk, m0 = q - l * nk;
        const int kl = max(l + 1, m0), km = min(l + 1, m0), ki = kl * (kl + 1) / 2 + km;
        const double e = ek[m0 + (l + 1) * nk], vq = dek[q];
        const double wt = (m0 == 0 || m0 == nk - 1) ? 2.0 : 4.0;
        const double wv = u.nf * wt * vq, wb = 2.0 * wv * vq;
        const double fb0 = f0Vb[q], fbL = f0Vb[nq + q], hb0 = hVb[q], hbL = hVb[nq + q];
        const double df0 = df0V[q], dfL = df0V[nq + q], dh0 = dhV[q], dhL = dhV[nq + q];
        cd v[8];
        // (1) f0V and hV samples 8 t - 1 .. 8 t + 8, their splines, one packed transform
        {
            double y[2][10], M[2][9];
            const S* const pf = f0T + (long)q * (L + 1) + 8 * t;
            const S* const ph = hT + (long)q * (L + 1) + 8 * t;
#pragma unroll
            for (int i = 0; i < 8; i++) {
                y[0][1 + i] = (double)pf[i];
                y[1][1 + i] = (double)ph[i];
            }
            const int im = (t == 0) ? 0 : -1;
            const double f_m = (double)pf[im], h_m = (double)ph[im], f_p = (double)pf[8], h_p = (double)ph[8];
            if (t == 0) {
                y[0][1] = fb0;
                y[1][1] = hb0;
            }
            y[0][0] = f_m;
            y[1][0] = h_m;
            // sample 0 of the chunk's left neighbour is the FP64 boundary value (thread 0 alone holds it)
            y[0][9] = (t == NT - 1) ? fbL : f_p;
            y[1][9] = (t == NT - 1) ? hbL : h_p;
            const double d0[2] = {df0, dh0}, dN[2] = {dfL, dhL};
            pen_spline<L, NT, 2>(y, g, d0, dN, M, sx, zt, nullptr, t);
            if (t == 0) {
                ends[0] = M[0][0];
                ends[1] = M[1][0];
            }
            if (t == NT - 1) {
                ends[2] = M[0][8];
                ends[3] = M[1][8];
            }
            const cd p = tw[4 * t];  // exp(-8 pi i t / L)
#pragma unroll
            for (int i = 0; i < 8; i++)
                v[i] = p * cd{(M[0][i + 1] - M[0][i]) * g.ih, (M[1][i + 1] - M[1][i]) * g.ih};
        }
        // exp(-2 pi i (t + 1/2) s / L), s = 1, 2, 4: odd multiples of pi/L come from the half-step table
        pen_fft_dit<L>(v, Z, tw, conjg(twX[2 * t + 1]), tw[2 * t + 1], tw[4 * t + 2], t);
        // (2) slots n = t + NT m, m < 4, with D_{L-1-n} from thread NT - 1 - t (row 7 - m)
        wave_lds_order();
#pragma unroll
        for (int m = 0; m < 4; m++) Z[m * PS + t] = v[4 + m];
        SelfT raw[4];
        cd ts[4];
#pragma unroll
        for (int m = 0; m < 4; m++) {
            raw[m] = Self[(long)ki * H + t + NT * m];
            ts[m] = twS[t + NT * m];
        }
        c.e0 = mu - e;
        c.C2 = Sinf2[ki];
        c.C3 = Sinf3[ki];
        c.cj01 = -fb0 - fbL;
        c.cj1 = -hb0 - hbL;
        c.cj02 = df0 + dfL;
        c.cj2 = dh0 + dhL;
        __syncthreads();
        c.cj03 = -(ends[0] + ends[2]);
        c.cj3 = -(ends[1] + ends[3]);
        double sg = 0.0, s4 = 0.0, s5 = 0.0, sq = 0.0;
#pragma unroll
        for (int m = 0; m < 4; m++) {
            const cd D = v[m], E = Z[(3 - m) * PS + NT - 1 - t];
            const cd A = cd{0.5 * (D.x + E.x), -0.5 * (D.y - E.y)};
            const cd B = cd{0.5 * (D.y + E.y), 0.5 * (D.x - E.x)};
            const double kn = (2 * (t + NT * m) + 1) * u.piT;
            cd Gn, Jn;
            double qn0;
            jj_slot(c, A, B, ts[m], raw[m], kn, u.T, Gn, Jn, qn0);
            sq += qn0;
            sg += Gn.x;
            s4 += kn * Gn.y;
            s5 -= kn * Jn.y;
            v[m] = cd{Gn.x + Jn.y, Gn.y + Jn.x};                        // Gn + i conj(Jn)
            Z[(7 - m) * PS + t] = cd{Gn.x - Jn.y, Jn.x - Gn.y};  // the same of slot -n-1
            __builtin_amdgcn_sched_barrier(0);  // one slot after the other: fewer registers
        }
        aq += wv * sq;
        k0acc -= 4.0 * wt * u.nf * d2ek[m0 + (l + 1) * nk] * sg;
        // summed here: the compiler would otherwise hold all their operands up to the end of the point
        asm volatile("" : "+v"(aq), "+v"(k0acc));
        // the two sums over the slots that the end slopes need, one value per wavefront
        s4 = wave_total63(s4);
        s5 = wave_total63(s5);
        if (lane == 63) {
            sc[wave] = s4;
            sc[W + wave] = s5;
        }
        __syncthreads();
#pragma unroll
        for (int m = 4; m < 8; m++) v[m] = Z[m * PS + NT - 1 - t];
        __syncthreads();
        // (3) to imaginary time: v[m] = G(tau_j) + i J(tau_j), j = beta + NT m
        pen_fft_dif<L>(v, Z, tw, t);
        const int beta = pen_beta<L>(t);
        {
            // half a slot: exp(-i pi j / L)
            constexpr double c1 = 0.92387953251128675613, s1 = 0.38268343236508977173, r2 = 0.70710678118654752440;
            cd w[4];
            w[0] = conjg(twX[beta]);
            w[1] = w[0] * cd{c1, -s1};
            w[2] = w[0] * cd{r2, -r2};
            w[3] = w[0] * cd{s1, -c1};
#pragma unroll
            for (int m = 0; m < 4; m++) {
                v[m] = w[m] * v[m];
                v[m + 4] = mul_mi(w[m] * v[m + 4]);
            }
        }
        const JJPoles& pp = poles[q];
        const double Jbeta = pp.Jinf_beta - v[0].y;  // thread 0: J at beta from the slot sum at tau = 0
        const double t0 = beta * g.h;
        wave_lds_order();
        jj_poles_add<8>(v, pp, t0, u.dt, u.beta, Z + PS * pen_row<L>(t) + pen_o<L>(t), NT / 8);
        // (4) the products; G(tau_{L-j}) of j < L/2 through LDS (own rows: value j at row j mod 8, place j/8)
        double* const gz = (double*)Z;
        wave_lds_order();
#pragma unroll
        for (int m = 4; m < 8; m++) gz[2 * PS * pen_row<L>(t) + pen_o<L>(t) + (NT / 8) * m] = v[m].x;
        __syncthreads();
#pragma unroll
        for (int m = 0; m < 8; m++) add_lo(aM[m * NT + t], lM[m], wv * (v[m].x * v[m].y));
        const int rb = NT - beta;  // L - j = rb + NT (7 - m); for beta = 0 the next row up
        const double* const gr = gz + 2 * PS * (rb & 7) + (rb >> 3);
#pragma unroll
        for (int m = 0; m < 4; m++) {
            const bool z0 = (m == 0) && t == 0;
            const double gm = z0 ? 0.0 : gr[(NT / 8) * (7 - m)];
            // at tau = 0: G(0-) = G(0+) + 1
            const double x = z0 ? -(v[m].x + 1.0) : gm;
            add_lo(aB[m], lB[m], -wb * (v[m].x * x));
        }
        if (t == 0) {
            aH -= wb * (v[4].x * v[4].x);
            const double G0 = v[0].x, J0 = v[0].y;
            double S4 = 0.0, S5 = 0.0;
#pragma unroll
            for (int i = 0; i < W; i++) {
                S4 += sc[i];
                S5 += sc[W + i];
            }
            S4 *= 2.0;
            S5 *= 2.0;
            const double dGp = S4 + pp.dGp, dGm = -S4 + pp.dGm, dJ0 = S5 + pp.dJ0, dJb = -S5 + pp.dJb;
            tot[0] += wv * (dGp * J0 + G0 * dJ0);
            tot[1] += wv * (dGm * Jbeta - (G0 + 1.0) * dJb);
            tot[2] -= wv * ((G0 + 1.0) * Jbeta);
            tot[3] += wb * (dGp * (G0 + 1.0) + G0 * dGm);
            k0acc -= 2.0 * wt * u.nf * d2ek[m0 + (l + 1) * nk] * pp.k0r;
        }
    }
    double* const c1 = part + (long)blk * 2 * NWB;
    double* const c2 = c1 + NWB;
    // (5) the splines of the summed samples and (6) the packed transform of their moments
    int t = tid;
    asm volatile("" : "+v"(t));
    const int beta = pen_beta<L>(t);
    double* const Y1 = (double*)Z;
    double* const Y2 = Y1 + P8::YS;
    __syncthreads();
    float* const l1 = (float*)aM;  // the low-order parts, once the sums are read
    float* const l2 = l1 + L;
    double am[8];
#pragma unroll
    for (int m = 0; m < 8; m++) am[m] = aM[m * NT + t];
    __syncthreads();
#pragma unroll
    for (int m = 0; m < 8; m++) {
        const int j = beta + NT * m;
        Y1[j + (j >> 3)] = am[m];
        l1[j] = lM[m];
        if (m < 4) {
            Y2[j + (j >> 3)] = aB[m];
            Y2[(L - j) + ((L - j) >> 3)] = aB[m];
            l2[j] = lB[m];
            if (j > 0) l2[L - j] = lB[m];
        }
    }
    if (t == 0) {
        Y1[9 * NT] = tot[2];
        Y2[H + H / 8] = aH;
        l2[H] = 0.0f;
    }
    __syncthreads();
    const double MJ1 = Y1[0] - Y1[9 * NT], dchi = tot[3];
    cd v[8];
    double bsum;
    {
        double y[2][10], M[2][9], integ[2];
        float yl[2][10];
#pragma unroll
        for (int k = 0; k < 2; k++) {
            const double* const Y = (k == 0 ? Y1 : Y2) + 9 * t;
            const float* const l = (k == 0 ? l1 : l2) + 8 * t;
            yl[k][0] = (t > 0) ? l[-1] : 0.0f;
#pragma unroll
            for (int i = 0; i < 8; i++) yl[k][1 + i] = l[i];
            yl[k][9] = (t < NT - 1) ? l[8] : (k == 0) ? 0.0f : l2[0];
            y[k][0] = (t > 0) ? Y[-2] : 0.0;
#pragma unroll
            for (int i = 0; i < 8; i++) y[k][1 + i] = Y[i];
            y[k][9] = Y[9];
        }
        const double d0[2] = {tot[0], dchi}, dN[2] = {tot[1], -dchi};
        pen_spline<L, NT, 2>(y, g, d0, dN, M, sx, zt, integ, t, yl);
        bsum = integ[1];
        if (t == 0) ends[0] = M[0][0];
        if (t == NT - 1) ends[1] = M[0][8];
#pragma unroll
        for (int i = 0; i < 8; i++)
            v[i] = cd{M[0][i], M[1][i]};
    }
    bsum = wave_total63(bsum);
    aq = wave_total63(aq);
    if (lane == 63) {
        sc[2 * W + wave] = bsum;
        sc[3 * W + wave] = aq;
    }
    pen_fft_dit<L>(v, Z, tw, tw[t], tw[2 * t], tw[4 * t], t);
    wave_lds_order();
#pragma unroll
    for (int m = 0; m < 4; m++) Z[m * PS + t] = v[4 + m];
    __syncthreads();
    const double MJ3 = ends[0] - ends[1];
    auto row_n = [&](int n, cd Fn, cd Fq) { jj_rows(c1, c2, n, Fn, Fq, twX[n], MJ1, MJ3, dchi, 2.0 * u.piT, g.ih); };
    // L - n = NT - t + NT (7 - m); for t = 0 the next row's first column
    const cd* const zq = Z + NT - t + (t == 0 ? 1 : 0);
#pragma unroll
    for (int m = 0; m < 4; m++)
        if (t + NT * m > 0) row_n(t + NT * m, v[m], zq[(3 - m) * PS]);
    if (t == 0) {
        double s0 = 0.0, s1 = 0.0;
#pragma unroll
        for (int i = 0; i < W; i++) {
            s0 += sc[2 * W + i];
            s1 += sc[3 * W + i];
        }
        c1[0] = -s0;
        c2[0] = -2.0 * s1 * u.beta;
        int nh = H + t;
        asm volatile("" : "+v"(nh));
        row_n(nh, v[4], v[4]);
        inf1 += 2.0 * dchi;
        inf2 += 2.0 * MJ1;
        inf4 -= 2.0 * MJ3;
    }
    k0acc = wave_total63(k0acc);
    if (lane == 63) sc[wave] = k0acc;
    __syncthreads();
    if (tid == 0) {
        double s = 0.0;
        for (int i = 0; i < W; i++) s += sc[i];
        scal[blk * 4 + 0] = s;
        scal[blk * 4 + 1] = inf1;
        scal[blk * 4 + 2] = inf2;
        scal[blk * 4 + 3] = inf4;
    }
}

// The same for L <= 256 on one wavefront per workgroup (its barriers are free), thread t holding j = t + 64 i.  Two waves
// per SIMD: uncapped, L = 16 and 32 take 276 registers and leave room for one.
template <int L, typename S, typename SelfT>
__global__ void __launch_bounds__(64, 2)
    k_jj_pencil_short(const double* __restrict__ ek, const double* __restrict__ dek, const double* __restrict__ d2ek,
                      const S* __restrict__ hT, const S* __restrict__ f0T, const double* __restrict__ dhV,
                      const double* __restrict__ df0V, const double* __restrict__ hVb,
                      const double* __restrict__ f0Vb, const JJPoles* __restrict__ poles,
                      const SelfT* __restrict__ Self, const double* __restrict__ Sinf2,
                      const double* __restrict__ Sinf3, const double* __restrict__ Sinfp, int N, double T, double mu,
                      const cd* __restrict__ tw, const cd* __restrict__ twX, const cd* __restrict__ twS,
                      const cd* __restrict__ phT, double* part, double* scal, JJGroups gr, int kp,
                      const double* __restrict__ dsc)
{
    if (dsc) mu = dsc[kPscMu + 1];
    constexpr int NT = 64, H = L / 2, NWB = H + 1, PER = (L + NT - 1) / NT;
    __shared__ __align__(16) double Yb[2 * (L + 1)];
    __shared__ cd X[L];
    __shared__ double ES[2 * (2 * NT + 8)];
    double* const Y1 = Yb;
    double* const Y2 = Yb + (L + 1);
    cd* const Wk = (cd*)Yb;  // L complex values, used while Y1, Y2 are free
    const int nk = N / 2 + 1;
    const long nq = (long)nk * (nk - 2);
    const double nf = 1.0 / ((double)N * N);
    const double hstep = 1.0 / (L * T), ihstep = L * T, iT = 1.0 / T, dt = iT / PER;
    const int tid = threadIdx.x;
    const int blk = xcd_remap(blockIdx.x, gridDim.x);
    const long nblk = gridDim.x;
    JJPoint c;
    c.Sinf = Sinfp[0];
    double k0acc = 0.0, inf1 = 0.0, inf2 = 0.0, inf4 = 0.0;
    const int i0 = gr.order ? gr.first[blk] : 0, ni = gr.order ? gr.first[blk + 1] - i0 : kp;
    // every lane holds the sums over the points: end slopes, sample L of the Maki-Thompson spline
    double aM[PER], aB[PER], aq = 0.0, gd0 = 0.0, gdN = 0.0, YL = 0.0, dchi = 0.0;
#pragma unroll
    for (int i = 0; i < PER; i++) aM[i] = aB[i] = 0.0;
#pragma unroll 1
    for (int kk = 0; kk < ni; kk++) {
        const long q = gr.order ? (long)gr.order[i0 + kk] : (long)blk + kk * nblk;
        if (q >= nq) break;
        const int l = (int)(q / nk), m0 = (int)(q % nk);
        const long ki = fold_idx(l + 1, m0, N);
        const double vq = dek[q];
        const double wt = (m0 == 0 || m0 == nk - 1) ? 2.0 : 4.0;
        const double wv = nf * wt * vq, wb = 2.0 * wv * vq;
        const double fb0 = f0Vb[q], fbL = f0Vb[nq + q], hb0 = hVb[q], hbL = hVb[nq + q];
        const double df0 = df0V[q], dfL = df0V[nq + q], dh0 = dhV[q], dhL = dhV[nq + q];
        for (int j = tid; j <= L; j += NT) {
            Y1[j] = (j == 0) ? fb0 : (j == L) ? fbL : (double)f0T[q * (L + 1) + j];
            Y2[j] = (j == 0) ? hb0 : (j == L) ? hbL : (double)hT[q * (L + 1) + j];
        }
        __syncthreads();
        {
            double* const ys[2] = {Y1, Y2};
            const double d0s[2] = {df0, dh0}, dNs[2] = {dfL, dhL};
            block_spline_fixed<L, NT, 2>(ys, hstep, d0s, dNs, ES, nullptr);
        }
        for (int j = tid; j < L; j += NT)
            X[j] = twX[j] * cd{(Y1[j + 1] - Y1[j]) * ihstep, (Y2[j + 1] - Y2[j]) * ihstep};
        c.cj03 = -(Y1[0] + Y1[L]);
        c.cj3 = -(Y2[0] + Y2[L]);
        c.e0 = mu - ek[m0 + (l + 1) * nk];
        c.C2 = Sinf2[ki];
        c.C3 = Sinf3[ki];
        c.cj01 = -fb0 - fbL;
        c.cj1 = -hb0 - hbL;
        c.cj02 = df0 + dfL;
        c.cj2 = dh0 + dhL;
        __syncthreads();
        block_fft_pp<L, NT>(X, Wk, +1, tw);
        double sg = 0.0, s4 = 0.0, s5 = 0.0, sq = 0.0;
        for (int n = tid; n < H; n += NT) {
            const cd F = X[n], E = X[L - 1 - n];
            const cd A = cd{0.5 * (F.x + E.x), 0.5 * (F.y - E.y)};
            const cd B = cd{0.5 * (F.y + E.y), -0.5 * (F.x - E.x)};
            const double kn = (2 * n + 1) * kPi * T;
            cd Gn, Jn;
            double qn0;
            jj_slot(c, A, B, twS[n], Self[ki * H + n], kn, T, Gn, Jn, qn0);
            sq += qn0;
            sg += Gn.x;
            s4 += kn * Gn.y;
            s5 -= kn * Jn.y;
            Wk[H + n] = cd{Gn.x + Jn.y, Gn.y + Jn.x};  // Gn + i conj(Jn), and of slot -n-1
            Wk[H - 1 - n] = cd{Gn.x - Jn.y, Jn.x - Gn.y};
        }
        aq += wv * sq;
        k0acc -= 4.0 * wt * nf * d2ek[m0 + (l + 1) * nk] * sg;
        s4 = 2.0 * wave_sum(s4);
        s5 = 2.0 * wave_sum(s5);
        __syncthreads();
        block_fft_pp<L, NT>(Wk, X, -1, tw);
        const JJPoles& pp = poles[q];
        const double Jbeta = pp.Jinf_beta - Wk[0].y;
        const double t0 = tid * hstep;
        cd v[PER];
#pragma unroll
        for (int i = 0; i < PER; i++) {
            const int j = tid + NT * i;
            v[i] = (j < L) ? phT[j] * Wk[j] : cd{0.0, 0.0};
        }
        if (tid < L) jj_poles_add<PER>(v, pp, t0, dt, iT, X + tid, NT);
#pragma unroll
        for (int i = 0; i < PER; i++)
            if (tid + NT * i < L) X[tid + NT * i] = v[i];
        __syncthreads();
        const double G0 = X[0].x, J0 = X[0].y;
#pragma unroll
        for (int i = 0; i < PER; i++) {
            const int j = tid + NT * i;
            if (j < L) {
                // at tau = 0: G(0-) = G(0+) + 1
                const double x = (j == 0) ? -(G0 + 1.0) : X[L - j].x;
                aM[i] += wv * (v[i].x * v[i].y);
                aB[i] -= wb * (v[i].x * x);
            }
        }
        const double dGp = s4 + pp.dGp, dGm = -s4 + pp.dGm, dJ0 = s5 + pp.dJ0, dJb = -s5 + pp.dJb;
        gd0 += wv * (dGp * J0 + G0 * dJ0);
        gdN += wv * (dGm * Jbeta - (G0 + 1.0) * dJb);
        YL -= wv * ((G0 + 1.0) * Jbeta);
        dchi += wb * (dGp * (G0 + 1.0) + G0 * dGm);
        if (tid == 0) k0acc -= 2.0 * wt * nf * d2ek[m0 + (l + 1) * nk] * pp.k0r;
        __syncthreads();
    }
    double* const c1 = part + (long)blk * 2 * NWB;
    double* const c2 = c1 + NWB;
#pragma unroll
    for (int i = 0; i < PER; i++) {
        const int j = tid + NT * i;
        if (j < L) {
            Y1[j] = aM[i];
            Y2[j] = aB[i];
            if (j == 0) {
                Y1[L] = YL;
                Y2[L] = aB[0];
            }
        }
    }
    __syncthreads();
    const double MJ1 = Y1[0] - Y1[L];
    double integ[2];
    {
        double* const ys[2] = {Y1, Y2};
        const double d0s[2] = {gd0, dchi}, dNs[2] = {gdN, -dchi};
        block_spline_fixed<L, NT, 2>(ys, hstep, d0s, dNs, ES, integ);
    }
    const double MJ3 = Y1[0] - Y1[L];
    const double bub0 = wave_sum(integ[1]), q0 = 2.0 * iT * wave_sum(aq);
    for (int j = tid; j < L; j += NT) X[j] = cd{Y1[j], Y2[j]};
    __syncthreads();
    block_fft_pp<L, NT>(X, Wk, -1, tw);
    for (int n = tid; n <= H; n += NT) {
        if (n == 0) {
            c1[0] = -bub0;
            c2[0] = -q0;
        } else {
            jj_rows(c1, c2, n, X[n], X[L - n], twX[n], MJ1, MJ3, dchi, 2.0 * kPi * T, ihstep);
        }
    }
    inf1 += 2.0 * dchi;
    inf2 += 2.0 * MJ1;
    inf4 -= 2.0 * MJ3;
    k0acc = wave_sum(k0acc);
    if (tid == 0) {
        scal[blk * 4 + 0] = k0acc;
        scal[blk * 4 + 1] = inf1;
        scal[blk * 4 + 2] = inf2;
        scal[blk * 4 + 3] = inf4;
    }
}

// kx = 0 and kx = pi rows of the diamagnetic term (cond_opt.cpp:3993-4173); block b:
// row l = (b < nk ? 0 : nk-1), m = b % nk
template <typename SelfT>
__global__ void k_kx0_rows(const double* __restrict__ ek, const double* __restrict__ d2ek, const SelfT* __restrict__ Self,
                           const double* __restrict__ Sinf2, const double* __restrict__ Sinf3,
                           const double* __restrict__ Sinfp, int N, int L, double T, double mu, double* out,
                           const double* __restrict__ dsc)
{
    if (dsc) mu = dsc[kPscMu + 1];
    __shared__ double sc[16];
    const int nk = N / 2 + 1;
    const int l = (blockIdx.x < nk) ? 0 : nk - 1, m = blockIdx.x % nk;
    const long ki = fold_idx(l, m, N);
    const double C2 = Sinf2[ki], C3 = Sinf3[ki], Sinf = Sinfp[0];
    const double e = ek[m + l * nk];
    const int H = L / 2;
    // Re of the sum over all slots: twice that of n >= 0, the slots -n-1 being the conjugates (both halves with
    // divisions: 13.0 us at 16 x 128, 19.9 at 256 x 2048 mixed; now 6.9, 12.3)
    double k0[1] = {0.0};
    for (int n = threadIdx.x; n < H; n += blockDim.x) {
        const double kn = (2 * n + 1) * kPi * T, ik = rcp_nr(kn);
        const cd sg = sigma_ik(Self[ki * H + n], Sinf, C2, C3, ik);
        k0[0] += 2.0 * (sdiv_rcp(T, cd{mu - e - sg.x, kn - sg.y}).x - sdiv_rcp(T, cd{mu - e, kn + Sinf * ik}).x);
    }
    block_sum_k<1>(k0, sc);
    if (threadIdx.x == 0) {
        const Poles P = make_poles(e, mu, Sinf, 0.0, T);
        const cd f1m = (P.r1.x > 0) ? P.a1 * cexpd(-(P.r1 / T)) / P.den1 : P.a1 / P.den1;
        const cd f2m = (P.r2.x > 0) ? P.a2 * cexpd(-(P.r2 / T)) / P.den2 : P.a2 / P.den2;
        const double k0r = k0[0] + (f1m + f2m).x;
        double wt = 2;
        if (m == 0 || m == nk - 1) wt = wt / 2;
        out[blockIdx.x] = -2.0 * wt / ((double)N * N) * d2ek[m + l * nk] * k0r;
    }
}

// ================================================================== launchers
hipError_t launch_jj_poles(const Grid& g, const DevArrays& d, double mu, hipStream_t s, const double* dsc)
{
    const double dt = 1.0 / (jj_samples(g.Nw) * g.T);
    hipLaunchKernelGGL(k_jj_poles, dim3((unsigned)((g.nq + 127) / 128)), dim3(128), 0, s, d.ek, d.hVb, d.Sinf, g.N,
                       g.T, mu, dt, (JJPoles*)d.poles, dsc);
    return hipGetLastError();
}

hipError_t launch_jj_pencil(const Grid& g, const DevArrays& d, double mu, double* part, double* scal,
                            const JJGroups& gr, hipStream_t s, const double* dsc)
{
    const int kp = jj_points(g.nq);
    const unsigned nblk = gr.order ? (unsigned)gr.n : (unsigned)jj_blocks(g.nq);
    const PenStep step = pen_step(1.0 / (g.Nw * g.T));
    const JJScale sc = {g.T, kPi * g.T, 1.0 / g.T, 1.0 / ((double)g.N * g.N), 1.0 / (jj_samples(g.Nw) * g.T)};
    DISPATCH_S(g.prec, {
        if (g.Nw <= 256) {
            DISPATCH_L_SHORT(g.Nw, hipLaunchKernelGGL((k_jj_pencil_short<LL, SS, ST>), dim3(nblk), dim3(64), 0, s,
                             d.ek, d.dek, d.d2ek, (const SS*)d.hT, (const SS*)d.f0T, d.dhV, d.df0V, d.hVb, d.f0Vb,
                             (const JJPoles*)d.poles, (const ST*)d.Self, d.Sinf2, d.Sinf3, d.Sinf, g.N, g.T, mu,
                             d.twN, d.twX, d.twS, d.ph, part, scal, gr, kp, dsc));
        } else {
            DISPATCH_L_LONG(g.Nw, hipLaunchKernelGGL((k_jj_pencil<LL, SS, ST>), dim3(nblk), dim3(Pen<LL>::NT), 0, s,
                            d.ek, d.dek, d.d2ek, (const SS*)d.hT, (const SS*)d.f0T, d.dhV, d.df0V, d.hVb, d.f0Vb,
                            (const JJPoles*)d.poles, (const ST*)d.Self, d.Sinf2, d.Sinf3, d.Sinf, g.N, step, sc, mu,
                            d.twN, d.twX, d.twS, part, scal, gr, kp, dsc));
        }
    });
    return hipGetLastError();
}

hipError_t launch_kx0_rows(const Grid& g, const DevArrays& d, double mu, hipStream_t s, const double* dsc,
                           double* out)
{
    DISPATCH_S(g.prec, {
        hipLaunchKernelGGL(k_kx0_rows<ST>, dim3(2 * g.nk), dim3(256), 0, s, d.ek, d.d2ek, (const ST*)d.Self, d.Sinf2,
                           d.Sinf3, d.Sinf, g.N, g.Nw, g.T, mu, out ? out : d.kx0part, dsc);
    });
    return hipGetLastError();
}

}  // namespace tpsc
