// tpsc_al.hip -- Aslamazov-Larkin term Lambda_jj3(iq_n) of the current-current correlation
// (cond_opt.cpp:4292-6467, chi3 = true) on gfx950, FP64 throughout.
//
// Set-up (once per call):
//   k_al_grt_slab    G0(r,-tau) on the wedge, tau_j = j beta/Nw, and its slopes (:4374-4445)
//   k_al_hg_slab     hG(q,tau) = DST x DCT [h(r,tau) G0(r,-tau)], slopes (:5159-5261)
//   k_al_hw_pencil   hG(q,iq_p), p < Nw/2, and its 1/qn^2 coefficient hg2 (:5266-5330)
// Per boson frequency q_n of the sparse set (:5350-6400):
//   k_al_HG_pencil   HG(q,iq_p) = Gamma(q,iq_p) [hG(p) - hG(p+n)] / [chi0(p) - chi0(p+n)] on the
//                    window p in [-Nw/2 - n/2, Nw/2 - n/2), to tau with the two-pole tail
//   k_al_prod_slab   HG(r,tau) G0(r,-tau) back to k, slopes
//   k_al_k_pencil    spline + shifted fermionic transform of the product, then the sum over k and
//                    w_m of v_k G(k,iw_m) G(k,iw_m+iq_n) [HG - HG2], HG2 the conjugate of HG
//                    at -w_m
// Layout: slab-major arrays [tau][q] feed the slab kernels, point-major rows [q][tau] feed the
// pencils (k_transpose in between); complex tau arrays are two real planes (re, im).
// Lambda grid q = m + l*nk: kx = (l+1) pi/(nk-1), ky = m pi/(nk-1), nq = nk (nk-2).
#include "tpsc_launch.hpp"
#include "tpsc_pencil.hpp"

namespace tpsc {

#define AL_PEN_THREADS 256

// Block j <= Nw: Grt[j*nk8 + w] = G0(r_w, -tau_j) (cond_opt.cpp:4396-4400).  Block Nw+1: dGrt[w] = d/dtau
// G0(r,-tau) at tau = 0 (x G0(k,0-), :4417-4421) and dGrt[nk8 + w] = eps(r) - mu0 delta_r0 - dGrt[w] at
// tau = beta.
template <int N>
__global__ void __launch_bounds__(SlabShape<N>::NT)
    k_al_grt_slab(const unsigned* __restrict__ wt, const double* __restrict__ ekw, const double* __restrict__ fw,
                  const double* __restrict__ er, double mu0, double T, int Nw, double* Grt, double* dGrt)
{
    constexpr long nk8 = (long)(N / 2 + 1) * (N / 2 + 2) / 2;
    extern __shared__ double smem[];
    double* slab = smem;
    cd* tw = slab_tw<N>(slab);
    fill_twiddles<N>(tw);
    const int j = blockIdx.x;
    const double t = (j <= Nw) ? (double)j / (T * Nw) : 0.0, bt = 1.0 / T - t;
    each_wedge<N>(wt, [&](int a, int b, int i) {
        const double x = ekw[i] - mu0;
        const double g = g0_exp(x, bt, t) * fw[i];
        slab[a] = slab[b] = (j <= Nw) ? g : x * g;
    });
    __syncthreads();
    slab_r2r_2d<double, N, 0>(slab, tw);
    each_wedge<N>(wt, [&](int a, int, int i) {
        const double v = slab[a];
        if (j <= Nw) {
            Grt[(long)j * nk8 + i] = v;
        } else {
            dGrt[i] = v;
            dGrt[nk8 + i] = ((i == 0) ? -mu0 : er[i]) - v;
        }
    });
}

// Block j <= Nw: hGs[j*nq + q] = DST x DCT [h(r,tau_j) G0(r,-tau_j)] with h(r,tau) the
// DST x DCT of the k-space integrand (cond_opt.cpp:4302-4330, 5231-5261).
// Blocks Nw+1+side: slope at tau = 0 / beta of the same product (:5159-5229),
// dh(r) G0(r,-tau_b) + h(r,tau_b) dG0(r,-tau_b), dh(k) = -x h(k), back to q -> dhG[side*nq + q].
template <int N>
__global__ void __launch_bounds__(SlabShape<N>::NT)
    k_al_hg_slab(const unsigned* __restrict__ wt, const double* __restrict__ ekw, const double* __restrict__ fw,
                 const double* __restrict__ vw, const double* __restrict__ Grt, const double* __restrict__ dGrt,
                 double mu0, double T, int Nw, double* hGs, double* dhG)
{
    constexpr int nk = N / 2 + 1;
    constexpr long nq = (long)nk * (nk - 2);
    constexpr int nk8 = nk * (nk + 1) / 2, PER = wedge_per_thread<N>();
    extern __shared__ double smem[];
    double* slab = smem;
    cd* tw = slab_tw<N>(slab);
    fill_twiddles<N>(tw);
    const int b = blockIdx.x;
    const int jt = (b <= Nw) ? b : ((b == Nw + 1) ? 0 : Nw);
    const double t = (double)jt / (T * Nw), bt = 1.0 / T - t;
    each_wedge<N>(wt, [&](int o, int p, int i) {
        const double g = g0_exp(ekw[i] - mu0, t, bt) * fw[i];
        slab[o] = g * vw[i];
        slab[p] = g * vw[nk8 + i];
    });
    const double* g = Grt + (long)jt * nk8;
    __syncthreads();
    slab_r2r_2d<double, N, 1>(slab, tw);
    if (b <= Nw) {
        each_wedge<N>(wt, [&](int o, int p, int i) {
            const double v = g[i], ra = slab[o] * v, rb = slab[p] * v;
            slab[o] = ra;
            slab[p] = rb;
        });
        __syncthreads();
        slab_r2r_2d<double, N, 1>(slab, tw);
        double* out = hGs + (long)b * nq;
        each_lambda<N>([&](int l, int m, int s) { out[s] = slab[at<N>(l + 1, m)]; });
        return;
    }
    const int side = b - Nw - 1;
    double sa[PER], sb[PER];
    each_wedge_slot<N>(wt, [&](int o, int p, int i, int c) {
        const double v = dGrt[side * nk8 + i];
        sa[c] = slab[o] * v;
        sb[c] = slab[p] * v;
    });
    __syncthreads();
    each_wedge<N>(wt, [&](int o, int p, int i) {
        const double x = ekw[i] - mu0, v = -x * g0_exp(x, t, bt) * fw[i];
        slab[o] = v * vw[i];
        slab[p] = v * vw[nk8 + i];
    });
    __syncthreads();
    slab_r2r_2d<double, N, 1>(slab, tw);
    each_wedge_slot<N>(wt, [&](int o, int p, int i, int c) {
        const double ra = slab[o] * g[i] + sa[c], rb = slab[p] * g[i] + sb[c];
        slab[o] = ra;
        slab[p] = rb;
    });
    __syncthreads();
    slab_r2r_2d<double, N, 1>(slab, tw);
    each_lambda<N>([&](int l, int m, int s) { dhG[side * nq + s] = slab[at<N>(l + 1, m)]; });
}

// Per Lambda point q: clamped spline of hG(q,tau_j), j = 0..L, slopes dhG; hw[q*H] = twice its
// integral, hw[q*H + p] = 2 Re[(1 - e^{-2 pi i p/L}) F_p], F = FORWARD DFT of 6a_j, 0 < p < H;
// hg2[q] = 2 (dhG(0) - dhG(beta)) (cond_opt.cpp:5266-5330).  hGp: point-major rows [q][j].
template <int L>
__global__ void __launch_bounds__(AL_PEN_THREADS)
    k_al_hw_pencil(const double* __restrict__ hGp, const double* __restrict__ dhG, long nq, double T,
                   const cd* __restrict__ tw, const cd* __restrict__ twM, double* hw, double* hg2)
{
    constexpr int NT = AL_PEN_THREADS;
    constexpr int H = L / 2;
    __shared__ double Y[L + 1];
    __shared__ cd X[L];
    __shared__ double ES[2 * NT + 8];
    __shared__ double sc[NT / 64];
    const long q = blockIdx.x;
    const int tid = threadIdx.x;
    const double h = 1.0 / (L * T);
    const double* row = hGp + q * (L + 1);
    for (int j = tid; j <= L; j += NT) Y[j] = row[j];
    const double d0 = dhG[q], dN = dhG[nq + q];
    __syncthreads();
    double integ[1] = {0.0};
    {
        double* const ys[1] = {Y};
        block_spline_fixed<L, NT, 1>(ys, h, &d0, &dN, ES, integ);
    }
    const double tot = block_sum(integ[0], sc);
    for (int j = tid; j < L; j += NT) X[j] = cd{(Y[j + 1] - Y[j]) / h, 0.0};
    __syncthreads();
    block_fft<L, NT>(X, -1, tw);
    double* o = hw + q * H;
    if (tid == 0) {
        o[0] = 2 * tot;
        hg2[q] = 2 * (d0 - dN);
    }
    for (int p = 1 + tid; p < H; p += NT) {
        const cd f = twM[p] * X[p];
        o[p] = 2 * f.x;
    }
}

// Per Lambda point q and boson index nn (cond_opt.cpp:5350-5620):
//   HG_j = Gamma(p1) D_j, D_j = [hG(p1) - hG(p2)]/[chi0(p1) - chi0(p2)], p1 = j (j < H - nn/2) or
//   j - L, p2 = p1 + nn; at p1 = -nn/2 (nn even, chi0(p1) = chi0(p2)) the Richardson value
//   (4 D_{j-1} - D_{j-2})/3; Gamma = 3 Usp chi_sp + Uch chi_ch.
//   HG(q,tau_t) = FORWARD DFT_t [T (HG_j - Hinf_j)] + hg2 tail(tau_t), Hinf the two-pole
//   asymptote, tail its imaginary-time form; slopes at 0+ and beta-.
// HG_j is real and the tail real and even about beta/2 (spin poles +-i a: cos(a(beta/2 - tau))/(2a sin(a beta/2)),
// charge poles +-c: (e^{-c tau} + e^{-c(beta - tau)})/(2c(e^{-c beta} - 1))), so HG(q,beta - tau) = conj HG(q,tau): only
// t <= H is formed, and everything that the reference builds from HG(beta - tau) is a conjugate.
// chiwP: chi0(q,iq_p) point-major [w][p], p <= H.  Writes HGp planes [c][q][t], t <= H, and the slope at 0+
// dHq[c*nq + q] (at beta-: -re, +im).
struct ALInput {  // one point's T (HG_j - Hinf_j)
    const double *cw, *hv;
    double ci, ci2, g2, Usp, Uch, T, tpT;
    int nn, nc, L;
    __device__ __forceinline__ double chi0(int p) const
    {
        p = abs(p);
        if (p <= L / 2) return cw[p];
        const double iw = rcp_nr(tpT * p), iw2 = iw * iw;
        return (ci + ci2 * iw2) * iw2;
    }
    __device__ __forceinline__ double hG(int p) const
    {
        p = abs(p);
        if (p == 0) return hv[0];
        const double iw = rcp_nr(tpT * p), iw2 = iw * iw;
        return (-g2 + hv[(p < L / 2) ? p : L / 2 - 1] * iw2) * iw2;
    }
    __device__ __forceinline__ int p1(int j) const { return (j < L / 2 - nc) ? j : j - L; }
    __device__ __forceinline__ double D(int j) const
    {
        const int a = p1(j), b = a + nn;
        return (hG(a) - hG(b)) * rcp_nr(chi0(a) - chi0(b));
    }
    // dr accumulates -w_j f_j
    __device__ __forceinline__ double f(int j, double& dr) const
    {
        const int p = p1(j);
        const double c1 = chi0(p);
        const double G = 3 * Usp * c1 * rcp_nr(1.0 - Usp * c1 / 2) + Uch * c1 * rcp_nr(1.0 + Uch * c1 / 2);
        const double Dj = (nn % 2 == 0 && p == -(nn / 2)) ? (4 * D(j - 1) - D(j - 2)) / 3.0 : D(j);
        const double wn = tpT * p, w2 = wn * wn;
        const double Hinf = g2 * (3.0 * Usp * rcp_nr(-w2 + 0.5 * Usp * ci) - Uch * rcp_nr(w2 + 0.5 * Uch * ci));
        const double v = T * (G * Dj - Hinf);
        dr -= wn * v;
        return v;
    }
};
// g2 x the tail at tau
struct ALTail {
    double a, c, hb, beta, ks, kc;
    __device__ __forceinline__ ALTail(double Usp, double Uch, double ci, double g2, double T)
    {
        beta = 1.0 / T;
        hb = 0.5 * beta;
        a = sqrt(0.5 * Usp * ci);
        c = sqrt(0.5 * Uch * ci);
        ks = 3.0 * Usp * g2 / (2.0 * a * sin(a * hb));
        kc = Uch * g2 / (2.0 * c * (exp(-c * beta) - 1.0));
    }
    __device__ __forceinline__ double at(double tau) const
    {
        return ks * cos(a * (hb - tau)) + kc * (exp(-c * tau) + exp(-c * (beta - tau)));
    }
};

template <int L>
__global__ void __launch_bounds__(AL_PEN_THREADS)
    k_al_HG_pencil_short(const double* __restrict__ chiwP, const double* __restrict__ chi0inf,
                         const double* __restrict__ chi0inf2, const double* __restrict__ hw,
                         const double* __restrict__ hg2, int N, double T, double Usp, double Uch, int nn,
                         const cd* __restrict__ tw, double* HGp, double* dHq)
{
    constexpr int NT = AL_PEN_THREADS;
    constexpr int H = L / 2;
    __shared__ double cw[H + 1], hv[H];
    __shared__ cd X[L];
    __shared__ double sc[NT / 64];
    const int nk = N / 2 + 1;
    const long nq = (long)nk * (nk - 2);
    const long q = blockIdx.x;
    const int tid = threadIdx.x;
    const int l = (int)(q / nk), m = (int)(q % nk);
    const long r = fold_idx(l + 1, m, N);
    for (int p = tid; p <= H; p += NT) cw[p] = chiwP[r * (H + 1) + p];
    for (int p = tid; p < H; p += NT) hv[p] = hw[q * H + p];
    const ALInput in = {cw, hv, chi0inf[r], chi0inf2[r], hg2[q], Usp, Uch, T, 2.0 * kPi * T, nn, nn / 2, L};
    __syncthreads();
    double dr = 0.0;
    for (int j = tid; j < L; j += NT) X[j] = cd{in.f(j, dr), 0.0};
    const double dtauH0 = block_sum(dr, sc);
    block_fft<L, NT>(X, -1, tw);
    const ALTail tail(Usp, Uch, in.ci, in.g2, T);
    double* Pr = HGp + q * (H + 1);
    double* Pi = Pr + nq * (H + 1);
    for (int t = tid; t <= H; t += NT) {
        Pr[t] = X[t].x + tail.at(t / (L * T));
        Pi[t] = X[t].y;
    }
    if (tid == 0) {
        dHq[q] = 0.5 * in.g2 * (3.0 * Usp + Uch);
        dHq[nq + q] = dtauH0;
    }
}

// The same for L >= 1024: the DFT of the real HG_j as one of length H = L/2 of z_i = f_2i + i f_2i+1, in registers
// (tpsc_pencil.hpp): X_t = (Z_t + conj Z_{H-t})/2 - (i/2) e^{-2 pi i t/L} (Z_t - conj Z_{H-t}).
// What bounds it: FP64 VALU (the ratios).  128^2 x 1024: 47 us a frequency (length-L LDS FFT, all tau: 82).
template <int L>
__global__ void __launch_bounds__(L / 16, 3)
    k_al_HG_pencil(const double* __restrict__ chiwP, const double* __restrict__ chi0inf,
                   const double* __restrict__ chi0inf2, const double* __restrict__ hw, const double* __restrict__ hg2,
                   int N, double T, double Usp, double Uch, int nn, const cd* __restrict__ tw, double* HGp, double* dHq)
{
    constexpr int H = L / 2, NT = Pen<H>::NT, W = Pen<H>::W, PS = Pen<H>::PS;
    __shared__ __align__(16) cd Z[Pen<H>::ZD / 2];
    __shared__ double sc[W];
    const int nk = N / 2 + 1;
    const long nq = (long)nk * (nk - 2);
    const int q = blockIdx.x, t = threadIdx.x;
    const int l = q / nk, m0 = q - l * nk;
    const long r = fold_idx(l + 1, m0, N);
    const ALInput in = {chiwP + r * (H + 1), hw + (long)q * H, chi0inf[r], chi0inf2[r], hg2[q], Usp, Uch, T, 2.0 * kPi * T, nn, nn / 2, L};
    double dr = 0.0;
    cd v[8];
#pragma unroll 1
    for (int m = 0; m < 8; m++) {  // through the thread's own LDS cells: one copy of the code, few registers
        const int j = 2 * (t + NT * m);
        const double f0 = in.f(j, dr), f1 = in.f(j + 1, dr);
        Z[m * PS + t] = cd{f0, f1};
    }
    wave_lds_order();
#pragma unroll
    for (int m = 0; m < 8; m++) v[m] = Z[m * PS + t];
    dr = wave_total63(dr);
    if ((t & 63) == 63) sc[t >> 6] = dr;
    pen_fft_dif<H, 2>(v, Z, tw, t);
    wave_lds_order();
    // element j at row j mod 8, place j/8: the thread's own cells
#pragma unroll
    for (int m = 0; m < 8; m++) Z[PS * pen_row<H>(t) + pen_o<H>(t) + (NT / 8) * m] = v[m];
    __syncthreads();
    const ALTail tail(Usp, Uch, in.ci, in.g2, T);
    double* const Pr = HGp + (long)q * (H + 1);
    double* const Pi = Pr + nq * (H + 1);
    auto z = [&](int j) { return Z[(j & 7) * PS + (j >> 3)]; };
#pragma unroll 1
    for (int j = t; j <= H; j += NT) {
        const cd A = z(j & (H - 1)), B = conjg(z((H - j) & (H - 1))), s = A + B, d = tw[j] * (A - B);
        Pr[j] = 0.5 * (s.x + d.y) + tail.at(j / (L * T));
        Pi[j] = 0.5 * (s.y - d.x);
    }
    if (t == 0) {
        double d0 = 0.0;
        for (int i = 0; i < W; i++) d0 += sc[i];
        dHq[q] = 0.5 * in.g2 * (3.0 * Usp + Uch);
        dHq[nq + q] = d0;
    }
}

// Products of HG(r,tau) with G0(r,-tau), back to k (cond_opt.cpp:5622-5905, 6000-6170).  The reference's second
// product, HG(r,beta-tau) G0(r,-tau), is the conjugate of the first and is not formed.
// Blocks b < 2(H+1): t = b/2 <= H, part c = b%2 (re, im):
//   S = DST x DCT [HG_c(q,tau_t)/N^2] (q -> r), then P_c(k,tau_t) = DST x DCT [S G0(r,-tau_t)] and, from the same
//   S, P_c(k,tau_L-t) = +-DST x DCT [S G0(r,-tau_{L-t})] (+ re, - im).
// Blocks 2(H+1) + 2 side + c: the slopes of P at tau = 0 / beta from HG(r,tau_b) dG0(r,-tau_b) + dHG(r) G0(r,-tau_b),
// with HG(r,beta) = conj HG(r,0) and dHG(r,beta) = -conj dHG(r,0).
// Planes: HGs [c][t][q], t <= H; Ps [c][t][q], t <= L; dHq [c][q]; dP [side][c][q].
// What bounds it: latency at 3 to 4 workgroups per CU (128^2: 38 KB of LDS each), so up to 128^2 the registers are
// capped for four waves per SIMD (108 us against 122 uncapped and 143 for five at 128^2 x 1024; both products and
// all tau before: 228).
template <int N>
__global__ void __launch_bounds__(SlabShape<N>::NT, (N <= 128 ? 4 : 1))
    k_al_prod_slab(const unsigned* __restrict__ wt, const double* __restrict__ HGs, const double* __restrict__ dHq,
                   const double* __restrict__ Grt, const double* __restrict__ dGrt, int L, double* Ps, double* dP)
{
    constexpr int nk = N / 2 + 1;
    constexpr long nq = (long)nk * (nk - 2);
    constexpr long nk8 = (long)nk * (nk + 1) / 2;
    constexpr int PER = wedge_per_thread<N>();
    const double nf = 1.0 / ((double)N * N);
    extern __shared__ double smem[];
    double* slab = smem;
    cd* tw = slab_tw<N>(slab);
    fill_twiddles<N>(tw);
    const int H = L / 2, b = blockIdx.x, c = b & 1;
    const bool main_blk = b < 2 * (H + 1);
    const int t = main_blk ? b >> 1 : 0, side = main_blk ? 0 : (b - 2 * (H + 1)) >> 1;
    const double* src = HGs + ((long)c * (H + 1) + t) * nq;
    const double f = (side && c) ? -nf : nf;
    each_lambda<N>([&](int l, int m, int s) { slab[at<N>(l + 1, m)] = f * src[s]; });
    __syncthreads();
    slab_r2r_2d<double, N, 1>(slab, tw);
    double sa[PER], sb[PER];  // HG(r,tau) at (l, m) and (m, l) of the thread's points
    each_wedge_slot<N>(wt, [&](int o, int p, int, int i) {
        sa[i] = slab[o];
        sb[i] = slab[p];
    });
    __syncthreads();
    if (main_blk) {
#pragma unroll 1
        for (int pass = 0; pass < 2; pass++) {
            if (pass && t == H) break;
            const int tg = pass ? L - t : t;
            const double* g = Grt + (long)tg * nk8;
            const double sgn = (pass && c) ? -1.0 : 1.0;
            each_wedge_slot<N>(wt, [&](int o, int p, int w, int i) {
                const double gw = sgn * g[w];
                slab[o] = sa[i] * gw;
                slab[p] = sb[i] * gw;
            });
            __syncthreads();
            slab_r2r_2d<double, N, 1>(slab, tw);
            double* out = Ps + ((long)c * (L + 1) + tg) * nq;
            each_lambda<N>([&](int l, int m, int s) { out[s] = slab[at<N>(l + 1, m)]; });
            __syncthreads();
        }
        return;
    }
    const double* dg = dGrt + side * nk8;
    const double* dsrc = dHq + (long)c * nq;
    const double fd = (side && !c) ? -nf : nf;
    each_lambda<N>([&](int l, int m, int s) { slab[at<N>(l + 1, m)] = fd * dsrc[s]; });
    __syncthreads();
    slab_r2r_2d<double, N, 1>(slab, tw);
    const double* g = Grt + (long)(side ? L : 0) * nk8;
    each_wedge_slot<N>(wt, [&](int o, int p, int w, int i) {
        const double ra = slab[o] * g[w] + sa[i] * dg[w], rb = slab[p] * g[w] + sb[i] * dg[w];
        slab[o] = ra;
        slab[p] = rb;
    });
    __syncthreads();
    slab_r2r_2d<double, N, 1>(slab, tw);
    double* out = dP + (long)(side * 2 + c) * nq;
    each_lambda<N>([&](int l, int m, int s) { out[s] = slab[at<N>(l + 1, m)]; });
}

// Dyson G(k, i w_f) = 1/(i w_f + mu - e - Sigma(k,iw_f)), Sigma from the stored form for
// |f + 1/2| < H, from its moments beyond, conjugated for f < 0 (cond_opt.cpp:6314-6377)
template <typename SelfT>
__device__ __forceinline__ cd al_G(const SelfT* __restrict__ Self, long ki, int H, int f, double C2, double C3,
                                   double Sinf, double e0, double piT)
{
    const int g = (f >= 0) ? f : -f - 1;
    const double kn = (2 * g + 1) * piT;
    const cd sg = (g < H) ? sigma_kw(Self, ki * H + g, Sinf, C2, C3, kn) : sigma_mom(Sinf, C2, C3, cd{0.0, 0.0}, kn);
    const cd G = sdiv_rcp(1.0, cd{e0 - sg.x, kn - sg.y});
    return (f < 0) ? conjg(G) : G;
}

// Per Lambda point k (cond_opt.cpp:5907-6400): clamped splines of P re, im with the slopes dP, and
//   V(s) = HG(k, i w_s) = -i (z_0 + z_L)/w - (z'_0 + z'_L)/w^2 + i (z''_0 + z''_L)/w^3 + (1 - e^{-i w beta/L}) F_s/w^4,
// F = FORWARD DFT of e^{-i pi t/L} 6a_t (re + i im).  The second function of the reference, HG2(k, i w_f) from the
// conjugate of P, is conj V(-f-1), so its sum over the window f = j (j < H - nn/2) or j - L is
//   sum over s = f + nn of G(s - nn) G(s) [V(s) - conj V(nn - 1 - s)],
// and the term of nn - 1 - s is minus the conjugate of that of s: contrib[k] = Re[-i U T wt v_k / (N^2 2 qn) sum] takes
// the upper half, s = nn/2 + i (nn/2 rounded down), twice; for odd nn, i = 0 (its own partner) and i = H (partner
// outside the window) once.
struct ALPoint {
    cd cw, ds, dd;  // z_0 + z_L, slopes, second derivatives
    double piT;
    // V(s) from F_s; x = 1 - e^{i w beta/L}
    __device__ __forceinline__ cd V(int s, cd F, cd x) const
    {
        const double iw = rcp_nr((2 * s + 1) * piT), iw2 = iw * iw;
        return cd{(cw.y - ds.x * iw - dd.y * iw2) * iw, (-cw.x - ds.y * iw + dd.x * iw2) * iw} +
               (conjg(x) * F) * (iw2 * iw2);
    }
};

template <int L, typename SelfT>
__global__ void __launch_bounds__(AL_PEN_THREADS)
    k_al_k_pencil_short(const double* __restrict__ Pp, const double* __restrict__ dP, const double* __restrict__ ek,
                        const double* __restrict__ dek, const SelfT* __restrict__ Self,
                        const double* __restrict__ Sinf2, const double* __restrict__ Sinf3,
                        const double* __restrict__ Sinfp, int N, double T, double mu, double U, int nn,
                        const cd* __restrict__ tw, const cd* __restrict__ twX, const cd* __restrict__ twS,
                        double* contrib)
{
    constexpr int H = L / 2, NT = AL_PEN_THREADS;
    __shared__ double Yb[2 * (L + 1)];
    __shared__ cd X[L];
    __shared__ double ES[2 * (2 * NT + 8)];
    __shared__ double sc[NT / 64];
    const int nk = N / 2 + 1;
    const long nq = (long)nk * (nk - 2);
    const long k = blockIdx.x;
    const int tid = threadIdx.x;
    const int l = (int)(k / nk), m = (int)(k % nk);
    const long ki = fold_idx(l + 1, m, N);
    const double hstep = 1.0 / (L * T), ih = L * T;
    const int nc = nn / 2;
    double* const Y0 = Yb;
    double* const Y1 = Yb + (L + 1);
    const double* const row = Pp + k * (L + 1);
    for (int j = tid; j <= L; j += NT) {
        Y0[j] = row[j];
        Y1[j] = row[nq * (L + 1) + j];
    }
    const double d0[2] = {dP[k], dP[nq + k]}, dN[2] = {dP[2 * nq + k], dP[3 * nq + k]};  // dP [side][c][q]
    __syncthreads();
    ALPoint p;
    p.piT = kPi * T;
    p.cw = cd{Y0[0] + Y0[L], Y1[0] + Y1[L]};
    p.ds = cd{d0[0] + dN[0], d0[1] + dN[1]};
    __syncthreads();
    {
        double* const ys[2] = {Y0, Y1};
        block_spline_fixed<L, NT, 2>(ys, hstep, d0, dN, ES, nullptr);
    }
    p.dd = cd{Y0[0] + Y0[L], Y1[0] + Y1[L]};
    for (int t = tid; t < L; t += NT)
        X[t] = conjg(twX[t]) * cd{(Y0[t + 1] - Y0[t]) * ih, (Y1[t + 1] - Y1[t]) * ih};
    __syncthreads();
    block_fft<L, NT>(X, -1, tw);
    const double C2 = Sinf2[ki], C3 = Sinf3[ki], Sinf = Sinfp[0], e0 = mu - ek[m + (l + 1) * nk];
    double acc = 0.0;
    for (int i = tid; i <= H; i += NT) {
        const bool odd = nn & 1;
        const double w = (i == H) ? (odd ? 1.0 : 0.0) : (odd && i == 0) ? 1.0 : 2.0;
        if (w == 0.0) continue;
        const int s = nc + i, s2 = nn - 1 - s;
        const int a = s & (L - 1), b = s2 & (L - 1);
        const cd d = p.V(s, X[a], twS[a]) - conjg(p.V(s2, X[b], twS[b]));
        const cd g = al_G(Self, ki, H, s - nn, C2, C3, Sinf, e0, p.piT) * al_G(Self, ki, H, s, C2, C3, Sinf, e0, p.piT);
        acc += w * (g.x * d.y + g.y * d.x);
    }
    acc = block_sum(acc, sc);
    if (tid == 0) {
        const double wt = (m == 0 || m == nk - 1) ? 2.0 : 4.0;
        const double qn = 2.0 * nn * kPi * T;
        contrib[k] = U * T * wt * dek[k] / ((double)N * N * 2.0 * qn) * acc;
    }
}

// The same for L >= 512 in registers (tpsc_pencil.hpp).  128^2 x 1024: 37 us a frequency (four splines,
// two LDS FFTs, the whole window: 395).
template <int L, typename SelfT>
__global__ void __launch_bounds__(Pen<L>::NT, 3)
    k_al_k_pencil(const double* __restrict__ Pp, const double* __restrict__ dP, const double* __restrict__ ek,
                  const double* __restrict__ dek, const SelfT* __restrict__ Self, const double* __restrict__ Sinf2,
                  const double* __restrict__ Sinf3, const double* __restrict__ Sinfp, int N, PenStep g, double T,
                  double mu, double U, int nn, const cd* __restrict__ tw, const cd* __restrict__ twX,
                  const cd* __restrict__ twS, double* contrib)
{
    constexpr int H = L / 2, NT = Pen<L>::NT, W = Pen<L>::W, PS = Pen<L>::PS;
    __shared__ __align__(16) cd Z[Pen<L>::ZD / 2];
    __shared__ double sx[6 * W], sc[W], ends[8];
    __shared__ SplineTab<8> zt;
    const int nk = N / 2 + 1, nq = nk * (nk - 2);
    const int k = blockIdx.x, t = threadIdx.x;
    zt.fill(t);  // ordered by the barrier of the spline
    const int l = k / nk, m0 = k - l * nk;
    const long ki = fold_idx(l + 1, m0, N);
    const int nc = nn / 2;
    const double d0[2] = {dP[k], dP[nq + k]}, dN[2] = {dP[2 * nq + k], dP[3 * nq + k]};  // dP [side][c][q]
    cd v[8];
    {
        double y[2][10], M[2][9];
        const double* const r0 = Pp + (long)k * (L + 1) + 8 * t;
        const double* const r1 = r0 + (long)nq * (L + 1);
#pragma unroll
        for (int i = 0; i < 9; i++) {
            y[0][1 + i] = r0[i];
            y[1][1 + i] = r1[i];
        }
        y[0][0] = r0[t > 0 ? -1 : 0];
        y[1][0] = r1[t > 0 ? -1 : 0];
        pen_spline<L, NT, 2>(y, g, d0, dN, M, sx, zt, nullptr, t);
        if (t == 0) {
            ends[0] = y[0][1];
            ends[1] = y[1][1];
            ends[2] = M[0][0];
            ends[3] = M[1][0];
        }
        if (t == NT - 1) {
            ends[4] = y[0][9];
            ends[5] = y[1][9];
            ends[6] = M[0][8];
            ends[7] = M[1][8];
        }
        const cd h = tw[4 * t];  // exp(-8 pi i t / L)
#pragma unroll
        for (int i = 0; i < 8; i++) v[i] = h * cd{(M[0][i + 1] - M[0][i]) * g.ih, (M[1][i + 1] - M[1][i]) * g.ih};
    }
    pen_fft_dit<L>(v, Z, tw, conjg(twX[2 * t + 1]), tw[2 * t + 1], tw[4 * t + 2], t);
    wave_lds_order();
#pragma unroll
    for (int m = 0; m < 8; m++) Z[m * PS + t] = v[m];  // F_s, s = t + NT m
    __syncthreads();
    ALPoint p;
    p.piT = kPi * T;
    p.cw = cd{ends[0] + ends[4], ends[1] + ends[5]};
    p.dd = cd{ends[2] + ends[6], ends[3] + ends[7]};
    p.ds = cd{d0[0] + dN[0], d0[1] + dN[1]};
    const double C2 = Sinf2[ki], C3 = Sinf3[ki], Sinf = Sinfp[0], e0 = mu - ek[m0 + (l + 1) * nk];
    double acc = 0.0;
    const bool odd = nn & 1;
    auto F = [&](int s) { return Z[(s / NT) * PS + (s & (NT - 1))]; };
#pragma unroll 1
    for (int i = t; i < H + (odd ? 1 : 0); i += NT) {
        const double w = (odd && (i == 0 || i == H)) ? 1.0 : 2.0;
        const int s = nc + i, s2 = nn - 1 - s;
        const int a = s & (L - 1), b = s2 & (L - 1);
        const cd d = p.V(s, F(a), twS[a]) - conjg(p.V(s2, F(b), twS[b]));
        const cd gg = al_G(Self, ki, H, s - nn, C2, C3, Sinf, e0, p.piT) * al_G(Self, ki, H, s, C2, C3, Sinf, e0, p.piT);
        acc += w * (gg.x * d.y + gg.y * d.x);
    }
    acc = wave_total63(acc);
    if ((t & 63) == 63) sc[t >> 6] = acc;
    __syncthreads();
    if (t == 0) {
        double s = 0.0;
        for (int i = 0; i < W; i++) s += sc[i];
        const double wt = (m0 == 0 || m0 == nk - 1) ? 2.0 : 4.0;
        const double qn = 2.0 * nn * kPi * T;
        contrib[k] = U * T * wt * dek[k] / ((double)N * N * 2.0 * qn) * s;
    }
}

// ================================================================== launchers
#define AL_DISPATCH_N(N, ...)                                       \
    switch (N) {                                                    \
        case 4: { constexpr int NN = 4; __VA_ARGS__; } break;       \
        case 8: { constexpr int NN = 8; __VA_ARGS__; } break;       \
        case 12: { constexpr int NN = 12; __VA_ARGS__; } break;     \
        case 24: { constexpr int NN = 24; __VA_ARGS__; } break;     \
        case 48: { constexpr int NN = 48; __VA_ARGS__; } break;     \
        case 96: { constexpr int NN = 96; __VA_ARGS__; } break;     \
        case 192: { constexpr int NN = 192; __VA_ARGS__; } break;   \
        case 16: { constexpr int NN = 16; __VA_ARGS__; } break;     \
        case 32: { constexpr int NN = 32; __VA_ARGS__; } break;     \
        case 64: { constexpr int NN = 64; __VA_ARGS__; } break;     \
        case 128: { constexpr int NN = 128; __VA_ARGS__; } break;   \
        case 256: { constexpr int NN = 256; __VA_ARGS__; } break;   \
        default: return hipErrorInvalidValue;                       \
    }
// Nw <= 2048 (the launchers refuse larger ones)
#define AL_DISPATCH_HW(Lv, ...) \
    switch (Lv) { TPSC_LS_256(__VA_ARGS__) TPSC_CASE_L(512, __VA_ARGS__) TPSC_CASE_L(1024, __VA_ARGS__) \
                  TPSC_CASE_L(2048, __VA_ARGS__) default: return hipErrorInvalidValue; }
#define AL_DISPATCH_FROM1024(Lv, ...) \
    switch (Lv) { TPSC_CASE_L(1024, __VA_ARGS__) TPSC_CASE_L(2048, __VA_ARGS__) default: return hipErrorInvalidValue; }
#define AL_DISPATCH_FROM512(Lv, ...) \
    switch (Lv) { TPSC_CASE_L(512, __VA_ARGS__) TPSC_CASE_L(1024, __VA_ARGS__) TPSC_CASE_L(2048, __VA_ARGS__) \
                  default: return hipErrorInvalidValue; }

template <typename K>
static void al_set_lds(K kern, size_t bytes)
{
    (void)hipFuncSetAttribute(reinterpret_cast<const void*>(kern), hipFuncAttributeMaxDynamicSharedMemorySize,
                              (int)bytes);
}

hipError_t launch_al_setup(const Grid& g, const DevArrays& d, const ALArrays& a, double mu0, hipStream_t s)
{
    AL_DISPATCH_N(g.N, {
        constexpr size_t lds = slab_bytes(NN, sizeof(double));
        al_set_lds(k_al_grt_slab<NN>, lds);
        hipLaunchKernelGGL(k_al_grt_slab<NN>, dim3(g.Nw + 2), dim3(SlabShape<NN>::NT), lds, s, d.wt, d.ekw, d.fw, d.er,
                           mu0, g.T, g.Nw, a.Grt, a.dGrt);
        al_set_lds(k_al_hg_slab<NN>, lds);
        hipLaunchKernelGGL(k_al_hg_slab<NN>, dim3(g.Nw + 3), dim3(SlabShape<NN>::NT), lds, s, d.wt, d.ekw, d.fw, d.vw,
                           a.Grt, a.dGrt, mu0, g.T, g.Nw, a.Ps, a.dhG);
    });
    hipError_t e = launch_transpose_d(a.Ps, a.Pp, g.nq, g.Nw + 1, s);
    if (e != hipSuccess) return e;
    AL_DISPATCH_HW(g.Nw, {
        hipLaunchKernelGGL(k_al_hw_pencil<LL>, dim3((unsigned)g.nq), dim3(AL_PEN_THREADS), 0, s, a.Pp, a.dhG, g.nq,
                           g.T, d.twN, d.twM, a.hw, a.hg2);
    });
    // chi0(q,iq_p) point-major for the per-frequency pencils
    return launch_transpose_d(d.chiw, a.chiwP, g.nk8, g.nwb, s);
}

hipError_t launch_al_freq(const Grid& g, const DevArrays& d, const ALArrays& a, double Usp, double Uch, double mu,
                          double U, long n, double* contrib, hipStream_t s)
{
    const int nn = (int)n, H = g.Nw / 2;
    const long plane = (long)(g.Nw + 1) * g.nq, half = (long)(H + 1) * g.nq;
    const unsigned nq = (unsigned)g.nq;
    if (g.Nw <= 512) {
        DISPATCH_L_TO512(g.Nw, hipLaunchKernelGGL(k_al_HG_pencil_short<LL>, dim3(nq), dim3(AL_PEN_THREADS), 0, s, a.chiwP,
                         d.chi0inf, d.chi0inf2, a.hw, a.hg2, g.N, g.T, Usp, Uch, nn, d.twN, a.Pp, a.dHq));
    } else {
        AL_DISPATCH_FROM1024(g.Nw, hipLaunchKernelGGL(k_al_HG_pencil<LL>, dim3(nq), dim3(LL / 16), 0, s, a.chiwP,
                             d.chi0inf, d.chi0inf2, a.hw, a.hg2, g.N, g.T, Usp, Uch, nn, d.twN, a.Pp, a.dHq));
    }
    hipError_t e = launch_transpose_d2(a.Pp, a.HGs, a.Pp + half, a.HGs + half, H + 1, (int)g.nq, s);
    if (e != hipSuccess) return e;
    AL_DISPATCH_N(g.N, {
        constexpr size_t lds = slab_bytes(NN, sizeof(double));
        al_set_lds(k_al_prod_slab<NN>, lds);
        hipLaunchKernelGGL(k_al_prod_slab<NN>, dim3(2 * (H + 1) + 4), dim3(SlabShape<NN>::NT), lds, s, d.wt, a.HGs, a.dHq,
                           a.Grt, a.dGrt, g.Nw, a.Ps, a.dP);
    });
    if ((e = launch_transpose_d2(a.Ps, a.Pp, a.Ps + plane, a.Pp + plane, g.nq, g.Nw + 1, s)) != hipSuccess) return e;
    const PenStep step = pen_step(1.0 / (g.Nw * g.T));
    DISPATCH_S(g.prec, {
        if (g.Nw <= 256) {
            DISPATCH_L_SHORT(g.Nw, hipLaunchKernelGGL((k_al_k_pencil_short<LL, ST>), dim3(nq), dim3(AL_PEN_THREADS), 0, s,
                             a.Pp, a.dP, d.ek, d.dek, (const ST*)d.Self, d.Sinf2, d.Sinf3, d.Sinf, g.N, g.T, mu, U, nn,
                             d.twN, d.twX, d.twS, contrib));
        } else {
            AL_DISPATCH_FROM512(g.Nw, hipLaunchKernelGGL((k_al_k_pencil<LL, ST>), dim3(nq), dim3(Pen<LL>::NT), 0, s, a.Pp,
                                a.dP, d.ek, d.dek, (const ST*)d.Self, d.Sinf2, d.Sinf3, d.Sinf, g.N, step, g.T, mu, U,
                                nn, d.twN, d.twX, d.twS, contrib));
        }
    });
    return hipGetLastError();
}

}  // namespace tpsc
