// tpsc_kernels.hip -- HIP kernels of the TPSC hot path for gfx950.
//
// Stage map (tpsc_tau.hip holds the chi0, V and Sigma pencils, tpsc_jj.hip the Lambda pencils; reference =
// dbergeron1/TPSC_conductivity):
//   k_mu0_root                   green0.cpp:182-203, 240-262 finite-lattice density and the mu0 root
//   k_chi0_tau0, k_chi0_slab     chi0.cpp:310-559   G0(k,+-tau) -> G(r,+-tau) -> chi0(r,tau) -> chi0(q,tau)
//   k_sum_rule*, k_sr_*          chi.cpp:738-830    sum-rule traces and the searches for Usp, Uch
//   k_vertex_slab                chi.cpp:85-170     V(r,iqn)
//   k_sigma_bnd, k_sigma_slab    green.cpp:1743-1892 Sigma(k,tau), end values and slopes
//   k_trace_*, k_mu_search       green.cpp:2929-3282 traces for mu and consistency checks
//   k_hf0_bnd, k_hV_slab         cond_opt.cpp:2584-3180 Lambda_jj: hV, f0V
// Slab kernels hold one (nk x nk) slab in LDS (151 KB at N=256 in FP64) and transform it with
// register FFTs of line pairs.
// Precision: S is the storage and slab-arithmetic type of the tau arrays (chi0(q,tau),
// chi0(r,tau), V, Sigma(k,tau), h, f0); chi0(q,iqn) is stored in FP64 in both paths.  S = double
// is the FP64 path.  S = float is the mixed path: the slab transforms and pointwise products run
// in FP32, while the tau = 0 / beta boundary data, the spline moments, the tail moments, the pencil Fourier sums, the root-finder reductions
// and the Lambda_jj Matsubara sums stay in FP64.  Self holds the remainder R(k,n) as FP64
// complex (S = double) or the assembled Sigma(k,iwn) as FP32 complex (S = float).
#include <algorithm>
#include <unordered_map>

#include "tpsc_launch.hpp"
#include "tpsc_pencil.hpp"

namespace tpsc {

// waves per SIMD a slab kernel is compiled for: two FP32 workgroups (76 KB of LDS and ten wavefronts
// each at N = 256) share a CU within 96 VGPRs; an FP64 slab (151 KB) runs alone, within 168
template <typename S>
constexpr int slab_occ() { return sizeof(S) == sizeof(float) ? 5 : 1; }

// ================================================================== small helpers
__global__ void k_fill_tw(cd* tw, int L)
{
    const int t = blockIdx.x * blockDim.x + threadIdx.x;
    if (t < L) {
        double s, c;
        sincospi(2.0 * (double)t / (double)L, &s, &c);
        tw[t] = cd{c, -s};
    }
}

// sum n partials in a fixed order (single block)
__global__ void k_finalize(const double* __restrict__ part, int n, double* out)
{
    __shared__ double sc[16];
    double a = 0.0;
    for (int i = threadIdx.x; i < n; i += blockDim.x) a += part[i];
    a = block_sum(a, sc);
    if (threadIdx.x == 0) out[0] = a;
}

// out[b] = sum of the n partials part[b*n .. b*n+n) in a fixed order; one block per value
__global__ void k_finalize_k(const double* __restrict__ part, int n, double* out)
{
    __shared__ double sc[16];
    const double* p = part + (long)blockIdx.x * n;
    double a = 0.0;
    for (int i = threadIdx.x; i < n; i += blockDim.x) a += p[i];
    a = block_sum(a, sc);
    if (threadIdx.x == 0) out[blockIdx.x] = a;
}

// ================================================================== device-driven root search
// mirror (mapped host memory) = {status, root, x, passes, f, f', lo, hi} of the search: written
// here with status "running", and by the step that settles it (one system-scope write per
// search instead of one per pass)
// chi0max != nullptr (the Usp search): the bracket is (0, 2/chi0max - 2 eps) from the device
// maximum of chi0, with the start s0.x kept when it lies inside and the midpoint otherwise, so
// that the host need not wait for chi0max before the first pass
// a0src (device Usp, may be null): a0 = uch_a0(a0A, nsr, U, *a0src); mu0p (may be null): the
// state's mu0 from the device
__device__ __forceinline__ HalleyState halley_begin(const RootInit& in)
{
    HalleyState s = in.s0;
    if (in.chi0max) {
        const double lo = 0.0, hi = 2.0 / in.chi0max[0] - 2 * DBL_EPSILON;
        const double x0 = (in.s0.x > lo && in.s0.x < hi) ? in.s0.x : 0.5 * (lo + hi);
        s = halley_start(x0, lo, hi, in.s0.itmax, in.s0.a0, in.s0.a1);
        s.T = in.s0.T;
        s.mu0 = in.s0.mu0;
    }
    if (in.mu0p) s.mu0 = *in.mu0p;
    if (in.a0src) s.a0 = uch_a0(in.a0A, in.nsr, in.U, *in.a0src);
    return s;
}
__device__ __forceinline__ void halley_mirror(const HalleyState& s, double* mirror)
{
    mirror[0] = s.status;
    mirror[1] = s.root;
    mirror[2] = s.x;
    mirror[3] = s.ne;
    mirror[4] = s.f;
    mirror[5] = s.f1;
    mirror[6] = s.lo;
    mirror[7] = s.hi;
}
__global__ void k_halley_init(HalleyState* st, RootInit in, double* mirror)
{
    const HalleyState s = halley_begin(in);
    *st = s;
    mirror[0] = s.status;
    mirror[1] = s.root;
    mirror[2] = s.x;
    mirror[3] = s.ne;
}

// A whole search in one workgroup of 1024 threads, for grids whose passes would be launch-bound: at most npass
// evaluations, pass(x, acc) adding this thread's part of {f, f', f''}, from values that the kernel keeps in registers.
// What bounds it: the latency of a pass's reduction (two barriers) and update.  A search of five passes
// over 5800 terms takes 16 us; five pass kernels take 33 us and their launches.
constexpr int kSearchThreads = 1024;
template <typename Pass>
__device__ __forceinline__ HalleyState search_block(const HalleyState& s0, int npass, const Pass& pass)
{
    constexpr int NWV = kSearchThreads / 64;  // 16: the wavefront sums of one value fill a DPP row
    __shared__ HalleyState s;
    __shared__ double sc[3 * NWV];
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    if (threadIdx.x < 3 * NWV) sc[threadIdx.x] = 0.0;  // a smaller workgroup leaves the other wavefronts' places zero
    if (threadIdx.x == 0) s = s0;
    __syncthreads();
    for (int k = 0; k < npass && s.status == kRootRunning; k++) {
        double acc[3] = {0.0, 0.0, 0.0};
        pass(s.x, acc);
#pragma unroll
        for (int i = 0; i < 3; i++) acc[i] = wave_total63(acc[i]);
        if (lane == 63)
#pragma unroll
            for (int i = 0; i < 3; i++) sc[i * NWV + wave] = acc[i];
        __syncthreads();
        if (wave == 0) {
            const double v = row_total15((lane < 3 * NWV) ? sc[lane] : 0.0);
            const double f[3] = {lane_get(v, 15), lane_get(v, 31), lane_get(v, 47)};
            if (lane == 0) halley_update(s, f);
        }
        __syncthreads();
    }
    return s;
}
__device__ __forceinline__ void search_end(const HalleyState& s, HalleyState* st, double* mirror)
{
    if (threadIdx.x != 0) return;
    *st = s;
    halley_mirror(s, mirror);
}

// One Halley step after a pass, by one workgroup of 256 threads: the three partial sums of
// part[k * n + i] (k = 0, 1, 2), each in the order of k_finalize_k, the update of st, and the
// outcome in mirror once the search has settled.  A settled search is left as it is.
__device__ __forceinline__ void halley_step_block(const double* part, int n, HalleyState* st, double* mirror,
                                                  double* sc)
{
    const HalleyState s0 = *st;
    if (s0.status != kRootRunning) return;
    double v[3] = {0.0, 0.0, 0.0};
    for (int i = threadIdx.x; i < n; i += blockDim.x) {
        v[0] += part[i];
        v[1] += part[(long)n + i];
        v[2] += part[2L * n + i];
    }
    block_sum_k<3>(v, sc);
    if (threadIdx.x == 0) {
        HalleyState s = s0;
        halley_update(s, v);
        *st = s;
        if (s.status != kRootRunning) halley_mirror(s, mirror);
    }
}

// True in the workgroup of a pass that finishes last, once every workgroup's partial sums acc[k] -> part[k * nblk + b]
// (stored here by its thread 0) are visible to it; that workgroup resets the ticket for the next pass.  No workgroup
// waits for another: the others return at once.  The sums are stored at agent scope, past the XCD's L2, and have
// arrived when the ticket is taken: no workgroup needs a release fence (a write-back of its whole L2), and only the
// last one acquires.  That order is gfx950's (an agent-scope store is acknowledged past the L2, and s_waitcnt waits for
// it), not the language's: only such stores may carry a pass's results to the last workgroup.
__device__ __forceinline__ bool last_workgroup(unsigned* ticket, unsigned nblk, unsigned b, const double acc[3],
                                               double* part)
{
    __shared__ unsigned last;
    if (threadIdx.x == 0) {
        for (int k = 0; k < 3; k++)
            __hip_atomic_store(part + (long)k * nblk + b, acc[k], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        asm volatile("" ::: "memory");
        __builtin_amdgcn_s_waitcnt(0);  // the stores have been acknowledged
        asm volatile("" ::: "memory");
        last = __hip_atomic_fetch_add(ticket, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) == nblk - 1;
    }
    __syncthreads();
    if (!last) return false;
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "agent");
    if (threadIdx.x == 0) __hip_atomic_store(ticket, 0u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    return true;
}

// the Halley step as a kernel of its own, launched after a trace pass of more than kFusedStepMax workgroups
__global__ void __launch_bounds__(256) k_halley_step(const double* part, int n, HalleyState* st, double* mirror)
{
    __shared__ double sc[3 * 4];
    halley_step_block(part, n, st, mirror, sc);
}

// ================================================================== chi0 slabs
// tau = 0 slice plus the tau-derivative data (chi0.cpp:323-447); one block.
// The boundary data are tail moments: this kernel runs in FP64 for both precisions and
// only rounds the slice-0 values it stores into the S arrays.
template <int N, typename S>
__global__ void __launch_bounds__(SlabShape<N>::NT)
    k_chi0_tau0(const unsigned* __restrict__ wt, const double* __restrict__ ekw, const double* __restrict__ fw,
                const double* __restrict__ er, const double* __restrict__ mu0p, double T, S* chi, S* chirt,
                double* dchirt0, double* dGrt0p, double* dchiqt0, double* chirt0)
{
    const double mu0 = *mu0p, beta = 1.0 / T;
    extern __shared__ double smem[];
    double* slab = smem;
    cd* tw = slab_tw<N>(slab);
    fill_twiddles<N>(tw);
    // d/dtau G(r,0+) = DCT[-x G0(k,0) / N^2]
    each_wedge<N>(wt, [&](int a, int b, int i) {
        const double x = ekw[i] - mu0;
        slab[a] = slab[b] = x * g0_exp(x, 0.0, beta) * fw[i];
    });
    __syncthreads();
    slab_r2r_2d<double, N, 0>(slab, tw);
    each_wedge<N>(wt, [&](int a, int, int i) { dGrt0p[i] = slab[a]; });
    __syncthreads();
    // G(r,0)
    each_wedge<N>(wt, [&](int a, int b, int i) { slab[a] = slab[b] = -g0_exp(ekw[i] - mu0, 0.0, beta) * fw[i]; });
    __syncthreads();
    slab_r2r_2d<double, N, 0>(slab, tw);
    // chi0(r,0) and its transform (each thread replaces the points it read and keeps their G(r,0))
    double G0r[wedge_per_thread<N>()];
    each_wedge_slot<N>(wt, [&](int a, int b, int i, int k) {
        const double g = slab[a];
        G0r[k] = g;
        const double c = (i == 0) ? -2.0 * g * (g + 1.0) : -2.0 * g * g;
        chirt[i] = (S)c;
        chirt0[i] = c;
        slab[a] = slab[b] = c;
    });
    __syncthreads();
    slab_r2r_2d<double, N, 0>(slab, tw);
    // d/dtau chi0(r,0) and its transform
    each_wedge_slot<N>(wt, [&](int a, int b, int i, int k) {
        chi[i] = (S)slab[a];
        const double g = G0r[k], dGp = dGrt0p[i];  // written above by this thread
        const double dGm = ((i == 0) ? -mu0 : er[i]) - dGp;
        const double v = (i == 0) ? -2.0 * (dGp * (1.0 + g) + dGm * g) : -2.0 * (dGp * g + dGm * g);
        dchirt0[i] = v;
        slab[a] = slab[b] = v;
    });
    __syncthreads();
    slab_r2r_2d<double, N, 0>(slab, tw);
    each_wedge<N>(wt, [&](int a, int, int i) { dchiqt0[i] = slab[a]; });
}

// slices j = 1 .. nwb-1 (chi0.cpp:454-559); block b handles j = b + 1
template <int N, typename S>
__global__ void __launch_bounds__(SlabShape<N>::NT, slab_occ<S>())
    k_chi0_slab(const unsigned* __restrict__ wt, const double* __restrict__ ekw, const double* __restrict__ fw,
                const double* __restrict__ mu0p, double T, int Nw, S* chi, S* chirt)
{
    const double mu0 = *mu0p;
    constexpr int nk = N / 2 + 1;
    constexpr long nk8 = (long)nk * (nk + 1) / 2;
    extern __shared__ double smem[];
    S* slab = (S*)smem;
    auto* tw = slab_tw<N>(slab);
    fill_twiddles<N>(tw);
    const int nwb = Nw / 2 + 1;
    const int j = blockIdx.x + 1;
    const double t = (j < nwb - 1) ? j / (Nw * T) : 1.0 / (2.0 * T), bt = 1.0 / T - t;
    S* cr = chirt + (long)j * nk8;
    S* cq = chi + (long)j * nk8;
    each_wedge<N>(wt, [&](int a, int b, int i) { slab[a] = slab[b] = (S)(-g0_exp(ekw[i] - mu0, t, bt) * fw[i]); });
    __syncthreads();
    slab_r2r_2d<S, N, 0>(slab, tw);
    if (j < nwb - 1) {
        S g[wedge_per_thread<N>()];  // G(r,t) of the thread's points
        each_wedge_slot<N>(wt, [&](int a, int, int, int c) { g[c] = slab[a]; });
        __syncthreads();
        each_wedge<N>(wt, [&](int a, int b, int i) { slab[a] = slab[b] = (S)(g0_exp(ekw[i] - mu0, bt, t) * fw[i]); });
        __syncthreads();
        slab_r2r_2d<S, N, 0>(slab, tw);
        // chi0(r,t) = -2 G(r,-t) G(r,t)
        each_wedge_slot<N>(wt, [&](int a, int b, int i, int c) {
            const S v = (S)(-2) * slab[a] * g[c];
            cr[i] = v;
            slab[a] = slab[b] = v;
        });
    } else {  // tau = beta/2: G(r,-t) = -G(r,t)
        each_wedge<N>(wt, [&](int a, int b, int i) {
            const S v = slab[a], c = (S)2 * v * v;
            cr[i] = c;
            slab[a] = slab[b] = c;
        });
    }
    __syncthreads();
    slab_r2r_2d<S, N, 0>(slab, tw);
    each_wedge<N>(wt, [&](int a, int, int i) { cq[i] = slab[a]; });
}

// ================================================================== chi0 maximum
// chi0max and its wedge position (chi0.cpp:703-717): largest value, ties to the
// larger packed index (the reference scans l, m downwards with a strict >).
// out2 (may be null): a second copy of the maximum
__global__ void k_chi0max(const double* __restrict__ chi, long nk8, double* out, int* imax, double* out2)
{
    __shared__ double sv[1024];
    __shared__ long si[1024];
    double best = 0.0;
    long bi = -1;
    for (long i = threadIdx.x; i < nk8; i += blockDim.x) {
        const double v = chi[i];
        if (v > best || (v == best && bi >= 0 && i > bi) ) {
            if (v > 0.0 || bi >= 0) {
                best = v;
                bi = i;
            }
        }
    }
    sv[threadIdx.x] = best;
    si[threadIdx.x] = bi;
    __syncthreads();
    for (int s = blockDim.x / 2; s > 0; s >>= 1) {
        if (threadIdx.x < s) {
            const double v2 = sv[threadIdx.x + s];
            const long i2 = si[threadIdx.x + s];
            if (i2 >= 0 && (v2 > sv[threadIdx.x] || (v2 == sv[threadIdx.x] && i2 > si[threadIdx.x]) ||
                            si[threadIdx.x] < 0)) {
                sv[threadIdx.x] = v2;
                si[threadIdx.x] = i2;
            }
        }
        __syncthreads();
    }
    if (threadIdx.x == 0) {
        out[0] = (si[0] >= 0) ? sv[0] : 0.0;
        imax[0] = (int)((si[0] >= 0) ? si[0] : 0);
        if (out2) out2[0] = out[0];
    }
}

// ================================================================== reductions
// sum-rule trace sum_{n=0}^{Nw} sum_q (w T/Nq) [chi/(1 + sU chi/2) - chi]  (chi.cpp:738-830)
// sU = -Usp for the spin channel, +Uch for the charge channel.  Grid: x over wedge points
// (256 per block), y over RG row groups; rows j = y, y+RG, ...  One partial per block.
__global__ void __launch_bounds__(256)
    k_sum_rule(const double* __restrict__ chi, const double* __restrict__ inf1, const double* __restrict__ inf2,
               const double* __restrict__ wq, int nk8, int nwmax, double T, double Nq, double sU, double* part)
{
    __shared__ double sc[16];
    const int q = blockIdx.x * 256 + threadIdx.x;
    double acc = 0.0;
    if (q < nk8) {
        const double w16 = 2.0 * wq[q];
        const double a1 = inf1[q], a2 = inf2[q];
        for (int j = blockIdx.y; j <= 2 * nwmax; j += gridDim.y) {
            const double w = (j == 0) ? 0.5 * w16 : w16;
            double c;
            if (j <= nwmax)
                c = chi[(long)j * nk8 + q];
            else {
                const double wn = 2 * j * kPi * T;
                c = a1 / (wn * wn) + a2 / (wn * wn * wn * wn);
            }
            acc += w * T / Nq * (c / (1 + sU * c / 2.0) - c);
        }
    }
    acc = block_sum(acc, sc);
    if (threadIdx.x == 0) part[blockIdx.y * gridDim.x + blockIdx.x] = acc;
}

// The same trace and its first two derivatives with respect to Ux, where sU = sgn * Ux:
// d/dUx [c/(1 + sU c/2)] = -sgn c^2/2 / (1 + sU c/2)^2, d2/dUx2 = c^3/2 / (1 + sU c/2)^3.
// Partials: part[k * nblk + blk], k = 0, 1, 2.  A thread sums its rows j = y, y + RG, ... in
// increasing j: the stored rows j <= nwmax in batches of kSR loads issued before any use (one
// dependent load per row would leave HBM idle), then the asymptotic rows, whose 1/wn^2 is
// common to the block.
constexpr int kSR = 8;
__device__ __forceinline__ void sum_rule3_term(double c, double w, double sU, double sgn, double acc[3])
{
    const double r = rcp_nr(1 + sU * c / 2.0);
    acc[0] += w * (c * r - c);
    acc[1] -= w * sgn * 0.5 * c * c * r * r;
    acc[2] += w * 0.5 * c * c * c * r * r * r;
}
// Rows of small chi: with y = -sU/2 and |y c| <= rho for every element of rows j >= n0,
//   c r - c = sum_{k>=1} y^k c^(k+1),  c^2 r^2 = sum_{k>=0} (k+1) y^k c^(k+2),
//   c^3 r^3 = sum_{k>=0} (k+1)(k+2)/2 y^k c^(k+3),   r = 1/(1 - y c),
// so their part of the three sums is a polynomial in y over the moments
// M_m(n0) = sum_{j>=n0} sum_q w c^m, m = 2..kSRK+3, stored once per chi0 (k_sr_moments,
// k_sr_suffix).  rho = 1/16 and kSRK = 18: the first omitted term of the c^3 r^3 series is
// below 210 * 16^-19 ~ 3e-21 of the moment M_3 it is measured against.  Every chi0(q,iqn) and
// its asymptotic continuation are positive, so the moments carry no cancellation.
constexpr double kSRRho = 1.0 / 16.0;
// Ux (and T) come from the root search st, so that a captured pass graph serves every point;
// a settled search leaves nothing to do.  The workgroup that finishes last takes the Halley step;
// large grids have fewer row groups (kSumRuleGrid).  srm != null: rows j >= n0(Ux) (all rows whose elements satisfy
// |Ux c/2| <= rho, from the suffix maxima srmax) are not read; workgroup (0, 0) adds their
// part from the suffix moments srm[n0].
__global__ void __launch_bounds__(256)
    k_sum_rule3(const double* __restrict__ chi, const double* __restrict__ inf1, const double* __restrict__ inf2,
                const double* __restrict__ wq, int nk8, int nwmax, double Nq, double sgn, HalleyState* st,
                double* part, unsigned* ticket, double* mirror, const double* __restrict__ srm,
                const double* __restrict__ srmax)
{
    __shared__ double sc[3 * 4];
    if (st->status != kRootRunning) return;
    const double Ux = st->x, T = st->T;
    const int q = blockIdx.x * 256 + threadIdx.x;
    const int RG = gridDim.y;
    const double sU = sgn * Ux;
    const int nrows = 2 * nwmax + 1;
    int n0 = nrows;
    if (srm) {
        // srmax is non-increasing in j: n0 = the number of rows above the threshold
        const double thr = kSRRho / (0.5 * fabs(Ux));
        double cnt = 0.0;
        for (int j = threadIdx.x; j < nrows; j += 256) cnt += (srmax[j] > thr) ? 1.0 : 0.0;
        n0 = (int)block_sum(cnt, sc);
    }
    double acc[3] = {0.0, 0.0, 0.0};
    if (q < nk8) {
        const double wb = 2.0 * wq[q] * T / Nq;
        const double a1 = inf1[q], a2 = inf2[q];
        const int jst = min(nwmax, n0 - 1), jas = min(2 * nwmax, n0 - 1);
        int j = blockIdx.y;
        for (; j + (kSR - 1) * RG <= jst; j += kSR * RG) {
            double c[kSR];
#pragma unroll
            for (int u = 0; u < kSR; u++) c[u] = chi[(long)(j + u * RG) * nk8 + q];
#pragma unroll
            for (int u = 0; u < kSR; u++) sum_rule3_term(c[u], (j + u * RG == 0) ? 0.5 * wb : wb, sU, sgn, acc);
        }
        for (; j <= jst; j += RG) sum_rule3_term(chi[(long)j * nk8 + q], (j == 0) ? 0.5 * wb : wb, sU, sgn, acc);
        for (; j <= jas; j += RG) {
            const double wn = 2 * j * kPi * T;
            const double i2 = rcp_nr(wn * wn);
            sum_rule3_term((a1 + a2 * i2) * i2, wb, sU, sgn, acc);
        }
    }
    if (srm && n0 < nrows && blockIdx.x == 0 && blockIdx.y == 0 && threadIdx.x == 0) {
        const double* M = srm + (long)n0 * kSRM;  // M[m - 2] = M_m(n0)
        const double y = -0.5 * sU;
        double f0 = 0.0, f1 = 0.0, f2 = 0.0;
        for (int k = kSRK; k >= 0; k--) {
            if (k >= 1) f0 = f0 * y + M[k - 1];
            f1 = f1 * y + (k + 1) * M[k];
            f2 = f2 * y + 0.5 * (k + 1) * (k + 2) * M[k + 1];
        }
        acc[0] += y * f0;
        acc[1] -= sgn * 0.5 * f1;
        acc[2] += 0.5 * f2;
    }
    block_sum_k<3>(acc, sc);
    const int nblk = gridDim.x * gridDim.y, b = blockIdx.y * gridDim.x + blockIdx.x;
    if (last_workgroup(ticket, nblk, b, acc, part)) halley_step_block(part, nblk, st, mirror, sc);
}

// The whole search in one workgroup: the nk8 (2 nwmax + 1) <= CN * 1024 values of chi0 and their weights are read
// once, CN per thread (no series part on such grids)
template <int CN>
__global__ void __launch_bounds__(kSearchThreads)
    k_sum_rule_search(const double* __restrict__ chi, const double* __restrict__ inf1, const double* __restrict__ inf2,
                      const double* __restrict__ wq, int nk8, int nwmax, double Nq, double sgn, HalleyState* st,
                      RootInit in, double* mirror, int npass)
{
    const HalleyState s0 = halley_begin(in);
    const double wT = 2.0 * s0.T / Nq;
    double c[CN], w[CN];
#pragma unroll
    for (int u = 0; u < CN; u++) {
        const int i = threadIdx.x + u * kSearchThreads, j = i / nk8, q = i - j * nk8;
        c[u] = w[u] = 0.0;
        if (j <= 2 * nwmax) {
            w[u] = (j == 0) ? 0.5 * wT * wq[q] : wT * wq[q];
            if (j <= nwmax) {
                c[u] = chi[i];
            } else {
                const double wn = 2 * j * kPi * s0.T;
                const double i2 = rcp_nr(wn * wn);
                c[u] = (inf1[q] + inf2[q] * i2) * i2;
            }
        }
    }
    const HalleyState r = search_block(s0, npass, [&](double Ux, double* acc) {
#pragma unroll
        for (int u = 0; u < CN; u++) sum_rule3_term(c[u], w[u], sgn * Ux, sgn, acc);
    });
    search_end(r, st, mirror);
}

// Row moments of the sum-rule terms (one workgroup per row j <= 2 nwmax, stored rows from chi,
// the rest from the asymptote a1/wn^2 + a2/wn^4 as k_sum_rule3 forms them): R[j][m - 2] =
// sum_q w_j wb_q c^m, m = 2..kSRK+3 (w_0 = 1/2), and rmax[j] = max_q |c|.
__global__ void __launch_bounds__(256)
    k_sr_moments(const double* __restrict__ chi, const double* __restrict__ inf1, const double* __restrict__ inf2,
                 const double* __restrict__ wq, int nk8, int nwmax, double Nq, double T, double* R, double* rmax)
{
    __shared__ double sc[kSRM * 4];
    const int j = blockIdx.x;
    double acc[kSRM];
#pragma unroll
    for (int m = 0; m < kSRM; m++) acc[m] = 0.0;
    double mx = 0.0;
    const double wn = 2 * j * kPi * T;
    const double i2 = (j > nwmax) ? rcp_nr(wn * wn) : 0.0;
    for (int q = threadIdx.x; q < nk8; q += 256) {
        const double wb = 2.0 * wq[q] * T / Nq * ((j == 0) ? 0.5 : 1.0);
        const double c = (j <= nwmax) ? chi[(long)j * nk8 + q] : (inf1[q] + inf2[q] * i2) * i2;
        // c^i, i < kSRM, as a product tree (c^i = c^h c^(i-h), h the largest power of two below
        // i): five multiplies deep instead of a chain of kSRM
        double cp[kSRM];
        cp[0] = 1.0;
        cp[1] = c;
#pragma unroll
        for (int i = 2; i < kSRM; i++) {
            const int h = 1 << (31 - __builtin_clz(i - 1));
            cp[i] = cp[h] * cp[i - h];
        }
        const double w2 = wb * c * c;
#pragma unroll
        for (int m = 0; m < kSRM; m++) acc[m] = fma(w2, cp[m], acc[m]);
        mx = fmax(mx, fabs(c));
    }
    block_sum_k<kSRM>(acc, sc);
    if (threadIdx.x == 0)
#pragma unroll
        for (int m = 0; m < kSRM; m++) R[(long)j * kSRM + m] = acc[m];
    // block maximum through the same scratch
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
#pragma unroll
    for (int o = 32; o >= 1; o >>= 1) mx = fmax(mx, __shfl_xor(mx, o, 64));
    if (lane == 0) sc[wave] = mx;
    __syncthreads();
    if (threadIdx.x == 0) rmax[j] = fmax(fmax(sc[0], sc[1]), fmax(sc[2], sc[3]));
}

// Suffix sums (columns 0..kSRM-1 of R, in place) and suffix maxima (rmax, in place) over the
// rows 0..nrows-1: column b of one workgroup of 1024 threads, thread t owning rows
// [t ch, t ch + ch); the thread totals are combined by a fixed-order scan, so the result does
// not depend on timing.
__global__ void __launch_bounds__(1024) k_sr_suffix(double* R, double* rmax, int nrows)
{
    __shared__ double tot[1024];
    const int b = blockIdx.x;  // b < kSRM: a moment column; b == kSRM: the maxima
    const bool ismax = b == kSRM;
    const int t = threadIdx.x;
    const int ch = (nrows + 1023) / 1024;
    constexpr int kMaxCh = 8;  // nrows <= 8192
    double v[kMaxCh];
    double s = 0.0;
    for (int i = ch - 1; i >= 0; i--) {
        const int j = t * ch + i;
        const double x = (j < nrows) ? (ismax ? rmax[j] : R[(long)j * kSRM + b]) : 0.0;
        s = ismax ? fmax(s, x) : s + x;
        v[i] = s;
    }
    tot[t] = s;
    __syncthreads();
    // inclusive suffix scan of the thread totals (Hillis-Steele, fixed order)
    for (int o = 1; o < 1024; o <<= 1) {
        const double a = tot[t], c = (t + o < 1024) ? tot[t + o] : 0.0;
        __syncthreads();
        tot[t] = ismax ? fmax(a, c) : a + c;
        __syncthreads();
    }
    const double after = (t + 1 < 1024) ? tot[t + 1] : 0.0;  // rows of the threads after t
    for (int i = 0; i < ch; i++) {
        const int j = t * ch + i;
        if (j < nrows) {
            if (ismax)
                rmax[j] = fmax(v[i], after);
            else
                R[(long)j * kSRM + b] = v[i] + after;
        }
    }
}

// green0::find_mu (green0.cpp:240-262) in one workgroup, on block-wide sums of the
// finite-lattice density n(mu) = (2/N^2) sum_wedge w f(eps - mu) (green0.cpp:182-203): every
// thread sees the same sums, so the control flow stays uniform.  One evaluation gives n - dens
// and its first two derivatives from the same exponential (f' = f(1-f)/T,
// f'' = f(1-f)(1-2f)/T^2), and the Halley iteration of tpsc_roots.hpp runs from the reference's
// start 0 in its bracket [-8, 8] (green0.cpp:248-257).  n(mu) is increasing, so it fails only
// when the root lies outside the bracket or the derivative underflows (no level within ~700 T
// of the iterate); the derivative-free bracketed search (bracket_root, which widens the
// interval) then takes over.  out = {found, mu0, evaluations}.
// Each thread keeps its K strided wedge points (eps, weight) in registers for all the
// evaluations; a padded slot has weight 0 and adds +0.  The launcher sizes the workgroup so
// that blockDim.x * K >= nk8: K = 1, 3, 9 for up to 1024, 3072, 9216 points (nine slots, division and LDS
// reductions for every size: 11.5, 17.1, 29.2 us a search on 45, 2145, 8385 points; now 7.4, 14.0, 28.1).
// The root goes to out (mapped host memory) and to the device slot mu0v, which the chi0 and
// h/f0 kernels read, so that the host need not wait for it; a failed search leaves mu0v as it
// was (the previous mu0).  A preset value (not NaN) is stored without a search.  fw (2 nk8): the
// Fermi factors of the slabs at that mu0.
template <int K>
__global__ void __launch_bounds__(1024) k_mu0_root(const double* __restrict__ ekw, const double* __restrict__ wq,
                                                   long nk8, double Nk2, double T, double dens, double preset,
                                                   double* out, double* mu0v, double* fw)
{
    __shared__ double sc[3 * 16];
    double e[K], w[K];
#pragma unroll
    for (int k = 0; k < K; k++) {
        const long i = threadIdx.x + (long)k * blockDim.x;
        e[k] = (i < nk8) ? ekw[i] : 0.0;
        w[k] = (i < nk8) ? 2.0 * wq[i] / Nk2 : 0.0;
    }
    const double iT = 1.0 / T;
    // f = 1/(e^{-|x|/T} + 1) / N^2 (x = eps - mu0) and f2 = (e^{-x/T} or 1) f^2 / (T N^2): the parts of
    // G0, h and f0 that do not depend on tau, once per mu0 for all the slabs
    auto weights = [&](double mu) {
#pragma unroll
        for (int k = 0; k < K; k++) {
            const long i = threadIdx.x + (long)k * blockDim.x;
            if (i < nk8) {
                const double x = e[k] - mu, ex = exp(-fabs(x) / T), f = 1.0 / (ex + 1.0);
                fw[i] = f / Nk2;
                fw[nk8 + i] = (x > 0 ? ex : 1.0) * f * f / (T * Nk2);
            }
        }
    };
    if (!isnan(preset)) {
        if (threadIdx.x == 0) {
            out[0] = 1.0;
            out[1] = preset;
            out[2] = 0.0;
            *mu0v = preset;
        }
        weights(preset);
        return;
    }
    // this thread's part of n(mu), n'(mu), n''(mu); e^{-|x|/T} so that the reciprocal's argument stays within 1..2
    auto density3 = [&](double mup, double* v) {
#pragma unroll
        for (int k = 0; k < K; k++) {
            const double x = e[k] - mup, ex = exp(-fabs(x) * iT), r = rcp_nr(1.0 + ex);
            const double f = (x > 0) ? ex * r : r, g = f * (1.0 - f) * iT;
            v[0] += w[k] * f;
            v[1] += w[k] * g;
            v[2] += w[k] * g * (1.0 - 2.0 * f) * iT;
        }
    };
    const HalleyState hs = search_block(halley_start(0.0, -8.0, 8.0, 60, -dens, 0.0), 60, density3);
    bool ok = hs.status == kRootConverged;
    double root = hs.root;
    int ne = hs.ne;
    if (!ok) {
        int nb = 0;
        auto density = [&](double mup) {
            double v[3] = {0.0, 0.0, 0.0};
            density3(mup, v);
            block_sum_k<3>(v, sc);
            return v[0] - dens;
        };
        ok = bracket_root(density, 0.0, -8.0, 8.0, nullptr, 1.0e-16, &root, &nb);
        ne += nb;
    }
    weights(ok ? root : *mu0v);
    if (threadIdx.x == 0) {
        out[0] = ok ? 1.0 : 0.0;
        out[1] = root;
        out[2] = ne;
        if (ok) *mu0v = root;
    }
}

// ================================================================== vertex V(r,tau)
// chi.cpp:85-119, block j = iqn index
template <int N, typename S>
__global__ void __launch_bounds__(SlabShape<N>::NT, slab_occ<S>())
    k_vertex_slab(const unsigned* __restrict__ wt, const double* __restrict__ chi, S* V, double normFact, double U, double Usp, double Uch,
                  const double* __restrict__ dsc)
{
    if (dsc) {
        Usp = dsc[kPscUsp + 1];
        Uch = dsc[kPscUch + 1];
    }
    constexpr int nk = N / 2 + 1;
    constexpr long nk8 = (long)nk * (nk + 1) / 2;
    extern __shared__ double smem[];
    S* slab = (S*)smem;
    auto* tw = slab_tw<N>(slab);
    fill_twiddles<N>(tw);
    const long j = blockIdx.x;
    each_wedge<N>(wt, [&](int a, int b, int i) {
        const double c = chi[i + j * nk8];
        const double csp = c / (1.0 - Usp * c / 2.0), cch = c / (1.0 + Uch * c / 2.0);
        slab[a] = slab[b] = (S)(normFact * U * (3.0 * Usp * (csp - c) + Uch * (cch - c)) / 8.0);
    });
    __syncthreads();
    slab_r2r_2d<S, N, 0>(slab, tw);
    each_wedge<N>(wt, [&](int a, int, int i) { V[i + j * nk8] = slab[a]; });
}

// ================================================================== self-energy
// Sigma_inf = -(Sigma(k=0,0) + Sigma(k=0,beta)) (green.cpp:1996); one thread
// Boundary data of Sigma(k,tau) in FP64, block b: side = b % 2 (0: tau = 0, 1: tau = beta),
// pass = b / 2: the slope dSigma/dtau (pass 0, green.cpp:1743-1817) or the value
// Sigma(k,tau_b) = DCT[G0(r,tau_b) V(r,0)] (pass 1, green.cpp:1822-1892 at j = 0, Nw;
// V(r,beta) = V(r,0)).  Each block transforms G0(k,tau_b) to r itself (the two passes of a
// side run side by side: two transforms in a row per block instead of three).
// G0(k,0+) = -1/(e^{-x/T}+1) and G0(k,beta-) = -1/(e^{x/T}+1), both over N^2.
template <int N>
__global__ void __launch_bounds__(SlabShape<N>::NT)
    k_sigma_bnd(const unsigned* __restrict__ wt, const double* __restrict__ ekw, const double* __restrict__ fw,
                const double* __restrict__ er, const double* __restrict__ V0, const double* __restrict__ dchirt0,
                const double* __restrict__ dGrt0p, double mu0, double T, double fact, double* dSig, double* Sb,
                const double* __restrict__ mu0p, double U, const double* __restrict__ dsc)
{
    if (mu0p) mu0 = *mu0p;
    if (dsc) fact = vfact(U, dsc[kPscUsp + 1], dsc[kPscUch + 1], 8.0);
    constexpr int nk = N / 2 + 1;
    constexpr long nk8 = (long)nk * (nk + 1) / 2;
    extern __shared__ double smem[];
    double* slab = smem;
    cd* tw = slab_tw<N>(slab);
    fill_twiddles<N>(tw);
    const int side = blockIdx.x & 1, pass = blockIdx.x >> 1;
    const double t = side ? 1.0 / T : 0.0, bt = side ? 0.0 : 1.0 / T;
    each_wedge<N>(wt, [&](int a, int b, int i) { slab[a] = slab[b] = -g0_exp(ekw[i] - mu0, t, bt) * fw[i]; });
    __syncthreads();
    slab_r2r_2d<double, N, 0>(slab, tw);
    each_wedge<N>(wt, [&](int a, int b, int i) {
        const double g = slab[a];
        const double v = V0[i];
        double r;
        if (pass == 1)
            r = g * v;
        else if (side == 0)
            r = fact * dchirt0[i] * g + v * dGrt0p[i];
        else {
            const double xi = (i == 0) ? -mu0 : er[i];
            r = -fact * dchirt0[i] * g + v * (-dGrt0p[i] + xi);
        }
        slab[a] = slab[b] = r;
    });
    __syncthreads();
    slab_r2r_2d<double, N, 0>(slab, tw);
    double* o = (pass == 0) ? dSig : Sb;
    each_wedge<N>(wt, [&](int a, int, int i) { o[i + side * nk8] = slab[a]; });
}

// Sigma(k,tau_j), j = 0..Nw (green.cpp:1822-1892): G0(k,tau) -> r, x V(r,|tau|), -> k
template <int N, typename S>
__global__ void __launch_bounds__(SlabShape<N>::NT, slab_occ<S>())
    k_sigma_slab(const unsigned* __restrict__ wt, const double* __restrict__ ekw, const double* __restrict__ fw,
                 const S* __restrict__ V, double mu0, double T, int Nw, S* Stau, const double* __restrict__ mu0p)
{
    if (mu0p) mu0 = *mu0p;
    constexpr int nk = N / 2 + 1;
    constexpr long nk8 = (long)nk * (nk + 1) / 2;
    extern __shared__ double smem[];
    S* slab = (S*)smem;
    auto* tw = slab_tw<N>(slab);
    fill_twiddles<N>(tw);
    const int j = blockIdx.x;
    const int nwb = Nw / 2 + 1;
    const int jv = (j < nwb) ? j : Nw - j;
    const double t = j / (Nw * T), bt = 1.0 / T - t;
    each_wedge<N>(wt, [&](int a, int b, int i) { slab[a] = slab[b] = (S)(-g0_exp(ekw[i] - mu0, t, bt) * fw[i]); });
    S v[wedge_per_thread<N>()];  // V(r,|tau|) of the thread's points, in flight during the transform
    load_wedge<N>(V + (long)jv * nk8, v);
    __syncthreads();
    slab_r2r_2d<S, N, 0>(slab, tw);
    each_wedge_slot<N>(wt, [&](int a, int b, int, int c) { slab[a] = slab[b] = slab[a] * v[c]; });
    __syncthreads();
    slab_r2r_2d<S, N, 0>(slab, tw);
    S* o = Stau + (long)j * nk8;
    each_wedge<N>(wt, [&](int a, int, int i) { o[i] = slab[a]; });
}

// phase tables of the pencil transforms, evaluated from the same double arguments as the
// reference: twX[j] = exp(i j pi/L) (green.cpp:1957, cond_opt.cpp:3290); twS[j] = 1 -
// exp(i a_j pi/L) with a_j = 2j+1 (j < L/2) or 2(j-L)+1 (green.cpp:2006,
// cond_opt.cpp:3305-3310); twM[n] = 1 - exp(-2 n i pi/L) (cond_opt.cpp:3731,3805);
// ph[j] = exp(i (j pi (L-1))/L) (cond_opt.cpp:3635), ph[L] = exp(i pi (L-1)) (:3693);
// tw4[n] = 4 sin^2((2n+1) pi/(2L)), n < L/2
__global__ void k_fill_tables(int L, cd* twX, cd* twS, cd* twM, double* tw4, cd* ph)
{
    const int j = blockIdx.x * blockDim.x + threadIdx.x;
    if (j < L) {
        twX[j] = cis(j * kPi / L);
        const double a = (j < L / 2) ? (2 * j + 1) * kPi / L : (2 * (j - L) + 1) * kPi / L;
        const cd e = cis(a);
        twS[j] = cd{1.0 - e.x, -e.y};
        const cd em = cis(-2 * j * kPi / L);
        twM[j] = cd{1.0 - em.x, -em.y};
        ph[j] = cis((j * kPi * (L - 1)) / L);
        if (j < L / 2) {
            const double sh = 2.0 * sin((2 * j + 1) * kPi / (2 * L));
            tw4[j] = sh * sh;
        }
    }
    if (j == L) ph[L] = cis(kPi * (L - 1));
}

// ================================================================== traces

// Trace reductions over (k, n).  Sigma(k,iwn) is stored point-major, Self[k*(Nw/2) + n], so
// one wavefront takes one wedge point and its lanes walk the frequencies (coalesced); a block
// of 256 threads covers 4 wedge points and writes one partial per value, summed afterwards
// in a fixed order (k_finalize, k_finalize_k).
constexpr int kTraceK = 4;  // wedge points per trace block

// traceDiffG(pmu) partials (green.cpp:3108-3182), n = 0..Nw
template <typename SelfT>
__global__ void __launch_bounds__(256)
    k_trace_diffG(const double* __restrict__ ekw, const double* __restrict__ wq, const SelfT* __restrict__ Self,
                  const double* __restrict__ Sinf2, const double* __restrict__ Sinf3,
                  const double* __restrict__ Sinf4, const double* __restrict__ Sinf, int nk8, int Nw, double T,
                  double mu0, double pmu, double* part)
{
    __shared__ double sc[16];
    const int lane = threadIdx.x & 63;
    const int q = blockIdx.x * kTraceK + (threadIdx.x >> 6);
    const int H = Nw / 2;
    double acc = 0.0;
    if (q < nk8) {
        const double Si = Sinf[0];
        const double e = ekw[q], w = 2.0 * wq[q];
        const double s2 = Sinf2[q], s3 = Sinf3[q], s4 = Sinf4[q];
        const SelfT* Sq = Self + (long)q * H;
        for (int j = lane; j <= Nw; j += 64) {
            const double wn = (2 * j + 1) * kPi * T;
            double rS, iS;
            if (j >= H) {
                rS = -s2 / (wn * wn) + s4 / (wn * wn * wn * wn);
                iS = -Si / wn + s3 / (wn * wn * wn);
            } else {
                const cd s = sigma_kw(Sq, j, Si, s2, s3, wn);
                rS = s.x;
                iS = s.y;
            }
            const double tmp = w / (((wn - iS) * (wn - iS) + (e - pmu + rS) * (e - pmu + rS)) *
                                    (wn * wn + (e - mu0) * (e - mu0)));
            acc += tmp * ((mu0 - pmu + rS) * (e - pmu + rS) * (e - mu0) + iS * (iS - 2 * wn) * (e - mu0) -
                          wn * wn * (mu0 - pmu + rS));
        }
    }
    acc = block_sum(acc, sc);
    if (threadIdx.x == 0) part[blockIdx.x] = acc;
}

// traceDiffG and its first two derivatives with respect to pmu.  With a = e - pmu + Re Sigma,
// b = wn - Im Sigma: Re G = -a/(a^2+b^2), d/dpmu Re G = (b^2-a^2)/(a^2+b^2)^2,
// d2/dpmu2 Re G = (6ab^2 - 2a^3)/(a^2+b^2)^3.  Partials part[k * nblk + blk], k = 0, 1, 2.
// A lane sums its frequencies j = lane, lane + 64, ... in increasing j: the stored ones
// (j < Nw/2) in batches of kTD loads issued before any use, then the asymptotic ones.
constexpr int kTD = 4;
__device__ __forceinline__ void trace_diffG3_term(double wn, double rS, double iS, double e, double c, double w,
                                                  double mu0, double pmu, double acc[3])
{
    const double a = e - pmu + rS, b = wn - iS;
    const double a2 = a * a, b2 = b * b, r = rcp_nr(a2 + b2);
    const double r0 = rcp_nr(wn * wn + c * c);
    // Re G - Re G0 = [c (a^2+b^2) - a (c^2+wn^2)] r r0, written without cancellation
    acc[0] += w * r * r0 * ((mu0 - pmu + rS) * a * c + iS * (iS - 2 * wn) * c - wn * wn * (mu0 - pmu + rS));
    acc[1] += w * (b2 - a2) * r * r;
    acc[2] += w * (6.0 * a * b2 - 2.0 * a * a2) * r * r * r;
}
// f(j, Sq[j]) for the stored frequencies j = lane, lane + 64, ... < H of a wavefront, in batches of kTD loads issued
// before any use
template <typename SelfT, typename Fn>
__device__ __forceinline__ void each_stored(const SelfT* __restrict__ Sq, int H, int lane, Fn&& f)
{
    int j = lane;
    for (; j + (kTD - 1) * 64 < H; j += kTD * 64) {
        SelfT v[kTD];
#pragma unroll
        for (int u = 0; u < kTD; u++) v[u] = Sq[j + u * 64];
#pragma unroll
        for (int u = 0; u < kTD; u++) f(j + u * 64, v[u]);
    }
    for (; j < H; j += 64) f(j, Sq[j]);
}
// pmu (and T, mu0) come from the root search st, so that a captured pass graph serves every
// point; a settled search leaves nothing to do.  ticket != null: the workgroup that finishes
// last takes the Halley step.
template <typename SelfT>
__global__ void __launch_bounds__(256)
    k_trace_diffG3(const double* __restrict__ ekw, const double* __restrict__ wq, const SelfT* __restrict__ Self,
                   const double* __restrict__ Sinf2, const double* __restrict__ Sinf3,
                   const double* __restrict__ Sinf4, const double* __restrict__ Sinf, int nk8, int Nw,
                   HalleyState* st, double* part, unsigned* ticket, double* mirror)
{
    __shared__ double sc[3 * 4];
    if (st->status != kRootRunning) return;
    const double pmu = st->x, T = st->T, mu0 = st->mu0;
    const int lane = threadIdx.x & 63;
    const int H = Nw / 2;
    double acc[3] = {0.0, 0.0, 0.0};
    const int q = blockIdx.x * kTraceK + (threadIdx.x >> 6);
    if (q < nk8) {
        const double Si = Sinf[0];
        const double e = ekw[q], w = 2.0 * wq[q];
        const double s2 = Sinf2[q], s3 = Sinf3[q], s4 = Sinf4[q];
        const double c = e - mu0;
        each_stored(Self + (long)q * H, H, lane, [&](int j, SelfT raw) {
            const double wn = (2 * j + 1) * kPi * T;
            const cd s = sigma_kw(&raw, 0, Si, s2, s3, wn);
            trace_diffG3_term(wn, s.x, s.y, e, c, w, mu0, pmu, acc);
        });
        for (int j = lane + ((H - lane + 63) / 64) * 64; j <= Nw; j += 64) {
            const double wn = (2 * j + 1) * kPi * T;
            const double iw = rcp_nr(wn), iw2 = iw * iw;
            trace_diffG3_term(wn, (-s2 + s4 * iw2) * iw2, (-Si + s3 * iw2) * iw, e, c, w, mu0, pmu, acc);
        }
    }
    block_sum_k<3>(acc, sc);
    if (ticket) {
        if (last_workgroup(ticket, gridDim.x, blockIdx.x, acc, part))
            halley_step_block(part, gridDim.x, st, mirror, sc);
    } else if (threadIdx.x == 0) {
        for (int k = 0; k < 3; k++) part[(long)k * gridDim.x + blockIdx.x] = acc[k];
    }
}
// The whole search in one workgroup: Sigma and the weights of the nk8 (Nw + 1) <= CN * 1024 terms, CN per thread
template <int CN, typename SelfT>
__global__ void __launch_bounds__(kSearchThreads)
    k_mu_search(const double* __restrict__ ekw, const double* __restrict__ wq, const SelfT* __restrict__ Self,
                const double* __restrict__ Sinf2, const double* __restrict__ Sinf3, const double* __restrict__ Sinf4,
                const double* __restrict__ Sinf, int nk8, int Nw, HalleyState* st, RootInit in, double* mirror,
                int npass)
{
    const HalleyState s0 = halley_begin(in);
    const double Si = Sinf[0];
    const int H = Nw / 2;
    double wn[CN], rS[CN], iS[CN], e[CN], w[CN];
#pragma unroll
    for (int u = 0; u < CN; u++) {
        const int i = threadIdx.x + u * kSearchThreads, q = i / (Nw + 1), j = i - q * (Nw + 1);
        wn[u] = (2 * j + 1) * kPi * s0.T;
        rS[u] = iS[u] = e[u] = w[u] = 0.0;
        if (q < nk8) {
            e[u] = ekw[q];
            w[u] = 2.0 * wq[q];
            if (j < H) {
                const cd s = sigma_kw(Self + (long)q * H, j, Si, Sinf2[q], Sinf3[q], wn[u]);
                rS[u] = s.x;
                iS[u] = s.y;
            } else {
                const double iw = rcp_nr(wn[u]), iw2 = iw * iw;
                rS[u] = (-Sinf2[q] + Sinf4[q] * iw2) * iw2;
                iS[u] = (-Si + Sinf3[q] * iw2) * iw;
            }
        }
    }
    const HalleyState r = search_block(s0, npass, [&](double pmu, double* acc) {
#pragma unroll
        for (int u = 0; u < CN; u++)
            trace_diffG3_term(wn[u], rS[u], iS[u], e[u], e[u] - s0.mu0, w[u], s0.mu0, pmu, acc);
    });
    search_end(r, st, mirror);
}

// Tr Sigma G0 (green.cpp:3018-3084) in one pass over Sigma: part[b] its main sum, part[nblk + b] the Sigma_inf correction
// (the n < Nw/2 terms plus one per k).  256^2 x 2048: 24 us mixed, 50 FP64 (a pass each: 2 x 27, 2 x 53)
template <typename SelfT>
__global__ void __launch_bounds__(256)
    k_trace_selfG0(const double* __restrict__ ekw, const double* __restrict__ wq, const SelfT* __restrict__ Self,
                   const double* __restrict__ Sinf2, const double* __restrict__ Sinf3, const double* __restrict__ Sinf,
                   int nk8, int Nw, double T, double mu0, double nk02, double* part)
{
    __shared__ double sc[2 * 4];
    const int lane = threadIdx.x & 63;
    const int q = blockIdx.x * kTraceK + (threadIdx.x >> 6);
    double acc[2] = {0.0, 0.0};
    if (q < nk8) {
        const double Si = Sinf[0], s2 = Sinf2[q], s3 = Sinf3[q];
        const double x = ekw[q] - mu0, w = wq[q] / nk02;
        each_stored(Self + (long)q * (Nw / 2), Nw / 2, lane, [&](int j, SelfT raw) {
            const double wn = (2 * j + 1) * kPi * T;
            const cd s = sigma_kw(&raw, 0, Si, s2, s3, wn);
            const double r = rcp_nr(wn * wn + x * x);
            acc[0] += r * (s.y * wn - s.x * x);
            acc[1] += r;
        });
        acc[0] *= w * T * 2;
        acc[1] *= w * Si * T * 2;
        if (lane == 0) {
            if (fabs(x) > 1.0e-12)
                acc[1] += w * Si * (1.0 / (exp(x / T) + 1.0) - 0.5) / x;
            else {
                const double ex = x < 0 ? exp(x / T) : exp(-x / T);
                acc[1] -= w * Si * ex / ((ex + 1.0) * (ex + 1.0) * T);
            }
        }
    }
    block_sum_k<2>(acc, sc);
    if (threadIdx.x == 0) {
        part[blockIdx.x] = acc[0];
        part[gridDim.x + blockIdx.x] = acc[1];
    }
}
// Tr Sigma G (green.cpp:2944-2976)
template <typename SelfT>
__global__ void __launch_bounds__(256)
    k_trace_selfG(const double* __restrict__ ekw, const double* __restrict__ wq, const SelfT* __restrict__ Self,
                  const double* __restrict__ Sinf2, const double* __restrict__ Sinf3, const double* __restrict__ Sinf,
                  int nk8, int Nw, double T, double mu, double nk02, double* part)
{
    __shared__ double sc[16];
    const int lane = threadIdx.x & 63;
    const int q = blockIdx.x * kTraceK + (threadIdx.x >> 6);
    double acc = 0.0;
    if (q < nk8) {
        const double Si = Sinf[0], s2 = Sinf2[q], s3 = Sinf3[q];
        const double x = ekw[q] - mu;
        each_stored(Self + (long)q * (Nw / 2), Nw / 2, lane, [&](int j, SelfT raw) {
            const double wn = (2 * j + 1) * kPi * T;
            const cd s = sigma_kw(&raw, 0, Si, s2, s3, wn);
            const double a = x + s.x, b = wn - s.y;
            acc += rcp_nr(a * a + b * b) * (s.y * b - s.x * a);
        });
        acc *= wq[q] * T * 2 / nk02;
    }
    acc = block_sum(acc, sc);
    if (threadIdx.x == 0) part[blockIdx.x] = acc;
}

// column sums of a row-major (nrows x ncols) partial table in a fixed order: a block of
// 16 columns (a cache line) x 64 row groups, row group partials added in order.  Bound by latency: ~1024 rows of few
// columns, so a thread's 16 rows are loaded at once (k_reduce_cols2
// at 128^2 x 1024 and 256^2 x 2048: 6.3, 7.2 us; 64 columns x 16 groups, one load after the other: 14, 20 us).
constexpr int kRedCols = 16, kRedRows = 1024 / kRedCols;
__device__ __forceinline__ void reduce_cols_block(const double* __restrict__ part, int nrows, int ncols, double* out,
                                                  int blk)
{
    __shared__ double t[kRedRows][kRedCols + 1];
    const int cx = threadIdx.x % kRedCols, ry = threadIdx.x / kRedCols;
    const int c = blk * kRedCols + cx;
    double a = 0.0;
    if (c < ncols)
        for (int r = ry; r < nrows; r += 16 * kRedRows) {
            double v[16];
#pragma unroll
            for (int u = 0; u < 16; u++) {
                const int rr = r + u * kRedRows;
                v[u] = (rr < nrows) ? part[(long)rr * ncols + c] : 0.0;
            }
#pragma unroll
            for (int u = 0; u < 16; u++) a += v[u];
        }
    t[ry][cx] = a;
    __syncthreads();
    if (ry == 0 && c < ncols) {
        double sum = 0.0;
#pragma unroll
        for (int i = 0; i < kRedRows; i++) sum += t[i][cx];
        out[c] = sum;
    }
}

__global__ void __launch_bounds__(1024) k_reduce_cols(const double* __restrict__ part, int nrows, int ncols,
                                                      double* out)
{
    reduce_cols_block(part, nrows, ncols, out, blockIdx.x);
}
// row ranges of one table (blockIdx.y < nbins), then all rows of another of four columns
__global__ void __launch_bounds__(1024) k_reduce_bins(const double* __restrict__ part, int ncols,
                                                      const int* __restrict__ row0, int nbins, double* out,
                                                      const double* __restrict__ scal, int nrows, double* oscal)
{
    const int b = blockIdx.y;
    if (b < nbins)
        reduce_cols_block(part + (long)row0[b] * ncols, row0[b + 1] - row0[b], ncols, out + (long)b * ncols,
                          blockIdx.x);
    else if (blockIdx.x == 0)
        reduce_cols_block(scal, nrows, 4, oscal, 0);
}
// two tables of the same row count in one launch (blocks of the first, then of the second);
// block 0 also copies ncopy doubles from csrc to cdst (null: nothing)
__global__ void __launch_bounds__(1024) k_reduce_cols2(const double* __restrict__ p1, int ncols1, double* o1,
                                                       const double* __restrict__ p2, int ncols2, double* o2,
                                                       int nrows, const double* __restrict__ csrc, int ncopy,
                                                       double* cdst)
{
    const int b1 = (ncols1 + kRedCols - 1) / kRedCols;
    if ((int)blockIdx.x < b1)
        reduce_cols_block(p1, nrows, ncols1, o1, blockIdx.x);
    else
        reduce_cols_block(p2, nrows, ncols2, o2, blockIdx.x - b1);
    if (csrc && blockIdx.x == 0)
        for (int i = threadIdx.x; i < ncopy; i += blockDim.x) cdst[i] = csrc[i];
}

// dispersion tables on the device (hamiltonien.cpp:49-68,125-155; green0 wedge weights).  wt[w]: the slab
// offsets of wedge point (l, m) (low half) and of (m, l) (high half), line stride LD.  vw, vw + nk8:
// v_x at (kx, ky) = (l, m) and (m, l), 0 at kx = 0 and pi, for the Lambda slabs.  Bound by the latency of the sines
// and cosines: four pairs per point serve every table (3.5 - 5.0 us; evaluated per table 7.8 - 11.8).
__global__ void k_model(int N, int LD, double t, double tp, double tpp, double t3, double* ek, double* ekw, double* wq,
                        double* er, double* d2ek, double* dek, unsigned* wt, double* vw)
{
    const int nk = N / 2 + 1;
    const long nk8 = (long)nk * (nk + 1) / 2;
    const long i = blockIdx.x * (long)blockDim.x + threadIdx.x;
    const double dk = kPi / (nk - 1);
    auto vx = [&](double sx, double s2x, double cy, double c2y) {
        return 2.0 * t * sx + 4.0 * tp * sx * cy + 4.0 * tpp * s2x + 4 * t3 * (2.0 * s2x * cy + c2y * sx);
    };
    if (i < (long)nk * nk) {
        const int l = (int)(i / nk), m = (int)(i % nk);
        const double kx = l * dk, ky = m * dk;
        double sx, cx, sy, cy, s2x, c2x, s2y, c2y;
        sincos(kx, &sx, &cx);
        sincos(ky, &sy, &cy);
        sincos(2 * kx, &s2x, &c2x);
        sincos(2 * ky, &s2y, &c2y);
        ek[i] = -2.0 * t * (cx + cy) - 4.0 * tp * cx * cy - 2.0 * tpp * (c2x + c2y) - 4 * t3 * (c2x * cy + c2y * cx);
        d2ek[i] = 2.0 * t * cx + 4.0 * tp * cx * cy + 8.0 * tpp * c2x + 4 * t3 * (4.0 * c2x * cy + c2y * cx);
        if (m <= l) {
            const long w = widx(l, m);
            ekw[w] = ek[i];
            wq[w] = wedge_weight(l, m, nk);
            er[w] = (w == 1) ? -t : (w == 2) ? -tp : (w == 3) ? -tpp : (w == 4) ? -t3 : 0.0;
            wt[w] = (unsigned)(m + l * LD) | ((unsigned)(l + m * LD) << 16);
            vw[w] = (l >= 1 && l <= nk - 2) ? vx(sx, s2x, cy, c2y) : 0.0;
            vw[nk8 + w] = (m >= 1 && m <= nk - 2) ? vx(sy, s2y, cx, c2x) : 0.0;
        }
        if (l >= 1 && l <= nk - 2) dek[i - nk] = vx(sx, s2x, cy, c2y);
    }
}

// ================================================================== Lambda_jj slabs
// The Lambda integrands h (which = 0) and f0 (1) of cond_opt.cpp:2697-2735, 2795-2827 at one tau without
// the velocity: with E = g0_exp(x, t, beta - t), fw = f/N^2 and fw2 = (e^{-x/T} or 1) f^2/(T N^2)
// (k_mu0_root), h = v E fw and f0 = v E (t fw - fw2).
__device__ __forceinline__ double lam_val(int which, double E, double t, double fw, double fw2)
{
    return E * (which == 0 ? fw : t * fw - fw2);
}

// Boundary data of hV and f0V in FP64 (cond_opt.cpp:2697-2735, 2745-3114 at tau = 0, beta).
// Block b: which = (b/2)%2 (0: h, 1: f0), side = b%2 (0: tau = 0, 1: tau = beta), part = b/4:
//   (1) h(r,tau_b) (or f0) by DST x DCT of the k-space integrand at t = 0 or beta
//   part 1: (2) the tau-derivative integrand -> r, combined with V(r,0), dchi0(r,0) -> k:
//       slopes dhV / df0V (cond_opt.cpp:2745-3014); dh/dtau = -x h, df0/dtau = -x f0 + h
//   part 0: (3) 2 h(r,tau_b) V(r,0) -> k: hVb / f0Vb, the tau = 0, beta values of hV / f0V
// Both parts of a (which, side) run (1) themselves and then side by side: three transforms in
// a row per block instead of four.  Independent of the tau slabs.
template <int N>
__global__ void __launch_bounds__(SlabShape<N>::NT)
    k_hf0_bnd(const unsigned* __restrict__ wt, const double* __restrict__ ekw, const double* __restrict__ fw,
              const double* __restrict__ vw, const double* __restrict__ V0, const double* __restrict__ dchirt0,
              double mu0, double T, double fact4, double* dhV, double* df0V, double* hVb, double* f0Vb,
              const double* __restrict__ mu0p, double U, const double* __restrict__ dsc)
{
    if (mu0p) mu0 = *mu0p;
    if (dsc) fact4 = vfact(U, dsc[kPscUsp + 1], dsc[kPscUch + 1], 4.0);
    constexpr int nk = N / 2 + 1;
    constexpr long nq = (long)nk * (nk - 2);
    constexpr int nk8 = nk * (nk + 1) / 2;
    extern __shared__ double smem[];
    double* slab = smem;
    cd* tw = slab_tw<N>(slab);
    fill_twiddles<N>(tw);
    const int which = (blockIdx.x >> 1) & 1, side = blockIdx.x & 1, part = blockIdx.x >> 2;
    const double t = side ? 1.0 / T : 0.0, bt = side ? 0.0 : 1.0 / T;
    // (1)
    each_wedge<N>(wt, [&](int a, int b, int i) {
        const double g = lam_val(which, g0_exp(ekw[i] - mu0, t, bt), t, fw[i], fw[nk8 + i]);
        slab[a] = g * vw[i];
        slab[b] = g * vw[nk8 + i];
    });
    __syncthreads();
    slab_r2r_2d<double, N, 1>(slab, tw);
    if (part == 0) {
        // (3), from h(r,tau_b) in place
        each_wedge<N>(wt, [&](int a, int b, int i) {
            const double v = 2.0 * V0[i], ha = slab[a] * v, hb = slab[b] * v;
            slab[a] = ha;
            slab[b] = hb;
        });
        __syncthreads();
        slab_r2r_2d<double, N, 1>(slab, tw);
        double* ob = ((which == 0) ? hVb : f0Vb) + side * nq;
        each_lambda<N>([&](int l, int m, int s) { ob[s] = slab[at<N>(l + 1, m)]; });
        return;
    }
    double ha[wedge_per_thread<N>()], hb[wedge_per_thread<N>()];  // h(r,tau_b) of the thread's points
    each_wedge_slot<N>(wt, [&](int a, int b, int, int c) {
        ha[c] = slab[a];
        hb[c] = slab[b];
    });
    __syncthreads();
    // (2)
    each_wedge<N>(wt, [&](int a, int b, int i) {
        const double x = ekw[i] - mu0, E = g0_exp(x, t, bt);
        double g = -x * lam_val(which, E, t, fw[i], fw[nk8 + i]);
        if (which == 1) g += E * fw[i];
        slab[a] = g * vw[i];
        slab[b] = g * vw[nk8 + i];
    });
    __syncthreads();
    slab_r2r_2d<double, N, 1>(slab, tw);
    const double sf = (side == 0) ? fact4 : -fact4;
    each_wedge_slot<N>(wt, [&](int a, int b, int i, int c) {
        const double v = 2.0 * V0[i], f = sf * dchirt0[i];
        const double ra = slab[a] * v + ha[c] * f, rb = slab[b] * v + hb[c] * f;
        slab[a] = ra;
        slab[b] = rb;
    });
    __syncthreads();
    slab_r2r_2d<double, N, 1>(slab, tw);
    double* o = ((which == 0) ? dhV : df0V) + side * nq;
    each_lambda<N>([&](int l, int m, int s) { o[s] = slab[at<N>(l + 1, m)]; });
}

// hV(k,tau_j) = DST x DCT [2 h(r,tau_j) V(r,|tau_j|)] with h(r,tau_j) = DST x DCT [h(k,tau_j)]
// (RODFT00 along kx, REDFT00 along ky; cond_opt.cpp:2697-2735, 2795-2827, 3029-3114), or f0V for
// which = 1, j = 1 .. Nw-1 (the end slices come from k_hf0_bnd).  h and f0 stay in LDS.  The pointwise
// phases run over the wedge: one exponential serves (kx, ky) and (ky, kx), and V(r) is read in order.
// Bound by the two transforms (VALU and LDS).  At 256^2 x 2048 the h and f0 slices took 976 + 844 us (FP64)
// and 628 + 399 us (FP32) as two kernels with h, f0 in global memory between them, two exponentials and
// two divisions per point and index; now 2 x 445 and 2 x 290 us beside the self-energy kernels (FP32 alone: 195).
template <int N, typename S>
__global__ void __launch_bounds__(SlabShape<N>::NT, slab_occ<S>())
    k_hV_slab(const unsigned* __restrict__ wt, const double* __restrict__ ekw, const double* __restrict__ fw,
              const double* __restrict__ vw, const double* __restrict__ mu0p, double T, int Nw,
              const S* __restrict__ V, int which, S* out)
{
    const double mu0 = *mu0p;
    constexpr int nk = N / 2 + 1;
    constexpr long nq = (long)nk * (nk - 2);
    constexpr int nk8 = nk * (nk + 1) / 2;
    extern __shared__ double smem[];
    S* slab = (S*)smem;
    auto* tw = slab_tw<N>(slab);
    fill_twiddles<N>(tw);
    const int j = blockIdx.x + 1;
    const int jv = (j > Nw / 2) ? Nw - j : j;
    const double t = (double)j / (T * Nw), bt = 1.0 / T - t;
    each_wedge<N>(wt, [&](int a, int b, int i) {
        const double g = lam_val(which, g0_exp(ekw[i] - mu0, t, bt), t, fw[i], fw[nk8 + i]);
        slab[a] = (S)(g * vw[i]);
        slab[b] = (S)(g * vw[nk8 + i]);
    });
    S v[wedge_per_thread<N>()];  // V(r,|tau|) of the thread's points, in flight during the transform
    load_wedge<N>(V + (long)jv * nk8, v);
    __syncthreads();
    slab_r2r_2d<S, N, 1>(slab, tw);
    each_wedge_slot<N>(wt, [&](int a, int b, int, int c) {
        const S va = (S)2 * slab[a] * v[c], vb = (S)2 * slab[b] * v[c];
        slab[a] = va;
        slab[b] = vb;
    });
    __syncthreads();
    slab_r2r_2d<S, N, 1>(slab, tw);
    S* o = out + (long)j * nq;
    each_lambda<N>([&](int l, int m, int s) { o[s] = slab[at<N>(l + 1, m)]; });
}

// ================================================================== transposes
// [j][q] (j < nj, q < nq) -> [q][j]: kTT x kTT tiles through LDS, both sides coalesced (a
// wave moves 64 consecutive elements of one row per access; 16 accesses per thread in flight).
// Rows of odd length (nq = nk (nk - 2), nj = Nw + 1) rule out vector accesses.  The Lambda
// pencils then read each tau-pencil as one contiguous row.  Two arrays per launch (grid z).
constexpr int kTT = 64;
template <typename S>
__global__ void __launch_bounds__(256) k_transpose(const S* __restrict__ in0, S* __restrict__ out0,
                                                   const S* __restrict__ in1, S* __restrict__ out1, long nq, int nj)
{
    const S* __restrict__ in = blockIdx.z ? in1 : in0;  // z: which of the two arrays
    S* __restrict__ out = blockIdx.z ? out1 : out0;
    __shared__ S t[kTT][kTT + 1];
    const long q0 = (long)blockIdx.x * kTT;
    const int j0 = blockIdx.y * kTT;
    const int tx = threadIdx.x & 63, ty = threadIdx.x >> 6;  // 64 x 4
    {
        // all 16 loads issued before the first LDS write
        const long q = q0 + tx;
        S v[kTT / 4];
#pragma unroll
        for (int r = 0; r < kTT / 4; r++) {
            const int j = j0 + ty + 4 * r;
            v[r] = (j < nj && q < nq) ? in[(long)j * nq + q] : S(0);
        }
#pragma unroll
        for (int r = 0; r < kTT / 4; r++) t[ty + 4 * r][tx] = v[r];
    }
    __syncthreads();
    const int j = j0 + tx;
#pragma unroll
    for (int r = 0; r < kTT; r += 4) {
        const long q = q0 + ty + r;
        if (j < nj && q < nq) out[q * nj + j] = t[tx][ty + r];
    }
}

// ================================================================== local Green function
// G_loc(iw_j) = sum over the wedge of (w_k/N^2) / (iw_j - e_k + mu - Sigma(k,iw_j)), j < Nw/2
// (green.cpp:209-266).  Thread = frequency j (Self is point-major, so a warp reads one k's
// row contiguously); blockIdx.y = k chunk: k = y, y + KCH, ...; partials
// part[y*2H + 2j + (0 re, 1 im)], y < kGlocChunks, summed over y in a fixed order by
// k_reduce_cols.
template <typename SelfT>
__global__ void __launch_bounds__(256)
    k_gloc(const double* __restrict__ ekw, const double* __restrict__ wq, const SelfT* __restrict__ Self,
           const double* __restrict__ Sinf2, const double* __restrict__ Sinf3, const double* __restrict__ Sinfp,
           long nk8, int H, double T, double mu, double nk02, double* part)
{
    const int j = blockIdx.x * blockDim.x + threadIdx.x;
    if (j >= H) return;
    const double wn = (2 * j + 1) * kPi * T;
    const double Sinf = Sinfp[0];
    double re = 0.0, im = 0.0;
    for (long k = blockIdx.y; k < nk8; k += gridDim.y) {
        const cd sg = sigma_kw(Self, k * H + j, Sinf, Sinf2[k], Sinf3[k], wn);
        const cd g = (wq[k] / nk02) / cd{mu - ekw[k] - sg.x, wn - sg.y};
        re += g.x;
        im += g.y;
    }
    double* o = part + (long)blockIdx.y * 2 * H;
    o[2 * j] = re;
    o[2 * j + 1] = im;
}

// ================================================================== launchers
// lattice sizes with compiled slab transforms: 2^k (4..256) and 3*2^k (12..192)
bool supported_N(int N)
{
    switch (N) {
        case 4: case 8: case 12: case 16: case 24: case 32: case 48: case 64: case 96: case 128: case 192: case 256:
            return true;
        default:
            return false;
    }
}
bool supported_Nw(int Nw)
{
    return Nw == 16 || Nw == 32 || Nw == 64 || Nw == 128 || Nw == 256 || Nw == 512 || Nw == 1024 || Nw == 2048 ||
           Nw == 4096;
}

#define DISPATCH_N(N, ...)                          \
    switch (N) {                                    \
        case 4: { constexpr int NN = 4; __VA_ARGS__; } break;     \
        case 8: { constexpr int NN = 8; __VA_ARGS__; } break;     \
        case 12: { constexpr int NN = 12; __VA_ARGS__; } break;   \
        case 24: { constexpr int NN = 24; __VA_ARGS__; } break;   \
        case 48: { constexpr int NN = 48; __VA_ARGS__; } break;   \
        case 96: { constexpr int NN = 96; __VA_ARGS__; } break;   \
        case 192: { constexpr int NN = 192; __VA_ARGS__; } break; \
        case 16: { constexpr int NN = 16; __VA_ARGS__; } break;   \
        case 32: { constexpr int NN = 32; __VA_ARGS__; } break;   \
        case 64: { constexpr int NN = 64; __VA_ARGS__; } break;   \
        case 128: { constexpr int NN = 128; __VA_ARGS__; } break; \
        case 256: { constexpr int NN = 256; __VA_ARGS__; } break; \
        default: return hipErrorInvalidValue;       \
    }
// the dynamic-LDS limit of a kernel, raised once to the largest size asked for (the attribute
// holds for the process; each host thread keeps its own record of what it has set)
template <typename K>
static void set_lds(K kern, size_t bytes)
{
    thread_local std::unordered_map<const void*, size_t> done;
    const void* f = reinterpret_cast<const void*>(kern);
    size_t& have = done[f];
    if (have >= bytes) return;
    (void)hipFuncSetAttribute(f, hipFuncAttributeMaxDynamicSharedMemorySize, (int)bytes);
    have = bytes;
}

hipError_t launch_fill_tw(const DevArrays& d, int L, hipStream_t s)
{
    hipLaunchKernelGGL(k_fill_tw, dim3((L + 255) / 256), dim3(256), 0, s, d.twN, L);
    hipLaunchKernelGGL(k_fill_tables, dim3((L + 256) / 256), dim3(256), 0, s, L, d.twX, d.twS, d.twM, d.tw4, d.ph);
    return hipGetLastError();
}

hipError_t launch_chi0_tau0(const Grid& g, const DevArrays& d, hipStream_t s)
{
    const size_t lds = slab_bytes(g.N, sizeof(double));
    DISPATCH_S(g.prec, DISPATCH_N(g.N, {
        set_lds(k_chi0_tau0<NN, SS>, lds);
        hipLaunchKernelGGL((k_chi0_tau0<NN, SS>), dim3(1), dim3(SlabShape<NN>::NT), lds, s, d.wt, d.ekw, d.fw,
                           d.er, d.mu0v, g.T, (SS*)d.chi, (SS*)d.chirt, d.dchirt0, d.dGrt0p, d.dchiqt0, d.chirt0);
    }));
    return hipGetLastError();
}

hipError_t launch_chi0_slab(const Grid& g, const DevArrays& d, hipStream_t s)
{
    DISPATCH_S(g.prec, DISPATCH_N(g.N, {
        constexpr size_t lds = slab_bytes(NN, sizeof(SS));
        set_lds(k_chi0_slab<NN, SS>, lds);
        hipLaunchKernelGGL((k_chi0_slab<NN, SS>), dim3(g.nwb - 1), dim3(SlabShape<NN>::NT), lds, s, d.wt, d.ekw, d.fw,
                           d.mu0v, g.T, g.Nw, (SS*)d.chi, (SS*)d.chirt);
    }));
    return hipGetLastError();
}

hipError_t launch_chi0max(const Grid& g, const DevArrays& d, hipStream_t s, double* out2)
{
    hipLaunchKernelGGL(k_chi0max, dim3(1), dim3(1024), 0, s, d.chiw, g.nk8, d.red, d.imax, out2);
    return hipGetLastError();
}

static dim3 red_grid(const Grid& g) { return dim3((unsigned)((g.nk8 + 255) / 256), kRowGroups); }
static dim3 trace_grid(const Grid& g) { return dim3((unsigned)((g.nk8 + kTraceK - 1) / kTraceK)); }

hipError_t launch_sum_rule(const Grid& g, const DevArrays& d, double sU, double* out, hipStream_t s)
{
    int np = 0;
    const hipError_t e = launch_sum_rule_part(g.N, g.Nw, g.T, d.chiw, d.chi0inf, d.chi0inf2, d.wq, sU, d.part, &np, s);
    if (e != hipSuccess) return e;
    hipLaunchKernelGGL(k_finalize, dim3(1), dim3(256), 0, s, d.part, np, out);
    return hipGetLastError();
}

int sum_rule_parts(int N) { return (int)((((long)(N / 2 + 1) * (N / 2 + 2) / 2) + 255) / 256) * kRowGroups; }

hipError_t launch_sum_rule_part(int N, int Nw, double T, const double* chiw, const double* inf1, const double* inf2,
                                const double* wq, double sU, double* part, int* nparts, hipStream_t s)
{
    const int nk = N / 2 + 1;
    const long nk8 = (long)nk * (nk + 1) / 2;
    const double Nq = 4.0 * (nk - 1) * (nk - 1);
    const dim3 gr((unsigned)((nk8 + 255) / 256), kRowGroups);
    hipLaunchKernelGGL(k_sum_rule, gr, dim3(256), 0, s, chiw, inf1, inf2, wq, (int)nk8, Nw / 2, T, Nq, sU, part);
    *nparts = (int)(gr.x * gr.y);
    return hipGetLastError();
}

hipError_t launch_halley_init(HalleyState* st, const RootInit& in, double* mirror, hipStream_t s)
{
    hipLaunchKernelGGL(k_halley_init, dim3(1), dim3(1), 0, s, st, in, mirror);
    return hipGetLastError();
}

hipError_t launch_sum_rule3_pass(const Grid& g, const DevArrays& d, double sgn, double* mirror, hipStream_t s)
{
    const double Nq = 4.0 * (g.nk - 1) * (g.nk - 1);
    dim3 gr = red_grid(g);
    while (gr.x * gr.y > (unsigned)kSumRuleGrid && gr.y > 1) gr.y /= 2;
    const bool series = d.srm && g.nk8 * g.nwb >= kSRMinElems;  // the moments exist (launch_sr_moments)
    hipLaunchKernelGGL(k_sum_rule3, gr, dim3(256), 0, s, d.chiw, d.chi0inf, d.chi0inf2, d.wq, (int)g.nk8, g.Nw / 2,
                       Nq, sgn, d.root, d.part, d.ticket, mirror, series ? d.srm : nullptr,
                       series ? d.srmax : nullptr);
    return hipGetLastError();
}

hipError_t launch_sum_rule_search(const Grid& g, const DevArrays& d, double sgn, const RootInit& in, double* mirror,
                                  int npass, hipStream_t s)
{
    if (sum_in_one(g)) {
        const long n = g.nk8 * (g.Nw + 1);
        const double Nq = 4.0 * (g.nk - 1) * (g.nk - 1);
#define SUM_SEARCH(CN)                                                                                              \
    hipLaunchKernelGGL(k_sum_rule_search<CN>, dim3(1), dim3(kSearchThreads), 0, s, d.chiw, d.chi0inf, d.chi0inf2,   \
                       d.wq, (int)g.nk8, g.Nw / 2, Nq, sgn, d.root, in, mirror, npass)
        if (n <= 4 * kSearchThreads)
            SUM_SEARCH(4);
        else if (n <= 8 * kSearchThreads)
            SUM_SEARCH(8);
        else
            SUM_SEARCH(kSumOneMax / kSearchThreads);
#undef SUM_SEARCH
        return hipGetLastError();
    }
    hipError_t e = launch_halley_init(d.root, in, mirror, s);
    for (int k = 0; k < npass && e == hipSuccess; k++) e = launch_sum_rule3_pass(g, d, sgn, mirror, s);
    return e;
}

hipError_t launch_sr_moments(const Grid& g, const DevArrays& d, hipStream_t s)
{
    if (!d.srm || g.nk8 * g.nwb < kSRMinElems) return hipSuccess;
    const double Nq = 4.0 * (g.nk - 1) * (g.nk - 1);
    const int nrows = g.Nw + 1;  // 2 nwmax + 1
    if (nrows > 8192) return hipErrorInvalidValue;
    hipLaunchKernelGGL(k_sr_moments, dim3(nrows), dim3(256), 0, s, d.chiw, d.chi0inf, d.chi0inf2, d.wq, (int)g.nk8,
                       g.Nw / 2, Nq, g.T, d.srm, d.srmax);
    hipLaunchKernelGGL(k_sr_suffix, dim3(kSRM + 1), dim3(1024), 0, s, d.srm, d.srmax, nrows);
    return hipGetLastError();
}

hipError_t launch_model(const Grid& g, const DevArrays& d, double t, double tp, double tpp, double t3,
                        hipStream_t s)
{
    const long n = (long)g.nk * g.nk;
    hipLaunchKernelGGL(k_model, dim3((unsigned)((n + 255) / 256)), dim3(256), 0, s, g.N, slab_dims(g.N).LD, t, tp,
                       tpp, t3, d.ek, d.ekw, d.wq, d.er, d.d2ek, d.dek, d.wt, d.vw);
    return hipGetLastError();
}

hipError_t launch_reduce_cols(const double* part, int nrows, int ncols, double* out, hipStream_t s)
{
    hipLaunchKernelGGL(k_reduce_cols, dim3((ncols + kRedCols - 1) / kRedCols), dim3(1024), 0, s, part, nrows, ncols, out);
    return hipGetLastError();
}

hipError_t launch_reduce_bins(const double* part, int ncols, const int* row0, int nbins, double* out, const double* scal,
                              int nrows, double* oscal, hipStream_t s)
{
    hipLaunchKernelGGL(k_reduce_bins, dim3((ncols + kRedCols - 1) / kRedCols, nbins + 1), dim3(1024), 0, s, part, ncols,
                       row0, nbins, out, scal, nrows, oscal);
    return hipGetLastError();
}

hipError_t launch_reduce_cols2(const double* p1, int ncols1, double* o1, const double* p2, int ncols2, double* o2,
                               int nrows, hipStream_t s, const double* csrc, int ncopy, double* cdst)
{
    const unsigned nb = (unsigned)((ncols1 + kRedCols - 1) / kRedCols + (ncols2 + kRedCols - 1) / kRedCols);
    hipLaunchKernelGGL(k_reduce_cols2, dim3(nb), dim3(1024), 0, s, p1, ncols1, o1, p2, ncols2, o2, nrows, csrc, ncopy,
                       cdst);
    return hipGetLastError();
}

hipError_t launch_mu0_root(const Grid& g, const DevArrays& d, double n, double preset, double* out, hipStream_t s)
{
    const double Nk2 = 4.0 * (g.nk - 1) * (g.nk - 1);
    const int K = (g.nk8 <= 1024) ? 1 : (g.nk8 <= 3072) ? 3 : 9;
    const long waves = (g.nk8 + 64L * K - 1) / (64L * K);
    if (waves > 16) return hipErrorInvalidValue;
    auto* const kern = (K == 1) ? k_mu0_root<1> : (K == 3) ? k_mu0_root<3> : k_mu0_root<9>;
    hipLaunchKernelGGL(kern, dim3(1), dim3((unsigned)(64 * waves)), 0, s, d.ekw, d.wq, g.nk8, Nk2, g.T, n, preset, out,
                       d.mu0v, d.fw);
    return hipGetLastError();
}

hipError_t launch_vertex_slab(const Grid& g, const DevArrays& d, double U, double Usp, double Uch, hipStream_t s,
                              const double* dsc)
{
    const double normFact = g.T / ((double)g.N * g.N);
    DISPATCH_S(g.prec, DISPATCH_N(g.N, {
        constexpr size_t lds = slab_bytes(NN, sizeof(SS));
        set_lds(k_vertex_slab<NN, SS>, lds);
        hipLaunchKernelGGL((k_vertex_slab<NN, SS>), dim3(g.nwb), dim3(SlabShape<NN>::NT), lds, s, d.wt, d.chiw, (SS*)d.V,
                           normFact, U, Usp, Uch, dsc);
    }));
    return hipGetLastError();
}

hipError_t launch_sigma_bnd(const Grid& g, const DevArrays& d, double mu0, double fact, hipStream_t s,
                            const double* mu0p, double U, const double* dsc)
{
    const size_t lds = slab_bytes(g.N, sizeof(double));
    DISPATCH_N(g.N, {
        set_lds(k_sigma_bnd<NN>, lds);
        hipLaunchKernelGGL(k_sigma_bnd<NN>, dim3(4), dim3(SlabShape<NN>::NT), lds, s, d.wt, d.ekw, d.fw, d.er, d.V0,
                           d.dchirt0, d.dGrt0p, mu0, g.T, fact, d.dSig, d.Sb, mu0p, U, dsc);
    });
    return hipGetLastError();
}

hipError_t launch_sigma_slab(const Grid& g, const DevArrays& d, double mu0, hipStream_t s, const double* mu0p)
{
    DISPATCH_S(g.prec, DISPATCH_N(g.N, {
        constexpr size_t lds = slab_bytes(NN, sizeof(SS));
        set_lds(k_sigma_slab<NN, SS>, lds);
        hipLaunchKernelGGL((k_sigma_slab<NN, SS>), dim3(g.Nw + 1), dim3(SlabShape<NN>::NT), lds, s, d.wt, d.ekw, d.fw,
                           (const SS*)d.V, mu0, g.T, g.Nw, (SS*)d.Stau, mu0p);
    }));
    return hipGetLastError();
}

hipError_t launch_trace_diffG(const Grid& g, const DevArrays& d, double pmu, double mu0, double* out,
                              hipStream_t s)
{
    const dim3 gr = trace_grid(g);
    DISPATCH_S(g.prec, {
        hipLaunchKernelGGL(k_trace_diffG<ST>, gr, dim3(256), 0, s, d.ekw, d.wq, (const ST*)d.Self, d.Sinf2, d.Sinf3,
                           d.Sinf4, d.Sinf, (int)g.nk8, g.Nw, g.T, mu0, pmu, d.part);
    });
    hipLaunchKernelGGL(k_finalize, dim3(1), dim3(256), 0, s, d.part, (int)(gr.x * gr.y), out);
    return hipGetLastError();
}

hipError_t launch_trace_diffG3_pass(const Grid& g, const DevArrays& d, double* mirror, hipStream_t s)
{
    const dim3 gr = trace_grid(g);
    const bool fused = gr.x <= (unsigned)kFusedStepMax;
    DISPATCH_S(g.prec, {
        hipLaunchKernelGGL(k_trace_diffG3<ST>, gr, dim3(256), 0, s, d.ekw, d.wq, (const ST*)d.Self, d.Sinf2, d.Sinf3,
                           d.Sinf4, d.Sinf, (int)g.nk8, g.Nw, d.root, d.part, fused ? d.ticket : nullptr, mirror);
    });
    if (!fused) hipLaunchKernelGGL(k_halley_step, dim3(1), dim3(256), 0, s, d.part, (int)gr.x, d.root, mirror);
    return hipGetLastError();
}

hipError_t launch_mu_search(const Grid& g, const DevArrays& d, const RootInit& in, double* mirror, int npass,
                            hipStream_t s)
{
    if (mu_in_one(g)) {
        const long n = g.nk8 * (g.Nw + 1);
#define MU_SEARCH(CN)                                                                                              \
    hipLaunchKernelGGL((k_mu_search<CN, ST>), dim3(1), dim3(kSearchThreads), 0, s, d.ekw, d.wq, (const ST*)d.Self, \
                       d.Sinf2, d.Sinf3, d.Sinf4, d.Sinf, (int)g.nk8, g.Nw, d.root, in, mirror, npass)
        DISPATCH_S(g.prec, {
            if (n <= 4 * kSearchThreads)
                MU_SEARCH(4);
            else
                MU_SEARCH(kMuOneMax / kSearchThreads);
        });
#undef MU_SEARCH
        return hipGetLastError();
    }
    hipError_t e = launch_halley_init(d.root, in, mirror, s);
    for (int k = 0; k < npass && e == hipSuccess; k++) e = launch_trace_diffG3_pass(g, d, mirror, s);
    return e;
}

hipError_t launch_trace_selfG0(const Grid& g, const DevArrays& d, double mu0, double* out, hipStream_t s)
{
    const double nk02 = 4.0 * (g.nk - 1) * (g.nk - 1);
    const dim3 gr = trace_grid(g);
    DISPATCH_S(g.prec, {
        hipLaunchKernelGGL(k_trace_selfG0<ST>, gr, dim3(256), 0, s, d.ekw, d.wq, (const ST*)d.Self, d.Sinf2, d.Sinf3,
                           d.Sinf, (int)g.nk8, g.Nw, g.T, mu0, nk02, d.part);
    });
    hipLaunchKernelGGL(k_finalize_k, dim3(2), dim3(256), 0, s, d.part, (int)gr.x, out);
    return hipGetLastError();
}

hipError_t launch_trace_selfG(const Grid& g, const DevArrays& d, double mu, double* out, hipStream_t s)
{
    const double nk02 = 4.0 * (g.nk - 1) * (g.nk - 1);
    const dim3 gr = trace_grid(g);
    DISPATCH_S(g.prec, {
        hipLaunchKernelGGL(k_trace_selfG<ST>, gr, dim3(256), 0, s, d.ekw, d.wq, (const ST*)d.Self, d.Sinf2, d.Sinf3,
                           d.Sinf, (int)g.nk8, g.Nw, g.T, mu, nk02, d.part);
    });
    hipLaunchKernelGGL(k_finalize, dim3(1), dim3(256), 0, s, d.part, (int)gr.x, out);
    return hipGetLastError();
}

hipError_t launch_hf0_bnd(const Grid& g, const DevArrays& d, double mu0, double fact4, hipStream_t s,
                          const double* mu0p, double U, const double* dsc)
{
    const size_t lds = slab_bytes(g.N, sizeof(double));
    DISPATCH_N(g.N, {
        set_lds(k_hf0_bnd<NN>, lds);
        hipLaunchKernelGGL(k_hf0_bnd<NN>, dim3(8), dim3(SlabShape<NN>::NT), lds, s, d.wt, d.ekw, d.fw, d.vw, d.V0,
                           d.dchirt0, mu0, g.T, fact4, d.dhV, d.df0V, d.hVb, d.f0Vb, mu0p, U, dsc);
    });
    return hipGetLastError();
}

hipError_t launch_hV_slab(const Grid& g, const DevArrays& d, int which, hipStream_t s)
{
    DISPATCH_S(g.prec, DISPATCH_N(g.N, {
        constexpr size_t lds = slab_bytes(NN, sizeof(SS));
        set_lds(k_hV_slab<NN, SS>, lds);
        hipLaunchKernelGGL((k_hV_slab<NN, SS>), dim3(g.Nw - 1), dim3(SlabShape<NN>::NT), lds, s, d.wt, d.ekw, d.fw,
                           d.vw, d.mu0v, g.T, g.Nw, (const SS*)d.V, which, (SS*)(which == 0 ? d.h : d.f0));
    }));
    return hipGetLastError();
}

hipError_t launch_jj_transpose(const Grid& g, const DevArrays& d, hipStream_t s)
{
    const dim3 gr((unsigned)((g.nq + kTT - 1) / kTT), (unsigned)((g.Nw + 1 + kTT - 1) / kTT), 2);
    DISPATCH_S(g.prec, {
        hipLaunchKernelGGL(k_transpose<SS>, gr, dim3(256), 0, s, (const SS*)d.h, (SS*)d.hT, (const SS*)d.f0,
                           (SS*)d.f0T, g.nq, g.Nw + 1);
    });
    return hipGetLastError();
}

// out[i] = (float)in[i]
__global__ void k_narrow(const double* __restrict__ in, float* __restrict__ out, long n)
{
    for (long i = blockIdx.x * (long)blockDim.x + threadIdx.x; i < n; i += (long)gridDim.x * blockDim.x)
        out[i] = (float)in[i];
}

hipError_t launch_narrow(const double* in, float* out, long n, hipStream_t s)
{
    const long nb = std::min<long>((n + 255) / 256, 4096);
    hipLaunchKernelGGL(k_narrow, dim3((unsigned)std::max<long>(nb, 1)), dim3(256), 0, s, in, out, n);
    return hipGetLastError();
}

// out[r*ntheta + b] = sum over k < n with bins[k] == b of part[r*n + k], in increasing k
__global__ void __launch_bounds__(256) k_sum_rows_binned(const double* __restrict__ part, int n,
                                                         const int* __restrict__ bins, int ntheta, double* out)
{
    __shared__ double sc[16];
    const int r = blockIdx.x, b = blockIdx.y;
    const double* row = part + (long)r * n;
    double a = 0.0;
    for (int k = threadIdx.x; k < n; k += 256)
        if (bins[k] == b) a += row[k];
    a = block_sum(a, sc);
    if (threadIdx.x == 0) out[(long)r * ntheta + b] = a;
}

hipError_t launch_sum_rows_binned(const double* part, int nrows, int n, const int* bins, int ntheta, double* out,
                                  hipStream_t s)
{
    if (nrows <= 0) return hipSuccess;
    hipLaunchKernelGGL(k_sum_rows_binned, dim3(nrows, ntheta), dim3(256), 0, s, part, n, bins, ntheta, out);
    return hipGetLastError();
}

hipError_t launch_gloc(const Grid& g, const DevArrays& d, double mu, double* part, double* out, hipStream_t s)
{
    const int H = g.Nw / 2;
    const double nk02 = 4.0 * (g.nk - 1) * (g.nk - 1);
    DISPATCH_S(g.prec, {
        hipLaunchKernelGGL(k_gloc<ST>, dim3((H + 255) / 256, kGlocChunks), dim3(256), 0, s, d.ekw, d.wq,
                           (const ST*)d.Self, d.Sinf2, d.Sinf3, d.Sinf, g.nk8, H, g.T, mu, nk02, part);
    });
    return launch_reduce_cols(part, kGlocChunks, 2 * H, out, s);
}

// [r][c] (nrows x ncols) -> [c][r]
hipError_t launch_transpose_d(const double* in, double* out, long ncols, int nrows, hipStream_t s)
{
    const dim3 gr((unsigned)((ncols + kTT - 1) / kTT), (unsigned)((nrows + kTT - 1) / kTT));
    hipLaunchKernelGGL(k_transpose<double>, gr, dim3(256), 0, s, in, out, in, out, ncols, nrows);  // grid z = 1
    return hipGetLastError();
}

// the same for two arrays
hipError_t launch_transpose_d2(const double* in0, double* out0, const double* in1, double* out1, long ncols, int nrows,
                               hipStream_t s)
{
    const dim3 gr((unsigned)((ncols + kTT - 1) / kTT), (unsigned)((nrows + kTT - 1) / kTT), 2);
    hipLaunchKernelGGL(k_transpose<double>, gr, dim3(256), 0, s, in0, out0, in1, out1, ncols, nrows);
    return hipGetLastError();
}

// out[r] = sum of part[r*n .. r*n+n) in a fixed order, r < nrows
hipError_t launch_sum_rows(const double* part, int nrows, int n, double* out, hipStream_t s)
{
    if (nrows <= 0) return hipSuccess;
    hipLaunchKernelGGL(k_finalize_k, dim3(nrows), dim3(256), 0, s, part, n, out);
    return hipGetLastError();
}

}  // namespace tpsc
