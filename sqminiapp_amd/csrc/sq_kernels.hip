// sq_kernels.hip -- gfx950 kernels of the SQ hot path.
//
// One workgroup runs the whole Lanczos recurrence of one grid node's cube
// (persistent over the N_qp+1 H applications) and then takes the next node;
// the Lanczos vectors live in a per-workgroup slice of HBM that stays resident
// in the L2/Infinity cache while the node is processed.  Per H application:
//   gather  : A[img][ch] = sum_{cube & box} v * chi   (one wavefront per image,
//             DPP/shuffle reduction, no atomics -> deterministic)
//   alpha   : per atom, from the A of its images (collapsed or KB slots)
//   apply   : u = sum over the 6*order+1 stencil columns in ascending column
//             order, + diag(L)+V_eff, then + chi*alpha over the images covering
//             the point in ascending image order (the reference's order)
//   reduce  : a = <v,u>, then w = u - a v - b vprev, b = ||w||
// This file is compiled with -ffp-contract=off: in the FP64 form every
// product and sum rounds as written.  The FP32 form uses explicit fmaf.
#include <hip/hip_runtime.h>
#include <stdint.h>

#include <algorithm>
#include <climits>
#include <mutex>

#include "sq_device_common.h"

namespace sqamd {

template <typename T, int NLM>
__global__ void __launch_bounds__(kWG) lanczos_kernel(KParams P)
{
    extern __shared__ __align__(16) unsigned char smem[];
    int *img_list = reinterpret_cast<int *>(smem);
    double *A = reinterpret_cast<double *>(smem + P.lds_A);
    double *alpha = reinterpret_cast<double *>(smem + P.lds_alpha);
    double *red = reinterpret_cast<double *>(smem + P.lds_red);
    short *local_of = reinterpret_cast<short *>(smem + P.lds_local);
    __shared__ int s_count;

    const int nx = P.nloc[0], ny = P.nloc[1];
    const int nc = P.nc;
    const float invx = 1.0f / (float)nx, invy = 1.0f / (float)ny;
    // three vectors per workgroup: v, vprev (raw, with scales) and u = H v
    T *buf0 = reinterpret_cast<T *>(P.scratch) + (size_t)blockIdx.x * 3 * nc;
    T *buf1 = buf0 + nc;
    T *Bu = buf1 + nc;
    const T *diag_ext = reinterpret_cast<const T *>(P.diag_ext);
    const T *chi = reinterpret_cast<const T *>(P.chi);

    __shared__ int s_near[kRecMax], s_nnear;
    for (long r = blockIdx.x; r < P.node_count; r += gridDim.x) {
        const long id = P.node_list ? (long)P.node_list[r] : P.node_begin + r;
        int node[3];
        node_coords(P, id, node);
        int cube_lo[3] = {node[0] - P.hw[0], node[1] - P.hw[1], node[2] - P.hw[2]};
        // images whose box meets this cube, ascending (ordered compaction)
        if (threadIdx.x == 0) s_count = 0;
        __syncthreads();
        for (int base = 0; base < P.n_images; base += kWG) {
            const int g = base + threadIdx.x;
            bool hit = false;
            if (g < P.n_images) {
                const int4 lo4 = P.img_lo[g], dm4 = P.img_dim[g];
                hit = lo4.x <= cube_lo[0] + P.nloc[0] - 1 && lo4.x + dm4.x - 1 >= cube_lo[0] &&
                      lo4.y <= cube_lo[1] + P.nloc[1] - 1 && lo4.y + dm4.y - 1 >= cube_lo[1] &&
                      lo4.z <= cube_lo[2] + P.nloc[2] - 1 && lo4.z + dm4.z - 1 >= cube_lo[2];
            }
            const unsigned long long bal = __ballot(hit);
            const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
            const int before = __popcll(bal & ((1ull << lane) - 1ull));
            int *wcnt = reinterpret_cast<int *>(red);
            if (lane == 0) wcnt[wave] = __popcll(bal);
            __syncthreads();
            int off = s_count;
            for (int w = 0; w < wave; w++) off += wcnt[w];
            if (hit) {
                const int li = off + before;
                if (li < P.img_cap) { img_list[li] = g; local_of[g] = (short)li; }
            }
            __syncthreads();
            if (threadIdx.x == 0) {
                int t = s_count;
                for (int w = 0; w < kWaves; w++) t += wcnt[w];
                s_count = t;
            }
            __syncthreads();
        }
        const int nimg = s_count;
        if (nimg > P.img_cap) {  // the host sized img_cap from the geometry; flag the node
            if (threadIdx.x == 0) P.status[id] = 4;
            __syncthreads();
            continue;
        }
        if (P.rec) {
            if (record_near(P, r, img_list, nimg, node, s_near, &s_nnear) > P.rec_slots) {
                if (threadIdx.x == 0) P.status[id] = 4;
                __syncthreads();
                continue;
            }
        }
        // Lanczos start: v = e_center, vprev = 0
        for (int p = threadIdx.x; p < nc; p += kWG) { buf0[p] = T(0); buf1[p] = T(0); }
        __syncthreads();
        if (threadIdx.x == 0) buf0[P.center] = T(1);
        __syncthreads();
        T *Bv = buf0, *Bvp = buf1;
        T sv = T(1), svp = T(0);
        double bprev = 0.0;
        double *out_a = P.out_a + id * (P.nqp + 1), *out_b = P.out_b + id * (P.nqp + 1);
        int status = 0;
        for (int step = 0; step <= P.nqp; step++) {
            gather_images<T, NLM>(P, img_list, nimg, cube_lo, Bv, sv, chi, A);
            __syncthreads();
            images_alpha<NLM>(P, img_list, nimg, A, alpha);
            __syncthreads();
            if (P.rec) record_step(P, r, step, s_near, s_nnear, alpha, NLM);
            double pa = 0.0;
            CSum ca{0.f, 0.f};
            for (int p = threadIdx.x; p < nc; p += kWG) {
                const int jk = fdiv(p, nx, invx);
                const int li = p - jk * nx;
                const int lk = fdiv(jk, ny, invy);
                const int lj = jk - lk * ny;
                const int64_t E = ((int64_t)(cube_lo[2] + lk - P.ext0[2]) * P.extn[1] + (cube_lo[1] + lj - P.ext0[1])) *
                                      P.extn[0] + (cube_lo[0] + li - P.ext0[0]);
                const T u = apply_point<T, NLM>(P, p, li, lj, lk, cube_lo, Bv, sv, diag_ext, chi, local_of, alpha, E);
                Bu[p] = u;
                const T vc = sv * Bv[p];
                if constexpr (sizeof(T) == 8) pa += vc * u;
                else ca = csum_add_prod(ca, vc, u);
            }
            double a;
            if constexpr (sizeof(T) == 8) a = block_sum(pa, red);
            else a = block_csum(ca, red);
            // w = (u - a v) - bprev vprev, written over vprev's storage
            const T ta = T(-a), tb = T(-bprev);
            double pb = 0.0;
            CSum cb{0.f, 0.f};
            for (int p = threadIdx.x; p < nc; p += kWG) {
                const T vc = sv * Bv[p];
                const T vpc = svp * Bvp[p];
                const T u = Bu[p];
                T w;
                if constexpr (sizeof(T) == 8) {
                    w = u + ta * vc;
                    w = w + tb * vpc;
                    pb += w * w;
                } else {
                    w = fmaf(ta, vc, u);
                    w = fmaf(tb, vpc, w);
                    cb = csum_add_prod(cb, w, w);
                }
                Bvp[p] = w;
            }
            double bb;
            if constexpr (sizeof(T) == 8) bb = block_sum(pb, red);
            else bb = block_csum(cb, red);
            const double b = sqrt(bb);
            if (threadIdx.x == 0) { out_a[step] = a; out_b[step] = b; }
            if (b == 0.0) { status = 7; break; }
            // rotate: v <- w / b, vprev <- v
            T *t = Bv; Bv = Bvp; Bvp = t;
            svp = sv;
            sv = T(1.0 / b);
            bprev = b;
        }
        if (threadIdx.x == 0) P.status[id] = status;
        __syncthreads();
    }
}

// One H application on one node (device vectors x, y of nc entries):
// y = H x, or with nonlocal_only y += V_nl x, each point's projector terms
// added onto its incoming y in ascending image order as Mult_NonlocalVector
// accumulates into V2 (lsdft_matvec.cc:110-142).
template <typename T, int NLM>
__global__ void __launch_bounds__(kWG) apply_kernel(KParams P, long id, const T *x, T *y, int nonlocal_only)
{
    extern __shared__ __align__(16) unsigned char smem[];
    int *img_list = reinterpret_cast<int *>(smem);
    double *A = reinterpret_cast<double *>(smem + P.lds_A);
    double *alpha = reinterpret_cast<double *>(smem + P.lds_alpha);
    short *local_of = reinterpret_cast<short *>(smem + P.lds_local);
    const int nx = P.nloc[0], ny = P.nloc[1];
    const float invx = 1.0f / (float)nx, invy = 1.0f / (float)ny;
    int node[3];
    node_coords(P, id, node);
    int cube_lo[3] = {node[0] - P.hw[0], node[1] - P.hw[1], node[2] - P.hw[2]};
    if (threadIdx.x == 0) {
        int n = 0;
        for (int g = 0; g < P.n_images; g++) {
            const int4 lo4 = P.img_lo[g], dm4 = P.img_dim[g];
            bool hit = lo4.x <= cube_lo[0] + P.nloc[0] - 1 && lo4.x + dm4.x - 1 >= cube_lo[0] &&
                       lo4.y <= cube_lo[1] + P.nloc[1] - 1 && lo4.y + dm4.y - 1 >= cube_lo[1] &&
                       lo4.z <= cube_lo[2] + P.nloc[2] - 1 && lo4.z + dm4.z - 1 >= cube_lo[2];
            if (hit && n < P.img_cap) { img_list[n] = g; local_of[g] = (short)n; }
            n += hit;
        }
        reinterpret_cast<int *>(smem + P.lds_red)[0] = n;
    }
    __syncthreads();
    const int nimg = reinterpret_cast<int *>(smem + P.lds_red)[0];
    if (nimg > P.img_cap) { if (threadIdx.x == 0) P.status[0] = 4; return; }
    __syncthreads();
    gather_images<T, NLM>(P, img_list, nimg, cube_lo, x, T(1), reinterpret_cast<const T *>(P.chi), A);
    __syncthreads();
    images_alpha<NLM>(P, img_list, nimg, A, alpha);
    __syncthreads();
    for (int p = threadIdx.x; p < P.nc; p += blockDim.x) {
        const int jk = fdiv(p, nx, invx);
        const int li = p - jk * nx;
        const int lk = fdiv(jk, ny, invy);
        const int lj = jk - lk * ny;
        const int64_t E = ((int64_t)(cube_lo[2] + lk - P.ext0[2]) * P.extn[1] + (cube_lo[1] + lj - P.ext0[1])) * P.extn[0] +
                          (cube_lo[0] + li - P.ext0[0]);
        y[p] = apply_point<T, NLM>(P, p, li, lj, lk, cube_lo, x, T(1), reinterpret_cast<const T *>(P.diag_ext),
                                   reinterpret_cast<const T *>(P.chi), local_of, alpha, E, !nonlocal_only,
                                   nonlocal_only ? y[p] : T(0));
    }
}

// r = sqrt(g g + f f), s = f / r, c = g / r, each correctly rounded as the
// operators round them.  One approximate 1/sqrt serves all three: coupled
// Newton steps (Goldschmidt) give sqrt(x) and 1/(2 sqrt(x)), two residual
// corrections round the root, one more Newton step rounds 1/r, and the residual
// of each quotient rounds it (Markstein, IBM J. Res. Dev. 34, 1990).  That needs
// operands away from the ends of the exponent range; others (zeros among them)
// take the operators, whose range scaling costs a third of the chain.
__device__ __forceinline__ void rotation(double f, double g, double &r, double &s, double &c)
{
    const double x = g * g + f * f;
    const double af = fabs(f), ag = fabs(g);
    if (fmin(af, ag) > 0x1p-300 && fmax(af, ag) < 0x1p300) {
        const double y = __builtin_amdgcn_rsq(x);
        double q = x * y, h = 0.5 * y;
        const double t = fma(-h, q, 0.5);
        q = fma(q, t, q);
        h = fma(h, t, h);
        q = fma(fma(-q, q, x), h, q);
        r = fma(fma(-q, q, x), h, q);
        h = h + h;
        h = fma(fma(-r, h, 1.0), h, h);
        h = fma(fma(-r, h, 1.0), h, h);
        const double qf = f * h, qg = g * h;
        s = fma(fma(-r, qf, f), h, qf);
        c = fma(fma(-r, qg, g), h, qg);
    } else {
        r = sqrt(x);
        s = f / r;
        c = g / r;
    }
}

// Implicit QL, one tridiagonal a lane (TridiagEigenVecSolve_NodesAndWeights,
// lsdft_tools.cc:912-1026).  Only row 0 of the eigenvector matrix is carried:
// the reference's rotations update each row of z independently, so row 0 -- the
// one the weights w_i = z[0][i]^2 use -- is the same number sequence.
//
// Bound by the chain of one rotation (rotation(), about 400
// clocks) times the rotations of a tridiagonal (5000 at n = 80), so what counts
// is that nothing else joins the chain and that many chains run side by side.
// The next rotation's entries are read ahead, and the test for a small
// off-diagonal, which the reference repeats from l on after every sweep, is
// made inside the sweep, where d and e become final; a scan before each sweep
// and the operators in place of rotation() took 13.3 ms for 16384 x n = 80, which
// take 3.4 to 3.8 now.  The rows d, e and z lie in LDS (ql_kernel) or, for batches of which
// LDS holds only a part at a time, in device memory (ql_kernel_mem); ql_lanes.

// Tridiagonals t0 .. t0 + mine - 1, one a lane; d, e and z of lane k at
// rows[i * pitch + k], i in [0, nmax), [nmax, 2 nmax) and [2 nmax, 3 nmax).  The
// outputs may be the inputs: a tridiagonal is read before any is written.
__device__ __forceinline__ void ql_rules(double *rows, const unsigned pitch, const double *a, const double *bsub, int nmax,
                                         int stride, long t0, int mine, double *lam, double *w, double *lmin, double *lmax,
                                         int *status, const int *nsteps)
{
    const int lane = threadIdx.x;
    for (int q = lane; q < mine * nmax; q += 64) {
        const int k = q / nmax, i = q - k * nmax;
        rows[i * pitch + k] = a[(t0 + k) * stride + i];
        rows[(nmax + i) * pitch + k] = bsub[(t0 + k) * stride + i];
        rows[(2 * nmax + i) * pitch + k] = i == 0 ? 1.0 : 0.0;
    }
    __syncthreads();
    const long t = t0 + lane;
    // a node that stopped early has a Gauss rule of nsteps[t] nodes; the rest of
    // its row is padded with weight zero at its largest node
    int n = nmax, bad = 0;
    if (lane < mine) {
        if (nsteps) n = max(1, min(nmax, nsteps[t]));
        double *const d = rows + lane, *const e = rows + nmax * pitch + lane, *const z = rows + 2 * nmax * pitch + lane;
#define D(i) d[(unsigned)(i) * pitch]
#define EE(i) e[(unsigned)(i) * pitch]
#define Z(i) z[(unsigned)(i) * pitch]
        EE(n - 1) = 0.0;
        auto small = [](double ei, double di, double dn) {
            const double dd = fabs(di) + fabs(dn);
            return (double)(fabs(ei) + dd) == dd;
        };
        int next = -1;   // the first small off-diagonal from l on, where the last sweep found it
        for (int l = 0; l < n && !bad; l++) {
            for (int iter = 0;;) {
                int m = next;
                if (m < l) {
                    m = l;
                    for (double dm = D(l); m <= n - 2; m++) {
                        const double dn = D(m + 1);
                        if (small(EE(m), dm, dn)) break;
                        dm = dn;
                    }
                    next = m;
                }
                if (m == l) break;
                if (iter++ == 50) { bad = 5; break; }
                const double el = EE(l);
                double g = (D(l + 1) - D(l)) / (2.0 * el);
                double r = sqrt(g * g + 1.0);
                double dnext = D(m);   // d(i + 1) before rotation i
                g = dnext - D(l) + el / (g + (g >= 0.0 ? fabs(r) : -fabs(r)));
                double s = 1.0, c = 1.0, p = 0.0, znext = Z(m), dfinal = 0.0;
                double di = D(m - 1), ei = EE(m - 1), zi = Z(m - 1);
                int i = m - 1, above = m;   // above: the first small off-diagonal past l so far
                for (;;) {
                    // entries of rotation i - 1 (row 0 again on the last one)
                    const int k = max(i - 1, 0);
                    const double dk = D(k), ek = EE(k), zk = Z(k);
                    const double f = s * ei, b = c * ei;
                    rotation(f, g, r, s, c);
                    EE(i + 1) = r;
                    if (r == 0.0) {
                        D(i + 1) = dnext - p;
                        Z(i + 1) = znext;
                        EE(m) = 0.0;
                        break;
                    }
                    g = dnext - p;
                    const double rr = (di - g) * s + 2.0 * c * b;
                    p = s * rr;
                    const double dn = g + p;   // d(i + 1), final
                    D(i + 1) = dn;
                    g = c * rr - b;
                    Z(i + 1) = s * zi + c * znext;
                    znext = c * zi - s * znext;
                    if (i + 1 < m && small(r, dn, dfinal)) above = i + 1;
                    dfinal = dn;
                    dnext = di;
                    if (i == l) break;
                    i--;
                    di = dk;
                    ei = ek;
                    zi = zk;
                }
                if (r == 0.0) { next = -1; continue; }
                const double dl = dnext - p;
                D(l) = dl;
                Z(l) = znext;
                EE(l) = g;
                EE(m) = 0.0;
                next = above;
                if (small(g, dl, dfinal)) break;
            }
        }
        double emin = D(0), emax = D(0);
        for (int i = 1; i < n; i++) {
            const double di = D(i);
            if (di > emax) emax = di;
            else if (di < emin) emin = di;
        }
        status[t] = bad;
        if (!bad) {
            lmin[t] = emin;
            lmax[t] = emax;
            for (int i = n; i < nmax; i++) {
                D(i) = emax;
                Z(i) = 0.0;
            }
        }
#undef D
#undef EE
#undef Z
    }
    // a tridiagonal that did not converge leaves its outputs untouched
    const unsigned long long failed = __ballot(bad != 0);
    __syncthreads();
    for (int q = lane; q < mine * nmax; q += 64) {
        const int k = q / nmax, i = q - k * nmax;
        if (failed >> k & 1) continue;
        const double zi = rows[(2 * nmax + i) * pitch + k];
        lam[(t0 + k) * nmax + i] = rows[i * pitch + k];
        w[(t0 + k) * nmax + i] = zi * zi;
    }
}

// Rows in LDS; only `lanes` lanes of a wavefront work, so that a batch spreads over
// all SIMDs and few tridiagonals wait for each other's sweeps.
__global__ void __launch_bounds__(64) ql_kernel(const double *a, const double *bsub, int nmax, int stride, long count,
                                                int lanes, double *lam, double *w, double *lmin, double *lmax, int *status,
                                                const int *nsteps)
{
    extern __shared__ double rows[];   // d, e, z: [3][nmax][lanes]
    const long t0 = (long)blockIdx.x * lanes;
    ql_rules(rows, lanes, a, bsub, nmax, stride, t0, (int)min((long)lanes, count - t0), lam, w, lmin, lmax, status, nsteps);
}

// Rows in device memory, 3 nmax x pitch doubles at ws: 64 tridiagonals a wavefront, and
// the wavefront's next ones in the same place.
__global__ void __launch_bounds__(64) ql_kernel_mem(const double *a, const double *bsub, int nmax, int stride, long count,
                                                    unsigned pitch, double *ws, double *lam, double *w, double *lmin,
                                                    double *lmax, int *status, const int *nsteps)
{
    double *const rows = ws + blockIdx.x * 64u;
    for (long t0 = blockIdx.x * 64L; t0 < count; t0 += gridDim.x * 64L) {
        ql_rules(rows, pitch, a, bsub, nmax, stride, t0, (int)min(64L, count - t0), lam, w, lmin, lmax, status, nsteps);
        __syncthreads();
    }
}

// ------------------------------------------------ density / Fermi / energy
__device__ __forceinline__ double fermi_occ(double x)  // 1/(1+e^x)
{
    if (x > 0) { double t = exp(-x); return t / (1.0 + t); }
    return 1.0 / (1.0 + exp(x));
}
__device__ __forceinline__ double fermi_ent(double x)  // f ln f + (1-f) ln(1-f)
{
    double ax = fabs(x), t = exp(-ax);
    return -log1p(t) - ax * t / (1.0 + t);
}

constexpr int kRedThreads = 256;

// A block's partial of sum w f(beta (lam - lf)) over its chunk
__device__ __forceinline__ void occupation_block(const double *lam, const double *w, long nq, double beta, double lf,
                                                 double *partial, double *red)
{
    const long chunk = (nq + gridDim.x - 1) / gridDim.x;
    const long q0 = blockIdx.x * chunk, q1 = min(nq, q0 + chunk);
    double s = 0.0;
    for (long q = q0 + threadIdx.x; q < q1; q += blockDim.x) s += w[q] * fermi_occ(beta * (lam[q] - lf));
    s = wave_sum(s);
    if ((threadIdx.x & 63) == 0) red[threadIdx.x >> 6] = s;
    __syncthreads();
    if (threadIdx.x == 0) {
        double t = 0.0;
        for (int k = 0; k < kRedThreads / 64; k++) t += red[k];
        partial[blockIdx.x] = t;
    }
}

// One electron count of the Fermi bisection, N(lf) = 2 sum w f, on [lambda_min
// - 1, lambda_max + 1] to 1e-14 (relative) in at most 200 halvings.  A launch
// first takes the decision that the last count calls for -- every block for
// itself, from the last launch's partials and state, so no launch is spent on
// it -- and then counts at the new midpoint.  Count k leaves its state at state[k
// & 1] and its partials in the (k + 2) % 3-th of three places: no block of a launch
// writes what another still reads.  count: -2 at the lower end, -1 at the upper
// end, then 0 (brackets, first midpoint), 1, ...  A halving takes 5 us where a rule
// set is small, 8 and 11 for the rules of 7872 and 15744 grid nodes; the count, its sum and
// a look by the host took 60, on the device 16 in two launches.
__global__ void __launch_bounds__(kRedThreads) fermi_count(const double *lam, const double *w, long nq, double beta,
                                                           double nelec, const double *range, int count, BisState *state,
                                                           double *partial)
{
    __shared__ double red[kRedThreads / 64], sm[ordered_lds(kRedBlocksDev)];
    const int nb = gridDim.x;
    double *const mine = partial + (count + 2) % 3 * nb;
    if (count < 0) {
        occupation_block(lam, w, nq, beta, count == -2 ? range[0] - 1.0 : range[1] + 1.0, mine, red);
        return;
    }
    BisState b;
    if (count == 0) {
        b.lo = range[0] - 1.0;
        b.hi = range[1] + 1.0;
        b.mid = 0.0;
        b.done = b.bad = b.count = 0;
        const double glo = 2.0 * ordered_total(partial, nb, sm);
        const double ghi = 2.0 * ordered_total(partial + nb, nb, sm);
        if (glo - nelec > 0 || ghi - nelec < 0) b.bad = b.done = 1;
    } else {
        b = state[(count - 1) & 1];
        if (!b.done) {
            const double g = 2.0 * ordered_total(partial + (count + 1) % 3 * nb, nb, sm);
            if (g - nelec > 0) b.hi = b.mid;
            else b.lo = b.mid;
            if (++b.count >= 200) b.done = 1;
        }
    }
    if (!b.done) {
        b.mid = 0.5 * (b.lo + b.hi);
        if (b.hi - b.lo <= 1e-14 * (fabs(b.mid) > 1.0 ? fabs(b.mid) : 1.0)) b.done = 1;
    }
    b.lf = 0.5 * (b.lo + b.hi);
    if (threadIdx.x == 0 && blockIdx.x == 0) state[count & 1] = b;
    if (!b.done) occupation_block(lam, w, nq, beta, b.mid, mine, red);
}

// sum of partials in index order -> out[0]
__global__ void __launch_bounds__(64) ordered_sum(const double *partial, int n, double scale, double *out)
{
    __shared__ double sm[ordered_lds(kRedBlocksDev)];
    const double s = ordered_total(partial, n, sm);
    if (threadIdx.x == 0) out[0] = scale * s;
}

// per node: rho = (2/dV) sum_i w f; partials of sum w lam f and sum w S(f).  The
// block's threads form the terms of its nodes' rules together, a node's own
// thread adds them in order: one thread a node, as before, left 8 of 256 busy
// with the exponentials (3840 nodes: 12 us, and 90 before).
__global__ void __launch_bounds__(kRedThreads) density_energy(const double *lam, const double *w, long n_nodes, int nqp,
                                                              double beta, const double *lf_dev, double two_over_dv,
                                                              double *rho, double *part_e, double *part_s)
{
    constexpr int kTerms = 1024;
    __shared__ double tr[kTerms], te[kTerms], ts[kTerms];
    __shared__ double re[kRedThreads / 64], rs[kRedThreads / 64];
    const double lf = *lf_dev;
    const long chunk = (n_nodes + gridDim.x - 1) / gridDim.x;
    const long p0 = blockIdx.x * chunk, p1 = min(n_nodes, p0 + chunk);
    double se = 0.0, ss = 0.0;
    for (long base = p0; base < p1; base += blockDim.x) {
        const int rows = (int)min((long)blockDim.x, p1 - base), width = min(nqp, kTerms / rows);
        const bool mine = (int)threadIdx.x < rows;
        double sr = 0.0;
        for (int i0 = 0; i0 < nqp; i0 += width) {
            const int cols = min(width, nqp - i0);
            for (int k = threadIdx.x; k < rows * cols; k += blockDim.x) {
                const int row = k / cols;
                const long q = (base + row) * nqp + i0 + (k - row * cols);
                const double x = beta * (lam[q] - lf);
                const double f = fermi_occ(x);
                tr[k] = w[q] * f;
                te[k] = w[q] * lam[q] * f;
                ts[k] = w[q] * fermi_ent(x);
            }
            __syncthreads();
            if (mine)
                for (int i = 0; i < cols; i++) {
                    const int k = threadIdx.x * cols + i;
                    sr += tr[k];
                    se += te[k];
                    ss += ts[k];
                }
            __syncthreads();
        }
        if (rho && mine) rho[base + threadIdx.x] = two_over_dv * sr;
    }
    se = wave_sum(se);
    ss = wave_sum(ss);
    if ((threadIdx.x & 63) == 0) { re[threadIdx.x >> 6] = se; rs[threadIdx.x >> 6] = ss; }
    __syncthreads();
    if (threadIdx.x == 0) {
        double a = 0.0, b = 0.0;
        for (int k = 0; k < kRedThreads / 64; k++) { a += re[k]; b += rs[k]; }
        part_e[blockIdx.x] = a;
        part_s[blockIdx.x] = b;
    }
}

// min/max of lambda over all nodes (bracket of the Fermi level)
__global__ void __launch_bounds__(1024) lam_range(const double *lmin, const double *lmax, long n, double *out)
{
    __shared__ double smin[16], smax[16];
    double a = 1e300, b = -1e300;
    for (long p = threadIdx.x; p < n; p += blockDim.x) { a = fmin(a, lmin[p]); b = fmax(b, lmax[p]); }
    for (int off = 32; off > 0; off >>= 1) {
        a = fmin(a, __shfl_xor(a, off, 64));
        b = fmax(b, __shfl_xor(b, off, 64));
    }
    if ((threadIdx.x & 63) == 0) {
        smin[threadIdx.x >> 6] = a;
        smax[threadIdx.x >> 6] = b;
    }
    __syncthreads();
    if (threadIdx.x == 0) {
        for (int k = 1; k < 16; k++) { a = fmin(a, smin[k]); b = fmax(b, smax[k]); }
        out[0] = a;
        out[1] = b;
    }
}

// ------------------------------------------------------------ launchers
template <typename T, int NLM>
static hipError_t launch_lanczos_nlm(const KParams &P, int grid, size_t lds, hipStream_t st)
{
    hipLaunchKernelGGL((lanczos_kernel<T, NLM>), dim3(grid), dim3(kWG), lds, st, P);
    return hipGetLastError();
}

hipError_t launch_lanczos(const KParams &P, int precision, int grid, size_t lds, hipStream_t st)
{
    if (P.nlm_max <= 6) {
        if (precision == 0) return launch_lanczos_nlm<double, 6>(P, grid, lds, st);
        return launch_lanczos_nlm<float, 6>(P, grid, lds, st);
    }
    if (P.nlm_max <= kMaxChannels) {
        if (precision == 0) return launch_lanczos_nlm<double, kMaxChannels>(P, grid, lds, st);
        return launch_lanczos_nlm<float, kMaxChannels>(P, grid, lds, st);
    }
    return hipErrorInvalidValue;
}

hipError_t launch_apply(const KParams &P, long id, const double *x, double *y, int nonlocal_only, size_t lds,
                        hipStream_t st)
{
    if (P.nlm_max <= 6)
        hipLaunchKernelGGL((apply_kernel<double, 6>), dim3(1), dim3(kWG), lds, st, P, id, x, y, nonlocal_only);
    else if (P.nlm_max <= kMaxChannels)
        hipLaunchKernelGGL((apply_kernel<double, kMaxChannels>), dim3(1), dim3(kWG), lds, st, P, id, x, y,
                           nonlocal_only);
    else return hipErrorInvalidValue;
    return hipGetLastError();
}

// Tridiagonals a wavefront of ql_kernel takes, 0: ql_kernel_mem.  LDS while the
// batch runs in one round: the fewest lanes with which every wavefront has a CU to
// itself (n = 80: 33 take 2.8 ms one a wavefront and 3.8 sixteen a wavefront; 4096
// take 4.6 sixteen a wavefront and 5.4 eight), else 16 on four wavefronts a CU
// (16384: 3.8, against 4.3 with 32).  Past that device memory, whose latency
// other wavefronts hide (LDS form, memory form; n = 80: 16384 take 3.8 and 4.6 ms,
// 20000 9.3 and 5.4, 200000 51 and 22; n = 256: 1024 take 36 and 41, 4096 71 and 48,
// 24576 329 and 60).
static int ql_lanes(int n, long count)
{
    const size_t row = (size_t)3 * n * sizeof(double);
    int lanes = 1;
    while (lanes < 32 && (count + lanes - 1) / lanes > 256) lanes <<= 1;
    if ((count + lanes - 1) / lanes <= 256 && lanes * row <= 65536) return lanes;
    return (count + 15) / 16 <= 1024 && 16 * row <= 40960 ? 16 : 0;
}

// Wavefronts of ql_kernel_mem: up to eight a CU, the batch in rounds past that
static long ql_mem_grid(long count) { return std::min<long>((count + 63) / 64, 2048); }

size_t ql_workspace_bytes(int n, long count)
{
    return ql_lanes(n, count) ? 0 : (size_t)3 * n * std::min(count, 64 * ql_mem_grid(count)) * sizeof(double);
}

hipError_t launch_ql(const double *a, const double *b, int n, int stride, long count, double *lam, double *w,
                     double *lmin, double *lmax, int *status, double *ws, hipStream_t st, const int *nsteps)
{
    if (n < 1 || n > kMaxNqp || count <= 0) return hipErrorInvalidValue;
    const int lanes = ql_lanes(n, count);
    if (lanes == 0) {
        if (!ws) return hipErrorInvalidValue;
        const long grid = ql_mem_grid(count);
        hipLaunchKernelGGL(ql_kernel_mem, dim3((unsigned)grid), dim3(64), 0, st, a, b, n, stride, count,
                           (unsigned)std::min(count, 64 * grid), ws, lam, w, lmin, lmax, status, nsteps);
        return hipGetLastError();
    }
    const long blocks = (count + lanes - 1) / lanes;
    // LDS for the rows, and no less than keeps a CU from taking more workgroups than its share
    const size_t rows = (size_t)lanes * 3 * n * sizeof(double);
    const size_t share = blocks > 512 ? 40960 : 65536;
    hipLaunchKernelGGL(ql_kernel, dim3((unsigned)blocks), dim3(64), std::max(rows, share), st, a, b, n, stride, count,
                       lanes, lam, w, lmin, lmax, status, nsteps);
    return hipGetLastError();
}

hipError_t launch_fermi_count(const double *lam, const double *w, long nq, double beta, double nelec, const double *range,
                              int count, BisState *state, double *partial, hipStream_t st)
{
    hipLaunchKernelGGL(fermi_count, dim3(kRedBlocksDev), dim3(kRedThreads), 0, st, lam, w, nq, beta, nelec, range, count,
                       state, partial);
    return hipGetLastError();
}

hipError_t launch_density_energy(const double *lam, const double *w, long n_nodes, int nqp, double beta,
                                 const double *lf_dev, double two_over_dv, double *rho, double *partial, double *out2,
                                 hipStream_t st)
{
    double *const part_e = partial, *const part_s = partial + kRedBlocksDev;
    hipLaunchKernelGGL(density_energy, dim3(kRedBlocksDev), dim3(kRedThreads), 0, st, lam, w, n_nodes, nqp, beta, lf_dev,
                       two_over_dv, rho, part_e, part_s);
    hipLaunchKernelGGL(ordered_sum, dim3(1), dim3(64), 0, st, part_e, kRedBlocksDev, 2.0, out2);
    hipLaunchKernelGGL(ordered_sum, dim3(1), dim3(64), 0, st, part_s, kRedBlocksDev, 2.0 / beta, out2 + 1);
    return hipGetLastError();
}

hipError_t launch_lam_range(const double *lmin, const double *lmax, long n, double *out, hipStream_t st)
{
    hipLaunchKernelGGL(lam_range, dim3(1), dim3(1024), 0, st, lmin, lmax, n, out);
    return hipGetLastError();
}

// ------------------------------------------------- QL without allocation
// Workspace of sq_tridiag_nodes_weights_noalloc: a static device array of
// kNoAllocScratchBytes, one copy per GPU at its own address, held until the
// process ends.  In host code `scratch` names a host-side stand-in, never the
// device memory: its address on each device comes from hipGetSymbolAddress
// (noalloc_scratch_init, once per device, with that device current) and only
// that address is handed to kernels.
static __device__ __align__(256) unsigned char scratch[kNoAllocScratchBytes];

namespace {
std::mutex g_scratch_mu;
void *g_scratch_dev[kNoAllocMaxDevices];

size_t align256(size_t x) { return (x + 255) & ~(size_t)255; }
}  // namespace

hipError_t noalloc_scratch_init(int device)
{
    if (device < 0 || device >= kNoAllocMaxDevices) return hipErrorInvalidDevice;
    std::lock_guard<std::mutex> lock(g_scratch_mu);
    if (g_scratch_dev[device]) return hipSuccess;
    void *p = nullptr;
    const hipError_t e = hipGetSymbolAddress(&p, HIP_SYMBOL(scratch));
    if (e != hipSuccess) return e;
    if (!p) return hipErrorInvalidSymbol;
    g_scratch_dev[device] = p;
    return hipSuccess;
}

void *noalloc_scratch(int device)
{
    if (device < 0 || device >= kNoAllocMaxDevices) return nullptr;
    std::lock_guard<std::mutex> lock(g_scratch_mu);
    return g_scratch_dev[device];
}

// workspace layout: [3][n][count] doubles, the rows of ql_kernel_mem (which never
// takes more) | status[count] | the index of the first failed tridiagonal (long long)
size_t noalloc_ql_bytes(int n, long count)
{
    return align256((size_t)3 * n * count * sizeof(double)) + align256((size_t)count * sizeof(int)) + 256;
}

// Index of the first tridiagonal whose QL did not converge, -1 when none
// (one workgroup; each thread scans its stride in ascending order).
__global__ void __launch_bounds__(256) first_failure(const int *status, long count, long long *out)
{
    __shared__ long long m[256];
    long long best = -1;
    for (long i = threadIdx.x; i < count; i += 256)
        if (status[i]) { best = i; break; }
    m[threadIdx.x] = best < 0 ? LLONG_MAX : best;
    __syncthreads();
    for (int s = 128; s > 0; s >>= 1) {
        if ((int)threadIdx.x < s) m[threadIdx.x] = min(m[threadIdx.x], m[threadIdx.x + s]);
        __syncthreads();
    }
    if (threadIdx.x == 0) out[0] = m[0] == LLONG_MAX ? -1 : m[0];
}

hipError_t launch_ql_noalloc(void *ws, const double *a, const double *b, int n, long count, double *lam, double *w,
                             double *lmin, double *lmax, long long **first_bad, hipStream_t st)
{
    if (!ws || n < 1 || n > kMaxNqp || count <= 0 || noalloc_ql_bytes(n, count) > kNoAllocScratchBytes)
        return hipErrorInvalidValue;
    unsigned char *base = static_cast<unsigned char *>(ws);
    int *status = reinterpret_cast<int *>(base + align256((size_t)3 * n * count * sizeof(double)));
    long long *bad = reinterpret_cast<long long *>(reinterpret_cast<unsigned char *>(status) +
                                                   align256((size_t)count * sizeof(int)));
    hipError_t e = launch_ql(a, b, n, n, count, lam, w, lmin, lmax, status, static_cast<double *>(ws), st);
    if (e != hipSuccess) return e;
    hipLaunchKernelGGL(first_failure, dim3(1), dim3(256), 0, st, status, count, bad);
    *first_bad = bad;
    return hipGetLastError();
}

}  // namespace sqamd
