// sq_mlp.hip -- the initial-density network: descriptors, forward (FP32 and
// BF16-storage), deltas, gradient sums and the Adam step.
//
// No counterpart in the reference (its SCF, declared only, would start from
// the superposed atomic densities, lsdft_readfiles.cc:1026-1040).  The network
// predicts the SCF's correction to that superposition at every cell point
// from Behler-type symmetry functions of the Mg atoms within rf = 8 bohr of
// the point (the point is the centre; fc(r) = (cos(pi r/rf) + 1)/2):
//   radial   f_k = sum_J exp(-((r_J - mu_k)/s)^2) fc(r_J),  mu_k = k rf/15, s = rf/15, k < 16
//   angular  g_a = 2^(1-zeta) sum_{J<L} (1 + lam cos t_JL)^zeta exp(-eta (r_J^2 + r_L^2)) fc(r_J) fc(r_L)
//            over eta in {0.005, 0.02}, zeta in {1, 2, 4, 16}, lam = +-1 (16 functions)
//   y = w3 . silu(W2 silu(W1 xhat + b1) + b2) + b3,  xhat = (f - mean) * rstd,  silu(z) = z/(1 + e^-z)
// Parameters packed W1[H][K], b1[H], W2[H][H], b2[H], w3[H], b3 (6337 floats
// for K = 32, H = 64): they sit in LDS, and FMA chains carry a point through the
// layers.  The layers are 32x64 and 64x64 -- far below an MFMA tile's worth of reuse
// per point -- and the whole forward over a cell is microseconds, so plain FMA is the
// right tool here.
// Training (FP32, full batch): deltas per point, then all gradient sums over points
// in one pass over point chunks, with double partial sums and a fixed-order second
// pass (deterministic), then Adam.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <type_traits>

#include "sq_kernels.h"
#include "sq_projectors.h"

namespace sqamd {

namespace {

template <int K, int H>
constexpr int param_count() { return H * K + H + H * H + H + H + 1; }

// float -> bfloat16 -> float, round to nearest even (finite inputs)
__device__ __forceinline__ float to_bf16(float x)
{
    unsigned u = __float_as_uint(x);
    u = (u + 0x7FFFu + ((u >> 16) & 1u)) & 0xFFFF0000u;
    return __uint_as_float(u);
}

constexpr int kRad = 16, kAng = 16, kMaxNb = 96;   // descriptor split; neighbours within rf of one point

constexpr int kBrick[3] = {8, 8, 4}, kCand = 512;   // points of a block; images a block lists at a time

// One point a thread, a brick of points a block.  The block first lists, in
// order, the images that can lie within rf of its brick, then every thread
// takes its neighbours from that list.  Bound by the exponentials of 14 neighbours and
// their pairs: the cell of 128 atoms takes 0.31 ms; 4.6 with each point against all 3348
// images.
__global__ void __launch_bounds__(256) mlp_features(const double4 *__restrict__ img, int nimg, int G0, int G1, int G2,
                                                    double h0, double h1, double h2, double R0, double R1, double R2,
                                                    double rf, float *__restrict__ out, int *__restrict__ overflow)
{
    __shared__ double cx[kCand], cy[kCand], cz[kCand];
    __shared__ int wcount[4];
    const int nb0 = (G0 + kBrick[0] - 1) / kBrick[0], nb1 = (G1 + kBrick[1] - 1) / kBrick[1];
    const int b = blockIdx.x, t = threadIdx.x, lane = t & 63, wave = t >> 6;
    const int i0 = b % nb0 * kBrick[0], j0 = b / nb0 % nb1 * kBrick[1], k0 = b / nb0 / nb1 * kBrick[2];
    const int i = i0 + t % kBrick[0], j = j0 + t / kBrick[0] % kBrick[1], k = k0 + t / (kBrick[0] * kBrick[1]);
    const bool inside = i < G0 && j < G1 && k < G2;
    const double x = h0 * i - R0, y = h1 * j - R1, z = h2 * k - R2;
    // the brick's corners, and a bound that rounding cannot bring an image of a neighbour past
    const double xa = h0 * i0 - R0, xb = h0 * min(i0 + kBrick[0], G0) - R0;
    const double ya = h1 * j0 - R1, yb = h1 * min(j0 + kBrick[1], G1) - R1;
    const double za = h2 * k0 - R2, zb = h2 * min(k0 + kBrick[2], G2) - R2;
    const double reach = rf * rf * (1.0 + 1e-6);
    const double s = rf / (kRad - 1);
    double f[kRad + kAng];
#pragma unroll
    for (int q = 0; q < kRad + kAng; q++) f[q] = 0.0;
    double nx[kMaxNb], ny[kMaxNb], nz[kMaxNb], nr[kMaxNb], nf[kMaxNb];
    int nn = 0, listed = 0;
    for (int base = 0; base < nimg; base += 256) {
        double4 X = make_double4(0.0, 0.0, 0.0, 0.0);
        bool near = false;
        if (base + t < nimg) {
            X = img[base + t];
            const double ex = fmax(0.0, fmax(xa - X.x, X.x - xb)), ey = fmax(0.0, fmax(ya - X.y, X.y - yb));
            const double ez = fmax(0.0, fmax(za - X.z, X.z - zb));
            near = ex * ex + ey * ey + ez * ez <= reach;
        }
        const unsigned long long m = __ballot(near);
        if (lane == 0) wcount[wave] = __popcll(m);
        __syncthreads();
        int at = listed + __popcll(m & ((1ull << lane) - 1));
        for (int w = 0; w < 4; w++) {
            if (w < wave) at += wcount[w];
            listed += wcount[w];
        }
        if (near) { cx[at] = X.x; cy[at] = X.y; cz[at] = X.z; }
        __syncthreads();
        if (listed <= kCand - 256 && base + 256 < nimg) continue;   // room for the next 256
        if (inside)
            for (int a = 0; a < listed; a++) {
                const double dx = cx[a] - x, dy = cy[a] - y, dz = cz[a] - z;
                const double r = sqrt(dx * dx + dy * dy + dz * dz);
                if (!(r < rf)) continue;
                const double fc = 0.5 * (cos(M_PI * r / rf) + 1.0);
#pragma unroll
                for (int q = 0; q < kRad; q++) {
                    const double u = (r - q * rf / (kRad - 1)) / s;
                    f[q] += exp(-(u * u)) * fc;
                }
                if (nn < kMaxNb) { nx[nn] = dx; ny[nn] = dy; nz[nn] = dz; nr[nn] = r; nf[nn] = fc; }
                nn++;
            }
        listed = 0;
        __syncthreads();
    }
    if (!inside) return;
    if (nn > kMaxNb) { atomicAdd(overflow, 1); nn = kMaxNb; }
    const double eta[2] = {0.005, 0.02};
    for (int a = 0; a < nn; a++) {
        const double ax = nx[a], ay = ny[a], az = nz[a], ar = nr[a], af = nf[a];
        for (int c2 = a + 1; c2 < nn; c2++) {
            const double c = (ax * nx[c2] + ay * ny[c2] + az * nz[c2]) / (ar * nr[c2]);
            const double rr = ar * ar + nr[c2] * nr[c2];
            const double w = af * nf[c2];
#pragma unroll
            for (int ie = 0; ie < 2; ie++) {
                const double e = exp(-eta[ie] * rr) * w;
#pragma unroll
                for (int il = 0; il < 2; il++) {
                    const double p1 = 1.0 + (il ? -c : c), p2 = p1 * p1, p4 = p2 * p2, p16 = (p4 * p4) * (p4 * p4);
                    // zeta = 1, 2, 4, 16 with 2^(1-zeta)
                    f[kRad + (ie * 4 + 0) * 2 + il] += p1 * e;
                    f[kRad + (ie * 4 + 1) * 2 + il] += 0.5 * p2 * e;
                    f[kRad + (ie * 4 + 2) * 2 + il] += 0.125 * p4 * e;
                    f[kRad + (ie * 4 + 3) * 2 + il] += 0x1p-15 * p16 * e;
                }
            }
        }
    }
    const long p = ((long)k * G1 + j) * G0 + i;
#pragma unroll
    for (int q = 0; q < kRad + kAng; q++) out[p * (kRad + kAng) + q] = (float)f[q];
}

// A point a thread, a brick of points a block, which lists in order the images whose box
// meets the brick.  A point's sum runs over its images in order, so it is the host's
// (build_atomic_density), bit for bit.  Bound by the bisection's chain of loads, the more
// the fewer bricks a cell has, so four images' bisections run side by side (two bricks
// of 108 points: 0.58 ms, 0.67 one after the other; 660 points: 0.18 and 0.25).  The
// cell of 128 atoms takes 72 us, and 3 ms on 16 host threads.
constexpr int kBeside = 4;

__global__ void __launch_bounds__(256) superposed_density(const DensityImage *__restrict__ img, int nimg,
                                                          const DensityType *__restrict__ types,
                                                          const double *__restrict__ tab, int G0, int G1, int G2, double h0,
                                                          double h1, double h2, double R0, double R1, double R2,
                                                          double *__restrict__ rho, int *__restrict__ status)
{
    __shared__ int list[kCand], wcount[4];
    const int nb0 = (G0 + kBrick[0] - 1) / kBrick[0], nb1 = (G1 + kBrick[1] - 1) / kBrick[1];
    const int b = blockIdx.x, t = threadIdx.x, lane = t & 63, wave = t >> 6;
    const int i0 = b % nb0 * kBrick[0], j0 = b / nb0 % nb1 * kBrick[1], k0 = b / nb0 / nb1 * kBrick[2];
    const int i = i0 + t % kBrick[0], j = j0 + t / kBrick[0] % kBrick[1], k = k0 + t / (kBrick[0] * kBrick[1]);
    const bool inside = i < G0 && j < G1 && k < G2;
    double sum = 0.0;
    int listed = 0;
    for (int base = 0; base < nimg; base += 256) {
        bool near = false;
        if (base + t < nimg) {
            const DensityImage &im = img[base + t];
            near = im.lo[0] < i0 + kBrick[0] && im.hi[0] >= i0 && im.lo[1] < j0 + kBrick[1] && im.hi[1] >= j0 &&
                   im.lo[2] < k0 + kBrick[2] && im.hi[2] >= k0;
        }
        const unsigned long long m = __ballot(near);
        if (lane == 0) wcount[wave] = __popcll(m);
        __syncthreads();
        int at = listed + __popcll(m & ((1ull << lane) - 1));
        for (int w = 0; w < 4; w++) {
            if (w < wave) at += wcount[w];
            listed += wcount[w];
        }
        if (near) list[at] = base + t;
        __syncthreads();
        if (listed <= kCand - 256 && base + 256 < nimg) continue;   // room for the next 256
        if (inside)
            for (int a = 0; a < listed; a += kBeside) {
                const double *x[kBeside];
                double r[kBeside];
                int n[kBeside], lo[kBeside], hi[kBeside];   // bisection: lower_bound; n = 0: nothing to add
#pragma unroll
                for (int u = 0; u < kBeside; u++) {
                    const DensityImage &im = img[list[min(a + u, listed - 1)]];
                    const DensityType T = types[im.at];
                    x[u] = tab + T.off;
                    const double dx = h0 * i - R0 - im.X[0], dy = h1 * j - R1 - im.X[1], dz = h2 * k - R2 - im.X[2];
                    r[u] = sqrt(dx * dx + dy * dy + dz * dz);
                    const bool in = a + u < listed && i >= im.lo[0] && i <= im.hi[0] && j >= im.lo[1] && j <= im.hi[1] &&
                                    k >= im.lo[2] && k <= im.hi[2] && r[u] <= x[u][T.n - 1];
                    if (in && !(r[u] >= x[u][0])) *status = 3;
                    n[u] = in && r[u] >= x[u][0] ? T.n : 0;
                    lo[u] = 0;
                    hi[u] = n[u];
                }
                for (bool more = true; more;) {
                    more = false;
#pragma unroll
                    for (int u = 0; u < kBeside; u++) {
                        const int mid = (lo[u] + hi[u]) >> 1;
                        const bool open = lo[u] < hi[u], less = x[u][mid] < r[u];   // x[0] of a closed one without knots
                        lo[u] = open && less ? mid + 1 : lo[u];
                        hi[u] = open && !less ? mid : hi[u];
                        more = more || lo[u] < hi[u];
                    }
                }
#pragma unroll
                for (int u = 0; u < kBeside; u++)
                    if (n[u]) {
                        double v;
                        spline_cubic(x[u], x[u] + n[u], x[u] + 2 * n[u], n[u], lo[u], r[u], &v);
                        sum += v;
                    }
            }
        listed = 0;
        __syncthreads();
    }
    if (inside) rho[((long)k * G1 + j) * G0 + i] = sum;
}

__global__ void __launch_bounds__(256) guess_add(double *__restrict__ rho, const float *__restrict__ y,
                                                 const double *__restrict__ sum, double ne, double dV, double scale, long n)
{
    const double f = ne / (*sum * dV);
    for (long q = blockIdx.x * 256L + threadIdx.x; q < n; q += gridDim.x * 256L)
        rho[q] = fmax(0.0, rho[q] * f + scale * (double)y[q]);
}

__global__ void __launch_bounds__(256) guess_scale(double *__restrict__ rho, const double *__restrict__ sum, double ne,
                                                   double dV, long n)
{
    const double tot = *sum * dV;
    if (!(tot > 0.0)) return;
    const double f = ne / tot;
    for (long q = blockIdx.x * 256L + threadIdx.x; q < n; q += gridDim.x * 256L) rho[q] *= f;
}

__device__ __forceinline__ float silu(float z) { return z / (1.0f + expf(-z)); }
__device__ __forceinline__ float dsilu(float z)
{
    const float sg = 1.0f / (1.0f + expf(-z));
    return sg * (1.0f + z * (1.0f - sg));
}

// A point's layers by four wavefronts, a quarter of each layer's outputs a wavefront
// (a lane a point, 64 points a block), four outputs' chains side by side; the
// activations change hands through LDS.  Each output's chain runs over its inputs in
// order.  Bound by the chains' latency where the rows are few: 18720 rows take 30 us, and
// 60 with a point's whole network in one thread; 153504 rows in BF16 86 and 89.
constexpr int kPts = 64, kOut = 4;   // points of a block; outputs side by side

template <int K, int H, bool B16>
__global__ void __launch_bounds__(256) mlp_forward(const float *__restrict__ X, long N, const float *__restrict__ P,
                                                   const float *__restrict__ mean, const float *__restrict__ rstd,
                                                   float *__restrict__ H1, float *__restrict__ H2, float *__restrict__ Z1,
                                                   float *__restrict__ Z2, float *__restrict__ Y)
{
    constexpr int NP = param_count<K, H>(), Q = H / 4;
    static_assert(K % 4 == 0 && Q % kOut == 0, "rows of four weights, quarters of four outputs");
    __shared__ __attribute__((aligned(16))) float w[NP];
    __shared__ float ex[H][kPts];
    for (int q = threadIdx.x; q < NP; q += blockDim.x) w[q] = B16 ? to_bf16(P[q]) : P[q];
    const int lane = threadIdx.x & 63, o0 = (threadIdx.x >> 6) * Q;
    const long n = (long)blockIdx.x * kPts + lane;
    const bool has = n < N;
    const float *W1 = w, *b1 = W1 + H * K, *W2 = b1 + H, *b2 = W2 + H * H, *w3 = b2 + H, *b3 = w3 + H;
    float a[H];   // inputs of the layer at hand
    {
        const float *x = X + (has ? n : N - 1) * K;
#pragma unroll
        for (int q = 0; q < K; q++) {
            float v = x[q];
            if (mean) v = (v - mean[q]) * rstd[q];
            a[q] = B16 ? to_bf16(v) : v;
        }
    }
    __syncthreads();
    // outputs o .. o + kOut - 1 of a layer with M inputs
    auto chains = [&](const float *W, const float *b, auto M, int o, float s[kOut]) {
        constexpr int n_in = decltype(M)::value;
#pragma unroll
        for (int k = 0; k < kOut; k++) s[k] = b[o + k];
#pragma unroll
        for (int q = 0; q < n_in; q += 4)
#pragma unroll
            for (int k = 0; k < kOut; k++) {
                const float4 c = *reinterpret_cast<const float4 *>(W + (o + k) * n_in + q);
                s[k] = fmaf(c.x, a[q], s[k]);
                s[k] = fmaf(c.y, a[q + 1], s[k]);
                s[k] = fmaf(c.z, a[q + 2], s[k]);
                s[k] = fmaf(c.w, a[q + 3], s[k]);
            }
    };
    // kOut outputs' activations to LDS, and to the rows a backward pass needs
    auto activate = [&](int o, const float s[kOut], float *Hn, float *Zn) {
        float t[kOut];
#pragma unroll
        for (int k = 0; k < kOut; k++) {
            t[k] = silu(s[k]);
            if (B16) t[k] = to_bf16(t[k]);
            ex[o + k][lane] = t[k];
        }
        if (Hn && has) *reinterpret_cast<float4 *>(Hn + n * H + o) = make_float4(t[0], t[1], t[2], t[3]);
        if (Zn && has) *reinterpret_cast<float4 *>(Zn + n * H + o) = make_float4(s[0], s[1], s[2], s[3]);
    };
#pragma unroll 1
    for (int o = o0; o < o0 + Q; o += kOut) {
        float s[kOut];
        chains(W1, b1, std::integral_constant<int, K>(), o, s);
        activate(o, s, H1, Z1);
    }
    __syncthreads();
#pragma unroll
    for (int i = 0; i < H; i++) a[i] = ex[i][lane];
    __syncthreads();
#pragma unroll 1
    for (int o = o0; o < o0 + Q; o += kOut) {
        float s[kOut];
        chains(W2, b2, std::integral_constant<int, H>(), o, s);
        activate(o, s, H2, Z2);
    }
    __syncthreads();
    if (o0 || !has) return;
    float y = b3[0];
#pragma unroll
    for (int j = 0; j < H; j++) y = fmaf(w3[j], ex[j][lane], y);
    Y[n] = y;
}

// L = (1/2N) sum (y - t)^2: d3 = (y - t)/N, d2 = d3 w3 silu'(z2), d1 = (W2^T d2) silu'(z1);
// split as the forward pass (18720 rows: 17 us, and 36 with a point a thread)
template <int K, int H>
__global__ void __launch_bounds__(256) mlp_deltas(const float *__restrict__ Z1, const float *__restrict__ Z2,
                                                  const float *__restrict__ Y, const float *__restrict__ T, long N,
                                                  const float *__restrict__ P, float *__restrict__ D1,
                                                  float *__restrict__ D2, float *__restrict__ D3)
{
    constexpr int Q = H / 4;
    __shared__ __attribute__((aligned(16))) float w2[H * H];
    __shared__ float w3[H], ex[H][kPts];
    const float *W2g = P + H * K + H, *w3g = W2g + H * H + H;
    for (int q = threadIdx.x; q < H * H; q += blockDim.x) w2[q] = W2g[q];
    for (int q = threadIdx.x; q < H; q += blockDim.x) w3[q] = w3g[q];
    __syncthreads();
    const int lane = threadIdx.x & 63, o0 = (threadIdx.x >> 6) * Q;
    const long n = (long)blockIdx.x * kPts + lane;
    const bool has = n < N;
    const long row = (has ? n : N - 1) * H;
    const float d3 = has ? (Y[n] - T[n]) / (float)N : 0.0f;
    if (has && o0 == 0) D3[n] = d3;
#pragma unroll
    for (int o = o0; o < o0 + Q; o += kOut) {
        const float4 z = *reinterpret_cast<const float4 *>(Z2 + row + o);
        const float zz[kOut] = {z.x, z.y, z.z, z.w};
        float d[kOut];
#pragma unroll
        for (int k = 0; k < kOut; k++) {
            d[k] = d3 * w3[o + k] * dsilu(zz[k]);
            ex[o + k][lane] = d[k];
        }
        if (has) *reinterpret_cast<float4 *>(D2 + row + o) = make_float4(d[0], d[1], d[2], d[3]);
    }
    __syncthreads();
#pragma unroll 1
    for (int o = o0; o < o0 + Q; o += kOut) {
        float s[kOut] = {0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll 16
        for (int j = 0; j < H; j++) {
            const float4 c = *reinterpret_cast<const float4 *>(w2 + j * H + o);
            const float d = ex[j][lane];
            s[0] = fmaf(c.x, d, s[0]);
            s[1] = fmaf(c.y, d, s[1]);
            s[2] = fmaf(c.z, d, s[2]);
            s[3] = fmaf(c.w, d, s[3]);
        }
        const float4 z = *reinterpret_cast<const float4 *>(Z1 + row + o);
        if (has)
            *reinterpret_cast<float4 *>(D1 + row + o) =
                make_float4(s[0] * dsilu(z.x), s[1] * dsilu(z.y), s[2] * dsilu(z.z), s[3] * dsilu(z.w));
    }
}

// The gradient sums over the points of one chunk, in double: W1 += d1 x^T, b1 +=
// d1, W2 += d2 h1^T, b2 += d2, w3 += h2 d3, b3 += d3 and, last, sum d3^2.  A tile of
// points' rows lies in LDS; a thread keeps a 4 x 4 piece of W2 and a 4 x 2 piece of
// W1 in registers, so a point costs it four LDS reads and 24 multiply-adds, and a
// column sum is one thread's.  Bound by the latency of a point's reads, with a
// wavefront a SIMD: 18720 points take 33 us and the sum over chunks 6; one launch a
// matrix, a thread an element and every operand from L2 took 58 + 16 each, seven times.
constexpr int kGradTile = 32;

template <int K, int H>
__global__ void __launch_bounds__(256) grad_partial(const float *__restrict__ X, const float *__restrict__ H1,
                                                    const float *__restrict__ H2, const float *__restrict__ D1,
                                                    const float *__restrict__ D2, const float *__restrict__ D3, long N,
                                                    long chunk, double *__restrict__ partial)
{
    static_assert(H == 64 && K == 32, "256 threads cover a 64 x 64 and a 64 x 32 matrix");
    __shared__ __attribute__((aligned(16))) float sx[kGradTile * K], sh1[kGradTile * H], sh2[kGradTile * H],
        sd1[kGradTile * H], sd2[kGradTile * H], sd3[kGradTile];
    const int t = threadIdx.x, row = t / 16 * 4, c2 = t % 16 * 4, c1 = t % 16 * 2, lane = t & 63, wave = t >> 6;
    double g2[4][4] = {}, g1[4][2] = {}, col = 0.0;
    const long n0 = blockIdx.x * chunk, n1 = min(N, n0 + chunk);
    for (long base = n0; base < n1; base += kGradTile) {
        const int rows = (int)min((long)kGradTile, n1 - base);
        for (int q = t; q < rows * H; q += 256) {
            sh1[q] = H1[base * H + q];
            sh2[q] = H2[base * H + q];
            sd1[q] = D1[base * H + q];
            sd2[q] = D2[base * H + q];
        }
        for (int q = t; q < rows * K; q += 256) sx[q] = X[base * K + q];
        if (t < rows) sd3[t] = D3[base + t];
        __syncthreads();
#pragma unroll 4
        for (int n = 0; n < rows; n++) {
            const float4 a2 = *(const float4 *)(sd2 + n * H + row), b2 = *(const float4 *)(sh1 + n * H + c2);
            const float4 a1 = *(const float4 *)(sd1 + n * H + row);
            const float2 b1 = *(const float2 *)(sx + n * K + c1);
            const double p2[4] = {a2.x, a2.y, a2.z, a2.w}, q2[4] = {b2.x, b2.y, b2.z, b2.w};
            const double p1[4] = {a1.x, a1.y, a1.z, a1.w}, q1[2] = {b1.x, b1.y};
#pragma unroll
            for (int i = 0; i < 4; i++) {
#pragma unroll
                for (int j = 0; j < 4; j++) g2[i][j] = fma(p2[i], q2[j], g2[i][j]);
#pragma unroll
                for (int j = 0; j < 2; j++) g1[i][j] = fma(p1[i], q1[j], g1[i][j]);
            }
            // column sums: b1, b2 and w3 by a wavefront each, b3 and the squares by two lanes of the last
            const double d3 = sd3[n];
            if (wave == 0) col += sd1[n * H + lane];
            else if (wave == 1) col += sd2[n * H + lane];
            else if (wave == 2) col = fma((double)sh2[n * H + lane], d3, col);
            else col = fma(d3, lane ? d3 : 1.0, col);
        }
        __syncthreads();
    }
    double *const out = partial + (size_t)blockIdx.x * (param_count<K, H>() + 1);
    double *const oW2 = out + H * K + H, *const ob2 = oW2 + H * H;
#pragma unroll
    for (int i = 0; i < 4; i++) {
#pragma unroll
        for (int j = 0; j < 4; j++) oW2[(row + i) * H + c2 + j] = g2[i][j];
#pragma unroll
        for (int j = 0; j < 2; j++) out[(row + i) * K + c1 + j] = g1[i][j];
    }
    if (wave == 0) out[H * K + lane] = col;
    else if (wave == 1) ob2[lane] = col;
    else if (wave == 2) ob2[H + lane] = col;
    else if (lane < 2) ob2[2 * H + lane] = col;
}

// out[e] = sum of the chunks' partials: 16 threads an element, each over every 16th
// chunk, then in order
__global__ void __launch_bounds__(1024) sum_chunks(const double *__restrict__ partial, int nchunk, int m,
                                                   double *__restrict__ out)
{
    __shared__ double sm[16][64];
    const int lane = threadIdx.x & 63, part = threadIdx.x >> 6, e = blockIdx.x * 64 + lane;
    double s = 0.0;
    if (e < m)
#pragma unroll 8
        for (int c = part; c < nchunk; c += 16) s += partial[(size_t)c * m + e];
    sm[part][lane] = s;
    __syncthreads();
    if (part || e >= m) return;
    for (int k = 1; k < 16; k++) s += sm[k][lane];
    out[e] = s;
}

__global__ void adam_step(float *__restrict__ p, const double *__restrict__ g, float *__restrict__ m, float *__restrict__ v,
                          int n, float lr, float b1, float b2, float eps, float c1, float c2)
{
    const int q = blockIdx.x * blockDim.x + threadIdx.x;
    if (q >= n) return;
    const float gq = (float)g[q];
    const float mq = b1 * m[q] + (1.0f - b1) * gq;
    const float vq = b2 * v[q] + (1.0f - b2) * gq * gq;
    m[q] = mq;
    v[q] = vq;
    p[q] -= lr * (mq / c1) / (sqrtf(vq / c2) + eps);
}

}  // namespace

int mlp_param_count(int K, int H) { return H * K + H + H * H + H + H + 1; }

hipError_t launch_mlp_features(const double4 *img, int nimg, const int G[3], const double h[3], const double R[3], int K,
                               double rf, float *out, int *overflow, hipStream_t st)
{
    if (K != kMlpK || kRad + kAng != kMlpK) return hipErrorInvalidValue;
    unsigned blocks = 1;
    for (int d = 0; d < 3; d++) blocks *= (G[d] + kBrick[d] - 1) / kBrick[d];
    hipLaunchKernelGGL(mlp_features, dim3(blocks), dim3(256), 0, st, img, nimg, G[0], G[1], G[2], h[0], h[1], h[2], R[0],
                       R[1], R[2], rf, out, overflow);
    return hipGetLastError();
}

hipError_t launch_superposed(const DensityImage *img, int nimg, const DensityType *types, const double *tab, const int G[3],
                             const double h[3], const double R[3], double *rho, int *status, hipStream_t st)
{
    unsigned blocks = 1;
    for (int d = 0; d < 3; d++) blocks *= (G[d] + kBrick[d] - 1) / kBrick[d];
    hipLaunchKernelGGL(superposed_density, dim3(blocks), dim3(256), 0, st, img, nimg, types, tab, G[0], G[1], G[2], h[0],
                       h[1], h[2], R[0], R[1], R[2], rho, status);
    return hipGetLastError();
}

static dim3 cell_grid(long n) { return dim3((unsigned)std::min<long>(4096, (n + 255) / 256)); }

hipError_t launch_guess_add(double *rho, const float *y, const double *sum, double ne, double dV, double scale, long n,
                            hipStream_t st)
{
    hipLaunchKernelGGL(guess_add, cell_grid(n), dim3(256), 0, st, rho, y, sum, ne, dV, scale, n);
    return hipGetLastError();
}

hipError_t launch_guess_scale(double *rho, const double *sum, double ne, double dV, long n, hipStream_t st)
{
    hipLaunchKernelGGL(guess_scale, cell_grid(n), dim3(256), 0, st, rho, sum, ne, dV, n);
    return hipGetLastError();
}

hipError_t launch_mlp_forward(const float *X, long N, const float *P, const float *mean, const float *rstd, float *H1,
                              float *H2, float *Z1, float *Z2, float *Y, int bf16, hipStream_t st)
{
    if (N <= 0) return hipSuccess;
    const dim3 g((unsigned)((N + kPts - 1) / kPts)), b(256);
    if (bf16) hipLaunchKernelGGL((mlp_forward<kMlpK, kMlpH, true>), g, b, 0, st, X, N, P, mean, rstd, H1, H2, Z1, Z2, Y);
    else hipLaunchKernelGGL((mlp_forward<kMlpK, kMlpH, false>), g, b, 0, st, X, N, P, mean, rstd, H1, H2, Z1, Z2, Y);
    return hipGetLastError();
}

hipError_t launch_mlp_deltas(const float *Z1, const float *Z2, const float *Y, const float *T, long N, const float *P,
                             float *D1, float *D2, float *D3, hipStream_t st)
{
    if (N <= 0) return hipSuccess;
    hipLaunchKernelGGL((mlp_deltas<kMlpK, kMlpH>), dim3((unsigned)((N + kPts - 1) / kPts)), dim3(256), 0, st, Z1, Z2, Y, T, N, P,
                       D1, D2, D3);
    return hipGetLastError();
}

// Chunks of the gradient sums: one a CU where each then has 32 points or more
int mlp_grad_chunks(long N) { return (int)std::max<long>(1, std::min<long>(256, N / kGradTile)); }

hipError_t launch_mlp_grad(const float *X, const float *H1, const float *H2, const float *D1, const float *D2,
                           const float *D3, long N, double *partial, double *out, hipStream_t st)
{
    if (N <= 0) return hipErrorInvalidValue;
    const int nchunk = mlp_grad_chunks(N), m = mlp_param_count(kMlpK, kMlpH) + 1;
    hipLaunchKernelGGL((grad_partial<kMlpK, kMlpH>), dim3(nchunk), dim3(256), 0, st, X, H1, H2, D1, D2, D3, N,
                       (N + nchunk - 1) / nchunk, partial);
    hipLaunchKernelGGL(sum_chunks, dim3((m + 63) / 64), dim3(1024), 0, st, partial, nchunk, m, out);
    return hipGetLastError();
}

hipError_t launch_adam(float *p, const double *g, float *m, float *v, int n, float lr, int t, hipStream_t st)
{
    const float b1 = 0.9f, b2 = 0.999f;
    const float c1 = 1.0f - powf(b1, (float)t), c2 = 1.0f - powf(b2, (float)t);
    hipLaunchKernelGGL(adam_step, dim3((unsigned)((n + 255) / 256)), dim3(256), 0, st, p, g, m, v, n, lr, b1, b2, 1e-8f, c1, c2);
    return hipGetLastError();
}

}  // namespace sqamd
