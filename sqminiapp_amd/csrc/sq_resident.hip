// sq_resident.hip -- the resident Lanczos kernel (FP64): one workgroup runs the whole recurrence of one grid node with its Lanczos
// vectors on chip; one thread owns one (x,y) column of the cube.
//   v      the current vector: the lower nl planes in LDS, the rest in a slice
//          of scratch (29^3: 17 of 29 planes);
//   r      the previous vector, then the vector being built: the thread's whole
//          column in registers, indexed statically (the z loops are unrolled to
//          NZ planes and guarded by the cube's nz).
// Per step: gather (one wavefront an image, image by image from a ticket) ->
// alpha -> r := -b r, scatter of chi alpha into r -> march over the planes, two at
// a time, r += (L + diag) v: the pair staged in LDS inside a zero halo gives the x
// and y neighbours, and its own values are pushed into the planes of r that they
// neighbour in z, so no window of v is held -> a = <v, r>, r -= a v, ||r||, v and r
// change places.  a is taken from r = H v - b v_prev, Paige's form of the
// recurrence: it equals <v, H v> up to rounding, v being orthogonal to v_prev.
//
// What it replaces: the batched kernel streams its vectors (B x 195 KB in FP64)
// through the Infinity Cache and moved 5.4 TB/s past the L2, the rate a plain
// copy reaches (5.1 TB/s), so the pass was bound by that
// traffic; here projector tables, the diagonal and the planes that do not fit LDS
// cross the L2 (29^3: 578 KB a node and step, 3.0 vectors where the batched kernel moves
// 13.8; the scratch planes are written past it every step).
//
// Projector tables: radial pairs (t0, t2) of each image's box trimmed to the
// reach of the radial functions, with kResPad zero planes below and above, so
// a group of four planes that meets the box needs no masks.  Images are sorted
// by the z of their centre: a column visits its images in that order, so at
// the wavefront level the k-th images of neighbouring columns lie at nearby
// heights and whole groups of planes are skipped together.
#include "sq_device_common.h"
#include "sq_resident.h"

namespace sqamd {

namespace {

// Cross-lane moves on the vector ALU (no LDS): rotate within rows of 16 lanes.
template <int N>
__device__ __forceinline__ double row_ror(double x)
{
    const int lo = __builtin_amdgcn_update_dpp(0, __double2loint(x), 0x120 + N, 0xf, 0xf, true);
    const int hi = __builtin_amdgcn_update_dpp(0, __double2hiint(x), 0x120 + N, 0xf, 0xf, true);
    return __hiloint2double(hi, lo);
}
// sum over each row of 16 lanes, in every lane of the row
__device__ __forceinline__ double row_sum(double x)
{
    x += row_ror<8>(x);
    x += row_ror<4>(x);
    x += row_ror<2>(x);
    x += row_ror<1>(x);
    return x;
}
__device__ __forceinline__ double lane_value(double x, int lane)
{
    return __hiloint2double(__builtin_amdgcn_readlane(__double2hiint(x), lane),
                            __builtin_amdgcn_readlane(__double2loint(x), lane));
}
// sum over the wavefront, the same value in every lane
__device__ __forceinline__ double wave_total(double x)
{
    x = row_sum(x);
    return (lane_value(x, 0) + lane_value(x, 16)) + (lane_value(x, 32) + lane_value(x, 48));
}

// Two values' sums over halves of the wavefront in one register: lanes 0-31
// hold a(l) + a(l+32), lanes 32-63 b(l-32) + b(l).
__device__ __forceinline__ double fold32(double a, double b)
{
    const auto l = __builtin_amdgcn_permlane32_swap(__double2loint(a), __double2loint(b), false, false);
    const auto h = __builtin_amdgcn_permlane32_swap(__double2hiint(a), __double2hiint(b), false, false);
    return __hiloint2double((int)h[0], (int)l[0]) + __hiloint2double((int)h[1], (int)l[1]);
}
// the same over neighbouring rows of 16 lanes: even rows hold a, odd rows b
__device__ __forceinline__ double fold16(double a, double b)
{
    const auto l = __builtin_amdgcn_permlane16_swap(__double2loint(a), __double2loint(b), false, false);
    const auto h = __builtin_amdgcn_permlane16_swap(__double2hiint(a), __double2hiint(b), false, false);
    return __hiloint2double((int)h[0], (int)l[0]) + __hiloint2double((int)h[1], (int)l[1]);
}

// Sum over the workgroup of one double a thread, every thread receiving it:
// wavefront partials through LDS, added as one row of NW values.  One barrier;
// the caller alternates between two buffers.
template <int NW>
__device__ __forceinline__ double group_sum(double x, double *red)
{
    x = wave_total(x);
    if ((threadIdx.x & 63) == 0) red[threadIdx.x >> 6] = x;
    __syncthreads();
    const int k = threadIdx.x & 15;
    const double s = row_sum(k < NW ? red[k] : 0.0);
    return lane_value(s, 0);
}

// LDS row pitch of the staged pair of planes: a halo of 6 on both sides fits to 33
// columns, and on a 29-column cube lanes that cross a row's end stay on consecutive banks.
// A pair brings both planes' neighbour in one read, which costs no more than the read
// of one plane's (29^3: march 63 thousand clocks a step plane by plane).
constexpr int kPitch = 45;

// Staged pairs of planes at a time: with two a plane pair costs one barrier, which is
// worth the planes of v it takes from LDS (29^3: march 57 -> 48 thousand clocks a step, the
// other phases 7 more) where one workgroup has the CU to itself.
constexpr int stage_buffers(int wg) { return wg == 1024 ? 2 : 1; }

// The launch parameters read afresh from the kernel-argument segment: each phase
// of a step takes its own opaque view, so its scalars live in that phase only.
// Kept alive across the step loop they overflow the scalar registers, and the
// stencil weights come back lane by lane in every plane.
typedef const __attribute__((address_space(4))) ResParams *ParamView;
__device__ __forceinline__ ParamView params()
{
    ParamView p = (ParamView)__builtin_amdgcn_kernarg_segment_ptr();
    asm volatile("" : "+s"(p));
    return p;
}
// a value the compiler may not look through
#define SQ_OPAQUE(x) asm volatile("" : "+s"(x))
#define SQ_OPAQUE_V(x) asm volatile("" : "+v"(x))

}  // namespace

// LDS tables of one node's images
struct ResLds {
    double A[kResMaxImages][6];      // gathered sums, then the scatter's coefficients
    double org[kResMaxImages][3];    // cube origin relative to the image's centre
    int lo[kResMaxImages];           // box origin in the cube, a byte an axis
    int dim[kResMaxImages];          // box size, a byte an axis; type
    int off[kResMaxImages];          // radial pair of cube point (0,0,0)
    unsigned char head[kResMaxImages];   // first entry of the same atom
    unsigned char next[kResMaxImages];   // next entry of the same atom, 255 at the last
    double red[2][16];
    int atom[kResMaxImages], id[kResMaxImages];
    unsigned char slot[kResMaxImages];   // force pass: the image's row of the record, 255 without one
    double ab[2][kMaxNqp + 1];           // early exit: the tridiagonal so far
    double g[kMatsubara][2];             // and the last check's Matsubara terms
    long next_row;
    int count, ticket, flag;
};

template <int WG, int NZ>
__global__ void __launch_bounds__(WG) __attribute__((amdgpu_waves_per_eu(4, 4))) lanczos_resident(ResParams)
{
    constexpr int NW = WG / 64, O = 6, NLM = 6, MW = kResMaxImages / 32;
    constexpr int PX = kPitch, NB = stage_buffers(WG);
    // planes a gather trip loads ahead: what the registers hold beside the column r (1024 threads,
    // 29^3: 168.7, 172.8 and 170.9 thousand clocks a step with 3, 4 and 2; 512 threads, 21^3: 99.6
    // and 98.8 with 3 and 4)
    constexpr int UG = WG == 1024 ? 3 : 4;
    constexpr int UC = 4;   // planes of a scatter group
    constexpr int UD = 4;   // planes of a dot or update chunk
    typedef double V2 __attribute__((ext_vector_type(2)));
    // LDS and device pointers by address space: a load from one or the other must
    // not be merged into a flat load
    typedef __attribute__((address_space(3))) double ST;
    typedef __attribute__((address_space(1))) double GT;
    typedef const __attribute__((address_space(1))) V2 GV2;
    typedef const __attribute__((address_space(1))) char GC;   // the table by 32-bit byte offsets
    typedef __attribute__((address_space(3))) V2 SV2;
    __shared__ ResLds S;
    extern __shared__ __align__(16) unsigned char smem[];
    ST *const vl = (ST *)smem;   // [nl][ncol], then the two staged planes
    // N planes of a column of v from z0 on; planes past the cube repeat its last.  nl is a
    // multiple of the chunks or nz, so a chunk lies in LDS or in scratch as a whole.
    auto load_planes = [](auto &v, int z0, int col, const ST *lds, const GT *mem, int nl, int nz, int ncol) {
        constexpr int N = sizeof(v) / sizeof(double);
        if (z0 < nl) {
#pragma unroll
            for (int u = 0; u < N; u++) v[u] = lds[min(z0 + u, nz - 1) * ncol + col];
        } else {
#pragma unroll
            for (int u = 0; u < N; u++) v[u] = (mem + min(z0 + u, nz - 1) * ncol)[(unsigned)col];
        }
    };

    const int tid = threadIdx.x, lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    // this thread's column, packed (threads past the last do the last column's work
    // over again and store the same values; only the sums leave them out); each phase unpacks
    // it behind an opaque copy, so what it derives does not stay alive between phases
    int cij;
    bool has, live;           // the thread, its wavefront own columns
    {
        const ParamView P = params();
        const int nx = P->nloc[0], ny = P->nloc[1], ncol = nx * ny;
        has = tid < ncol;
        live = wave * 64 < ncol;
        const int col = has ? tid : ncol - 1;
        cij = col / nx << 16 | (col % nx);
        ST *const stage = vl + ((P->nl * ncol + 1) & ~1);
        for (int q = tid; q < 2 * NB * PX * (ny + 2 * O); q += WG) stage[q] = 0;   // the halo stays zero
    }
    int q_at = 0;
    for (;;) {
        // ---- work queue: eight contiguous parts of the node range, one per XCD
        if (tid == 0) {
            const ParamView P = params();
            const long part = (P->node_count + 7) / 8;
            const int home = blockIdx.x & 7;
            long r = -1;
            for (; q_at < 8; q_at++) {
                const int x = (home + q_at) & 7;
                const long lo = x * part, hi = min(P->node_count, lo + part);
                if (lo >= hi) continue;
                const long k = atomicAdd(&P->queue[x], 1);
                if (lo + k < hi) { r = lo + k; break; }
            }
            S.next_row = r;
            S.count = 0;
            S.ticket = 0;
        }
        __syncthreads();
        const int row = __builtin_amdgcn_readfirstlane((int)S.next_row);
        if (row < 0) break;
        int id;
        {
            const ParamView P = params();
            id = __builtin_amdgcn_readfirstlane(P->node_list ? P->node_list[row] : (int)P->node_begin + row);
        }
        int ebase;               // the cube's first point in the extended diagonal
        unsigned cmask[MW];      // the images whose projector reaches the column
        int nimg;
        {
            const ParamView P = params();
            const int nx = P->nloc[0], ny = P->nloc[1], nz = P->nloc[2], nl = P->nl, ncol = nx * ny;
            const int lxb = P->box_n[0], lyb = P->box_n[1];
            const int c0 = P->box0[0] + id % lxb - P->hw[0], c1 = P->box0[1] + id / lxb % lyb - P->hw[1],
                      c2 = P->box0[2] + id / (lxb * lyb) - P->hw[2];
            const double hx = P->hgrid[0], hy = P->hgrid[1], hz = P->hgrid[2];
            const int ci = cij & 0xffff, cj = cij >> 16, col = cj * nx + ci;
            // ---- images whose box meets the cube, in list order
            for (int base = 0; base < P->n_images; base += WG) {
                const int g = base + tid;
                bool hit = false;
                ResImage im;
                if (g < P->n_images) {
                    im = P->img[g];
                    hit = im.lo[0] <= c0 + nx - 1 && im.lo[0] + im.dim[0] - 1 >= c0 && im.lo[1] <= c1 + ny - 1 &&
                          im.lo[1] + im.dim[1] - 1 >= c1 && im.lo[2] <= c2 + nz - 1 && im.lo[2] + im.dim[2] - 1 >= c2;
                }
                const unsigned long long bal = __ballot(hit);
                const int before = __popcll(bal & ((1ull << lane) - 1ull));
                int *wcnt = reinterpret_cast<int *>(S.red);
                if (lane == 0) wcnt[wave] = __popcll(bal);
                __syncthreads();
                int li = S.count + before;
                for (int w = 0; w < wave; w++) li += wcnt[w];
                if (hit && li < kResMaxImages) {
                    const int lx = im.lo[0] - c0, ly = im.lo[1] - c1, lz = im.lo[2] - c2;
                    S.lo[li] = (lx & 255) | (ly & 255) << 8 | (lz & 255) << 16;
                    S.dim[li] = im.dim[0] | im.dim[1] << 8 | im.dim[2] << 16 | im.type << 24;
                    S.off[li] = im.off + ((kResPad - lz) * im.dim[1] - ly) * im.dim[0] - lx;
                    S.org[li][0] = hx * c0 - P->range[0] - im.cen[0];
                    S.org[li][1] = hy * c1 - P->range[1] - im.cen[1];
                    S.org[li][2] = hz * c2 - P->range[2] - im.cen[2];
                    S.atom[li] = im.atom;
                    S.id[li] = im.id;
                    S.slot[li] = 255;
                }
                __syncthreads();
                if (tid == 0) {
                    int t = S.count;
                    for (int w = 0; w < NW; w++) t += wcnt[w];
                    S.count = t;
                }
                __syncthreads();
            }
            nimg = __builtin_amdgcn_readfirstlane(S.count);
            if (nimg > kResMaxImages) {   // the host checked the geometry; flag the node
                __syncthreads();
                if (tid == 0) P->status[id] = 4;
                continue;
            }
            // ---- images of one atom, linked in list order
            if (tid < nimg) {
                int h = tid, nxt = 255;
                for (int q = nimg - 1; q >= 0; q--)
                    if (S.atom[q] == S.atom[tid]) {
                        if (q > tid) nxt = q;
                        h = min(h, q);
                    }
                S.head[tid] = (unsigned char)h;
                S.next[tid] = (unsigned char)nxt;
            }
            // ---- force pass: the images whose box holds the node get a row of the record (the
            // host counted the whole boxes, so the trimmed ones never exceed rec_slots)
            if (P->rec) {
                if (tid == 0) {
                    int n = 0;
                    for (int q = 0; q < nimg; q++) {
                        const int lo = S.lo[q], dm = S.dim[q];
                        const int bx = P->hw[0] - (signed char)(lo & 255), by = P->hw[1] - (signed char)(lo >> 8 & 255),
                                  bz = P->hw[2] - (signed char)(lo >> 16 & 255);
                        if ((unsigned)bx < (unsigned)(dm & 255) && (unsigned)by < (unsigned)(dm >> 8 & 255) &&
                            (unsigned)bz < (unsigned)(dm >> 16 & 255)) {
                            if (n < P->rec_slots) {
                                S.slot[q] = (unsigned char)n;
                                P->rec_img[(long)row * P->rec_slots + n] = S.id[q];
                            }
                            n++;
                        }
                    }
                    for (int q = n; q < P->rec_slots; q++) P->rec_img[(long)row * P->rec_slots + q] = -1;
                }
                __syncthreads();
            }
#pragma unroll
            for (int w = 0; w < MW; w++) cmask[w] = 0u;
            const double xi = hx * ci, yj = hy * cj;
            for (int li = 0; li < nimg; li++) {
                const int lo = S.lo[li], dm = S.dim[li];
                const int bx = ci - (signed char)(lo & 255), by = cj - (signed char)(lo >> 8 & 255);
                const float x = (float)(S.org[li][0] + xi), y = (float)(S.org[li][1] + yj);
                const bool in = (unsigned)bx < (unsigned)(dm & 255) && (unsigned)by < (unsigned)(dm >> 8 & 255) &&
                                x * x + y * y < P->rt2;
#pragma unroll
                for (int w = 0; w < MW; w++)
                    if (w == (li >> 5) && in) cmask[w] |= 1u << (li & 31);
            }
            // ---- Lanczos start: v = e_center
            {
                GT *const gvn = (GT *)P->scratch + ((long)blockIdx.x * (nz - nl) - nl) * ncol;
                const int cen = P->center;
                for (int z = 0; z < nz; z++) {
                    const int p = z * ncol + col;
                    if (z < nl) vl[p] = p == cen ? 1 : 0;
                    else gvn[p] = p == cen ? 1 : 0;
                }
            }
            ebase = ((c2 - P->ext0[2]) * P->extn[1] + (c1 - P->ext0[1])) * P->extn[0] + (c0 - P->ext0[0]);
        }
        double r[NZ];
#pragma unroll
        for (int z = 0; z < NZ; z++) r[z] = 0;
        double sv = 1.0, svp = 0.0, bprev = 0.0;   // v = sv * stored, previous = svp * r
        int status = 0, nq = 0, checks = 0;   // nq: Gauss nodes of a rule that stops early
        __syncthreads();
        for (int step = 0;; step++) {
            // ---- gather: sum_{box & cube} v chi_ch; one (x,y) column of the box a lane,
            // four sums over z (t0, t2, t2 z, t2 z^2), then the channels from the
            // column's constants and one reduction over the lanes
            {
                const ParamView P = params();
                const int nx = P->nloc[0], ny = P->nloc[1], nz = P->nloc[2], nl = P->nl, ncol = nx * ny;
                const GT *const gvn = (const GT *)P->scratch + ((long)blockIdx.x * (nz - nl) - nl) * ncol;
                const GC *const tab = (const GC *)P->tab;
                const double hx = P->hgrid[0], hy = P->hgrid[1], hz = P->hgrid[2];
                const float rt2 = P->rt2;
                for (;;) {
                    int li = 0;
                    if (lane == 0) li = atomicAdd(&S.ticket, 1);
                    li = __builtin_amdgcn_readfirstlane(li);
                    if (li >= nimg) break;
                    const int lo = __builtin_amdgcn_readfirstlane(S.lo[li]), dm = __builtin_amdgcn_readfirstlane(S.dim[li]);
                    const int lx = (signed char)(lo & 255), ly = (signed char)(lo >> 8 & 255), lz = (signed char)(lo >> 16 & 255);
                    const int dx = dm & 255, dy = dm >> 8 & 255, dz = dm >> 16 & 255;
                    const unsigned ts = dx * dy * 16u;
                    const int x0 = max(lx, 0), nbx = min(lx + dx, nx) - x0;
                    const int y0 = max(ly, 0), nby = min(ly + dy, ny) - y0;
                    const int z0 = max(lz, 0), z1 = min(lz + dz, nz);
                    const int nxy = nbx * nby;
                    const float inv = 1.0f / (float)nbx;
                    const int off = __builtin_amdgcn_readfirstlane(S.off[li]) + z0 * dx * dy;
                    const double oz = lane_value(S.org[li][2], 0);
                    double acc[NLM];
#pragma unroll
                    for (int ch = 0; ch < NLM; ch++) acc[ch] = 0;
                    for (int q0 = 0; q0 < nxy; q0 += 64) {
                        const int q = min(q0 + lane, nxy - 1);
                        const int yi = fdiv(q, nbx, inv);
                        const int cx = x0 + q - yi * nbx, cy = y0 + yi;
                        const double x = S.org[li][0] + hx * cx, y = S.org[li][1] + hy * cy;
                        if (q0 + lane >= nxy || !((float)x * (float)x + (float)y * (float)y < rt2)) continue;
                        unsigned tp = (off + cy * dx + cx) * 16u;
                        int vp = z0 * ncol + cy * nx + cx;
                        double s0 = 0, s1 = 0, s2 = 0, s3 = 0;
                        auto add = [&](V2 t, double v, double z) {
                            const double zz = fma(hz, z, oz);
                            const double p = t.y * v, pz = p * zz;
                            s0 = fma(t.x, v, s0);
                            s1 += p;
                            s2 += pz;
                            s3 = fma(pz, zz, s3);
                        };
                        auto walk = [&](int z, int zb, auto v) {
                            double zd = z;
#pragma unroll 1
                            for (; z < zb; z += UG) {
                                V2 t[UG];
                                double vv[UG];
#pragma unroll
                                for (int u = 0; u < UG; u++)
                                    if (z + u < zb) {   // uniform
                                        t[u] = *(GV2 *)(tab + (tp + u * ts));
                                        vv[u] = v[vp + u * ncol];
                                    }
#pragma unroll
                                for (int u = 0; u < UG; u++)
                                    if (z + u < zb) add(t[u], vv[u], zd + u);
                                const int n = min(UG, zb - z);
                                tp += n * ts;
                                vp += n * ncol;
                                zd += UG;
                            }
                        };
                        if (z0 < nl) walk(z0, min(z1, nl), vl);
                        if (z1 > nl) walk(max(z0, nl), z1, gvn);
                        const double C = 1.092548430592079, C20 = 0.315391565252520, C22 = 0.546274215296040;
                        acc[0] += s0;
                        acc[1] = fma(C * (x * y), s1, acc[1]);
                        acc[2] = fma(C * y, s2, acc[2]);
                        acc[3] = fma(C20, fma(-(x * x) - y * y, s1, 2 * s3), acc[3]);
                        acc[4] = fma(C * x, s2, acc[4]);
                        acc[5] = fma(C22 * (x * x - y * y), s1, acc[5]);
                    }
                    // six channels over 64 lanes: rows 0..3 of f hold channels 0, 2, 1, 3, rows 0 and 2 of g 4 and 5
                    const double f01 = fold32(acc[0], acc[1]), f23 = fold32(acc[2], acc[3]), f45 = fold32(acc[4], acc[5]);
                    const double f = row_sum(fold16(f01, f23)), g = row_sum(fold16(f45, f45));
                    if ((lane & 15) == 0) {
                        const int row = lane >> 4;
                        S.A[li][(row & 1) << 1 | row >> 1] = f * sv;   // the sums used the stored v
                        if (!(row & 1)) S.A[li][4 + (row >> 1)] = g * sv;
                    }
                }
            }
            __syncthreads();
            // ---- per atom (at its first list entry): alpha, and over its images' sums the
            // scatter's column-independent coefficients:
            // chi alpha = t0 K0 + t2 (xy K1 + xx K2 + yy K3) + t2 z (y K4 + x K5) - t2 z^2 (K2 + K3)
            if (tid == 0) S.ticket = 0;
            if (tid < nimg) {
                const ParamView P = params();
                if (S.head[tid] == tid) {
                    const double *gam = P->gamma_ch + (S.dim[tid] >> 24 & 255) * kMaxChannels;
                    double a6[NLM], al = 0.0;
#pragma unroll
                    for (int ch = 0; ch < NLM; ch++) a6[ch] = 0.0;
                    for (int q = tid; q < kResMaxImages; q = S.next[q])
#pragma unroll
                        for (int ch = 0; ch < NLM; ch++) a6[ch] += S.A[q][ch];
#pragma unroll
                    for (int ch = 0; ch < NLM; ch++) {
                        a6[ch] = gam[ch] * a6[ch];
                        al += a6[ch];
                    }
                    if (P->mode == 0)   // one coefficient per atom
#pragma unroll
                        for (int ch = 0; ch < NLM; ch++) a6[ch] = al;
                    const double C = 1.092548430592079, C20 = 0.315391565252520, C22 = 0.546274215296040;
                    const double a1 = a6[1], a2 = a6[2], a3 = a6[3], a4 = a6[4], a5 = a6[5];
                    const double k6[NLM] = {a6[0], C * a1, fma(C22, a5, -(C20 * a3)), fma(-C22, a5, -(C20 * a3)), C * a2, C * a4};
                    for (int q = tid; q < kResMaxImages; q = S.next[q]) {
                        double *k = reinterpret_cast<double *>(S.A[q]);
#pragma unroll
                        for (int ch = 0; ch < NLM; ch++) k[ch] = k6[ch];
                        if (P->rec && S.slot[q] != 255 && step < P->nqp) {
                            double *dst = P->rec + (((long)row * P->nqp + step) * P->rec_slots + S.slot[q]) * NLM;
#pragma unroll
                            for (int ch = 0; ch < NLM; ch++) dst[ch] = a6[ch];
                        }
                    }
                }
            }
            __syncthreads();
            // ---- r := -b r + sum over the column's images of chi alpha
            if (live) {
                const ParamView P = params();
                const int nz = P->nloc[2];
                const GC *const tab = (const GC *)P->tab;
                const double hz = P->hgrid[2];
                int cc = cij;
                SQ_OPAQUE_V(cc);
                const int ci = cc & 0xffff, cj = cc >> 16;
                const double xi = P->hgrid[0] * ci, yj = P->hgrid[1] * cj;
                const float rt2 = P->rt2, ihz = 1.0f / (float)hz;
                const double tb = -bprev * svp;
#pragma unroll
                for (int z = 0; z < NZ; z++) r[z] = tb * r[z];
#pragma unroll 1
                for (int wd = 0; wd < MW; wd++) {
                    unsigned m = cmask[0];
#pragma unroll
                    for (int q = 1; q < MW; q++) m = wd == q ? cmask[q] : m;
                    while (m) {
                        const int li = (wd << 5) + __ffs(m) - 1;
                        m &= m - 1u;
                        const int lo = S.lo[li], dm = S.dim[li];
                        const int dx = dm & 255;
                        const unsigned ts = (dm >> 8 & 255) * dx * 16u;
                        const double *k6 = reinterpret_cast<const double *>(S.A[li]);
                        const double oz = S.org[li][2];
                        const double x = (S.org[li][0] + xi), y = (S.org[li][1] + yj);
                        const double k0 = k6[0];
                        const double p0 = fma(x * y, k6[1], fma(x * x, k6[2], (y * y) * k6[3]));
                        const double p1 = fma(y, k6[4], x * k6[5]);
                        const double p2 = -(k6[2] + k6[3]);
                        // planes of the column the projector reaches
                        const float xf = (float)x, yf = (float)y;
                        const float half = sqrtf(fmaxf(rt2 - xf * xf - yf * yf, 0.0f));
                        const int lz = (signed char)(lo >> 16 & 255);
                        const int zl = max(max(lz, 0), (int)ceilf(((float)-oz - half) * ihz));
                        const int zh = min(min(lz + (dm >> 16 & 255), nz) - 1, (int)floorf(((float)-oz + half) * ihz));
                        unsigned tp = (S.off[li] + cj * dx + ci) * 16u;
#pragma unroll
                        for (int z0 = 0; z0 < NZ; z0 += UC) {
                            if (zl < z0 + UC && zh >= z0) {
                                V2 t[UC];
#pragma unroll
                                for (int u = 0; u < UC; u++) t[u] = *(GV2 *)(tab + (tp + u * ts));
                                const double zr = fma(hz, (double)z0, oz);
#pragma unroll
                                for (int u = 0; u < UC; u++)
                                    if (z0 + u < NZ) {
                                        const double z = fma(hz, (double)u, zr);
                                        r[z0 + u] = fma(t[u].x, k0, fma(t[u].y, fma(z, fma(z, p2, p1), p0), r[z0 + u]));
                                    }
                            }
                            tp += UC * ts;
                        }
                    }
                }
            }
            // ---- march: r += (L + diag) v
            {
                const ParamView P = params();
                const int nz = P->nloc[2], nl = P->nl, ncol = P->nloc[0] * P->nloc[1];
                const GT *const gvn = (const GT *)P->scratch + ((long)blockIdx.x * (nz - nl) - nl) * ncol;
                const GT *const diag = (const GT *)P->diag_ext;
                const int eplane = P->extn[1] * P->extn[0];
                const int sbuf = PX * (P->nloc[1] + 2 * O);
                SV2 *const stage = (SV2 *)(vl + ((nl * ncol + 1) & ~1));
                int cc = cij;
                SQ_OPAQUE_V(cc);
                const int ci = cc & 0xffff, cj = cc >> 16, col = cj * P->nloc[0] + ci;
                // the stencil footprint's top-left corner in the staged plane: every neighbour
                // lies at a constant non-negative offset
                SV2 *const scol = stage + cj * PX + ci;
                double wt[3][O];
#pragma unroll
                for (int d = 0; d < 3; d++)
#pragma unroll
                    for (int l = 0; l < O; l++) wt[d][l] = P->cw[d][l + 1];
                const double s = sv;
                if (live) {
                    // Two planes at a time, staged side by side: a 16-byte read brings a neighbour
                    // of both.  Plane pointers advance as scalars; vl's plane offset likewise.  The
                    // pair's second plane may lie past the cube: it is zero then.
                    const int dcol = cj * P->extn[0] + ci;
                    // v and the diagonal at plane z, or at the last; z is opaque, so no plane's
                    // addresses are worked out before its turn
                    auto load = [&](int z, double &v, double &d) {
                        SQ_OPAQUE(z);
                        const int k = min(z, nz - 1);
                        d = (diag + (ebase + k * eplane))[(unsigned)dcol];
                        if (k < nl) v = vl[k * ncol + col];
                        else v = (gvn + k * ncol)[(unsigned)col];
                    };
                    double n0, n1, d0, d1;
                    load(0, n0, d0);
                    load(1, n1, d1);
#pragma unroll
                    for (int z = 0; z < NZ; z += 2) {
                        if (z < nz) {   // uniform
                            const double va = s * n0, vb = z + 1 < nz ? s * n1 : 0.0, da = d0, db = d1;
                            SV2 *const sc = NB == 2 && (z & 2) ? scol + sbuf : scol;
                            if (NB == 1 && z) __syncthreads();   // the last pair has been read
                            sc[O * PX + O] = V2{va, vb};
                            load(z + 2, n0, d0);
                            load(z + 3, n1, d1);
                            __syncthreads();
                            double xa = da * va, xb = db * vb, ya = 0, yb = 0;
#pragma unroll
                            for (int l = 1; l <= O; l++) {
                                const V2 xm = sc[O * PX + O - l], xp = sc[O * PX + O + l];
                                const V2 ym = sc[(O - l) * PX + O], yp = sc[(O + l) * PX + O];
                                xa = fma(wt[0][l - 1], xm.x + xp.x, xa);
                                xb = fma(wt[0][l - 1], xm.y + xp.y, xb);
                                ya = fma(wt[1][l - 1], ym.x + yp.x, ya);
                                yb = fma(wt[1][l - 1], ym.y + yp.y, yb);
                                if (z - l >= 0) r[z >= l ? z - l : 0] = fma(wt[2][l - 1], va, r[z >= l ? z - l : 0]);
                                if (z + l < NZ) r[z + l < NZ ? z + l : 0] = fma(wt[2][l - 1], va, r[z + l < NZ ? z + l : 0]);
                                if (z + 1 - l >= 0 && z + 1 < NZ)
                                    r[z + 1 >= l ? z + 1 - l : 0] = fma(wt[2][l - 1], vb, r[z + 1 >= l ? z + 1 - l : 0]);
                                if (z + 1 + l < NZ) r[z + 1 + l < NZ ? z + 1 + l : 0] = fma(wt[2][l - 1], vb, r[z + 1 + l < NZ ? z + 1 + l : 0]);
                            }
                            r[z] += xa + ya;
                            if (z + 1 < NZ) r[z + 1 < NZ ? z + 1 : 0] += xb + yb;
                        }
                    }
                } else {
                    for (int z = 0; z < nz; z += 2) {   // the staged planes of the others
                        if (NB == 1 && z) __syncthreads();
                        __syncthreads();
                    }
                }
            }
            // ---- a = <v, r>; r -= a v; ||r||; the vectors change places
            double a, pb = 0.0;
            {
                const ParamView P = params();
                const int nz = P->nloc[2], nl = P->nl, ncol = P->nloc[0] * P->nloc[1];
                const GT *const gvn = (const GT *)P->scratch + ((long)blockIdx.x * (nz - nl) - nl) * ncol;
                double pa = 0.0;
                int cc = cij;
                SQ_OPAQUE_V(cc);
                const int col = (cc >> 16) * P->nloc[0] + (cc & 0xffff);
                if (live) {
#pragma unroll
                    for (int z0 = 0; z0 < NZ; z0 += UD)
                        if (z0 < nz) {   // uniform
                            double v[UD];
                            load_planes(v, z0, col, vl, gvn, nl, nz, ncol);
#pragma unroll
                            for (int u = 0; u < UD; u++)
                                if (z0 + u < NZ && z0 + u < nz) pa = fma(v[u], r[z0 + u < NZ ? z0 + u : 0], pa);
                        }
                }
                a = group_sum<NW>(has ? pa : 0.0, S.red[0]) * sv;
            }
            if (live) {
                const ParamView P = params();
                const int nz = P->nloc[2], nl = P->nl, ncol = P->nloc[0] * P->nloc[1];
                GT *const gvn = (GT *)P->scratch + ((long)blockIdx.x * (nz - nl) - nl) * ncol;
                const double ta = -a * sv;
                int cc = cij;
                SQ_OPAQUE_V(cc);
                const int col = (cc >> 16) * P->nloc[0] + (cc & 0xffff);
#pragma unroll
                for (int z0 = 0; z0 < NZ; z0 += UD)
                    if (z0 < nz) {   // uniform
                        double v[UD];
                        load_planes(v, z0, col, vl, (const GT *)gvn, nl, nz, ncol);
#pragma unroll
                        for (int u = 0; u < UD; u++) {
                            const int z = z0 + u < NZ ? z0 + u : 0;
                            if (z0 + u < NZ && z0 + u < nz) {
                                const double w = fma(ta, v[u], r[z]);
                                pb = fma(w, w, pb);
                                if (z0 < nl) vl[z * ncol + col] = w;
                                else gvn[z * ncol + col] = w;
                                r[z] = v[u];
                            }
                        }
                    }
            }
            const double b = lane_value(sqrt(group_sum<NW>(has ? pb : 0.0, S.red[1])), 0);
            {
                const ParamView P = params();
                const int nqp = P->nqp;
                if (tid == 0) {
                    P->out_a[(long)id * (nqp + 1) + step] = a;
                    P->out_b[(long)id * (nqp + 1) + step] = b;
                }
                if (b == 0.0) { status = 7; break; }
                if (P->exit_tol > 0.0) {
                    // early exit: the lowest Matsubara terms of e1^double (lf + i w - double)^-1 e1 by the
                    // continued fraction, one a lane, against the last check's
                    if (tid == 0) {
                        S.ab[0][step] = a;
                        S.ab[1][step] = b;
                        S.flag = 0;
                    }
                    const int n = step + 1;
                    if (n >= P->exit_min && (n - P->exit_min) % P->exit_every == 0 && n < nqp) {
                        __syncthreads();
                        if (tid < kMatsubara) {
                            const double wm = (2 * tid + 1) * M_PI / P->exit_beta;
                            double tr = P->exit_lf - S.ab[0][n - 1], ti = wm;
                            for (int j = n - 2; j >= 0; j--) {
                                const double den = tr * tr + ti * ti, q2 = S.ab[1][j] * S.ab[1][j];
                                tr = (P->exit_lf - S.ab[0][j]) - q2 * tr / den;
                                ti = wm + q2 * ti / den;
                            }
                            const double den = tr * tr + ti * ti, gr = tr / den, gi = -ti / den;
                            const double dr = gr - S.g[tid][0], di = gi - S.g[tid][1];
                            const double d = (2.0 / P->exit_beta) * sqrt(dr * dr + di * di);
                            if (checks == 0 || !(d < P->exit_tol)) S.flag = 1;
                            S.g[tid][0] = gr;
                            S.g[tid][1] = gi;
                        }
                        __syncthreads();
                        if (__builtin_amdgcn_readfirstlane(S.flag) == 0) { nq = n; break; }
                        checks++;
                    }
                }
                if (step == nqp) break;
            }
            svp = sv;
            sv = lane_value(1.0 / b, 0);
            bprev = b;
        }
        if (tid == 0) {
            const ParamView P = params();
            P->status[id] = status;
            P->nsteps[id] = nq ? nq : P->nqp;
        }
        __syncthreads();
    }
}

#undef SQ_OPAQUE
#undef SQ_OPAQUE_V

// Builds: 512 threads for cubes of at most 512 columns (two workgroups a CU),
// 1024 for the rest; each unrolled to the smallest plane count that holds nz.
int resident_workgroup(const int nloc[3])
{
    const int ncol = nloc[0] * nloc[1];
    if (nloc[0] > kResMaxNz || nloc[1] > kResMaxNz || nloc[2] > kResMaxNz || ncol > 1024) return 0;
    return ncol <= 512 && nloc[2] <= 25 ? 512 : 1024;
}

void resident_lds(const int nloc[3], int nl, size_t *total, size_t *dynamic)
{
    const size_t vdoubles = (size_t)nl * nloc[0] * nloc[1], pair = 2 * (size_t)kPitch * (nloc[1] + 12);
    *dynamic = ((vdoubles + 1) / 2 * 2 + stage_buffers(resident_workgroup(nloc)) * pair) * sizeof(double);
    *total = *dynamic + sizeof(ResLds);
}

static const void *resident_build(const ResParams &P)
{
    const int wg = resident_workgroup(P.nloc), nz = P.nloc[2];
    if (wg == 0) return nullptr;
    if (wg == 512) return nz <= 21 ? (const void *)lanczos_resident<512, 21> : (const void *)lanczos_resident<512, 25>;
    if (nz <= 25) return (const void *)lanczos_resident<1024, 25>;
    return nz <= 29 ? (const void *)lanczos_resident<1024, 29> : (const void *)lanczos_resident<1024, 31>;
}

hipError_t launch_resident(const ResParams &P, int grid, size_t lds, hipStream_t st)
{
    const void *f = resident_build(P);
    if (!f || P.nl < 0 || P.nl > P.nloc[2]) return hipErrorInvalidValue;
    ResParams q = P;
    void *args[] = {&q};
    return hipLaunchKernel(f, dim3(grid), dim3(resident_workgroup(P.nloc)), args, lds, st);
}

int resident_occupancy(const ResParams &P, size_t lds)
{
    const void *f = resident_build(P);
    int n = 0;
    if (!f || hipOccupancyMaxActiveBlocksPerMultiprocessor(&n, f, resident_workgroup(P.nloc), lds) != hipSuccess) return 0;
    return n;
}

__global__ void __launch_bounds__(256) resident_tables(const ResImage *__restrict__ img, const int64_t *__restrict__ rad_off,
                                                       const int4 *__restrict__ box_lo, const int4 *__restrict__ box_dim,
                                                       const double *__restrict__ rad, double *__restrict__ tab)
{
    const ResImage im = img[blockIdx.x];
    const int4 lo = box_lo[im.id], dm = box_dim[im.id];
    const int np = im.dim[0] * im.dim[1] * (im.dim[2] + 2 * kResPad);
    for (int p = threadIdx.x; p < np; p += blockDim.x) {
        const int i = p % im.dim[0], j = p / im.dim[0] % im.dim[1], k = p / (im.dim[0] * im.dim[1]) - kResPad;
        double t0 = 0.0, t2 = 0.0;
        if (k >= 0 && k < im.dim[2]) {
            const int64_t q = ((int64_t)(im.lo[2] + k - lo.z) * dm.y + (im.lo[1] + j - lo.y)) * dm.x + (im.lo[0] + i - lo.x);
            t0 = rad[rad_off[im.id] + 2 * q];
            t2 = rad[rad_off[im.id] + 2 * q + 1];
        }
        const int64_t o = 2 * ((int64_t)im.off + p);
        tab[o] = t0;
        tab[o + 1] = t2;
    }
}

hipError_t launch_resident_tables(const ResImage *img, int n, const int64_t *rad_off, const int4 *box_lo, const int4 *box_dim,
                                  const double *rad, double *tab, hipStream_t st)
{
    if (n <= 0) return hipSuccess;
    hipLaunchKernelGGL(resident_tables, dim3(n), dim3(256), 0, st, img, rad_off, box_lo, box_dim, rad, tab);
    return hipGetLastError();
}

}  // namespace sqamd
