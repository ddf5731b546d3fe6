// sq_resident.h -- launch parameters of the resident Lanczos kernel
// (sq_resident.hip, FP64): one node a workgroup, its vectors kept on chip.
#pragma once
#include <hip/hip_runtime.h>
#include <stdint.h>

#include "sq_kernels.h"

namespace sqamd {

constexpr int kResMaxImages = 128;   // images one cube may meet (four mask words a column)
constexpr int kResPad = 3;           // zero planes below and above an image's table

// One projector image, trimmed to the points its radial factors reach.
struct ResImage {
    int lo[3], dim[3];   // trimmed box, global unwrapped indices
    int off;             // first radial pair of its padded table
    int atom, type, id;  // supercell atom, pseudopotential type, index in the setup's image list
    int pad[2];
    double cen[3];       // image position
    double pad2;
};

struct ResParams {
    int nloc[3], hw[3];
    int box0[3], box_n[3], ext0[3], extn[3];
    int center;                  // cube point of the node
    int nqp, mode;
    int n_images;
    int nl;                      // planes of v in LDS; the rest in the workgroup's scratch slice
    long node_begin, node_count;
    double hgrid[3], range[3];
    float rt2;                   // squared reach of the projectors
    double cw[3][7];             // stencil weights (x,y,z)
    const ResImage *img;         // sorted by z of the centre
    const void *tab;             // radial pairs (t0, t2) per padded box point
    const double *gamma_ch;      // [type][kMaxChannels]
    const void *diag_ext;
    void *scratch;               // (nz - nl) planes of T per workgroup
    double *out_a, *out_b;       // [node][nqp+1]
    int *status, *nsteps;        // [node]
    int *queue;                  // eight counters, zeroed before a launch
    // early exit (exit_tol > 0) and force-pass record (rec), as in KParams
    double exit_tol, exit_lf, exit_beta;
    int exit_min, exit_every;
    const int *node_list;        // [node_count] rank-box node ids (nullptr: node_begin + r)
    double *rec;                 // [node_count][nqp][rec_slots][6]
    int *rec_img;                // [node_count][rec_slots]
    int rec_slots;
};

// the longest side of a cube the kernel's builds hold
constexpr int kResMaxNz = 31;
// Workgroup (512 or 1024 threads) for a cube, 0 when the kernel does not hold it.
int resident_workgroup(const int nloc[3]);
// LDS bytes of a workgroup with nl planes of v resident: in all, and the dynamic part
void resident_lds(const int nloc[3], int nl, size_t *total, size_t *dynamic);
hipError_t launch_resident(const ResParams &P, int grid, size_t lds, hipStream_t st);
int resident_occupancy(const ResParams &P, size_t lds);
// Padded tables of the trimmed boxes from the radial factors of the whole boxes:
// src[g] = {first factor, lo, dim} of image id g.
hipError_t launch_resident_tables(const ResImage *img, int n, const int64_t *rad_off, const int4 *box_lo, const int4 *box_dim,
                                  const double *rad, double *tab, hipStream_t st);

}  // namespace sqamd
