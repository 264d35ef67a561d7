/*
 * A 16 x 16 TMz problem whose point detector names a cell far past the grid:
 * creating, stepping and reading it must work, and its samples stay zero.
 */
#include <stdio.h>
#include <string.h>

#include "chiml/chiml_dev.h"

#define N 16

int main(void) {
    const double dt = 0.01, ce[1] = {dt}, inveps[1] = {1.0}, ch[1] = {dt};
    const int flags[1] = {0}, poleset[1] = {-1};
    const int src_comp[1] = {2}, src_box[6] = {8, 9, 8, 9, 0, 1};
    const double src_amp[4] = {1.0, 0.0, 0.0, 0.0};
    const int det_interval[1] = {1}, det_npts[1] = {1}, det_comp[2] = {2, 2}, det_pow[1] = {0};
    const long long far_cell = 40000000000LL, det_cell[2] = {far_cell, far_cell};
    const double det_conv[1] = {1.0};
    chiml_problem_t p;
    memset(&p, 0, sizeof p);
    p.nx = p.ny = N;
    p.nz = 1;
    p.precision = 64;
    p.dt = dt;
    p.d[0] = p.d[1] = p.d[2] = 0.05;
    p.nsteps = 4;
    p.nmat_e[2] = 1;
    p.mat_e_ce[2] = ce;
    p.mat_e_inveps[2] = inveps;
    p.mat_e_flags[2] = flags;
    p.mat_e_poleset[2] = poleset;
    for (int k = 0; k < 2; ++k) {
        p.nmat_h[k] = 1;
        p.mat_h_ch[k] = ch;
    }
    p.nsrc = 1;
    p.src_comp = src_comp;
    p.src_box = src_box;
    p.src_amp = src_amp;
    p.ndet = 1;
    p.det_interval = det_interval;
    p.det_npts = det_npts;
    p.det_comp = det_comp;
    p.det_cell = det_cell;
    p.det_conv = det_conv;
    p.det_pow = det_pow;
    chiml_dev_t* ctx = NULL;
    if (chiml_dev_create(&p, &ctx) != CHIML_OK || chiml_dev_step(ctx, 3) != CHIML_OK || chiml_dev_sync(ctx) != CHIML_OK) {
        printf("%s\n", chiml_dev_global_error());
        return 1;
    }
    double v[8];
    size_t ns = 0;
    if (chiml_dev_read_points(ctx, 0, v, 8, &ns) != CHIML_OK || ns < 3) return 1;
    for (size_t k = 0; k < ns; ++k)
        if (v[k] != 0.0) return 1;
    chiml_dev_destroy(ctx);
    printf("OK\n");
    return 0;
}
