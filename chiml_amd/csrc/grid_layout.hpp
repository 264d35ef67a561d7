// How a grid is stored and swept on the device, shared by the device layer
// and the manager's byte accounting.
#pragma once

// Rows along x are stored in whole groups of W = 16 / sizeof(T) cells (one
// 16-byte access each) and the x CPML's psi regions are widened to whole
// groups with identity coefficients, so grids and slabs of any size take the
// W-cell kernels.  The padding cells of a row stay zero.
struct GridLayout {
    int W;       // cells per group
    bool vec;    // the W-cell kernels apply (else one thread per cell, rows as they are)
    int px;      // stored cells per row
    bool split;  // 3D: interior + CPML slab sweeps
    bool rows;   // split: the interior takes whole rows (x slabs inline), H and E one launch each
    bool cellwise;  // stepped alone with one thread per cell, though the W-cell kernels apply
};

inline int round_up(int n, int w) { return (n + w - 1) / w * w; }
inline int round_down(int n, int w) { return n / w * w; }

// psi_lo / psi_hi0: the largest lower end and the smallest upper start of the
// x psi regions over the components (T and nx - T for a CPML of T cells).
// The W-cell form needs the two widened regions not to reach into each other's
// unwidened part: a group belongs to one of them, or to neither.
inline GridLayout grid_layout(int nx, int ny, int nz, const int* T, int psi_lo, int psi_hi0, bool fp32, bool hmap) {
    GridLayout g;
    g.W = fp32 ? 4 : 2;
    const int lo = round_up(psi_lo, g.W), hi = round_down(psi_hi0, g.W);
    g.vec = !hmap && lo <= hi;
    g.px = g.vec ? round_up(nx, g.W) : nx;
    // (the sweeps number groups in 32 bits)
    g.split = g.vec && nz > 1 && nx > 2 * T[0] && ny > 2 * T[1] && nz > 2 * T[2] &&
              static_cast<double>(g.px / g.W) * (ny + 8) * nz < 4.0e9;
    const bool aligned = nx % g.W == 0 && T[0] % g.W == 0;
    // FP64 leaves the x slabs of aligned grids to the slab sweep, which
    // measured faster there (256^3: 0.603 against 0.619 ms per step)
    g.rows = g.split && (fp32 || !aligned);
    // Groups leave a small grid about one wave per SIMD, each waiting for memory
    // alone, so a small grid that had to be padded is stepped one thread per
    // cell.  (Aligned grids are not: their groups round both products of a curl,
    // the per-cell kernels fuse one, and FP32 metals amplify a change of
    // rounding.)  The line goes by the bytes of a component over the threads
    // launched (blocks of 64 x 4 cells: a row of 66 takes two).  us a step per
    // cell / in groups, FP32: 30^3 13.0/16.4, 64^3 15.4/17.9, 45x75x75 (1.46 MB)
    // 16.2/18.2, 33x85x81 (1.82) 18.7/17.9, 66x60x60 (1.84) 20.8/17.5, 72^3 (2.65)
    // 23.9/18.5; FP64: 50^3 (1.33) 16.1/16.8, 126x42x42 (1.89) 20.2/18.8, 65^3
    // 30.6/20.6.  FP32 2D grids that the tiles do not take (us of
    // the two kernels, with a source, a metal and a flux box): 67x65 8.8/10.3,
    // 257x255 9.0/11.3, 515x509 9.5/10.9, 701x699 equal; FP64 ones are equal at
    // every size.  A batch of such grids fills the chip and takes the groups where
    // it has a class (56^3, 72^3 and 88^3 FP32 together with three 2D grids: 72 and
    // 51 us a step); unaligned FP64 3D grids have none.
    const double threads = static_cast<double>(round_up(nx, 64)) * round_up(ny, 4) * nz;
    g.cellwise = (g.split || (g.vec && nz == 1 && fp32)) && !aligned && threads * (fp32 ? 4 : 8) < 1.48e6;
    return g;
}
