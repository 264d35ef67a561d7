// MI355X (gfx950) kernels and the C ABI of include/chiml/chiml_dev.h.
//
// One context = one device-resident domain.  Per step (the order of
// parallelFDTDFieldBase::step(), src/FDTD_MANAGER/parallelFDTDField.hpp:1228-1303):
//   1. H sweep     : H += curl E with CPML psi (updateH + updateHPML) and H
//                    sources; in 3D its first blocks advance the poles (updatePolE)
//   2. E sweep     : soft E sources, pole currents, E += curl H with CPML psi
//                    (addPul, updateE/updateD, updateEPML, D2E)
//                    3D FP32: k_h3_all / k_e3_all; 3D FP64: k_h3_int + k_h3_slab /
//                    k_e3_int + k_e3_slab; 2D: k_tile2 (several steps) or k_h2v / k_e2v;
//                    else k_update_h / k_update_e
//   3. emitters    : k_ml_addp, k_ml_entry, then k_ml_pop_finish on recording steps
//                    (parallelQEBase::addQE)
//   4. t_step += 1 : plain launches are given the step number by the host;
//                    inside captured graphs the H launch advances a two-slot
//                    device counter (advance_counter)
//   5. k_sample    : point detectors and DFT staging (dtc->output, flux->fieldIn)
//   6. k_dft_flush : every kDftBlock samples, F[s,f] += sum_k W[k,f] U[k,s]
//
// Formulation.  The reference keeps D for dispersive, emitter and
// PML-with-material cells and recomputes E = (D - sum P)/eps after every step
// (DtoU, src/UTIL/FDTD_up_eq.cpp:838-848).  Here E itself is the state:
// E' = E + (dt/eps) curl H - (1/eps) sum_p (P_p' - P_p), which is the same
// recursion in exact arithmetic, and each pole is advanced in current form
// J' = (alpha + xi - 1) P - xi J + gamma E, P' = P + J' with J = P - P_prev,
// which is UpdateLorPol's P' = alpha P + xi P_prev + gamma E rewritten
// (src/UTIL/FDTD_up_eq.cpp:425-448).  In FP32 this avoids the cancellation of
// large D and P in metals (a Drude pole's P grows without bound while E stays
// small).  The CPML uses the same b, c, kappa profiles and psi recursions as
// src/PML/parallelPML.hpp:693-765 and src/PML/parallelPML.cpp:12-40.
#include <hip/hip_runtime.h>

#include "grid_layout.hpp"
#include "qe_layout.hpp"

#include <algorithm>

#include <cmath>
#include <cstdio>
#include <cstdlib>
#include <cstring>
#include <map>
#include <memory>
#include <mutex>
#include <string>
#include <type_traits>
#include <vector>

#include "../../include/chiml/chiml_dev.h"

namespace {

constexpr int kDftBlock = 32;  // samples staged before one DFT contraction
constexpr int kMaxLevels = 8;

thread_local std::string g_err;  // last error of this host thread
// Stream capture of one context must not overlap calls that may synchronise
// the device from other threads (allocation, free, blocking copies): those
// would invalidate the capture.  Capture, create, destroy and the blocking
// reads take this lock; plain step launches do not.
std::mutex g_capture_mu;

#define HIP_TRY(expr)                                                                                \
    do {                                                                                             \
        hipError_t _e = (expr);                                                                      \
        if (_e != hipSuccess) {                                                                      \
            throw std::runtime_error(std::string(#expr) + ": " + hipGetErrorString(_e));            \
        }                                                                                            \
    } while (0)

struct DevBuf {
    void* p = nullptr;
    size_t bytes = 0;
    DevBuf() = default;
    DevBuf(const DevBuf&) = delete;
    DevBuf& operator=(const DevBuf&) = delete;
    ~DevBuf() {
        if (p) (void)hipFree(p);
    }
    // Zero-filled buffers are cleared on the owning context's stream, so the
    // clear is ordered before every kernel of that context and never waits
    // for other contexts sharing the device.
    void alloc(size_t b, hipStream_t zero_on, bool zero) {
        if (p) (void)hipFree(p);
        p = nullptr;
        bytes = b;
        if (b == 0) return;
        HIP_TRY(hipMalloc(&p, b));
        if (zero) HIP_TRY(hipMemsetAsync(p, 0, b, zero_on));
    }
    template <typename T>
    T* as() const { return static_cast<T*>(p); }
};

// ---------------------------------------------------------------- params ----
template <typename T>
struct PmlDev {
    const T* b[3];
    const T* cd[3];
    const T* kinv[3];
    T* psi[3];
    const T* psi_in[3];  // fused step: psi before the step (ping-pong for H); psi itself elsewhere
    int lo[3], hi0[3], hi1[3], S[3];
};

template <typename T>
struct StepArgs {
    T* F[6];  // Ex, Ey, Ez, Hx, Hy, Hz
    const T* G[6];  // fused step: the fields before the step (ping-pong); F itself elsewhere
    int nx, ny, nz;
    int px;  // cells per stored x row: nx, or nx rounded up to whole W-cell groups (the added cells stay zero)
    T inv_d[3];
    int Tp[3];
    const uint8_t* mat_e[3];
    const T* ce[3];
    const T* inveps[3];
    const int* flags[3];
    const int* poleset[3];
    const uint8_t* mat_h[3];
    const T* ch[3];
    const int* pole_count;
    const T* pole_coef;  // [set][kMaxPoles][3]
    T* P[3];
    T* J[3];
    T* jsum[3];  // pole-box sized: sum of the new pole currents of this step (split 3D path)
    int box[3][6];
    long long boxn[3];
    PmlDev<T> pml[6];
    int nsrc;
    const int* src_comp;
    const int* src_box;
    const T* src_amp;
    const int* step;
    int stepv;  // >= 0: the step number, passed by the host (plain launches); -1: read *step (captured graphs)
    int* step_next;  // captured graphs: the other counter slot, set to *step + 1 by the H launch
};

// The step number a launch works on: passed by the host for plain launches,
// read from the device counter inside captured graphs.
__device__ __forceinline__ int step_now(const int* p, int v) { return v >= 0 ? v : *p; }

// Inside captured graphs the step counter has two slots: step k's launches
// read slot k % 2, and the first block of its H launch writes slot (k+1) % 2,
// which nothing reads before the next step's launches (the sample and DFT
// launches of step k read it after the H launch, as the advanced step).
// Only the H kernels' ADV instantiations, launched by steps being captured,
// carry it, after their sweep: a store ahead of the sweep's loads keeps the
// compiler from proving the uniform ones unclobbered, and they become
// per-lane vector loads (the 256^3 FP32 H sweep took 8% longer), and even
// at the end the store cost plain launches 3%.
template <typename A>
__device__ __forceinline__ void advance_counter(const A& a) {
    if (a.step_next && blockIdx.x == 0 && blockIdx.y == 0 && blockIdx.z == 0 && threadIdx.x == 0 && threadIdx.y == 0 &&
        threadIdx.z == 0)
        *a.step_next = *a.step + 1;
}
// The same for a block bx of one simulation inside a batched launch.
template <typename A>
__device__ __forceinline__ void advance_counter_at(const A& a, long long bx) {
    if (a.step_next && bx == 0 && threadIdx.x == 0) *a.step_next = *a.step + 1;
}

__device__ __forceinline__ long long lidx(int x, int y, int z, int nx, int ny) {
    return x + static_cast<long long>(nx) * (y + static_cast<long long>(ny) * z);
}

// CPML term for one derivative direction a of component c:
// psi' = b psi + (c/d) dV (psi-carrying positions), term = dV/(kappa d) + psi'.
// Elsewhere in the PML region the term is dV/d (kappa = 1, no psi).
template <typename T>
struct PmlCell {
    T b, cd, kinv, psi;
    T* at = nullptr;  // null: no psi here
    __device__ __forceinline__ void load(const PmlDev<T>& p, int a, int pos, int x, int y, int z, int nx, int ny) {
        int s;
        if (pos < p.lo[a]) s = pos;
        else if (pos >= p.hi0[a] && pos < p.hi1[a]) s = p.lo[a] + pos - p.hi0[a];
        else return;
        long long pi;
        if (a == 0) pi = s + static_cast<long long>(p.S[0]) * (y + static_cast<long long>(ny) * z);
        else if (a == 1) pi = x + static_cast<long long>(nx) * (s + static_cast<long long>(p.S[1]) * z);
        else pi = x + static_cast<long long>(nx) * (y + static_cast<long long>(ny) * s);
        at = p.psi[a] + pi;
        psi = *at;
        b = p.b[a][pos];
        cd = p.cd[a][pos];
        kinv = p.kinv[a][pos];
    }
    __device__ __forceinline__ T term(T dV, T dVd) {
        if (!at) return dVd;
        psi = fma(b, psi, cd * dV);
        *at = psi;
        return fma(kinv, dVd, psi);
    }
};
template <typename T>
__device__ __forceinline__ T pml_term(const PmlDev<T>& p, int a, int pos, int x, int y, int z, int nx, int ny, T dV, T dVd) {
    PmlCell<T> q;
    q.load(p, a, pos, x, y, z, nx, ny);
    return q.term(dV, dVd);
}
// d1/dA - d2/dB of a cell with its CPML terms: one rounding less outside the
// CPML, as the compiler contracts the difference of two products
template <typename T>
__device__ __forceinline__ T curl_cell(PmlCell<T>& q1, PmlCell<T>& q2, bool inpml, T d1, T i1, T d2, T i2) {
    const T p1 = d1 * i1;
    if (!inpml) return fma(-i2, d2, p1);
    const T t1 = q1.term(d1, p1), t2 = q2.term(d2, d2 * i2);
    {
#pragma clang fp contract(off)
        return t1 - t2;
    }
}

template <typename T>
__device__ __forceinline__ T src_value(const StepArgs<T>& a, int comp, int x, int y, int z, int step) {
    T v = 0;
    for (int s = 0; s < a.nsrc; ++s) {
        if (a.src_comp[s] != comp) continue;
        const int* b = a.src_box + 6 * s;
        if (x >= b[0] && x < b[1] && y >= b[2] && y < b[3] && z >= b[4] && z < b[5]) v += a.src_amp[static_cast<long long>(step) * a.nsrc + s];
    }
    return v;
}

// src_value of the components c0 .. c0 + 2 of a cell
template <typename T>
__device__ __forceinline__ void src_values(const StepArgs<T>& a, int c0, int x, int y, int z, int step, T (&v)[3]) {
    for (int s = 0; s < a.nsrc; ++s) {
        const int c = a.src_comp[s] - c0;
        const int* b = a.src_box + 6 * s;
        if (!(x >= b[0] && x < b[1] && y >= b[2] && y < b[3] && z >= b[4] && z < b[5])) continue;
        const T amp = a.src_amp[static_cast<long long>(step) * a.nsrc + s];
#pragma unroll
        for (int k = 0; k < 3; ++k)
            if (c == k) v[k] += amp;
    }
}

// ----------------------------------------------------------- H update -------
// 3D: Hx += ch[(Ey(z+1)-Ey)/dz - (Ez(y+1)-Ez)/dy], Hy += ch[(Ez(x+1)-Ez)/dx -
// (Ex(z+1)-Ex)/dz], Hz += ch[(Ex(y+1)-Ex)/dy - (Ey(x+1)-Ey)/dx]; 2D TMz keeps
// the Ez terms of Hx and Hy (OneCompCurlK/J, src/UTIL/FDTD_up_eq.cpp:10-35).
//
// One thread per cell: small unaligned 3D grids, H maps and grids that no
// other kernel takes.  Few waves are in flight on a small grid, so the time is
// that of the longest chain of dependent accesses: every load of a cell is
// issued before its first store, which the next component's loads could not
// pass.  64^3 FP32 with a metal block and soft sources: H 6.8 -> 6.1 us, E
// 10.3 -> 9.2 us.
template <typename T, int DIM, bool HMAP, bool SRC>
__device__ __forceinline__ void update_h_cells(const StepArgs<T>& a) {
    const int x = blockIdx.x * blockDim.x + threadIdx.x;
    const int y = blockIdx.y * blockDim.y + threadIdx.y;
    const int z = blockIdx.z;
    const int nx = a.nx, ny = a.ny, nz = a.nz, px = a.px;
    if (x >= nx || y >= ny) return;
    const long long i = lidx(x, y, z, px, ny);
    const long long sy = px, sz = static_cast<long long>(px) * ny;
    const bool inpml = (x < a.Tp[0]) || (x >= nx - a.Tp[0]) || (y < a.Tp[1]) || (y >= ny - a.Tp[1]) ||
                       (DIM == 3 && ((z < a.Tp[2]) || (z >= nz - a.Tp[2])));
    int step = 0;
    if (SRC) step = step_now(a.step, a.stepv);
    const bool xin = x < nx - 1, yin = y < ny - 1;
    const T *Ex = a.F[0], *Ey = a.F[1], *Ez = a.F[2];
    T ch[3] = {};
    PmlCell<T> q[6];
    T sv[3] = {};
    if constexpr (DIM == 3) {
        const bool zin = z < nz - 1;
        const T ex = Ex[i], ey = Ey[i], ez = Ez[i];
        const T ezx = xin ? Ez[i + 1] : T(0), eyx = xin ? Ey[i + 1] : T(0);
        const T exy = yin ? Ex[i + sy] : T(0), ezy = yin ? Ez[i + sy] : T(0);
        const T exz = zin ? Ex[i + sz] : T(0), eyz = zin ? Ey[i + sz] : T(0);
        const T h0 = a.F[3][i], h1 = a.F[4][i], h2 = a.F[5][i];
#pragma unroll
        for (int c = 0; c < 3; ++c) ch[c] = HMAP ? a.ch[c][a.mat_h[c][i]] : a.ch[c][0];
        if (inpml) {
            if (yin && zin) {
                q[0].load(a.pml[3], 2, z, x, y, z, px, ny);
                q[1].load(a.pml[3], 1, y, x, y, z, px, ny);
            }
            if (xin && zin) {
                q[2].load(a.pml[4], 0, x, x, y, z, px, ny);
                q[3].load(a.pml[4], 2, z, x, y, z, px, ny);
            }
            if (xin && yin) {
                q[4].load(a.pml[5], 1, y, x, y, z, px, ny);
                q[5].load(a.pml[5], 0, x, x, y, z, px, ny);
            }
        }
        if (SRC) src_values(a, 3, x, y, z, step, sv);
        if (yin && zin) {
            T h = fma(ch[0], curl_cell(q[0], q[1], inpml, eyz - ey, a.inv_d[2], ezy - ez, a.inv_d[1]), h0);
            if (SRC) h += sv[0];
            a.F[3][i] = h;
        }
        if (xin && zin) {
            T h = fma(ch[1], curl_cell(q[2], q[3], inpml, ezx - ez, a.inv_d[0], exz - ex, a.inv_d[2]), h1);
            if (SRC) h += sv[1];
            a.F[4][i] = h;
        }
        if (xin && yin) {
            T h = fma(ch[2], curl_cell(q[4], q[5], inpml, exy - ex, a.inv_d[1], eyx - ey, a.inv_d[0]), h2);
            if (SRC) h += sv[2];
            a.F[5][i] = h;
        }
    } else {
        if (yin) {  // Hx
            const T dEz = Ez[i + sy] - Ez[i];
            T acc;
            if (!inpml) acc = -(dEz * a.inv_d[1]);
            else acc = -pml_term(a.pml[3], 1, y, x, y, z, px, ny, dEz, dEz * a.inv_d[1]);
            const T ch0 = HMAP ? a.ch[0][a.mat_h[0][i]] : a.ch[0][0];
            T h = a.F[3][i] + ch0 * acc;
            if (SRC) h += src_value(a, 3, x, y, z, step);
            a.F[3][i] = h;
        }
        if (xin) {  // Hy
            const T dEz = Ez[i + 1] - Ez[i];
            T acc;
            if (!inpml) acc = dEz * a.inv_d[0];
            else acc = pml_term(a.pml[4], 0, x, x, y, z, px, ny, dEz, dEz * a.inv_d[0]);
            const T ch1 = HMAP ? a.ch[1][a.mat_h[1][i]] : a.ch[1][0];
            T h = a.F[4][i] + ch1 * acc;
            if (SRC) h += src_value(a, 4, x, y, z, step);
            a.F[4][i] = h;
        }
    }
}

template <typename T, int DIM, bool HMAP, bool SRC, bool ADV>
__global__ void __launch_bounds__(256) k_update_h(StepArgs<T> a) {
    update_h_cells<T, DIM, HMAP, SRC>(a);
    if (ADV) advance_counter(a);
}

// ----------------------------------------------------------- E update -------
// What the E update of a component reads at its own cell.
template <typename T>
struct ECell {
    T ce, inveps, e;
    int fl, ps;
    __device__ __forceinline__ void load(const StepArgs<T>& a, int c, long long i) {
        const uint8_t id = a.mat_e[c] ? a.mat_e[c][i] : 0;
        e = a.F[c][i];
        ce = a.ce[c][id];
        fl = a.flags[c][id];
        ps = a.poleset[c][id];
        inveps = a.inveps[c][id];
    }
};
template <typename T>
__device__ __forceinline__ void e_finish(const StepArgs<T>& a, const ECell<T>& m, int c, long long i, int x, int y, int z, T acc, T src) {
    const int ps = m.ps;
    const T e_old = m.e;
    // A soft source on a D cell reaches the ADE but not E: D2E overwrites E
    // from D, which the source never touched (parallelFDTDField.hpp:1261-1281).
    const T e_base = (m.fl & CHIML_MAT_DCELL) ? e_old : e_old + src;
    const T e_ade = e_old + src;
    T jsum = 0;
    if (ps >= 0) {
        const int* bx = a.box[c];
        long long bi = (x - bx[0]) + static_cast<long long>(bx[1] - bx[0]) * ((y - bx[2]) + static_cast<long long>(bx[3] - bx[2]) * (z - bx[4]));
        const int np = a.pole_count[ps];
        const T* co = a.pole_coef + static_cast<long long>(ps) * CHIML_MAX_POLES * 3;
        for (int p = 0; p < np; ++p) {
            T* Pp = a.P[c] + p * a.boxn[c];
            T* Jp = a.J[c] + p * a.boxn[c];
            T P = Pp[bi], J = Jp[bi];
            T Jn = co[3 * p] * P + co[3 * p + 1] * J + co[3 * p + 2] * e_ade;
            Pp[bi] = P + Jn;
            Jp[bi] = Jn;
            jsum += Jn;
        }
    }
    a.F[c][i] = fma(-m.inveps, jsum, fma(m.ce, acc, e_base));
}

// 3D: Ex += ce[(Hz-Hz(y-1))/dy - (Hy-Hy(z-1))/dz], Ey += ce[(Hx-Hx(z-1))/dz -
// (Hz-Hz(x-1))/dx], Ez += ce[(Hy-Hy(x-1))/dx - (Hx-Hx(y-1))/dy] (TwoCompCurl,
// src/UTIL/FDTD_up_eq.cpp:26-35); the ghost border is zero (PEC).
template <typename T, int DIM, bool SRC>
__global__ void __launch_bounds__(256) k_update_e(StepArgs<T> a) {
    const int x = blockIdx.x * blockDim.x + threadIdx.x;
    const int y = blockIdx.y * blockDim.y + threadIdx.y;
    const int z = blockIdx.z;
    const int nx = a.nx, ny = a.ny, nz = a.nz, px = a.px;
    if (x >= nx || y >= ny) return;
    const long long i = lidx(x, y, z, px, ny);
    const long long sy = px, sz = static_cast<long long>(px) * ny;
    const bool inpml = (x < a.Tp[0]) || (x >= nx - a.Tp[0]) || (y < a.Tp[1]) || (y >= ny - a.Tp[1]) ||
                       (DIM == 3 && ((z < a.Tp[2]) || (z >= nz - a.Tp[2])));
    int step = 0;
    if (SRC) step = step_now(a.step, a.stepv);
    const T* Hx = a.F[3];
    const T* Hy = a.F[4];
    const T* Hz = a.F[5];
    T sv[3] = {};
    ECell<T> m[3];
    if constexpr (DIM == 3) {
        const bool xin = x < nx - 1, yin = y < ny - 1, zin = z < nz - 1;
        const T hx = Hx[i], hy = Hy[i], hz = Hz[i];
        const T hyx = x > 0 ? Hy[i - 1] : T(0), hzx = x > 0 ? Hz[i - 1] : T(0);
        const T hxy = y > 0 ? Hx[i - sy] : T(0), hzy = y > 0 ? Hz[i - sy] : T(0);
        const T hxz = z > 0 ? Hx[i - sz] : T(0), hyz = z > 0 ? Hy[i - sz] : T(0);
        PmlCell<T> q[6];
#pragma unroll
        for (int c = 0; c < 3; ++c) m[c].load(a, c, i);
        if (inpml) {
            if (xin) {
                q[0].load(a.pml[0], 1, y, x, y, z, px, ny);
                q[1].load(a.pml[0], 2, z, x, y, z, px, ny);
            }
            if (yin) {
                q[2].load(a.pml[1], 2, z, x, y, z, px, ny);
                q[3].load(a.pml[1], 0, x, x, y, z, px, ny);
            }
            if (zin) {
                q[4].load(a.pml[2], 0, x, x, y, z, px, ny);
                q[5].load(a.pml[2], 1, y, x, y, z, px, ny);
            }
        }
        if (SRC) src_values(a, 0, x, y, z, step, sv);
        const T i0 = a.inv_d[0], i1 = a.inv_d[1], i2 = a.inv_d[2];
        if (xin) e_finish(a, m[0], 0, i, x, y, z, curl_cell(q[0], q[1], inpml, hz - hzy, i1, hy - hyz, i2), sv[0]);
        if (yin) e_finish(a, m[1], 1, i, x, y, z, curl_cell(q[2], q[3], inpml, hx - hxz, i2, hz - hzx, i0), sv[1]);
        if (zin) e_finish(a, m[2], 2, i, x, y, z, curl_cell(q[4], q[5], inpml, hy - hyx, i0, hx - hxy, i1), sv[2]);
    } else {
        const T hx = Hx[i], hy = Hy[i];
        const T hyx = x > 0 ? Hy[i - 1] : T(0), hxy = y > 0 ? Hx[i - sy] : T(0);
        PmlCell<T> q[2];
        m[2].load(a, 2, i);
        if (inpml) {
            q[0].load(a.pml[2], 0, x, x, y, z, px, ny);
            q[1].load(a.pml[2], 1, y, x, y, z, px, ny);
        }
        if (SRC) src_values(a, 0, x, y, z, step, sv);
        e_finish(a, m[2], 2, i, x, y, z, curl_cell(q[0], q[1], inpml, hy - hyx, a.inv_d[0], hx - hxy, a.inv_d[1]), sv[2]);
    }
}

// ------------------------------------------------ 3D split kernels ---------
// The 3D field update is split by region: an interior box (whole x rows of
// the y/z interior, with CPML terms only where a row enters an x slab; in FP64
// on aligned grids the x/y/z interior) and the CPML slabs around it.  The
// whole-row form runs both regions of a field as one launch (k_h3_all /
// k_e3_all), the other as two (k_h3_int + k_h3_slab, k_e3_int + k_e3_slab).
// Every thread takes W consecutive x cells so that every field, psi and
// material access of a lane is one 16-byte load or store (W = 4 in FP32, 2 in
// FP64): on MI355X a plain copy reaches ~3.8 TB/s with 4-byte lanes and
// ~6.3 TB/s with 16-byte lanes.  Rows are stored in whole groups and the psi
// regions widened to whole groups (grid_layout.hpp; identity coefficients on
// the added positions), so that the W cells of a group share their CPML
// membership on every axis.  101x93x87 FP32 with a 10-cell CPML and a
// three-pole metal: one thread per cell 48.6 us a step, groups 27.1.
// The interior walk leaves out the y and z CPML terms at compile time, and
// blocks and groups are numbered in 32 bits: 256^3 FP32 with a 16-cell CPML
// 0.302 -> 0.284 ms a step (the 64-bit divisions of the numbering and the
// slab tests of every group cost the latency that the loads then wait for).
template <typename T>
struct MatLds {
    T ce, inveps;
    int flags, poleset;
};

template <typename T, int W>
struct alignas(sizeof(T) * W) Pk {
    T v[W];
};

template <typename T, int W>
__device__ __forceinline__ Pk<T, W> ldv(const T* p) {
    return *reinterpret_cast<const Pk<T, W>*>(p);
}
template <typename T, int W>
__device__ __forceinline__ void stv(T* p, const Pk<T, W>& v) {
    *reinterpret_cast<Pk<T, W>*>(p) = v;
}
// Streaming forms for the words a kernel touches once (its own cells' field
// values, CPML psi, pole currents, material ids): the nontemporal hint keeps
// them from displacing the neighbour rows and planes the other threads of
// the sweep still read from L2.  A grid whose six fields fit the 256 MB
// memory-side cache with room to spare does better without: the words of one
// sweep then come from that cache in the next.  Measured without and with the
// hint, us a step: FP32 128^3 51 and 58, 192^3 (170 MB) 123 and 135, 200^3
// 152 and 153, 224^3 215 and 196, 256^3 324 and 274; FP64 128^3 93 and 108,
// 152^3 (168 MB) 144 and 155, 160^3 172 and 166.  (Keeping only part of a
// larger grid's rows cached lost: 256^3 with 30% of the rows 295.)  Emitter
// state that each step streams counts with the fields.
constexpr bool streams_past_caches(double bytes) { return bytes > 185e6; }
template <typename T, int W>
using NtVec = T __attribute__((ext_vector_type(W)));
template <typename T, int W>
__device__ __forceinline__ Pk<T, W> ldv_nt(const T* p) {
    const NtVec<T, W> x = __builtin_nontemporal_load(reinterpret_cast<const NtVec<T, W>*>(p));
    Pk<T, W> r;
#pragma unroll
    for (int w = 0; w < W; ++w) r.v[w] = x[w];
    return r;
}
template <typename T, int W>
__device__ __forceinline__ void stv_nt(T* p, const Pk<T, W>& v) {
    NtVec<T, W> x;
#pragma unroll
    for (int w = 0; w < W; ++w) x[w] = v.v[w];
    __builtin_nontemporal_store(x, reinterpret_cast<NtVec<T, W>*>(p));
}
template <bool NT, typename T, int W>
__device__ __forceinline__ Pk<T, W> ldc(const T* p) {
    if constexpr (NT) return ldv_nt<T, W>(p);
    else return ldv<T, W>(p);
}
template <bool NT, typename T, int W>
__device__ __forceinline__ void stc(T* p, const Pk<T, W>& v) {
    if constexpr (NT) stv_nt<T, W>(p, v);
    else stv<T, W>(p, v);
}
template <typename T, int W>
__device__ __forceinline__ Pk<T, W> zpk() {
    Pk<T, W> r;
#pragma unroll
    for (int w = 0; w < W; ++w) r.v[w] = T(0);
    return r;
}

// Blocks are dealt to the 8 XCDs round robin in dispatch order; renumber
// them so that each XCD walks one contiguous eighth of the domain and the
// y/z neighbour rows a block reads were loaded into the same L2.
__device__ __forceinline__ int xcd_block(int b, int nb) {
    const int q = nb / 8, r = nb % 8, x = b % 8, k = b / 8;
    return (x < r ? x * (q + 1) : r * (q + 1) + (x - r) * q) + k;
}

// The cells of the group at x0 with x < nx - 1, as a bit mask (the components
// staggered along x have no point at nx - 1, nor in the row's padding).
template <int W>
__device__ __forceinline__ unsigned cells_below_last(int x0, int nx) {
    constexpr unsigned all = (1u << W) - 1;
    const int n = nx - 1 - x0;
    return n >= W ? all : (n > 0 ? (1u << n) - 1 : 0u);
}

// Does the group [x0, x0 + W) x {y} x {z} touch any source box?
template <typename T, int W>
__device__ __forceinline__ bool group_has_src(const StepArgs<T>& a, int x0, int y, int z) {
    for (int s = 0; s < a.nsrc; ++s) {
        const int* b = a.src_box + 6 * s;
        if (x0 < b[1] && b[0] < x0 + W && y >= b[2] && y < b[3] && z >= b[4] && z < b[5]) return true;
    }
    return false;
}

template <typename T>
__device__ __forceinline__ T ade_apply(const StepArgs<T>& a, int c, int ps, int x, int y, int z, T e_ade) {
    const int* bx = a.box[c];
    long long bi = (x - bx[0]) + static_cast<long long>(bx[1] - bx[0]) * ((y - bx[2]) + static_cast<long long>(bx[3] - bx[2]) * (z - bx[4]));
    const int np = a.pole_count[ps];
    const T* co = a.pole_coef + static_cast<long long>(ps) * CHIML_MAX_POLES * 3;
    T jsum = 0;
    for (int p = 0; p < np; ++p) {
        T* Pp = a.P[c] + p * a.boxn[c];
        T* Jp = a.J[c] + p * a.boxn[c];
        T P = Pp[bi], J = Jp[bi];
        T Jn = co[3 * p] * P + co[3 * p + 1] * J + co[3 * p + 2] * e_ade;
        Pp[bi] = P + Jn;
        Jp[bi] = Jn;
        jsum += Jn;
    }
    return jsum;
}

// E of one cell from its curl term, material and sources (the E-form of
// updatePolE + updateE/updateD + D2E).
template <typename T>
__device__ __forceinline__ T e_new(const StepArgs<T>& a, const MatLds<T>& m, int c, int x, int y, int z, T e_old, T acc, T src) {
    T e_base = (m.flags & CHIML_MAT_DCELL) ? e_old : e_old + src;
    T jsum = 0;
    if (m.poleset >= 0) jsum = ade_apply(a, c, m.poleset, x, y, z, e_old + src);
    return e_base + m.ce * acc - m.inveps * jsum;
}

template <typename T>
__device__ __forceinline__ void load_mat(const StepArgs<T>& a, MatLds<T> (*mt)[CHIML_MAX_MAT], const int* nm) {
    const int tid = threadIdx.x + blockDim.x * threadIdx.y;
    const int nt = blockDim.x * blockDim.y;
    for (int c = 0; c < 3; ++c)
        for (int k = tid; k < nm[c]; k += nt) mt[c][k] = MatLds<T>{a.ce[c][k], a.inveps[c][k], a.flags[c][k], a.poleset[c][k]};
    __syncthreads();
}

struct Box3 {
    int x0, x1, y0, y1, z0, z1;
    int by;  // rows per y band of the interior walk (0: one band)
};

// CPML term of derivative axis ax for the W cells of a group (pml_term for a
// group): term = dV/(kappa d) + psi' with psi' = b psi + (c/d) dV on psi
// positions, term = dV/d elsewhere.  psi is written back only for the cells
// in `valid` (cells the reference does not update keep their psi).
template <typename T, int W>
__device__ __forceinline__ void pml_group(const PmlDev<T>& p, int ax, int pos0, int x0, int y, int z, int nx, int ny, const T (&dV)[W],
                                          T invd, unsigned valid, T (&term)[W]) {
    int s;
    if (pos0 < p.lo[ax]) s = pos0;
    else if (pos0 >= p.hi0[ax] && pos0 < p.hi1[ax]) s = p.lo[ax] + pos0 - p.hi0[ax];
    else {
#pragma unroll
        for (int w = 0; w < W; ++w) term[w] = dV[w] * invd;
        return;
    }
    long long pi;
    if (ax == 0) pi = s + static_cast<long long>(p.S[0]) * (y + static_cast<long long>(ny) * z);
    else if (ax == 1) pi = x0 + static_cast<long long>(nx) * (s + static_cast<long long>(p.S[1]) * z);
    else pi = x0 + static_cast<long long>(nx) * (y + static_cast<long long>(ny) * s);
    Pk<T, W> ps = ldv_nt<T, W>(p.psi[ax] + pi);
#pragma unroll
    for (int w = 0; w < W; ++w) {
        const int pos = ax == 0 ? pos0 + w : pos0;
        const T psi = p.b[ax][pos] * ps.v[w] + p.cd[ax][pos] * dV[w];
        if (valid & (1u << w)) ps.v[w] = psi;
        term[w] = p.kinv[ax][pos] * (dV[w] * invd) + psi;
    }
    stv_nt<T, W>(p.psi[ax] + pi, ps);
}

// One CPML term of a group along derivative axis AX (pml_group's arithmetic):
// load() fetches psi and the profiles with the component's other loads, apply()
// forms the term and stores psi.  ON = false: a region without this term.
template <typename T, int W, int AX, bool ON, bool NT>
struct PsiTerm {
    int s;
    T* at;
    Pk<T, W> ps;
    T b[AX == 0 ? W : 1], cd[AX == 0 ? W : 1], ki[AX == 0 ? W : 1];
    __device__ __forceinline__ void load(const PmlDev<T>& p, int pos, int x0, int y, int z, int px, int ny) {
        s = -1;
        if (!ON) return;
        if (pos < p.lo[AX]) s = pos;
        else if (pos >= p.hi0[AX] && pos < p.hi1[AX]) s = p.lo[AX] + pos - p.hi0[AX];
        if (s < 0) return;
        long long pi;
        if (AX == 0) pi = s + static_cast<long long>(p.S[0]) * (y + static_cast<long long>(ny) * z);
        else if (AX == 1) pi = x0 + static_cast<long long>(px) * (s + static_cast<long long>(p.S[1]) * z);
        else pi = x0 + static_cast<long long>(px) * (y + static_cast<long long>(ny) * s);
        at = p.psi[AX] + pi;
        ps = ldc<NT, T, W>(at);
        if (AX == 0) {
            const Pk<T, W> vb = ldv<T, W>(p.b[0] + pos), vc = ldv<T, W>(p.cd[0] + pos), vk = ldv<T, W>(p.kinv[0] + pos);
#pragma unroll
            for (int w = 0; w < (AX == 0 ? W : 1); ++w) {
                b[w] = vb.v[w];
                cd[w] = vc.v[w];
                ki[w] = vk.v[w];
            }
        } else {
            b[0] = p.b[AX][pos];
            cd[0] = p.cd[AX][pos];
            ki[0] = p.kinv[AX][pos];
        }
    }
    // term = dV/d, or dV/(kappa d) + psi' on psi positions; cells outside
    // `valid` keep their psi
    __device__ __forceinline__ void apply(const T (&dV)[W], T invd, unsigned valid, T (&term)[W]) {
#pragma unroll
        for (int w = 0; w < W; ++w) term[w] = dV[w] * invd;
        if (!ON || s < 0) return;
#pragma unroll
        for (int w = 0; w < W; ++w) {
            const int k = AX == 0 ? w : 0;
            const T psi = fma(b[k], ps.v[w], cd[k] * dV[w]);
            if (valid & (1u << w)) ps.v[w] = psi;
            term[w] = fma(ki[k], term[w], psi);
        }
        stc<NT, T, W>(at, ps);
    }
};

// t1 - t2 of a curl.  FMA (grids whose rows or x CPML are no whole groups):
// cells outside the CPML keep the second product unrounded, as the per-cell
// kernels that swept such grids form it; FP32 metals amplify a change of
// rounding.  plain: the group's cells outside the CPML.
template <typename T, int W, bool FMA>
__device__ __forceinline__ void curl_of(const T (&t1)[W], const T (&t2)[W], const T (&d2)[W], T inv2, unsigned plain, T (&acc)[W]) {
// (a product that feeds the difference is rounded first, whatever the path)
#pragma clang fp contract(off)
#pragma unroll
    for (int w = 0; w < W; ++w) {
        acc[w] = t1[w] - t2[w];
        if (FMA && (plain & (1u << w))) acc[w] = fma(-inv2, d2[w], t1[w]);
    }
}

// The cells of the group with Tx <= x < nx - Tx, as a bit mask.
template <int W>
__device__ __forceinline__ unsigned cells_inside(int x0, int nx, int Tx) {
    unsigned m = 0;
#pragma unroll
    for (int w = 0; w < W; ++w)
        if (x0 + w >= Tx && x0 + w < nx - Tx) m |= 1u << w;
    return m;
}

// H update of the group (x0..x0+W-1, y, z): H += ch (curl E) (+ sources).
// PX / PYZ: the group may lie in an x / in a y or z CPML slab.
// nb: the next lane of the wave holds the next group of the same row, so the
// first value of that group comes by a lane shuffle instead of a load.
template <typename T, int W, bool PX, bool PYZ, bool SRC, bool FMA, bool NT>
__device__ __forceinline__ void h_group(const StepArgs<T>& a, int x0, int y, int z, bool nb = false) {
    const int nx = a.nx, ny = a.ny, nz = a.nz, px = a.px;
    const long long sy = px, sz = static_cast<long long>(px) * ny;
    const long long i = lidx(x0, y, z, px, ny);
    const T idx = a.inv_d[0], idy = a.inv_d[1], idz = a.inv_d[2];
    const T *Ex = a.F[0], *Ey = a.F[1], *Ez = a.F[2];
    const Pk<T, W> ex = ldv<T, W>(Ex + i), ey = ldv<T, W>(Ey + i), ez = ldv<T, W>(Ez + i);
    const bool last = x0 + W >= nx, yin = y < ny - 1, zin = z < nz - 1;
    const unsigned all = (1u << W) - 1, vx = cells_below_last<W>(x0, nx);  // vx: cells with x < nx - 1
    const unsigned plain = FMA && !PYZ ? cells_inside<W>(x0, nx, a.Tp[0]) : 0u;
    const T ez_nb = __shfl_down(ez.v[0], 1), ey_nb = __shfl_down(ey.v[0], 1);
    const bool src = SRC && group_has_src<T, W>(a, x0, y, z);
    const int step = src ? step_now(a.step, a.stepv) : 0;
    T d1[W], d2[W], t1[W], t2[W], acc[W];
    auto finish = [&](int c, Pk<T, W>& h, unsigned valid) {
        const T ch = a.ch[c][0];
#pragma unroll
        for (int w = 0; w < W; ++w) {
            if (!(valid & (1u << w))) continue;
            T hv = fma(ch, acc[w], h.v[w]);
            if (src) hv += src_value(a, 3 + c, x0 + w, y, z, step);
            h.v[w] = hv;
        }
        stc<NT, T, W>(a.F[3 + c] + i, h);
    };
    if (yin && zin) {  // Hx += ch [dEy/dz - dEz/dy]
        const Pk<T, W> eyz = ldv<T, W>(Ey + i + sz), ezy = ldv<T, W>(Ez + i + sy);
        Pk<T, W> h = ldc<NT, T, W>(a.F[3] + i);
        PsiTerm<T, W, 2, PYZ, NT> q1;
        PsiTerm<T, W, 1, PYZ, NT> q2;
        q1.load(a.pml[3], z, x0, y, z, px, ny);
        q2.load(a.pml[3], y, x0, y, z, px, ny);
#pragma unroll
        for (int w = 0; w < W; ++w) {
            d1[w] = eyz.v[w] - ey.v[w];
            d2[w] = ezy.v[w] - ez.v[w];
        }
        q1.apply(d1, idz, all, t1);
        q2.apply(d2, idy, all, t2);
        curl_of<T, W, FMA>(t1, t2, d2, idy, plain, acc);
        finish(0, h, all);
    }
    if (zin) {  // Hy += ch [dEz/dx - dEx/dz], x < nx - 1
        const Pk<T, W> exz = ldv<T, W>(Ex + i + sz);
        const T ezn = last ? T(0) : (nb ? ez_nb : Ez[i + W]);
        Pk<T, W> h = ldc<NT, T, W>(a.F[4] + i);
        PsiTerm<T, W, 0, PX, NT> q1;
        PsiTerm<T, W, 2, PYZ, NT> q2;
        q1.load(a.pml[4], x0, x0, y, z, px, ny);
        q2.load(a.pml[4], z, x0, y, z, px, ny);
#pragma unroll
        for (int w = 0; w < W; ++w) {
            d1[w] = (w + 1 < W ? ez.v[w + 1 < W ? w + 1 : w] : ezn) - ez.v[w];
            d2[w] = exz.v[w] - ex.v[w];
        }
        q1.apply(d1, idx, vx, t1);
        q2.apply(d2, idz, vx, t2);
        curl_of<T, W, FMA>(t1, t2, d2, idz, plain, acc);
        finish(1, h, vx);
    }
    if (yin) {  // Hz += ch [dEx/dy - dEy/dx], x < nx - 1
        const Pk<T, W> exy = ldv<T, W>(Ex + i + sy);
        const T eyn = last ? T(0) : (nb ? ey_nb : Ey[i + W]);
        Pk<T, W> h = ldc<NT, T, W>(a.F[5] + i);
        PsiTerm<T, W, 1, PYZ, NT> q1;
        PsiTerm<T, W, 0, PX, NT> q2;
        q1.load(a.pml[5], y, x0, y, z, px, ny);
        q2.load(a.pml[5], x0, x0, y, z, px, ny);
#pragma unroll
        for (int w = 0; w < W; ++w) {
            d1[w] = exy.v[w] - ex.v[w];
            d2[w] = (w + 1 < W ? ey.v[w + 1 < W ? w + 1 : w] : eyn) - ey.v[w];
        }
        q1.apply(d1, idy, vx, t1);
        q2.apply(d2, idx, vx, t2);
        curl_of<T, W, FMA>(t1, t2, d2, idx, plain, acc);
        finish(2, h, vx);
    }
}

template <int W, bool NT = true>
__device__ __forceinline__ Pk<uint8_t, W> load_ids(const uint8_t* m, long long i) {
    if (!m) {
        Pk<uint8_t, W> z;
#pragma unroll
        for (int w = 0; w < W; ++w) z.v[w] = 0;
        return z;
    }
    return ldc<NT, uint8_t, W>(m + i);
}

// E of the W cells of a group from their curl acc, materials,
// sources and poles: e_new for a group, with each pole's P and J of the
// group read and written as one aligned 16-byte access (the pole-state box
// is 4-aligned in x); cells without poles keep their stored values.
template <typename T, int W>
__device__ __forceinline__ Pk<T, W> e_finish_group(const StepArgs<T>& a, const MatLds<T> (*mt)[CHIML_MAX_MAT], int c, long long i, int x0,
                                               int y, int z, unsigned valid, const T (&acc)[W], bool src, int step) {
    const Pk<uint8_t, W> id = load_ids<W>(a.mat_e[c], i);
    Pk<T, W> e = ldv_nt<T, W>(a.F[c] + i);
    T jsum[W];
    bool anyp = false;
#pragma unroll
    for (int w = 0; w < W; ++w) {
        jsum[w] = T(0);
        anyp |= (mt[c][id.v[w]].poleset >= 0) && (valid & (1u << w));
    }
    if (anyp) {  // rare: groups that touch a dispersive object
        const int* bx = a.box[c];
        const long long bi = (x0 - bx[0]) + static_cast<long long>(bx[1] - bx[0]) * ((y - bx[2]) + static_cast<long long>(bx[3] - bx[2]) * (z - bx[4]));
        int np[W], npmax = 0;
#pragma unroll
        for (int w = 0; w < W; ++w) {
            const int ps = mt[c][id.v[w]].poleset;
            np[w] = (ps >= 0 && (valid & (1u << w))) ? a.pole_count[ps] : 0;
            npmax = max(npmax, np[w]);
        }
        for (int p = 0; p < npmax; ++p) {
            T* Pp = a.P[c] + p * a.boxn[c] + bi;
            T* Jp = a.J[c] + p * a.boxn[c] + bi;
            Pk<T, W> P = ldv_nt<T, W>(Pp), J = ldv_nt<T, W>(Jp);
#pragma unroll
            for (int w = 0; w < W; ++w) {
                if (p >= np[w]) continue;
                const int ps = mt[c][id.v[w]].poleset;
                const T* co = a.pole_coef + (static_cast<long long>(ps) * CHIML_MAX_POLES + p) * 3;
                const T sv = src ? src_value(a, c, x0 + w, y, z, step) : T(0);
                const T Jn = co[0] * P.v[w] + co[1] * J.v[w] + co[2] * (e.v[w] + sv);
                P.v[w] = P.v[w] + Jn;
                J.v[w] = Jn;
                jsum[w] += Jn;
            }
            stv_nt<T, W>(Pp, P);
            stv_nt<T, W>(Jp, J);
        }
    }
#pragma unroll
    for (int w = 0; w < W; ++w) {
        if (!(valid & (1u << w))) continue;
        const MatLds<T> m = mt[c][id.v[w]];
        const T sv = src ? src_value(a, c, x0 + w, y, z, step) : T(0);
        const T e_base = (m.flags & CHIML_MAT_DCELL) ? e.v[w] : e.v[w] + sv;
        e.v[w] = fma(-m.inveps, jsum[w], fma(m.ce, acc[w], e_base));
    }
    stv_nt<T, W>(a.F[c] + i, e);
    return e;
}

// E update of the group: the E-form of updateE/updateD + ADE + D2E per cell,
// the pole currents already advanced by ade_block.  PX, PYZ, FMA as in
// h_group; mt: the material tables in LDS.
// nb: the previous lane of the wave holds the previous group of the same row
template <typename T, int W, bool PX, bool PYZ, bool SRC, bool FMA, bool NT>
__device__ __forceinline__ void e_group(const StepArgs<T>& a, const MatLds<T> (*mt)[CHIML_MAX_MAT], int x0, int y, int z,
                                        bool nb = false) {
    const int nx = a.nx, ny = a.ny, nz = a.nz, px = a.px;
    const long long sy = px, sz = static_cast<long long>(px) * ny;
    const long long i = lidx(x0, y, z, px, ny);
    const T idx = a.inv_d[0], idy = a.inv_d[1], idz = a.inv_d[2];
    const T *Hx = a.F[3], *Hy = a.F[4], *Hz = a.F[5];
    const Pk<T, W> hx = ldv<T, W>(Hx + i), hy = ldv<T, W>(Hy + i), hz = ldv<T, W>(Hz + i);
    const bool yin = y < ny - 1, zin = z < nz - 1;
    const unsigned all = (1u << W) - 1, vx = cells_below_last<W>(x0, nx);
    const unsigned plain = FMA && !PYZ ? cells_inside<W>(x0, nx, a.Tp[0]) : 0u;
    const T hz_nb = __shfl_up(hz.v[W - 1], 1), hy_nb = __shfl_up(hy.v[W - 1], 1);
    const bool src = SRC && group_has_src<T, W>(a, x0, y, z);
    const int step = src ? step_now(a.step, a.stepv) : 0;
    T d1[W], d2[W], t1[W], t2[W], acc[W];
    auto finish = [&](int c, unsigned valid) {
        const Pk<uint8_t, W> id = load_ids<W, NT>(a.mat_e[c], i);
        Pk<T, W> e = ldc<NT, T, W>(a.F[c] + i);
        bool anyp = false;
#pragma unroll
        for (int w = 0; w < W; ++w) anyp |= (mt[c][id.v[w]].poleset >= 0) && (valid & (1u << w));
        Pk<T, W> js = zpk<T, W>();
        if (anyp) {  // rare: groups that touch a dispersive object
            const int* bx = a.box[c];
            const long long bi = (x0 - bx[0]) + static_cast<long long>(bx[1] - bx[0]) * ((y - bx[2]) + static_cast<long long>(bx[3] - bx[2]) * (z - bx[4]));
            js = ldv<T, W>(a.jsum[c] + bi);
        }
#pragma unroll
        for (int w = 0; w < W; ++w) {
            if (!(valid & (1u << w))) continue;
            const MatLds<T> m = mt[c][id.v[w]];
            const T sv = src ? src_value(a, c, x0 + w, y, z, step) : T(0);
            const T e_base = (m.flags & CHIML_MAT_DCELL) ? e.v[w] : e.v[w] + sv;
            const T jsum = m.poleset >= 0 ? js.v[w] : T(0);
            e.v[w] = fma(-m.inveps, jsum, fma(m.ce, acc[w], e_base));
        }
        stc<NT, T, W>(a.F[c] + i, e);
    };
    {  // Ex += ce [dHz/dy - dHy/dz], x < nx - 1
        const Pk<T, W> hzy = y > 0 ? ldv<T, W>(Hz + i - sy) : zpk<T, W>();
        const Pk<T, W> hyz = z > 0 ? ldv<T, W>(Hy + i - sz) : zpk<T, W>();
        PsiTerm<T, W, 1, PYZ, NT> q1;
        PsiTerm<T, W, 2, PYZ, NT> q2;
        q1.load(a.pml[0], y, x0, y, z, px, ny);
        q2.load(a.pml[0], z, x0, y, z, px, ny);
#pragma unroll
        for (int w = 0; w < W; ++w) {
            d1[w] = hz.v[w] - hzy.v[w];
            d2[w] = hy.v[w] - hyz.v[w];
        }
        q1.apply(d1, idy, vx, t1);
        q2.apply(d2, idz, vx, t2);
        curl_of<T, W, FMA>(t1, t2, d2, idz, plain, acc);
        finish(0, vx);
    }
    if (yin) {  // Ey += ce [dHx/dz - dHz/dx]
        const Pk<T, W> hxz = z > 0 ? ldv<T, W>(Hx + i - sz) : zpk<T, W>();
        const T hzm = x0 > 0 ? (nb ? hz_nb : Hz[i - 1]) : T(0);
        PsiTerm<T, W, 2, PYZ, NT> q1;
        PsiTerm<T, W, 0, PX, NT> q2;
        q1.load(a.pml[1], z, x0, y, z, px, ny);
        q2.load(a.pml[1], x0, x0, y, z, px, ny);
#pragma unroll
        for (int w = 0; w < W; ++w) {
            d1[w] = hx.v[w] - hxz.v[w];
            d2[w] = hz.v[w] - (w > 0 ? hz.v[w > 0 ? w - 1 : 0] : hzm);
        }
        q1.apply(d1, idz, all, t1);
        q2.apply(d2, idx, all, t2);
        curl_of<T, W, FMA>(t1, t2, d2, idx, plain, acc);
        finish(1, all);
    }
    if (zin) {  // Ez += ce [dHy/dx - dHx/dy]
        const Pk<T, W> hxy = y > 0 ? ldv<T, W>(Hx + i - sy) : zpk<T, W>();
        const T hym = x0 > 0 ? (nb ? hy_nb : Hy[i - 1]) : T(0);
        PsiTerm<T, W, 0, PX, NT> q1;
        PsiTerm<T, W, 1, PYZ, NT> q2;
        q1.load(a.pml[2], x0, x0, y, z, px, ny);
        q2.load(a.pml[2], y, x0, y, z, px, ny);
#pragma unroll
        for (int w = 0; w < W; ++w) {
            d1[w] = hy.v[w] - (w > 0 ? hy.v[w > 0 ? w - 1 : 0] : hym);
            d2[w] = hx.v[w] - hxy.v[w];
        }
        q1.apply(d1, idx, all, t1);
        q2.apply(d2, idy, all, t2);
        curl_of<T, W, FMA>(t1, t2, d2, idy, plain, acc);
        finish(2, all);
    }
}

// Pole update of the 3D split path, before the E kernels: one thread per
// W-cell group of component c's pole box (blk: block within the component),
// run by the first blocks of the H interior launch, so the few dispersive
// cells are spread over the whole chip instead of loading the XCDs whose
// part of the domain holds the object.  It advances P and J from
// E before its update (plus the soft source, as updatePolE sees it) and
// leaves the sum of the new currents per cell in jsum for the E kernels.
template <typename T, int W, bool SRC>
__device__ __forceinline__ void ade_block(const StepArgs<T>& a, int c, long long blk) {
    const int* bx = a.box[c];
    if (!a.jsum[c]) return;
    const int gw = (bx[1] - bx[0]) / W, ny = bx[3] - bx[2], nz = bx[5] - bx[4];
    const long long t = blk * blockDim.x + threadIdx.x;
    if (t >= static_cast<long long>(gw) * ny * nz) return;
    const long long r = t / gw;
    const int x0 = bx[0] + static_cast<int>(t - r * gw) * W;
    const int y = bx[2] + static_cast<int>(r % ny), z = bx[4] + static_cast<int>(r / ny);
    const long long bi = t * W;  // (x0 - bx0) + width * ((y - by0) + height * (z - bz0))
    const long long i = lidx(x0, y, z, a.px, a.ny);
    const Pk<uint8_t, W> id = load_ids<W>(a.mat_e[c], i);
    // the cells the E kernels update: Ex x < nx - 1, Ey y < ny - 1, Ez z < nz - 1
    unsigned valid = (1u << W) - 1;
    if (c == 0) valid = cells_below_last<W>(x0, a.nx);
    if ((c == 1 && y >= a.ny - 1) || (c == 2 && z >= a.nz - 1)) valid = 0;
    int ps[W], np[W], npmax = 0;
#pragma unroll
    for (int w = 0; w < W; ++w) {
        ps[w] = (valid & (1u << w)) ? a.poleset[c][id.v[w]] : -1;
        np[w] = ps[w] >= 0 ? a.pole_count[ps[w]] : 0;
        npmax = max(npmax, np[w]);
    }
    Pk<T, W> js = zpk<T, W>();
    if (npmax > 0) {
        const bool src = SRC && group_has_src<T, W>(a, x0, y, z);
        const int step = src ? step_now(a.step, a.stepv) : 0;
        const Pk<T, W> e = ldv<T, W>(a.F[c] + i);
        T ea[W];
#pragma unroll
        for (int w = 0; w < W; ++w) ea[w] = e.v[w] + (src ? src_value(a, c, x0 + w, y, z, step) : T(0));
        for (int p = 0; p < npmax; ++p) {
            T* Pp = a.P[c] + p * a.boxn[c] + bi;
            T* Jp = a.J[c] + p * a.boxn[c] + bi;
            Pk<T, W> P = ldv_nt<T, W>(Pp), J = ldv_nt<T, W>(Jp);
#pragma unroll
            for (int w = 0; w < W; ++w) {
                if (p >= np[w]) continue;
                const T* co = a.pole_coef + (static_cast<long long>(ps[w]) * CHIML_MAX_POLES + p) * 3;
                const T Jn = co[0] * P.v[w] + co[1] * J.v[w] + co[2] * ea[w];
                P.v[w] = P.v[w] + Jn;
                J.v[w] = Jn;
                js.v[w] += Jn;
            }
            stv_nt<T, W>(Pp, P);
            stv_nt<T, W>(Jp, J);
        }
    }
    stv<T, W>(a.jsum[c] + bi, js);
}

// Interior box, one group per thread, walked band by band: x fastest, then
// the by rows of a y band, then z, then the band.  With the XCD renumbering
// each XCD marches one band through z, so the rows of the previous and next
// planes a group reads are still in that XCD's L2 (a whole plane of six
// fields is larger than an L2).
template <typename T, int W>
__device__ __forceinline__ bool int_group(const Box3& b, int blk, int& x0, int& y, int& z, int& col) {
    const unsigned gw = (b.x1 - b.x0) / W, ny = b.y1 - b.y0, nz = b.z1 - b.z0;
    const unsigned by = b.by > 0 ? b.by : ny, nb = (ny + by - 1) / by;
    const unsigned t = static_cast<unsigned>(blk) * blockDim.x + threadIdx.x;
    unsigned r = t / gw;
    if (r >= by * nz * nb) return false;
    col = static_cast<int>(t - r * gw);
    x0 = b.x0 + col * W;
    const unsigned p = r / by, band = p / nz;
    z = b.z0 + static_cast<int>(p - band * nz);
    y = b.y0 + static_cast<int>(band * by + (r - p * by));
    return y < b.y1;  // the last band may be short
}

// FP64 interior (the x slabs are left to the slab kernel, so the interior
// carries no CPML code).  The first ade_blocks(ade_bpc) blocks run the pole update (ade_bpc blocks
// per E component, padded to a multiple of 8 so that the interior blocks
// keep their XCD numbering): it reads only E, which this kernel does not
// write, and its latency-bound blocks overlap the bandwidth-bound H sweep
// (15 us less than a launch of its own on the 256^3 step).
__host__ __device__ constexpr int ade_blocks(int ade_bpc) { return (3 * ade_bpc + 7) / 8 * 8; }

template <typename T, int W, bool SRC, bool NT>
__device__ __forceinline__ void h3_int_sweep(const StepArgs<T>& a, const Box3& b, int nib, int ade_bpc, int bx) {
    const int nade = ade_blocks(ade_bpc);
    if (bx < nade) {
        const int c = bx / max(ade_bpc, 1);
        if (c < 3) ade_block<T, W, SRC>(a, c, bx - c * ade_bpc);
        return;
    }
    int x0, y, z, col;
    if (!int_group<T, W>(b, xcd_block(bx - nade, nib), x0, y, z, col)) return;
    // consecutive threads walk a row: lane + 1 holds the next group unless this one ends the row
    const int lane = threadIdx.x & 63, gw = (b.x1 - b.x0) / W;
    h_group<T, W, false, false, SRC, false, NT>(a, x0, y, z, lane < 63 && col + 1 < gw);
}

template <typename T, int W, bool SRC, bool ADV, bool NT>
__global__ void __launch_bounds__(256) k_h3_int(StepArgs<T> a, Box3 b, int nib, int ade_bpc) {
    h3_int_sweep<T, W, SRC, NT>(a, b, nib, ade_bpc, blockIdx.x);
    if (ADV) advance_counter(a);
}

template <typename T, int W, bool SRC, bool NT>
__device__ __forceinline__ void e3_int_sweep(const StepArgs<T>& a, const MatLds<T> (*mt)[CHIML_MAX_MAT], const Box3& b, int bx, int nb) {
    int x0, y, z, col;
    if (!int_group<T, W>(b, xcd_block(bx, nb), x0, y, z, col)) return;
    const int lane = threadIdx.x & 63;
    e_group<T, W, false, false, SRC, false, NT>(a, mt, x0, y, z, lane > 0 && col > 0);
}

template <typename T, int W, bool SRC, bool NT>
__global__ void __launch_bounds__(256) k_e3_int(StepArgs<T> a, Box3 b, int nm0, int nm1, int nm2) {
    __shared__ MatLds<T> mt[3][CHIML_MAX_MAT];
    const int nm[3] = {nm0, nm1, nm2};
    load_mat(a, mt, nm);
    e3_int_sweep<T, W, SRC, NT>(a, mt, b, blockIdx.x, gridDim.x);
}

// CPML slab groups: the union of the z slabs, the y slabs inside the z range
// and the x slabs inside the y and z ranges, enumerated x fastest, in units
// of W-cell groups (gx = nx / W groups per row, gT = Tx / W per x slab).
struct SlabMap {
    int nx, ny, nz, Tx, Ty, Tz, W;  // nx: cells per stored row
    unsigned nA, nB, nC;  // group counts of the three regions
};

// col / rowlen: the group's place in a run of consecutive groups of one x
// row (rowlen 0 where rows are not walked whole: the x slabs)
__device__ __forceinline__ bool slab_group(const SlabMap& m, unsigned t, int& x0, int& y, int& z, int& col, int& rowlen) {
    if (t >= m.nA + m.nB + m.nC) return false;
    const unsigned gx = m.nx / m.W;
    rowlen = gx;
    if (t < m.nA) {  // z slabs: z in [0,Tz) U [nz-Tz,nz), all x, y
        const unsigned row = t / gx, k = row / m.ny;
        z = static_cast<int>(k) < m.Tz ? k : m.nz - 2 * m.Tz + k;
        y = row - k * m.ny;
        col = t - row * gx;
        x0 = col * m.W;
        return true;
    }
    t -= m.nA;
    if (t < m.nB) {  // y slabs inside the z interior
        const unsigned row = t / gx, w = 2 * m.Ty, k = row / w;
        z = m.Tz + k;
        const int yy = row - k * w;
        col = t - row * gx;
        x0 = col * m.W;
        y = yy < m.Ty ? yy : m.ny - 2 * m.Ty + yy;
        return true;
    }
    t -= m.nB;
    col = 0;
    rowlen = 0;
    // x slabs inside the y and z interiors
    const unsigned gT = 2 * (m.Tx / m.W), row = t / gT, nyi = m.ny - 2 * m.Ty, k = row / nyi;
    z = m.Tz + k;
    const int xx = static_cast<int>(t - row * gT) * m.W;
    y = m.Ty + static_cast<int>(row - k * nyi);
    x0 = xx < m.Tx ? xx : m.nx - 2 * m.Tx + xx;
    return true;
}

template <typename T, int W, bool SRC, bool NT>
__device__ __forceinline__ void h3_slab_sweep(const StepArgs<T>& a, const SlabMap& m, int bx, int nb) {
    int x0, y, z, col, rowlen;
    if (!slab_group(m, static_cast<unsigned>(xcd_block(bx, nb)) * blockDim.x + threadIdx.x, x0, y, z, col, rowlen)) return;
    // the z- and y-slab regions start on row boundaries (nA is whole rows), so
    // lane + 1 holds the next group of the row unless this one ends it
    h_group<T, W, true, true, SRC, false, NT>(a, x0, y, z, (threadIdx.x & 63) < 63 && col + 1 < rowlen);
}

template <typename T, int W, bool SRC, bool NT>
__global__ void __launch_bounds__(256) k_h3_slab(StepArgs<T> a, SlabMap m) {
    h3_slab_sweep<T, W, SRC, NT>(a, m, blockIdx.x, gridDim.x);
}

template <typename T, int W, bool SRC, bool NT>
__device__ __forceinline__ void e3_slab_sweep(const StepArgs<T>& a, const MatLds<T> (*mt)[CHIML_MAX_MAT], const SlabMap& m, int bx, int nb) {
    int x0, y, z, col, rowlen;
    if (!slab_group(m, static_cast<unsigned>(xcd_block(bx, nb)) * blockDim.x + threadIdx.x, x0, y, z, col, rowlen)) return;
    e_group<T, W, true, true, SRC, false, NT>(a, mt, x0, y, z);  // (the lane shuffle measured slower here)
}

template <typename T, int W, bool SRC, bool NT>
__global__ void __launch_bounds__(256) k_e3_slab(StepArgs<T> a, SlabMap m, int nm0, int nm1, int nm2) {
    __shared__ MatLds<T> mt[3][CHIML_MAX_MAT];
    const int nm[3] = {nm0, nm1, nm2};
    load_mat(a, mt, nm);
    e3_slab_sweep<T, W, SRC, NT>(a, mt, m, blockIdx.x, gridDim.x);
}

// Whole-row layout (GridLayout::rows): the whole 3D sweep of a field in one
// launch, [pole update | CPML slabs | interior] for H and [CPML slabs |
// interior] for E, each region starting on a multiple of 8 blocks so that
// every region keeps its XCD numbering.  The less efficient slab and pole
// blocks run first and overlap the interior stream, and two launch ramps and
// tails per step go away (5% on the 256^3 FP32 step).  Aligned FP64 grids keep
// separate launches: there the interior kernel carries no CPML code and runs
// at a higher occupancy than a merged kernel would.
template <typename T, int W, bool SRC, bool FMA, bool NT>
__device__ __forceinline__ void h3_all_sweep(const StepArgs<T>& a, const Box3& b, const SlabMap& m, int nib, int nsbp,
                                             int ade_bpc, int bx) {
    const int nade = ade_blocks(ade_bpc);
    if (bx < nade) {
        const int c = bx / max(ade_bpc, 1);
        if (c < 3) ade_block<T, W, SRC>(a, c, bx - c * ade_bpc);
        return;
    }
    bx -= nade;
    if (bx < nsbp) {
        int x0, y, z, col, rowlen;
        if (!slab_group(m, static_cast<unsigned>(xcd_block(bx, nsbp)) * blockDim.x + threadIdx.x, x0, y, z, col, rowlen)) return;
        h_group<T, W, true, true, SRC, FMA, NT>(a, x0, y, z, (threadIdx.x & 63) < 63 && col + 1 < rowlen);
        return;
    }
    bx -= nsbp;
    int x0, y, z, col;
    if (!int_group<T, W>(b, xcd_block(bx, nib), x0, y, z, col)) return;
    const int lane = threadIdx.x & 63, gw = (b.x1 - b.x0) / W;
    h_group<T, W, true, false, SRC, FMA, NT>(a, x0, y, z, lane < 63 && col + 1 < gw);
}

template <typename T, int W, bool SRC, bool ADV, bool FMA, bool NT>
__global__ void __launch_bounds__(256) k_h3_all(StepArgs<T> a, Box3 b, SlabMap m, int nib, int nsbp, int ade_bpc) {
    h3_all_sweep<T, W, SRC, FMA, NT>(a, b, m, nib, nsbp, ade_bpc, blockIdx.x);
    if (ADV) advance_counter(a);
}

template <typename T, int W, bool SRC, bool FMA, bool NT>
__device__ __forceinline__ void e3_all_sweep(const StepArgs<T>& a, const MatLds<T> (*mt)[CHIML_MAX_MAT], const Box3& b, const SlabMap& m,
                                             int nib, int nsbp, int bx) {
    if (bx < nsbp) {
        int x0, y, z, col, rowlen;
        if (!slab_group(m, static_cast<unsigned>(xcd_block(bx, nsbp)) * blockDim.x + threadIdx.x, x0, y, z, col, rowlen)) return;
        e_group<T, W, true, true, SRC, FMA, NT>(a, mt, x0, y, z);
        return;
    }
    bx -= nsbp;
    int x0, y, z, col;
    if (!int_group<T, W>(b, xcd_block(bx, nib), x0, y, z, col)) return;
    const int lane = threadIdx.x & 63;
    e_group<T, W, true, false, SRC, FMA, NT>(a, mt, x0, y, z, lane > 0 && col > 0);
}

template <typename T, int W, bool SRC, bool FMA, bool NT>
__global__ void __launch_bounds__(256) k_e3_all(StepArgs<T> a, Box3 b, SlabMap m, int nib, int nsbp, int nm0, int nm1, int nm2) {
    __shared__ MatLds<T> mt[3][CHIML_MAX_MAT];
    const int nm[3] = {nm0, nm1, nm2};
    load_mat(a, mt, nm);
    e3_all_sweep<T, W, SRC, FMA, NT>(a, mt, b, m, nib, nsbp, blockIdx.x);
}

// ------------------------------------------------------- fused 3D step ----
// One launch advances H and then E over the whole 3D domain, so that each
// field word is read once and written once per step (the split sweeps read
// E again in the H sweep and H again in the E sweep).  The fields are
// ping-ponged: old values come from a.G, new ones go to a.F, and so does the
// CPML psi of the H components (pml[3..5].psi_in -> psi); the E psi is
// updated in place.  A block owns a tile of `ty` whole x rows for `lz`
// consecutive planes and marches it through z.  Per plane it computes H for
// its rows and, without storing it, for the row below the tile; shares the
// plane through LDS; then computes E, which needs H at x-1 and y-1 (LDS) and
// at z-1 (registers, from the previous plane).  A segment's first plane
// takes H at z-1 from the same recomputation.  The reference's phase order
// (H, sources on H, pole update, E, parallelFDTDField.hpp:1228-1303) holds
// per cell: a cell's E is formed from H values that are final for the step.
constexpr int kFusedMaxThreads = 640;  // (ty + 1) * gx at most: 9 + 1 rows of 64 groups

struct FuseMap {
    int gx;        // W-cell groups per x row (nx / W)
    int ty;        // rows per tile
    int ntile;     // tiles along y
    int nseg;      // segments along z
    int lz;        // planes per segment
    int nthr;      // (ty + 1) * gx working threads of a block
    int ys0, ys1;  // rows outside [ys0, ys1) carry y CPML psi of some component
    int zs0, zs1;  // planes outside [zs0, zs1) carry z CPML psi of some component
    unsigned cstride;  // bytes between components of a field buffer (a.F[k] = a.F[0] + k N)
    int xpsi;          // the x-CPML psi of Hy, Hz, Ey and Ez exist (all four or none)
};

// CPML profiles of the fused kernel in LDS, by slab-compact position s
// (the psi array's own index along its axis): b, c/d and 1/kappa for each
// component and derivative axis that carries psi.  Staged at kernel entry,
// so the per-cell CPML terms read LDS instead of waiting on global loads.
constexpr int kFusedSlab = 64;  // psi positions per axis (both slabs) at most

template <typename T>
struct ProfLds {
    T v[6][3][3][kFusedSlab];  // [comp][axis][b, c/d, 1/kappa][s]
};

template <typename T>
__device__ __forceinline__ void load_prof_lds(const StepArgs<T>& a, ProfLds<T>& P) {
    const int tid = threadIdx.x;
    for (int k = tid; k < 6 * 3 * kFusedSlab; k += blockDim.x) {
        const int comp = k / (3 * kFusedSlab), ax = (k / kFusedSlab) % 3, sidx = k % kFusedSlab;
        const PmlDev<T>& p = a.pml[comp];
        T b = 0, cd = 0, ki = 1;
        if (p.psi[ax] && sidx < p.S[ax]) {
            const int pos = sidx < p.lo[ax] ? sidx : p.hi0[ax] + (sidx - p.lo[ax]);
            b = p.b[ax][pos];
            cd = p.cd[ax][pos];
            ki = p.kinv[ax][pos];
        }
        P.v[comp][ax][0][sidx] = b;
        P.v[comp][ax][1][sidx] = cd;
        P.v[comp][ax][2][sidx] = ki;
    }
}

// Slab-compact position of pos on axis ax, or -1 outside the psi region.
template <typename T>
__device__ __forceinline__ int psi_pos(const PmlDev<T>& p, int ax, int pos) {
    if (pos < p.lo[ax]) return pos;
    if (pos >= p.hi0[ax] && pos < p.hi1[ax]) return p.lo[ax] + pos - p.hi0[ax];
    return -1;
}

// Element index of the psi of the group at slab position s (s >= 0).
template <typename T>
__device__ __forceinline__ unsigned psi_index(const PmlDev<T>& p, int ax, int s, int x0, int y, int z, int nx, int ny) {
    if (ax == 0) return static_cast<unsigned>(s) + static_cast<unsigned>(p.S[0]) * (static_cast<unsigned>(y) + static_cast<unsigned>(ny) * z);
    if (ax == 1) return static_cast<unsigned>(x0) + static_cast<unsigned>(nx) * (static_cast<unsigned>(s) + static_cast<unsigned>(p.S[1]) * z);
    return static_cast<unsigned>(x0) + static_cast<unsigned>(nx) * (static_cast<unsigned>(y) + static_cast<unsigned>(ny) * s);
}

// CPML term of (comp, ax) for a group at slab position sp (-1: none) whose
// psi ps was loaded ahead, profiles from LDS; ps becomes the new psi (cells
// outside `valid` keep the old one).  pml_group's arithmetic.
template <typename T, int W>
__device__ __forceinline__ void psi_term_l(const ProfLds<T>& P, int comp, int ax, int sp, const T (&dV)[W], T invd, unsigned valid,
                                           Pk<T, W>& ps, T (&term)[W]) {
    if (sp < 0) {
#pragma unroll
        for (int w = 0; w < W; ++w) term[w] = dV[w] * invd;
        return;
    }
#pragma unroll
    for (int w = 0; w < W; ++w) {
        const int q = ax == 0 ? sp + w : sp;
        const T psi = P.v[comp][ax][0][q] * ps.v[w] + P.v[comp][ax][1][q] * dV[w];
        if (valid & (1u << w)) ps.v[w] = psi;
        term[w] = P.v[comp][ax][2][q] * (dV[w] * invd) + psi;
    }
}

// A y or z CPML term (rows / planes of the slabs, wave-uniform): load psi,
// update, store.
template <typename T, int W>
__device__ __forceinline__ void psi_yz_l(const StepArgs<T>& a, const ProfLds<T>& P, int comp, int ax, int pos0, int x0, int y, int z,
                                         const T (&dV)[W], T invd, unsigned valid, bool store, T (&term)[W]) {
    const PmlDev<T>& p = a.pml[comp];
    const int sp = psi_pos(p, ax, pos0);
    Pk<T, W> ps = zpk<T, W>();
    unsigned pi = 0;
    if (sp >= 0) {
        pi = psi_index(p, ax, sp, x0, y, z, a.nx, a.ny);
        ps = ldv_nt<T, W>(p.psi_in[ax] + pi);
    }
    psi_term_l<T, W>(P, comp, ax, sp, dV, invd, valid, ps, term);
    if (store && sp >= 0) stv_nt<T, W>(p.psi[ax] + pi, ps);
}

// The soft sources of one launch, staged in LDS at kernel entry with this
// step's amplitudes: inside the fused kernel's loop, which stores to global
// memory, uniform loads of the source table would become per-lane loads,
// each waited for.
template <typename T>
struct SrcLds {
    int n;
    int comp[CHIML_MAX_SRC];
    int box[CHIML_MAX_SRC][6];
    T amp[CHIML_MAX_SRC];
};

template <typename T>
__device__ __forceinline__ void load_src_lds(const StepArgs<T>& a, SrcLds<T>& S, int step) {
    const int tid = threadIdx.x;
    if (tid == 0) S.n = min(a.nsrc, CHIML_MAX_SRC);
    for (int k = tid; k < min(a.nsrc, CHIML_MAX_SRC); k += blockDim.x) {
        S.comp[k] = a.src_comp[k];
#pragma unroll
        for (int j = 0; j < 6; ++j) S.box[k][j] = a.src_box[6 * k + j];
        S.amp[k] = a.src_amp[static_cast<long long>(step) * a.nsrc + k];
    }
}

// group_has_src / src_value on the staged table
template <typename T, int W>
__device__ __forceinline__ bool group_has_src_l(const SrcLds<T>& S, int x0, int y, int z) {
    for (int s = 0; s < S.n; ++s) {
        const int* b = S.box[s];
        if (x0 < b[1] && b[0] < x0 + W && y >= b[2] && y < b[3] && z >= b[4] && z < b[5]) return true;
    }
    return false;
}
template <typename T>
__device__ __forceinline__ T src_value_l(const SrcLds<T>& S, int comp, int x, int y, int z) {
    T v = 0;
    for (int s = 0; s < S.n; ++s) {
        if (S.comp[s] != comp) continue;
        const int* b = S.box[s];
        if (x >= b[0] && x < b[1] && y >= b[2] && y < b[3] && z >= b[4] && z < b[5]) v += S.amp[s];
    }
    return v;
}

// The group's new E of component c from its curl terms (e_finish_group's
// arithmetic), with its material ids loaded ahead; the stores are the
// caller's.  PRE: the pole-current sum was left in jsum by the pole-update
// launch; otherwise the pole update runs here.  Cells outside `valid` keep
// their old value.
template <typename T, int W, bool PRE>
__device__ __forceinline__ Pk<T, W> e_new_group(const StepArgs<T>& a, const MatLds<T> (*mt)[CHIML_MAX_MAT], const SrcLds<T>& S, int c,
                                                int x0, int y, int z, unsigned valid, const T (&t1)[W], const T (&t2)[W], bool src,
                                                Pk<T, W> e, const Pk<uint8_t, W>& id) {
    T jsum[W];
    bool anyp = false;
#pragma unroll
    for (int w = 0; w < W; ++w) {
        jsum[w] = T(0);
        anyp |= (mt[c][id.v[w]].poleset >= 0) && (valid & (1u << w));
    }
    if (PRE && anyp) {
        const int* bx = a.box[c];
        const long long bi = (x0 - bx[0]) + static_cast<long long>(bx[1] - bx[0]) * ((y - bx[2]) + static_cast<long long>(bx[3] - bx[2]) * (z - bx[4]));
        const Pk<T, W> js = ldv<T, W>(a.jsum[c] + bi);
#pragma unroll
        for (int w = 0; w < W; ++w)
            if (mt[c][id.v[w]].poleset >= 0 && (valid & (1u << w))) jsum[w] = js.v[w];
    } else if (!PRE && anyp) {
        const int* bx = a.box[c];
        const long long bi = (x0 - bx[0]) + static_cast<long long>(bx[1] - bx[0]) * ((y - bx[2]) + static_cast<long long>(bx[3] - bx[2]) * (z - bx[4]));
        int np[W], npmax = 0;
#pragma unroll
        for (int w = 0; w < W; ++w) {
            const int ps = mt[c][id.v[w]].poleset;
            np[w] = (ps >= 0 && (valid & (1u << w))) ? a.pole_count[ps] : 0;
            npmax = max(npmax, np[w]);
        }
        for (int p = 0; p < npmax; ++p) {
            T* Pp = a.P[c] + p * a.boxn[c] + bi;
            T* Jp = a.J[c] + p * a.boxn[c] + bi;
            Pk<T, W> Pv = ldv_nt<T, W>(Pp), J = ldv_nt<T, W>(Jp);
#pragma unroll
            for (int w = 0; w < W; ++w) {
                if (p >= np[w]) continue;
                const int ps = mt[c][id.v[w]].poleset;
                const T* co = a.pole_coef + (static_cast<long long>(ps) * CHIML_MAX_POLES + p) * 3;
                const T sv = src ? src_value_l<T>(S, c, x0 + w, y, z) : T(0);
                const T Jn = co[0] * Pv.v[w] + co[1] * J.v[w] + co[2] * (e.v[w] + sv);
                Pv.v[w] = Pv.v[w] + Jn;
                J.v[w] = Jn;
                jsum[w] += Jn;
            }
            stv_nt<T, W>(Pp, Pv);
            stv_nt<T, W>(Jp, J);
        }
    }
#pragma unroll
    for (int w = 0; w < W; ++w) {
        if (!(valid & (1u << w))) continue;
        const MatLds<T> m = mt[c][id.v[w]];
        const T sv = src ? src_value_l<T>(S, c, x0 + w, y, z) : T(0);
        const T e_base = (m.flags & CHIML_MAT_DCELL) ? e.v[w] : e.v[w] + sv;
        e.v[w] = e_base + m.ce * (t1[w] - t2[w]) - m.inveps * jsum[w];
    }
    return e;
}

// Loads and stores at a byte offset from a base held in scalar registers
// (the 32-bit offset keeps one vector register per address).
template <typename T, int W>
__device__ __forceinline__ Pk<T, W> ldo(const T* base, unsigned off) {
    return *reinterpret_cast<const Pk<T, W>*>(reinterpret_cast<const char*>(base) + off);
}
template <typename T, int W>
__device__ __forceinline__ Pk<T, W> ldo_nt(const T* base, unsigned off) {
    return ldv_nt<T, W>(reinterpret_cast<const T*>(reinterpret_cast<const char*>(base) + off));
}
template <typename T, int W>
__device__ __forceinline__ void sto_nt(T* base, unsigned off, const Pk<T, W>& v) {
    stv_nt<T, W>(reinterpret_cast<T*>(reinterpret_cast<char*>(base) + off), v);
}
template <typename T>
__device__ __forceinline__ T ld1(const T* base, unsigned off) {
    return *reinterpret_cast<const T*>(reinterpret_cast<const char*>(base) + off);
}

template <typename T, int W>
struct FuseCarry {
    Pk<T, W> ex, ey, ez;  // E at the plane being updated
    Pk<T, W> hxp, hyp;    // new Hx, Hy one plane down
};

// New Hx and Hy of the group at a plane, not stored: the plane below a
// segment (one value per own row).  h_group's arithmetic.
template <typename T, int W, bool SRC>
__device__ __forceinline__ void fused_h_below(const StepArgs<T>& a, const SrcLds<T>& S, const ProfLds<T>& P, const T (&chv)[3], unsigned cs,
                                              int x0, int y, int z, Pk<T, W>& hx, Pk<T, W>& hy) {
    const int nx = a.nx, ny = a.ny, nz = a.nz;
    const unsigned ob = static_cast<unsigned>(lidx(x0, y, z, nx, ny)) * sizeof(T);
    const unsigned sy = nx * sizeof(T), sz = static_cast<unsigned>(nx) * ny * sizeof(T);
    const T* G = a.G[0];
    const bool last = x0 + W >= nx;
    const unsigned all = (1u << W) - 1, vx = last ? (all >> 1) : all;
    const Pk<T, W> ex = ldo<T, W>(G, ob), ey = ldo<T, W>(G, ob + cs), ez = ldo<T, W>(G, ob + 2 * cs);
    const Pk<T, W> exz = ldo<T, W>(G, ob + sz), eyz = ldo<T, W>(G, ob + cs + sz);
    const Pk<T, W> ezy = y < ny - 1 ? ldo<T, W>(G, ob + 2 * cs + sy) : zpk<T, W>();
    const T ezn = last ? T(0) : ld1<T>(G, ob + 2 * cs + W * sizeof(T));
    hx = ldo_nt<T, W>(G, ob + 3 * cs);
    hy = ldo_nt<T, W>(G, ob + 4 * cs);
    const bool src = SRC && group_has_src_l<T, W>(S, x0, y, z);
    T d1[W], d2[W], t1[W], t2[W];
    if (y < ny - 1 && z < nz - 1) {
#pragma unroll
        for (int w = 0; w < W; ++w) {
            d1[w] = eyz.v[w] - ey.v[w];
            d2[w] = ezy.v[w] - ez.v[w];
        }
        psi_yz_l<T, W>(a, P, 3, 2, z, x0, y, z, d1, a.inv_d[2], all, false, t1);
        psi_yz_l<T, W>(a, P, 3, 1, y, x0, y, z, d2, a.inv_d[1], all, false, t2);
#pragma unroll
        for (int w = 0; w < W; ++w) {
            T hv = hx.v[w] + chv[0] * (t1[w] - t2[w]);
            if (SRC && src) hv += src_value_l<T>(S, 3, x0 + w, y, z);
            hx.v[w] = hv;
        }
    }
    if (z < nz - 1) {
#pragma unroll
        for (int w = 0; w < W; ++w) {
            d1[w] = (w + 1 < W ? ez.v[w + 1] : ezn) - ez.v[w];
            d2[w] = exz.v[w] - ex.v[w];
        }
        psi_yz_l<T, W>(a, P, 4, 0, x0, x0, y, z, d1, a.inv_d[0], vx, false, t1);
        psi_yz_l<T, W>(a, P, 4, 2, z, x0, y, z, d2, a.inv_d[2], vx, false, t2);
#pragma unroll
        for (int w = 0; w < W; ++w) {
            if (!(vx & (1u << w))) continue;
            T hv = hy.v[w] + chv[1] * (t1[w] - t2[w]);
            if (SRC && src) hv += src_value_l<T>(S, 4, x0 + w, y, z);
            hy.v[w] = hv;
        }
    }
}

// One plane of the fused step for one thread's group (row y, cells x0..).
// Its memory traffic is in three phases, so that it waits for memory once:
// every load it needs (E one plane up, E of the row above and of the next
// group, old H, material ids, x-CPML psi) is issued first, from clamped
// addresses and without branches; then H is formed and shared through LDS,
// and after the block barrier E; every store comes last.  (One in-order
// counter tracks loads and stores alike, so a load issued after a store
// could not be waited for without waiting for the store.)  slab: the row
// or plane lies in a y or z CPML slab (wave-uniform), whose psi terms load
// and store in place; elsewhere those terms are plain differences.  The
// field buffers hold the six components cstride bytes apart (a.G[0], a.F[0]).
template <typename T, int W, bool SRC, bool PRE>
__device__ __forceinline__ void fused_plane(const StepArgs<T>& a, const MatLds<T> (*mt)[CHIML_MAX_MAT], const SrcLds<T>& S,
                                            const ProfLds<T>& P, const T (&chv)[3], T* L, int plane, unsigned cs, int r, int x0,
                                            int y, int z, bool row, bool own, bool work, bool slab, bool m_xpsi, FuseCarry<T, W>& st) {
    const int nx = a.nx, ny = a.ny, nz = a.nz;
    const unsigned sy = nx * sizeof(T), sz = static_cast<unsigned>(nx) * ny * sizeof(T);
    const int yc = min(max(y, 0), ny - 1);  // a row of the domain for the (unused) loads of rows outside it
    const long long i = lidx(x0, yc, z, nx, ny);
    const unsigned ob = static_cast<unsigned>(i) * sizeof(T);
    const T* G = a.G[0];
    T* F = a.F[0];
    const T idx = a.inv_d[0], idy = a.inv_d[1], idz = a.inv_d[2];
    const bool last = x0 + W >= nx;
    const unsigned all = (1u << W) - 1, vx = last ? (all >> 1) : all;  // cells with x < nx - 1
    const bool yin = y < ny - 1, zin = z < nz - 1;
    // ---- every load of the plane ----
    const unsigned oz = zin ? sz : 0u, oy = yin ? sy : 0u, ox = last ? 0u : W * sizeof(T);
    Pk<T, W> exz = ldo<T, W>(G, ob + oz), eyz = ldo<T, W>(G, ob + cs + oz), ezz = ldo<T, W>(G, ob + 2 * cs + oz);
    const Pk<T, W> exy = ldo<T, W>(G, ob + oy), ezy = ldo<T, W>(G, ob + 2 * cs + oy);
    T ezn = ld1<T>(G, ob + 2 * cs + ox), eyn = ld1<T>(G, ob + cs + ox);
    Pk<T, W> hx = ldo_nt<T, W>(G, ob + 3 * cs), hy = ldo_nt<T, W>(G, ob + 4 * cs), hz = ldo_nt<T, W>(G, ob + 5 * cs);
    const Pk<uint8_t, W> id0 = load_ids<W>(a.mat_e[0], i), id1 = load_ids<W>(a.mat_e[1], i), id2 = load_ids<W>(a.mat_e[2], i);
    // x psi of Hy, Hz, Ey, Ez (slab-compact positions, -1 outside the x slabs)
    const int sHy = zin ? psi_pos(a.pml[4], 0, x0) : -1, sHz = yin ? psi_pos(a.pml[5], 0, x0) : -1;
    const int sEy = yin ? psi_pos(a.pml[1], 0, x0) : -1, sEz = zin ? psi_pos(a.pml[2], 0, x0) : -1;
    const unsigned iHy = psi_index(a.pml[4], 0, max(sHy, 0), x0, yc, z, nx, ny), iHz = psi_index(a.pml[5], 0, max(sHz, 0), x0, yc, z, nx, ny);
    const unsigned iEy = psi_index(a.pml[1], 0, max(sEy, 0), x0, yc, z, nx, ny), iEz = psi_index(a.pml[2], 0, max(sEz, 0), x0, yc, z, nx, ny);
    const bool xpsi = m_xpsi;
    Pk<T, W> psHy = zpk<T, W>(), psHz = zpk<T, W>(), psEy = zpk<T, W>(), psEz = zpk<T, W>();
    if (xpsi) {
        psHy = ldv_nt<T, W>(a.pml[4].psi_in[0] + iHy);
        psHz = ldv_nt<T, W>(a.pml[5].psi_in[0] + iHz);
        psEy = ldv_nt<T, W>(a.pml[1].psi[0] + iEy);
        psEz = ldv_nt<T, W>(a.pml[2].psi[0] + iEz);
    }
    if (!zin) exz = eyz = ezz = zpk<T, W>();
    if (last) ezn = eyn = T(0);
    const bool src = SRC && row && group_has_src_l<T, W>(S, x0, y, z);
    // ---- H ----
    T d1[W], d2[W], t1[W], t2[W];
    const Pk<T, W>&ex = st.ex, &ey = st.ey, &ez = st.ez;
    if (yin && zin) {  // Hx += ch [dEy/dz - dEz/dy]
#pragma unroll
        for (int w = 0; w < W; ++w) {
            d1[w] = eyz.v[w] - ey.v[w];
            d2[w] = ezy.v[w] - ez.v[w];
        }
        if (slab) {
            psi_yz_l<T, W>(a, P, 3, 2, z, x0, yc, z, d1, idz, all, own, t1);
            psi_yz_l<T, W>(a, P, 3, 1, y, x0, yc, z, d2, idy, all, own, t2);
        } else {
#pragma unroll
            for (int w = 0; w < W; ++w) {
                t1[w] = d1[w] * idz;
                t2[w] = d2[w] * idy;
            }
        }
#pragma unroll
        for (int w = 0; w < W; ++w) {
            T hv = hx.v[w] + chv[0] * (t1[w] - t2[w]);
            if (SRC && src) hv += src_value_l<T>(S, 3, x0 + w, y, z);
            hx.v[w] = hv;
        }
    }
    if (own && zin) {  // Hy += ch [dEz/dx - dEx/dz], x < nx - 1
#pragma unroll
        for (int w = 0; w < W; ++w) {
            d1[w] = (w + 1 < W ? ez.v[w + 1] : ezn) - ez.v[w];
            d2[w] = exz.v[w] - ex.v[w];
        }
        psi_term_l<T, W>(P, 4, 0, sHy, d1, idx, vx, psHy, t1);
        if (slab) {
            psi_yz_l<T, W>(a, P, 4, 2, z, x0, yc, z, d2, idz, vx, true, t2);
        } else {
#pragma unroll
            for (int w = 0; w < W; ++w) t2[w] = d2[w] * idz;
        }
#pragma unroll
        for (int w = 0; w < W; ++w) {
            if (!(vx & (1u << w))) continue;
            T hv = hy.v[w] + chv[1] * (t1[w] - t2[w]);
            if (SRC && src) hv += src_value_l<T>(S, 4, x0 + w, y, z);
            hy.v[w] = hv;
        }
    }
    if (yin) {  // Hz += ch [dEx/dy - dEy/dx], x < nx - 1
#pragma unroll
        for (int w = 0; w < W; ++w) {
            d1[w] = exy.v[w] - ex.v[w];
            d2[w] = (w + 1 < W ? ey.v[w + 1] : eyn) - ey.v[w];
        }
        if (slab) {
            psi_yz_l<T, W>(a, P, 5, 1, y, x0, yc, z, d1, idy, vx, own, t1);
        } else {
#pragma unroll
            for (int w = 0; w < W; ++w) t1[w] = d1[w] * idy;
        }
        psi_term_l<T, W>(P, 5, 0, sHz, d2, idx, vx, psHz, t2);
#pragma unroll
        for (int w = 0; w < W; ++w) {
            if (!(vx & (1u << w))) continue;
            T hv = hz.v[w] + chv[2] * (t1[w] - t2[w]);
            if (SRC && src) hv += src_value_l<T>(S, 5, x0 + w, y, z);
            hz.v[w] = hv;
        }
    }
    if (!row) hx = hy = hz = zpk<T, W>();  // the zero ghost below the domain / past its last row
    if (work) {
        const int o = r * nx + x0;
        stv<T, W>(L + o, hx);
        stv<T, W>(L + plane + o, hy);
        stv<T, W>(L + 2 * plane + o, hz);
    }
    __syncthreads();
    // ---- E ----
    Pk<T, W> en0 = st.ex, en1 = st.ey, en2 = st.ez;
    if (own) {
        const int o = r * nx + x0;
        const Pk<T, W> hxy = ldv<T, W>(L + o - nx), hzy = ldv<T, W>(L + 2 * plane + o - nx);
        const T hym = x0 > 0 ? L[plane + o - 1] : T(0), hzm = x0 > 0 ? L[2 * plane + o - 1] : T(0);
        {  // Ex += ce [dHz/dy - dHy/dz], x < nx - 1
#pragma unroll
            for (int w = 0; w < W; ++w) {
                d1[w] = hz.v[w] - hzy.v[w];
                d2[w] = hy.v[w] - st.hyp.v[w];
            }
            if (slab) {
                psi_yz_l<T, W>(a, P, 0, 1, y, x0, y, z, d1, idy, vx, true, t1);
                psi_yz_l<T, W>(a, P, 0, 2, z, x0, y, z, d2, idz, vx, true, t2);
            } else {
#pragma unroll
                for (int w = 0; w < W; ++w) {
                    t1[w] = d1[w] * idy;
                    t2[w] = d2[w] * idz;
                }
            }
            en0 = e_new_group<T, W, PRE>(a, mt, S, 0, x0, y, z, vx, t1, t2, src, st.ex, id0);
        }
        if (yin) {  // Ey += ce [dHx/dz - dHz/dx]
#pragma unroll
            for (int w = 0; w < W; ++w) {
                d1[w] = hx.v[w] - st.hxp.v[w];
                d2[w] = hz.v[w] - (w > 0 ? hz.v[w - 1] : hzm);
            }
            if (slab) {
                psi_yz_l<T, W>(a, P, 1, 2, z, x0, y, z, d1, idz, all, true, t1);
            } else {
#pragma unroll
                for (int w = 0; w < W; ++w) t1[w] = d1[w] * idz;
            }
            psi_term_l<T, W>(P, 1, 0, sEy, d2, idx, all, psEy, t2);
            en1 = e_new_group<T, W, PRE>(a, mt, S, 1, x0, y, z, all, t1, t2, src, st.ey, id1);
        }
        if (zin) {  // Ez += ce [dHy/dx - dHx/dy]
#pragma unroll
            for (int w = 0; w < W; ++w) {
                d1[w] = hy.v[w] - (w > 0 ? hy.v[w - 1] : hym);
                d2[w] = hx.v[w] - hxy.v[w];
            }
            psi_term_l<T, W>(P, 2, 0, sEz, d1, idx, all, psEz, t1);
            if (slab) {
                psi_yz_l<T, W>(a, P, 2, 1, y, x0, y, z, d2, idy, all, true, t2);
            } else {
#pragma unroll
                for (int w = 0; w < W; ++w) t2[w] = d2[w] * idy;
            }
            en2 = e_new_group<T, W, PRE>(a, mt, S, 2, x0, y, z, all, t1, t2, src, st.ez, id2);
        }
    }
    // ---- every store of the plane ----
    if (own) {
        if (yin && zin) sto_nt<T, W>(F, ob + 3 * cs, hx);
        if (zin) {
            sto_nt<T, W>(F, ob + 4 * cs, hy);
            if (sHy >= 0) stv_nt<T, W>(a.pml[4].psi[0] + iHy, psHy);
        }
        if (yin) {
            sto_nt<T, W>(F, ob + 5 * cs, hz);
            if (sHz >= 0) stv_nt<T, W>(a.pml[5].psi[0] + iHz, psHz);
        }
        sto_nt<T, W>(F, ob, en0);
        if (yin) {
            sto_nt<T, W>(F, ob + cs, en1);
            if (sEy >= 0) stv_nt<T, W>(a.pml[1].psi[0] + iEy, psEy);
        }
        if (zin) {
            sto_nt<T, W>(F, ob + 2 * cs, en2);
            if (sEz >= 0) stv_nt<T, W>(a.pml[2].psi[0] + iEz, psEz);
        }
    }
    st.hxp = hx;
    st.hyp = hy;
    st.ex = exz;
    st.ey = eyz;
    st.ez = ezz;
}

template <typename T, int W, bool SRC, bool PRE, bool ADV>
__global__ void __launch_bounds__(kFusedMaxThreads) k_fused3(StepArgs<T> a, FuseMap m, int nm0, int nm1, int nm2) {
    __shared__ MatLds<T> mt[3][CHIML_MAX_MAT];
    __shared__ SrcLds<T> S;
    __shared__ ProfLds<T> P;
    extern __shared__ __align__(16) unsigned char fused_lds[];
    T* lds = reinterpret_cast<T*>(fused_lds);  // [2][3][(ty + 1) * nx]
    const int nm[3] = {nm0, nm1, nm2};
    const int step = SRC ? step_now(a.step, a.stepv) : 0;
    if (SRC) load_src_lds<T>(a, S, step);
    else if (threadIdx.x == 0) S.n = 0;
    load_prof_lds<T>(a, P);
    load_mat(a, mt, nm);  // (its barrier also publishes the source and profile tables)
    const T chv[3] = {a.ch[0][0], a.ch[1][0], a.ch[2][0]};
    const int nx = a.nx, ny = a.ny, nz = a.nz;
    const int item = xcd_block(blockIdx.x, gridDim.x);
    const int tile = item / m.nseg, seg = item - tile * m.nseg;
    const int z0 = seg * m.lz, z1 = min(z0 + m.lz, nz);
    const int tid = threadIdx.x;
    const bool work = tid < m.nthr;
    const int r = work ? tid / m.gx : 0, g = work ? tid - r * m.gx : 0;
    const int x0 = g * W, y = tile * m.ty - 1 + r;
    const bool row = work && y >= 0 && y < ny;  // a row of the domain
    const bool own = row && r > 0;              // a row this block updates (r = 0: the row below the tile)
    const bool yslab = y < m.ys0 || y >= m.ys1;
    const int plane = (m.ty + 1) * nx;
    const unsigned cs = m.cstride;
    FuseCarry<T, W> st;
    st.ex = st.ey = st.ez = st.hxp = st.hyp = zpk<T, W>();
    if (row) {
        const unsigned ob = static_cast<unsigned>(lidx(x0, y, z0, nx, ny)) * sizeof(T);
        st.ex = ldo<T, W>(a.G[0], ob);
        st.ey = ldo<T, W>(a.G[0], ob + cs);
        st.ez = ldo<T, W>(a.G[0], ob + 2 * cs);
        if (own && z0 > 0) fused_h_below<T, W, SRC>(a, S, P, chv, cs, x0, y, z0 - 1, st.hxp, st.hyp);
    }
    for (int z = z0; z < z1; ++z) {
        T* L = lds + (z & 1) * 3 * plane;
        fused_plane<T, W, SRC, PRE>(a, mt, S, P, chv, L, plane, cs, r, x0, y, z, row, own, work, yslab || z < m.zs0 || z >= m.zs1,
                                    m.xpsi != 0, st);
    }
    if (ADV) advance_counter(a);
}

// The pole update of the fused step, as a launch of its own before it
// (ade_block over the pole boxes; it reads E before the step, a.F = a.G).
template <typename T, int W, bool SRC>
__global__ void __launch_bounds__(256) k_ade3(StepArgs<T> a, int ade_bpc) {
    const int c = blockIdx.x / max(ade_bpc, 1);
    if (c < 3) ade_block<T, W, SRC>(a, c, blockIdx.x - c * ade_bpc);
}

// One set of DFT accumulators: its sampled cells, sampling interval and
// staging buffer [kDftBlock][n].
constexpr int kMaxDftGroups = 16;  // flux boxes + up to 15 frequency detectors; the table rides in the kernel arguments
template <typename T>
struct DftSample {
    int n, interval;
    const int* comp;
    const long long* cell;
    T* stage;
};

template <typename T>
struct SampleArgs {
    const T* F[6];
    const int* step;
    int stepv;  // as in StepArgs
    int ndet;
    const int* det_interval;
    const int* det_npts;
    const int* det_off;  // prefix sums of npts
    const int* det_comp;
    const long long* det_cell;
    const double* det_conv;
    const int* det_pow;
    const int* det_nf;             // fields per point
    const long long* det_eoff;     // per detector offset into det_comp / det_cell (pairs)
    int det_all1;                  // every detector reads one field: point t's cells are entries 2t, 2t + 1
    double* det_out;
    const long long* det_out_off;  // per detector offset into det_out
    const int* det_cap;            // per detector max samples
    int totpts;
    int ndft;  // sampled DFT cells over all groups
    int ndg;   // DFT groups (0: the flux boxes; then the frequency detectors)
    int gofs[kMaxDftGroups + 1];  // first sample thread of each group
    DftSample<T> dg[kMaxDftGroups];
};

// Stores detector point t's sample at `step` from its two field values u, v
// (fieldOutputFunction: conv/2 (u + v), or conv/2 (u^2 + v^2) for power).
template <typename T>
__device__ __forceinline__ void store_point(const SampleArgs<T>& a, int t, double u, double v, int step) {
    int d = 0;  // the detector of point t
    while (d + 1 < a.ndet && a.det_off[d + 1] <= t) ++d;
    if (step % a.det_interval[d] != 0) return;
    const int slot = step / a.det_interval[d];
    if (slot >= a.det_cap[d]) return;
    const double c = a.det_conv[d];
    double point = 0.0;
    if (a.det_pow[d]) {
        point = point + c / 2.0 * (u * u);
        point = point + c / 2.0 * (v * v);
    } else {
        point = point + c / 2.0 * u;
        point = point + c / 2.0 * v;
    }
    a.det_out[a.det_out_off[d] + static_cast<long long>(slot) * a.det_npts[d] + (t - a.det_off[d])] = point;
}

// 2D TMz on W-cell groups over the whole domain (CPML handled per group; the
// x-slab membership is uniform within a group as in 3D).
template <typename T, int W, bool SRC>
__device__ __forceinline__ void h2v_sweep(const StepArgs<T>& a, int bx, int nb) {
    const int nx = a.nx, ny = a.ny, px = a.px, gx = px / W;
    const unsigned t = static_cast<unsigned>(xcd_block(bx, nb)) * blockDim.x + threadIdx.x;
    const int y = static_cast<int>(t / static_cast<unsigned>(gx)), x0 = static_cast<int>(t - static_cast<unsigned>(y) * gx) * W;
    if (y >= ny) return;
    const long long i = x0 + static_cast<long long>(px) * y;
    const T* Ez = a.F[2];
    const Pk<T, W> ez = ldv<T, W>(Ez + i);
    const bool last = x0 + W >= nx;
    const unsigned all = (1u << W) - 1, vx = cells_below_last<W>(x0, nx);
    const bool src = SRC && group_has_src<T, W>(a, x0, y, 0);
    const int step = src ? step_now(a.step, a.stepv) : 0;
    T d[W], term[W];
    if (y < ny - 1) {  // Hx += ch [-dEz/dy]
        const Pk<T, W> ezy = ldv<T, W>(Ez + i + px);
        Pk<T, W> h = ldv<T, W>(a.F[3] + i);
#pragma unroll
        for (int w = 0; w < W; ++w) d[w] = ezy.v[w] - ez.v[w];
        pml_group<T, W>(a.pml[3], 1, y, x0, y, 0, px, ny, d, a.inv_d[1], all, term);
        const T ch = a.ch[0][0];
#pragma unroll
        for (int w = 0; w < W; ++w) {
            T hv = h.v[w] + ch * (-term[w]);
            if (src) hv += src_value(a, 3, x0 + w, y, 0, step);
            h.v[w] = hv;
        }
        stv<T, W>(a.F[3] + i, h);
    }
    {  // Hy += ch [dEz/dx], x < nx - 1
        const T ezn = last ? T(0) : Ez[i + W];
        Pk<T, W> h = ldv<T, W>(a.F[4] + i);
#pragma unroll
        for (int w = 0; w < W; ++w) d[w] = (w + 1 < W ? ez.v[w + 1] : ezn) - ez.v[w];
        pml_group<T, W>(a.pml[4], 0, x0, x0, y, 0, px, ny, d, a.inv_d[0], vx, term);
        const T ch = a.ch[1][0];
#pragma unroll
        for (int w = 0; w < W; ++w) {
            if (!(vx & (1u << w))) continue;
            T hv = h.v[w] + ch * term[w];
            if (src) hv += src_value(a, 4, x0 + w, y, 0, step);
            h.v[w] = hv;
        }
        stv<T, W>(a.F[4] + i, h);
    }
}

template <typename T, int W, bool SRC, bool ADV>
__global__ void __launch_bounds__(256) k_h2v(StepArgs<T> a) {
    h2v_sweep<T, W, SRC>(a, blockIdx.x, gridDim.x);
    if (ADV) advance_counter(a);
}

// DET: the deck's point detectors (single-cell, Ez / Hx / Hy) are sampled
// here, by the thread that owns each detector cell, at the advanced step:
// no separate sample launch (2D decks without flux boxes and with few points).
template <typename T, int W, bool SRC, bool DET, bool FMA>
__device__ __forceinline__ void e2v_sweep(const StepArgs<T>& a, const SampleArgs<T>& sa, const MatLds<T> (*mt)[CHIML_MAX_MAT], int bx, int nb) {
    const int ny = a.ny, px = a.px, gx = px / W;
    const unsigned t = static_cast<unsigned>(xcd_block(bx, nb)) * blockDim.x + threadIdx.x;
    const int y = static_cast<int>(t / static_cast<unsigned>(gx)), x0 = static_cast<int>(t - static_cast<unsigned>(y) * gx) * W;
    if (y >= ny) return;
    const long long i = x0 + static_cast<long long>(px) * y;
    const T *Hx = a.F[3], *Hy = a.F[4];
    const Pk<T, W> hx = ldv<T, W>(Hx + i), hy = ldv<T, W>(Hy + i);
    const Pk<T, W> hxy = y > 0 ? ldv<T, W>(Hx + i - px) : zpk<T, W>();
    const T hym = x0 > 0 ? Hy[i - 1] : T(0);
    const unsigned all = (1u << W) - 1;
    const bool src = SRC && group_has_src<T, W>(a, x0, y, 0);
    const int step = src ? step_now(a.step, a.stepv) : 0;
    T d1[W], d2[W], t1[W], t2[W];
#pragma unroll
    for (int w = 0; w < W; ++w) {
        d1[w] = hy.v[w] - (w > 0 ? hy.v[w - 1] : hym);
        d2[w] = hx.v[w] - hxy.v[w];
    }
    pml_group<T, W>(a.pml[2], 0, x0, x0, y, 0, px, ny, d1, a.inv_d[0], all, t1);
    pml_group<T, W>(a.pml[2], 1, y, x0, y, 0, px, ny, d2, a.inv_d[1], all, t2);
    T acc[W];
    const unsigned plain = FMA && y >= a.Tp[1] && y < ny - a.Tp[1] ? cells_inside<W>(x0, a.nx, a.Tp[0]) : 0u;
    curl_of<T, W, FMA>(t1, t2, d2, a.inv_d[1], plain, acc);
    const Pk<T, W> ez = e_finish_group<T, W>(a, mt, 2, i, x0, y, 0, all, acc, src, step);
    if (DET) {
        const int st = step_now(a.step, a.stepv) + 1;
        for (int p = 0; p < sa.totpts; ++p) {
            const long long cell = sa.det_cell[2 * p];
            if (cell < i || cell >= i + W) continue;
            const int w = static_cast<int>(cell - i), comp = sa.det_comp[2 * p];
            const double v = static_cast<double>(comp == 2 ? ez.v[w] : (comp == 3 ? hx.v[w] : hy.v[w]));
            store_point(sa, p, v, v, st);
        }
    }
}

template <typename T, int W, bool SRC, bool DET, bool FMA>
__global__ void __launch_bounds__(256) k_e2v(StepArgs<T> a, SampleArgs<T> sa, int nm2) {
    __shared__ MatLds<T> mt[3][CHIML_MAX_MAT];
    const int nm[3] = {0, 0, nm2};
    load_mat(a, mt, nm);
    e2v_sweep<T, W, SRC, DET, FMA>(a, sa, mt, blockIdx.x, gridDim.x);
}

// --------------------------------------------- 2D: several steps a launch ----
// A 2D TMz grid is small: a step of 256^2 cells moves 4 MB, and launches, not
// memory, set its time (two launches, 8.1 us a step).  k_tile2 advances up to
// kTileSteps steps in one launch.  A block loads a tile of the grid with a
// halo of kTileSteps cells on every side, keeps it in registers for all its
// steps and writes the tile's own cells to the other field buffer (the
// neighbours still read the old one); the halo cells are recomputed by every
// block that holds them, and their outermost ring goes stale by one cell per
// step.  A thread owns R consecutive rows of one column: the y neighbour is
// its own register except at the ends of its strip (one row through LDS per
// half step, one barrier each), the x neighbour is the next lane's register.
// The CPML psi of the tile's cells are registers too, pole states are in LDS.
// The arithmetic of a cell is that of h2v_sweep / e2v_sweep.
//
// A launch costs about 8 us of latency to get its tiles in and out and about
// 0.8 us a step.  Small grids take small tiles, one or two a CU (4x the cells
// in halos), large ones large tiles (1.8x).  A block has 8-16 waves of few
// rows: the same 32 x 32 tile with 4 rows a thread (1 wave per SIMD) measured
// 2.6 us a step, with 2 rows 1.85, with 1 row 1.7 but slower with poles;
// 16-step launches (64 x 48 tiles) 2.9.  us a step in long runs, two sweeps /
// tiles: 256^2 FP64 8.1/1.75, 301x243 FP32 with a metal cylinder 12.9/1.9, FP32
// 512^2 9.8/2.5, 1024^2 16.6/4.9, 2048^2 33.5/15.8, 6144^2 253/120; FP64 2048^2
// 58.7/32.4, 6144^2 485/279: no size was found from which the sweeps are faster
// (one or two steps at a time they are: tile_pays).
constexpr int kTileSteps = 8;
constexpr int kTileDet = 64;  // detector points of one tile at most
constexpr int kTileSets = 8;  // pole sets at most

// A detector point of a tile: its thread and row, and where its samples go.
struct TileDet {
    double conv;
    long long out;
    int thr, row, comp, interval, cap, npts, pow;
};

template <typename T>
struct TileArgs {
    const T *ez, *hx, *hy;  // current buffers
    T *ez_o, *hx_o, *hy_o;
    int nx, ny, px, ntx, Tx, Ty;
    T inv_dx, inv_dy;
    const T *ch0, *ch1;
    const uint8_t* mat;
    const T *ce, *inveps;
    const int *flags, *poleset;
    int nmat;
    // psi of Hx (y), Hy (x), Ez (x), Ez (y): region, profiles, current and next
    int lo[4], hi0[4], hi1[4], S[4];
    const T *b[4], *cd[4], *kinv[4], *psi[4];
    T* psi_o[4];
    int npole;  // poles of the largest set (0: no dispersive cell)
    int nset;   // pole sets
    const int* pole_count;
    const T* pole_coef;
    const T *P, *J;
    T *P_o, *J_o;
    int box[4];  // x0, x1, y0, y1 of the pole-state box
    long long boxn;
    int nsrc;
    const int *src_comp, *src_box;
    const T* src_amp;
    const int* step;
    int stepv;
    int* step_next;
    int nstep;  // steps of this launch, 1 .. kTileSteps
    const int* det_ofs;  // [ntx nty + 1]: each tile's range in det
    const TileDet* det;
    double* det_out;
    bool fma_curl;  // outside the CPML the curl's second product is fused (see enable_tiles)
};

// The next (up = true) or previous lane's value over the whole wave.  At the
// wave's ends, and between the two rows of a wave that holds two, the value
// is another cell's; those lanes hold the halo's outermost columns.
template <bool UP>
__device__ __forceinline__ float lane_nb(float v) {
    return __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(v), UP ? 0x130 : 0x138, 0xf, 0xf, false));
}
template <bool UP>
__device__ __forceinline__ double lane_nb(double v) {
    const long long l = __double_as_longlong(v);
    const int a = __builtin_amdgcn_update_dpp(0, static_cast<int>(l), UP ? 0x130 : 0x138, 0xf, 0xf, false);
    const int b = __builtin_amdgcn_update_dpp(0, static_cast<int>(l >> 32), UP ? 0x130 : 0x138, 0xf, 0xf, false);
    return __longlong_as_double((static_cast<long long>(b) << 32) | static_cast<unsigned>(a));
}

// Tile shape: RX columns, NS strips of R rows.
template <int RX, int R, int NS>
struct TileShape {
    static constexpr int rx = RX, r = R, ns = NS, ry = R * NS, threads = RX * NS;
    static constexpr int ux = RX - 2 * kTileSteps, uy = R * NS - 2 * kTileSteps;  // the tile's own cells
};

template <typename T, typename SH>
__device__ __forceinline__ void tile2_body(const TileArgs<T>& a, int bx, int nb) {
    constexpr int RX = SH::rx, R = SH::r, NS = SH::ns, K = kTileSteps, NT = SH::threads;
    static_assert(NT >= CHIML_MAX_MAT && NT >= 2 * SH::ry && NT >= kTileSets * CHIML_MAX_POLES * 3 && CHIML_MAX_SRC <= 64, "one thread per table entry");
    __shared__ T s_ez[NS][RX], s_hx[NS][RX];
    __shared__ MatLds<T> s_mt[CHIML_MAX_MAT];
    __shared__ T s_y[2][3][SH::ry];  // y CPML b, c/d, 1/kappa of Hx and Ez by row
    __shared__ T s_amp[K][CHIML_MAX_SRC];
    __shared__ int4 s_box[CHIML_MAX_SRC];  // x0, x1, y0, y1 of the sources that touch the tile
    __shared__ int s_comp[CHIML_MAX_SRC];
    __shared__ TileDet s_det[kTileDet];
    __shared__ T s_co[kTileSets * CHIML_MAX_POLES * 3];
    __shared__ int s_np[kTileSets];
    __shared__ int s_nsrc;
    extern __shared__ __align__(16) unsigned char tile_lds[];
    T* const s_P = reinterpret_cast<T*>(tile_lds);  // [npole][P, J][R][NT]
    const int tid = threadIdx.x, col = tid % RX, strip = tid / RX;
    const int tile = xcd_block(bx, nb);
    const int ty = tile / a.ntx, tx = tile - ty * a.ntx;
    const int x0 = tx * SH::ux - K, y0 = ty * SH::uy - K;
    const int x = x0 + col, yb = y0 + strip * R;
    const int nx = a.nx, ny = a.ny, px = a.px;
    const int step = step_now(a.step, a.stepv);
    const bool xin = x >= 0 && x < nx;
    // slab position of pos: psi 0 Hx along y, 1 Hy along x, 2 Ez along x, 3 Ez along y
    auto at = [&](int q, int pos) {
        if (pos < 0) return -1;
        if (pos < a.lo[q]) return pos;
        if (pos >= a.hi0[q] && pos < a.hi1[q]) return a.lo[q] + pos - a.hi0[q];
        return -1;
    };
    auto meets = [&](int q, int p0, int p1) { return a.S[q] > 0 && ((p0 < a.lo[q] && p1 > 0) || (p1 > a.hi0[q] && p0 < a.hi1[q])); };
    const bool xp = meets(1, x0, x0 + RX) || meets(2, x0, x0 + RX), yp = meets(0, y0, y0 + SH::ry) || meets(3, y0, y0 + SH::ry);
    // ---- every load of the tile, before the first wait ----
    T ez[R], hx[R], hy[R];
    unsigned id[R], in = 0;  // in: rows inside the grid
    const int xc = min(max(x, 0), nx - 1);
#pragma unroll
    for (int r = 0; r < R; ++r) {
        const int y = yb + r;
        const long long i = xc + static_cast<long long>(px) * min(max(y, 0), ny - 1);
        if (xin && y >= 0 && y < ny) in |= 1u << r;
        ez[r] = a.ez[i];
        hx[r] = a.hx[i];
        hy[r] = a.hy[i];
        id[r] = a.mat ? a.mat[i] : 0u;
    }
    T pxh[R], pxe[R], pyh[R], pye[R], xh[3] = {T(0), T(0), T(1)}, xe[3] = {T(0), T(0), T(1)}, yc[3] = {T(0), T(0), T(1)};
#pragma unroll
    for (int r = 0; r < R; ++r) pxh[r] = pxe[r] = pyh[r] = pye[r] = T(0);
    const int sxh = xin ? at(1, x) : -1, sxe = xin ? at(2, x) : -1;
    if (xp) {
        if (sxh >= 0) {
            xh[0] = a.b[1][x];
            xh[1] = a.cd[1][x];
            xh[2] = a.kinv[1][x];
        }
        if (sxe >= 0) {
            xe[0] = a.b[2][x];
            xe[1] = a.cd[2][x];
            xe[2] = a.kinv[2][x];
        }
#pragma unroll
        for (int r = 0; r < R; ++r) {
            const int y = min(max(yb + r, 0), ny - 1);
            if (sxh >= 0) pxh[r] = a.psi[1][sxh + static_cast<long long>(a.S[1]) * y];
            if (sxe >= 0) pxe[r] = a.psi[2][sxe + static_cast<long long>(a.S[2]) * y];
        }
    }
    if (yp) {
        if (tid < 2 * SH::ry) {
            const int q = tid < SH::ry ? 0 : 3, y = y0 + tid % SH::ry;
            if (y < ny && at(q, y) >= 0) {
                yc[0] = a.b[q][y];
                yc[1] = a.cd[q][y];
                yc[2] = a.kinv[q][y];
            }
        }
#pragma unroll
        for (int r = 0; r < R; ++r) {
            const int s0 = yb + r < ny ? at(0, yb + r) : -1, s3 = yb + r < ny ? at(3, yb + r) : -1;
            if (s0 >= 0) pyh[r] = a.psi[0][xc + static_cast<long long>(px) * s0];
            if (s3 >= 0) pye[r] = a.psi[3][xc + static_cast<long long>(px) * s3];
        }
    }
    MatLds<T> mt{T(0), T(0), 0, -1};
    if (tid < a.nmat) mt = MatLds<T>{a.ce[tid], a.inveps[tid], a.flags[tid], a.poleset[tid]};
    T co = T(0);
    int np = 0;
    if (a.npole) {
        if (tid < a.nset * CHIML_MAX_POLES * 3) co = a.pole_coef[tid];
        if (tid < a.nset) np = a.pole_count[tid];
    }
    const int d0 = a.det_ofs[tile], nd = min(a.det_ofs[tile + 1] - d0, kTileDet);
    TileDet det{};
    if (tid < nd) det = a.det[d0 + tid];
    const T ch0 = a.ch0[0], ch1 = a.ch1[0];
    int4 sb = make_int4(0, 0, 0, 0);
    int scomp = 0;
    T amp[K];
    if (tid < a.nsrc) {  // one lane per source
        sb = make_int4(a.src_box[6 * tid], a.src_box[6 * tid + 1], a.src_box[6 * tid + 2], a.src_box[6 * tid + 3]);
        scomp = a.src_comp[tid];
#pragma unroll
        for (int s = 0; s < K; ++s) amp[s] = a.src_amp[static_cast<long long>(step + min(s, a.nstep - 1)) * a.nsrc + tid];
    }
    // ---- tables to LDS ----
    if (tid < a.nmat) s_mt[tid] = mt;
    if (yp && tid < 2 * SH::ry)
        for (int k = 0; k < 3; ++k) s_y[tid < SH::ry ? 0 : 1][k][tid % SH::ry] = yc[k];
    if (a.npole) {
        if (tid < a.nset * CHIML_MAX_POLES * 3) s_co[tid] = co;
        if (tid < a.nset) s_np[tid] = np;
    }
    if (tid < nd) {
        // row .. pow as they are; interval counts down to the next sample, out is its place
        const int first = det.interval - step % det.interval, slot = (step + first) / det.interval;
        det.out += static_cast<long long>(slot) * det.npts;
        det.cap -= slot;
        det.thr |= det.row << 16;
        det.row = first - 1;  // launch step of the next sample
        s_det[tid] = det;
    }
    if (tid < 64) {  // the sources that touch the tile, in the table's order
        const bool hit = tid < a.nsrc && sb.x < x0 + RX && sb.y > x0 && sb.z < y0 + SH::ry && sb.w > y0;
        const unsigned long long m = __ballot(hit);
        if (hit) {
            const int n = __popcll(m & ((1ull << tid) - 1));
            s_box[n] = sb;
            s_comp[n] = scomp;
#pragma unroll
            for (int s = 0; s < K; ++s) s_amp[s][n] = amp[s];
        }
        if (tid == 0) s_nsrc = __popcll(m);
    }
    __syncthreads();
    // ---- what the steps need per row, in registers ----
    T ce[R], iev[R];
    unsigned prow = 0, drow = 0, sets = 0, nps = 0;  // dispersive rows, D rows, pole set and pole count (4 bits a row)
    unsigned long long dets = 0;                     // the thread's detector points
#pragma unroll
    for (int r = 0; r < R; ++r) {
        const MatLds<T> m = s_mt[id[r]];
        ce[r] = m.ce;
        iev[r] = m.inveps;
        const bool on = (in >> r) & 1u;
        if (!on) ez[r] = hx[r] = hy[r] = T(0);
        if (m.flags & CHIML_MAT_DCELL) drow |= 1u << r;
        if (a.npole && on && m.poleset >= 0) {
            prow |= 1u << r;
            sets |= static_cast<unsigned>(m.poleset) << (4 * r);
            const int n = s_np[m.poleset];
            nps |= static_cast<unsigned>(n) << (4 * r);
            const long long bi = (x - a.box[0]) + static_cast<long long>(a.box[1] - a.box[0]) * (yb + r - a.box[2]);
            for (int p = 0; p < n; ++p) {
                s_P[((2 * p) * R + r) * NT + tid] = a.P[p * a.boxn + bi];
                s_P[((2 * p + 1) * R + r) * NT + tid] = a.J[p * a.boxn + bi];
            }
        }
    }
    for (int q = 0; q < nd; ++q)
        if ((s_det[q].thr & 0xffff) == tid) dets |= 1ull << q;
    const int nsrc = s_nsrc;
    unsigned srows[3] = {0u, 0u, 0u};  // the rows that a source touches, per component (Ez, Hx, Hy)
    for (int k = 0; k < nsrc; ++k) {
        const int4 b = s_box[k];
        const int f = max(b.z - yb, 0), l = min(b.w - yb, R);
        if (x < b.x || x >= b.y || f >= l) continue;
        const unsigned rows = ((1u << l) - 1) & ~((1u << f) - 1);
        const int comp = s_comp[k];
#pragma unroll
        for (int c = 0; c < 3; ++c)
            if (comp == 2 + c) srows[c] |= rows;
    }
    auto src_at = [&](int comp, int s, int y) {
        T v = T(0);
        for (int k = 0; k < nsrc; ++k) {
            const int4 b = s_box[k];
            if (s_comp[k] == comp && x >= b.x && x < b.y && y >= b.z && y < b.w) v += s_amp[s][k];
        }
        return v;
    };
    const bool hyv = x < nx - 1, plain = x >= a.Tx && x < nx - a.Tx;  // plain: outside the x CPML
    // ---- the steps ----
    for (int s = 0; s < a.nstep; ++s) {
        s_ez[strip][col] = ez[0];
        __syncthreads();
        const T ez_up = strip + 1 < NS ? s_ez[strip + 1][col] : T(0);
#pragma unroll
        for (int r = 0; r < R; ++r) {
            const T dy = (r + 1 < R ? ez[r + 1 < R ? r + 1 : r] : ez_up) - ez[r];
            const T dx = lane_nb<true>(ez[r]) - ez[r];
            T ty_ = dy * a.inv_dy, tx_ = dx * a.inv_dx;
            const bool on = (in >> r) & 1u, hxon = on && yb + r < ny - 1, hyon = on && hyv;
            if (yp) {
                const int k = strip * R + r;
                const T psi = fma(s_y[0][0][k], pyh[r], s_y[0][1][k] * dy);
                if (hxon) pyh[r] = psi;
                ty_ = fma(s_y[0][2][k], ty_, psi);
            }
            if (xp) {
                const T psi = fma(xh[0], pxh[r], xh[1] * dx);
                if (hyon) pxh[r] = psi;
                tx_ = fma(xh[2], tx_, psi);
            }
            T vx = fma(ch0, -ty_, hx[r]), vy = fma(ch1, tx_, hy[r]);
            if ((srows[1] >> r) & 1u) vx += src_at(3, s, yb + r);
            if ((srows[2] >> r) & 1u) vy += src_at(4, s, yb + r);
            hx[r] = hxon ? vx : hx[r];
            hy[r] = hyon ? vy : hy[r];
        }
        s_hx[strip][col] = hx[R - 1];
        __syncthreads();
        const T hx_dn = strip > 0 ? s_hx[strip - 1][col] : T(0);
        T acc[R];
#pragma unroll
        for (int r = 0; r < R; ++r) {
            const T d1 = hy[r] - lane_nb<false>(hy[r]);
            const T d2 = hx[r] - (r > 0 ? hx[r > 0 ? r - 1 : 0] : hx_dn);
            T t1 = d1 * a.inv_dx, t2 = d2 * a.inv_dy;
            const bool fused = a.fma_curl && plain && yb + r >= a.Ty && yb + r < ny - a.Ty;
            const T accf = fma(-a.inv_dy, d2, t1);
            const bool on = (in >> r) & 1u;
            if (xp) {
                const T psi = fma(xe[0], pxe[r], xe[1] * d1);
                if (on) pxe[r] = psi;
                t1 = fma(xe[2], t1, psi);
            }
            if (yp) {
                const int k = strip * R + r;
                const T psi = fma(s_y[1][0][k], pye[r], s_y[1][1][k] * d2);
                if (on) pye[r] = psi;
                t2 = fma(s_y[1][2][k], t2, psi);
            }
            {
#pragma clang fp contract(off)
                acc[r] = fused ? accf : t1 - t2;
            }
        }
        if (prow | srows[0]) {  // rare: poles and sources; a row without either keeps the plain form
            T sv[R], jsum[R];
#pragma unroll
            for (int r = 0; r < R; ++r) {
                jsum[r] = T(0);
                sv[r] = (srows[0] >> r) & 1u ? src_at(2, s, yb + r) : T(0);
            }
            if (prow)
                for (int p = 0; p < a.npole; ++p) {
                    T Pv[R], Jv[R];
#pragma unroll
                    for (int r = 0; r < R; ++r) {
                        Pv[r] = s_P[((2 * p) * R + r) * NT + tid];
                        Jv[r] = s_P[((2 * p + 1) * R + r) * NT + tid];
                    }
#pragma unroll
                    for (int r = 0; r < R; ++r) {
                        if (p >= static_cast<int>((nps >> (4 * r)) & 15u)) continue;
                        const T* c = s_co + (((sets >> (4 * r)) & 15u) * CHIML_MAX_POLES + p) * 3;
                        const T Jn = fma(c[2], ez[r] + sv[r], fma(c[0], Pv[r], c[1] * Jv[r]));
                        s_P[((2 * p) * R + r) * NT + tid] = Pv[r] + Jn;
                        s_P[((2 * p + 1) * R + r) * NT + tid] = Jn;
                        jsum[r] += Jn;
                    }
                }
#pragma unroll
            for (int r = 0; r < R; ++r)
                if ((in >> r) & 1u) {
                    const T base = (drow >> r) & 1u ? ez[r] : ez[r] + sv[r];
                    ez[r] = fma(-iev[r], jsum[r], fma(ce[r], acc[r], base));
                }
        } else {
#pragma unroll
            for (int r = 0; r < R; ++r)
                if ((in >> r) & 1u) ez[r] = fma(ce[r], acc[r], ez[r]);
        }
        for (unsigned long long m = dets; m; m &= m - 1) {  // store_point's samples, at the advanced step
            TileDet& q = s_det[__ffsll(static_cast<long long>(m)) - 1];
            if (q.row != s) continue;
            const int row = q.thr >> 16;
            T f = T(0);
#pragma unroll
            for (int r = 0; r < R; ++r)
                if (r == row) f = q.comp == 2 ? ez[r] : (q.comp == 3 ? hx[r] : hy[r]);
            double u = static_cast<double>(f);
            if (q.pow) u = u * u;
            double point = q.conv / 2.0 * u;
            point = point + q.conv / 2.0 * u;
            if (q.cap > 0) a.det_out[q.out] = point;
            q.row = s + q.interval;
            q.out += q.npts;
            q.cap -= 1;
        }
    }
    // ---- the tile's own cells go to the other buffers ----
    const bool xown = xin && col >= K && col < RX - K;
#pragma unroll
    for (int r = 0; r < R; ++r) {
        const int row = strip * R + r, y = yb + r;
        if (!xown || row < K || row >= SH::ry - K || !((in >> r) & 1u)) continue;
        const long long i = x + static_cast<long long>(px) * y;
        a.ez_o[i] = ez[r];
        a.hx_o[i] = hx[r];
        a.hy_o[i] = hy[r];
        if (sxh >= 0) a.psi_o[1][sxh + static_cast<long long>(a.S[1]) * y] = pxh[r];
        if (sxe >= 0) a.psi_o[2][sxe + static_cast<long long>(a.S[2]) * y] = pxe[r];
        const int s0 = at(0, y), s3 = at(3, y);
        if (s0 >= 0) a.psi_o[0][x + static_cast<long long>(px) * s0] = pyh[r];
        if (s3 >= 0) a.psi_o[3][x + static_cast<long long>(px) * s3] = pye[r];
        if ((prow >> r) & 1u) {
            const long long bi = (x - a.box[0]) + static_cast<long long>(a.box[1] - a.box[0]) * (y - a.box[2]);
            for (int p = 0; p < static_cast<int>((nps >> (4 * r)) & 15u); ++p) {
                a.P_o[p * a.boxn + bi] = s_P[((2 * p) * R + r) * NT + tid];
                a.J_o[p * a.boxn + bi] = s_P[((2 * p + 1) * R + r) * NT + tid];
            }
        }
    }
}

template <typename T, typename SH>
__global__ void __launch_bounds__(SH::threads) k_tile2(TileArgs<T> a) {
    tile2_body<T, SH>(a, blockIdx.x, gridDim.x);
    if (a.step_next && blockIdx.x == 0 && threadIdx.x == 0) *a.step_next = step_now(a.step, a.stepv) + a.nstep;
}

// 32 x 32 cells (16 x 16 own), 64 x 32 (48 x 16), 64 x 64 (48 x 48; FP32 only,
// its FP64 registers spill: 1024^2 FP64 25 us a step, 16.5 with 64 x 32)
using TileS = TileShape<32, 2, 16>;
using TileM = TileShape<64, 2, 16>;
using TileL = TileShape<64, 4, 16>;

// ----------------------------------------------------- step counter ---------
// both slots: captured steps start on either
__global__ void k_set_step(int* step, int v) { step[0] = step[1] = v; }

// ----------------------------------------------- detectors and DFT ----------

template <typename T>
__device__ __forceinline__ void sample_at(const SampleArgs<T>& a, int t) {
    const int step = step_now(a.step, a.stepv);
    if (t < a.totpts && a.det_all1) {
        // the cells do not depend on the detector: their loads overlap its
        // search; a cell of -1 is the zero ghost beyond the domain
        const long long cu = a.det_cell[2 * t], cv = a.det_cell[2 * t + 1];
        store_point(a, t, cu >= 0 ? static_cast<double>(a.F[a.det_comp[2 * t]][cu]) : 0.0,
                    cv >= 0 ? static_cast<double>(a.F[a.det_comp[2 * t + 1]][cv]) : 0.0, step);
    } else if (t < a.totpts) {
        int d = 0;  // the detector of point t
        while (d + 1 < a.ndet && a.det_off[d + 1] <= t) ++d;
        if (step % a.det_interval[d] != 0) return;
        const int slot = step / a.det_interval[d];
        if (slot >= a.det_cap[d]) return;
        // the point's fields in order, each as the pair (point, offset cell)
        const int nf = a.det_nf[d];
        const long long e0 = a.det_eoff[d] + static_cast<long long>(t - a.det_off[d]) * nf;
        const double c = a.det_conv[d];
        double point = 0.0;
        for (int f = 0; f < nf; ++f) {
            const long long e = 2 * (e0 + f);
            const long long cu = a.det_cell[e], cv = a.det_cell[e + 1];
            const double u = cu >= 0 ? static_cast<double>(a.F[a.det_comp[e]][cu]) : 0.0;
            const double v = cv >= 0 ? static_cast<double>(a.F[a.det_comp[e + 1]][cv]) : 0.0;
            if (a.det_pow[d]) {
                point = point + c / 2.0 * (u * u);
                point = point + c / 2.0 * (v * v);
            } else {
                point = point + c / 2.0 * u;
                point = point + c / 2.0 * v;
            }
        }
        a.det_out[a.det_out_off[d] + static_cast<long long>(slot) * a.det_npts[d] + (t - a.det_off[d])] = point;
    } else if (t < a.totpts + a.ndft) {
        const int s = t - a.totpts;
        // constant group indices keep the group table in kernel arguments
#pragma unroll
        for (int g = 0; g < kMaxDftGroups; ++g) {
            if (g >= a.ndg) break;
            if (s < a.gofs[g] || s >= a.gofs[g + 1]) continue;
            const DftSample<T>& d = a.dg[g];
            const int j = s - a.gofs[g];
            if (step % d.interval == 0) {
                const int k = (step / d.interval) % kDftBlock;
                d.stage[static_cast<long long>(k) * d.n + j] = a.F[d.comp[j]][d.cell[j]];
            }
        }
    }
}

template <typename T>
__global__ void k_sample(SampleArgs<T> a) {
    sample_at<T>(a, blockIdx.x * blockDim.x + threadIdx.x);
}

// F[f][s] += sum_k exp(-i w_f t_k) U[k][s] over the staged samples k of the
// current block (parallelStorageFreqDTCReal::fieldIn rank-1 updates,
// src/DTC/parallelStorageFreqDTC.cpp:21-30, batched over kDftBlock steps).
// A thread owns one sampled cell: its staged samples sit in registers, the
// block's phasors in LDS, and the accumulators are stored frequency-major so
// that the read-modify-write of F is coalesced across threads.
constexpr int kDftFreqChunk = 64;

template <typename T>
__global__ void __launch_bounds__(256) k_dft_flush(const T* stage, const double* phasor, double* F, const int* stepp, int ndft, int nfreq,
                                                  int interval, int force, int step_override) {
    __shared__ double2 w[kDftBlock * kDftFreqChunk];
    const int step = step_override >= 0 ? step_override : *stepp;
    if (step % interval != 0 && !force) return;
    const int kmax = step / interval;
    if (!force && (kmax % kDftBlock) != kDftBlock - 1) return;
    const int kfirst = kmax - (kmax % kDftBlock);
    const int nk = kmax - kfirst + 1;
    const int s = blockIdx.x * blockDim.x + threadIdx.x;
    double u[kDftBlock];
#pragma unroll
    for (int k = 0; k < kDftBlock; ++k) u[k] = (s < ndft && k < nk) ? static_cast<double>(stage[static_cast<long long>(k) * ndft + s]) : 0.0;
    for (int f0 = 0; f0 < nfreq; f0 += kDftFreqChunk) {
        const int nfc = min(kDftFreqChunk, nfreq - f0);
        __syncthreads();
        // slots past the open block's last sample get zero weight (the phasor
        // table ends at the last sampled step, and 0 * garbage may be NaN)
        for (int t = threadIdx.x; t < kDftBlock * nfc; t += blockDim.x) {
            const int k = t / nfc, f = t % nfc;
            double2 v = make_double2(0.0, 0.0);
            if (k < nk) {
                const double* src = phasor + 2 * (static_cast<long long>(kfirst + k) * nfreq + f0 + f);
                v = make_double2(src[0], src[1]);
            }
            w[k * kDftFreqChunk + f] = v;
        }
        __syncthreads();
        if (s < ndft) {
            for (int f = 0; f < nfc; ++f) {
                double re = 0.0, im = 0.0;
#pragma unroll
                for (int k = 0; k < kDftBlock; ++k) {
                    const double2 ww = w[k * kDftFreqChunk + f];
                    re += ww.x * u[k];
                    im += ww.y * u[k];
                }
                double2* dst = reinterpret_cast<double2*>(F) + static_cast<long long>(f0 + f) * ndft + s;
                double2 acc = *dst;
                acc.x += re;
                acc.y += im;
                *dst = acc;
            }
        }
    }
}

// Flux through the faces of a box: the combined face fields (combineField,
// parallelFlux.hpp:325-395), Ej Hk* - Ek Hj* over nt^2, the integration weight,
// and a sum over the block's 256 points, one block row per frequency.  Each face
// starts on a block boundary and the host adds a face's blocks in order.  Reads
// 16 samples per point and frequency from the accumulators: a 61^3 box with 40
// frequencies is read in 1.0 ms, where copying the accumulators to the host and
// combining them there took 70 ms.
constexpr int kFluxFaces = 6;
struct FluxPlanDev {
    int nface, start[kFluxFaces + 1];  // first point (padded) of each face
    int npt[kFluxFaces];
    double cw[kFluxFaces][4];
    const int* ids;    // [16][start[nface]]
    const double* sw;  // [start[nface]]
};

__global__ void __launch_bounds__(256) k_flux_faces(FluxPlanDev pl, const double2* __restrict__ F, int ndft, double inv_nt2,
                                                    double2* __restrict__ partial) {
    __shared__ double2 red[256];
    const int total = pl.start[pl.nface], t = blockIdx.x * 256 + threadIdx.x;
    int f = 0;
    while (f + 1 < pl.nface && pl.start[f + 1] <= static_cast<int>(blockIdx.x) * 256) ++f;
    const double2* Ff = F + static_cast<long long>(blockIdx.y) * ndft;
    double2 v = make_double2(0.0, 0.0);
    if (t - pl.start[f] < pl.npt[f]) {
        double2 g[4];
#pragma unroll
        for (int c = 0; c < 4; ++c) {
            double2 acc = make_double2(0.0, 0.0);
#pragma unroll
            for (int k = 0; k < 4; ++k) {
                const int id = pl.ids[(c * 4 + k) * static_cast<long long>(total) + t];
                if (id < 0) continue;
                const double2 u = Ff[id];
                acc.x += pl.cw[f][c] * u.x;
                acc.y += pl.cw[f][c] * u.y;
            }
            g[c] = acc;
        }
        const double w = pl.sw[t] * inv_nt2;
        v.x = w * ((g[0].x * g[3].x + g[0].y * g[3].y) - (g[1].x * g[2].x + g[1].y * g[2].y));
        v.y = w * ((g[0].y * g[3].x - g[0].x * g[3].y) - (g[1].y * g[2].x - g[1].x * g[2].y));
    }
    red[threadIdx.x] = v;
    __syncthreads();
    for (int w = 128; w > 0; w >>= 1) {
        if (threadIdx.x < w) {
            red[threadIdx.x].x += red[threadIdx.x + w].x;
            red[threadIdx.x].y += red[threadIdx.x + w].y;
        }
        __syncthreads();
    }
    if (threadIdx.x == 0) partial[blockIdx.y * static_cast<long long>(gridDim.x) + blockIdx.x] = red[0];
}

// ------------------------------------------------------------ emitters ------
struct QeDev {
    int packed;             // rho and its history hold the upper triangle only (Hermitian)
    int N, nmem, nemit;
    const int* xyz;         // [nemit][3]
    const double2* h0;      // [nmem][N*N]
    const double2* mu;      // [3][N*N]
    int ngam;
    const int* gam_ptr;     // [N*N + 1]: the Lindblad entries of each row
    const int* gam_col;     // [ngam], by row
    const double* gam_val;
    double na, ih;          // ih = 1 / hbar
    double ab[4], am[4];    // dt/24 (55, -59, 37, -9) and dt/24 (9, 19, -5, 1): predictor and corrector weights
    int bmin[3], bn[3];     // emitter box
    double* Pbox[3];        // (bn+2)^3 node polarization, z-extent bn+1+zoff
    double* Aprev[3];       // per touched E cell (bn+1)^3 previous back-coupling
    double2* rho;           // [N*N][nmem*nemit]
    double2* hist;          // [4][N*N][nmem*nemit]
    int npop;
    const int* pop_flat;
    int pop_interval;
    double2* pop_partial;   // [npop][nblocks]
    double2* pop_out;       // [npop][cap]
    int pop_cap;
    int dim;
    const double* eps_node;
    int fold_addp;          // 2D: the density kernel does addP for its own emitter cell (no k_ml_addp launch)
};

// addP (src/UTIL/FDTD_up_eq.cpp:1367-1380) in increment form: a cell's
// back-coupling A = P(p)/(2 eps(p)) + P(p+off)/(2 eps(p+off)) is subtracted
// once per step from E derived from D, so E changes by A_prev - A_cur.
template <typename T>
__global__ void k_ml_addp(QeDev q, T* E0, T* E1, T* E2, int nx, int ny, int nz) {
    const int t = blockIdx.x * blockDim.x + threadIdx.x;
    const int c = blockIdx.y;
    T* E = c == 0 ? E0 : (c == 1 ? E1 : E2);
    if (!E) return;
    const int ex = q.bn[0] + 1, ey = q.bn[1] + 1, ez = (q.dim == 3) ? q.bn[2] + 1 : 1;
    if (t >= ex * ey * ez) return;
    const int x = t % ex, y = (t / ex) % ey, z = t / (ex * ey);
    // E cell at point (bmin - 1 + x, ...) <-> P box index (x, y, z)
    const int px = q.bmin[0] - 1 + x, py = q.bmin[1] - 1 + y, pz = (q.dim == 3) ? q.bmin[2] - 1 + z : 0;
    if (px < 0 || py < 0 || pz < 0 || px >= nx || py >= ny || pz >= nz) return;
    int off[3] = {0, 0, 0};
    if (q.dim == 3) off[c] = 1;
    const int PX = q.bn[0] + 2, PY = q.bn[1] + 2;
    const int zi = (q.dim == 3) ? z : 0;
    const double* P = q.Pbox[c];
    double p0 = P[x + PX * (y + PY * zi)];
    double p1 = P[(x + off[0]) + PX * ((y + off[1]) + PY * (zi + off[2]))];
    const long long i0 = px + static_cast<long long>(nx) * (py + static_cast<long long>(ny) * pz);
    int qx = px + off[0], qy = py + off[1], qz = pz + off[2];
    double e1 = (qx < nx && qy < ny && qz < nz) ? q.eps_node[qx + static_cast<long long>(nx) * (qy + static_cast<long long>(ny) * qz)] : 1.0;
    double A = 0.5 * p0 / q.eps_node[i0] + 0.5 * p1 / e1;
    double* Ap = q.Aprev[c] + t;
    double prev = *Ap;
    *Ap = A;
    E[i0] = static_cast<T>(static_cast<double>(E[i0]) + (prev - A));
}

__device__ __forceinline__ double2 cmul(double2 a, double2 b) { return make_double2(a.x * b.x - a.y * b.y, a.x * b.y + a.y * b.x); }
__device__ __forceinline__ double2 cadd(double2 a, double2 b) { return make_double2(a.x + b.x, a.y + b.y); }
__device__ __forceinline__ double2 cscale(double2 a, double s) { return make_double2(a.x * s, a.y * s); }

// Entry (i, j) of d rho/dt for the matrices H and X of one emitter in LDS
// (entry k of emitter t at [k EB + t], column-major): (i/hbar)(H X - X H)[i, j]
// + the entry's Lindblad row.
template <int N, int EB>
__device__ __forceinline__ double2 den_deriv(double ih, const double2* H, const double2* X, int i, int j, const int* col, const double* val,
                                             int g0, int g1) {
    double2 s1 = make_double2(0.0, 0.0), s2 = s1;
    // Up to five terms are written out; of more, three are in flight at a time.
    // 144,000 emitters, us a launch, in threes / written out: N = 4 packed
    // 52.7/47.4, N = 5 full 134/124 (one lane per column: 123), N = 6 packed in
    // fives 100 against 89, N = 8 packed 234 against 211.
#pragma unroll (N <= 5 ? N : 3)
    for (int k = 0; k < N; ++k) {
        s1 = cadd(s1, cmul(H[(i + k * N) * EB], X[(k + j * N) * EB]));
        s2 = cadd(s2, cmul(X[(i + k * N) * EB], H[(k + j * N) * EB]));
    }
    double2 out = make_double2(-(s1.y - s2.y) * ih, (s1.x - s2.x) * ih);
    for (int g = g0; g < g1; ++g) {
        const double2 v = X[col[g] * EB];
        out.x += v.x * val[g];
        out.y += v.y * val[g];
    }
    return out;
}

// Every emitter group (N >= 2): one lane per stored entry of rho and emitter,
// advanced by the Adams-Bashforth-Moulton predictor-corrector (PCABAM4,
// parallelQE.hpp:751-770) cold-started from zero history; the derivative
// history is a 4-slot ring instead of the reference's three copies per step
// (density.hpp:65-70).  Lanes are grouped by entry, lane = k EB + emitter, so
// every rho and history access of an entry is a contiguous run of EB complex
// words.  H = h0 - E.mu (formed once per member, each lane its entry) and the
// matrix being differentiated are shared through LDS, entry by entry with the
// emitters side by side: consecutive lanes read consecutive words, no bank is
// hit twice.
//
// PK (Hermitian packing): rho and the derivative history keep only the upper
// triangle, entry (i, j) with i <= j stored at j (j + 1) / 2 + i; a lane also
// writes the conjugate of its entry to the lower half of the shared matrices.
// rho stays exactly Hermitian, which the full form keeps up to rounding (the
// Lindblad sums of mirrored entries may add in another order).  Used when H0,
// the dipoles and the Lindblad operator preserve hermiticity; the derivative
// of a Hermitian rho is then Hermitian.
//
// The kernel moves 7 words per stored entry (338,560 six-level emitters,
// packed: 796 MB) and is bound by memory as long as enough waves are in flight
// to cover its phases (load, two derivatives, store), so a lane holds one entry
// (78 VGPRs, 6 waves per SIMD).  With one lane per column (236 VGPRs, 2 waves)
// the same launch took 407 us, now 231 (3.4 TB/s); the copy rate would allow
// 124.  4 waves per SIMD measured 275, blocks of 16 emitters 330.  32,768
// two-level emitters: 10.1 -> 6.8 us.
constexpr int kMlGamLds = 256;  // Lindblad entries staged in LDS (more are read from global memory)

__host__ __device__ constexpr int ml_store_words(int n, bool pk) { return pk ? n * (n + 1) / 2 : n * n; }
// emitters per block: the largest run whose lanes fit a block
__host__ __device__ constexpr int ml_emitters(int n, bool pk) {
    const int w = ml_store_words(n, pk);
    return w * 64 <= 1024 ? 64 : (w * 32 <= 1024 ? 32 : 16);
}
__host__ __device__ constexpr int ml_threads(int n, bool pk) { return (ml_store_words(n, pk) * ml_emitters(n, pk) + 63) / 64 * 64; }

template <typename T, int N, bool PK>
__global__ void __launch_bounds__(ml_threads(N, PK), 6) k_ml_entry(QeDev q, T* E0, T* E1, T* E2, int nx, int ny, int nz,
                                                                const int* stepp, int stepv) {
    constexpr int S = N * N, SP = ml_store_words(N, PK), EB = ml_emitters(N, PK);
    static_assert(SP >= 3, "the first three entries' lanes gather the field components");
    __shared__ double2 Hs[S * EB], Xs[S * EB];
    __shared__ double2 mus[3][S];
    __shared__ double ef[3][EB];
    __shared__ double2 pops[4][EB];
    __shared__ int gc_s[kMlGamLds];
    __shared__ double gv_s[kMlGamLds];
    const int k = threadIdx.x / EB, team = threadIdx.x - k * EB;  // stored entry and emitter
    const int e = blockIdx.x * EB + team;
    const bool act = k < SP && e < q.nemit;
    int i, j;
    if (PK) {
        j = 0;
        while ((j + 1) * (j + 2) / 2 <= k && j < N - 1) ++j;
        i = min(k - j * (j + 1) / 2, j);
    } else {
        j = min(k / N, N - 1);
        i = k - (k / N) * N;
    }
    const int kk = i + j * N;  // the entry's place in the full matrix
    const int step = step_now(stepp, stepv);
    const int u = step & 3;
    const int s0 = (u + 3) & 3, s1 = (u + 2) & 3, s2 = (u + 1) & 3, s3 = u;
    const long long ld = static_cast<long long>(q.nmem) * q.nemit;
    long long at = k * ld + e;  // the entry of member 0
    const long long slot = SP * ld;
    double2 rk = make_double2(0.0, 0.0), f0 = rk, f1 = rk, f2 = rk, f3 = rk;
    auto load = [&] {
        if (!act) return;
        rk = q.rho[at];
        f0 = q.hist[s0 * slot + at];
        f1 = q.hist[s1 * slot + at];
        f2 = q.hist[s2 * slot + at];
        f3 = q.hist[s3 * slot + at];
    };
    load();
    for (int t = threadIdx.x; t < 3 * S; t += blockDim.x) mus[t / S][t % S] = q.mu[t];
    const bool gam_lds = q.ngam <= kMlGamLds;
    if (gam_lds)
        for (int g = threadIdx.x; g < q.ngam; g += blockDim.x) {
            gc_s[g] = q.gam_col[g];
            gv_s[g] = q.gam_val[g];
        }
    const int* gc = gam_lds ? gc_s : q.gam_col;
    const double* gv = gam_lds ? gv_s : q.gam_val;
    const int g0 = act ? q.gam_ptr[kk] : 0, g1 = act ? q.gam_ptr[kk + 1] : 0;
    // the lanes of entries 0..2 gather E_x, E_y, E_z at their emitter
    T* const Ec = k == 0 ? E0 : (k == 1 ? E1 : (k == 2 ? E2 : nullptr));
    if (k < 3 && act) {
        const int px = q.xyz[3 * e], py = q.xyz[3 * e + 1], pz = q.xyz[3 * e + 2];
        double ev = 0.0;
        if (Ec) {
            const long long ip = px + static_cast<long long>(nx) * (py + static_cast<long long>(ny) * pz);
            ev = static_cast<double>(Ec[ip]);
            if (q.dim != 2) {
                // mean of the two Yee edges E_c(p) and E_c(p - e_c) (getE_TE)
                const int qx = px - (k == 0), qy = py - (k == 1), qz = pz - (k == 2);
                const double v1 = (qx >= 0 && qy >= 0 && qz >= 0) ? static_cast<double>(Ec[qx + static_cast<long long>(nx) * (qy + static_cast<long long>(ny) * qz)]) : 0.0;
                ev = 0.5 * ev + 0.5 * v1;
            } else if (q.fold_addp) {
                // k_ml_addp for this emitter's own E cell (in 2D no other
                // emitter's polarisation reaches it): E += A_prev - A
                const int bx = px - q.bmin[0] + 1, by = py - q.bmin[1] + 1;
                const double p0 = q.Pbox[2][bx + (q.bn[0] + 2) * by];
                const double A = 0.5 * p0 / q.eps_node[ip] + 0.5 * p0 / q.eps_node[ip];
                double* const Ap = q.Aprev[2] + bx + static_cast<long long>(q.bn[0] + 1) * by;
                const T en = static_cast<T>(ev + (*Ap - A));
                *Ap = A;
                Ec[ip] = en;
                ev = static_cast<double>(en);
            }
        }
        ef[k][team] = ev;
    }
    double2* const X = Xs + team;
    double2* const H = Hs + team;
    // population samples: every pop_interval steps while slots remain (QEPopDtc)
    const bool record = q.npop > 0 && step % q.pop_interval == 0 && step / q.pop_interval < q.pop_cap;
    double P = 0.0;
    if (record && k == 0)
        for (int jj = 0; jj < 4; ++jj) pops[jj][team] = make_double2(0.0, 0.0);
    __syncthreads();  // mu, the Lindblad entries and E are staged
    for (int m = 0; m < q.nmem; ++m) {
        double2 cr = rk;
        if (act) {
            double2 h = q.h0[m * S + kk];
#pragma unroll
            for (int c = 0; c < 3; ++c) {
                h.x -= ef[c][team] * mus[c][kk].x;
                h.y -= ef[c][team] * mus[c][kk].y;
            }
            H[kk * EB] = h;
            double2 pr = rk;
            pr = cadd(pr, cscale(f0, q.ab[0]));
            pr = cadd(pr, cscale(f1, q.ab[1]));
            pr = cadd(pr, cscale(f2, q.ab[2]));
            pr = cadd(pr, cscale(f3, q.ab[3]));
            X[kk * EB] = pr;
            if (PK && i < j) {
                H[(j + i * N) * EB] = make_double2(h.x, -h.y);
                X[(j + i * N) * EB] = make_double2(pr.x, -pr.y);
            }
            cr = cadd(cr, cscale(f0, q.am[1]));
            cr = cadd(cr, cscale(f1, q.am[2]));
            cr = cadd(cr, cscale(f2, q.am[3]));
        }
        __syncthreads();
        double2 fp = make_double2(0.0, 0.0);
        if (act) fp = den_deriv<N, EB>(q.ih, H, X, i, j, gc, gv, g0, g1);
        __syncthreads();
        if (act) {
            cr = cadd(cr, cscale(fp, q.am[0]));
            q.rho[at] = cr;
            X[kk * EB] = cr;
            if (PK && i < j) X[(j + i * N) * EB] = make_double2(cr.x, -cr.y);
        }
        __syncthreads();
        if (act) {
            fp = den_deriv<N, EB>(q.ih, H, X, i, j, gc, gv, g0, g1);
            q.hist[s3 * slot + at] = fp;
            if (k < 3 && Ec) {  // polarisation of the emitter: sum of Re(conj(rho) mu)
                double sacc = 0.0;
#pragma unroll
                for (int b = 0; b < N; ++b)
#pragma unroll
                    for (int a = 0; a < (PK ? b + 1 : N); ++a) {
                        // with packing the mirrored entry adds the same again (rho and mu Hermitian)
                        const double2 r = X[(a + b * N) * EB], mu = mus[k][a + b * N];
                        const double t = r.x * mu.x + r.y * mu.y;
                        sacc += (PK && a < b) ? 2.0 * t : t;
                    }
                P += q.na * sacc;
            }
            if (record && k == 0)
                for (int jj = 0; jj < q.npop; ++jj) pops[jj][team] = cadd(pops[jj][team], X[q.pop_flat[jj] * EB]);
        }
        if (m + 1 < q.nmem) {
            at += q.nemit;
            load();
            __syncthreads();  // Hs and Xs are rewritten by the next member
        }
    }
    if (k < 3 && act && Ec) {
        const int bx = q.xyz[3 * e] - q.bmin[0] + 1, by = q.xyz[3 * e + 1] - q.bmin[1] + 1, bz = (q.dim == 3) ? q.xyz[3 * e + 2] - q.bmin[2] + 1 : 0;
        q.Pbox[k][bx + (q.bn[0] + 2) * (by + (q.bn[1] + 2) * bz)] = P;
    }
    // Per-block population sums by the first EB lanes, in a fixed order;
    // k_ml_pop_finish adds the blocks' sums in a fixed order.  A finish inside
    // this launch (last block by an atomic ticket) needs a device-scope release
    // per block, which writes back the XCD's L2 each time and more than doubled
    // the launch.
    if (record && threadIdx.x < EB) {
        for (int jj = 0; jj < q.npop; ++jj) {
            double2 v = pops[jj][team];
#pragma unroll
            for (int w = EB / 2; w > 0; w >>= 1) {
                v.x += __shfl_down(v.x, w, EB);
                v.y += __shfl_down(v.y, w, EB);
            }
            if (threadIdx.x == 0) q.pop_partial[jj * gridDim.x + blockIdx.x] = v;
        }
    }
}

constexpr int kPopThreads = 1024;

// Populations of this step: block jb sums population j0 + jb's per-block
// partials (each thread a fixed strided subset, then a tree in LDS, so the
// order is the same every run) and stores the mean over the emitters.
__device__ __forceinline__ void pop_finish(const QeDev& q, const double2* __restrict__ partial, int nblocks, int j0, int jb, int step) {
    __shared__ double2 red[kPopThreads];
    if (step % q.pop_interval != 0 || step / q.pop_interval >= q.pop_cap) return;
    double2 sum = make_double2(0.0, 0.0);
    for (int b = threadIdx.x; b < nblocks; b += kPopThreads) sum = cadd(sum, partial[jb * nblocks + b]);
    red[threadIdx.x] = sum;
    __syncthreads();
    for (int w = kPopThreads / 2; w > 0; w >>= 1) {
        if (threadIdx.x < w) red[threadIdx.x] = cadd(red[threadIdx.x], red[threadIdx.x + w]);
        __syncthreads();
    }
    if (threadIdx.x == 0)
        q.pop_out[static_cast<long long>(j0 + jb) * q.pop_cap + step / q.pop_interval] = make_double2(red[0].x / q.nemit, red[0].y / q.nemit);
}

__global__ void __launch_bounds__(kPopThreads) k_ml_pop_finish(QeDev q, const double2* __restrict__ partial, int nblocks, int j0,
                                                                const int* stepp, int stepv) {
    pop_finish(q, partial, nblocks, j0, blockIdx.x, step_now(stepp, stepv));
}

// The population finish and the sample launch of a step in one: neither reads
// what the other writes, and each is a launch of a few us that a 2D emitter
// step has too many of (1024^2, 32,768 emitters: 25.5 -> 23.2 us a step).
template <typename T>
__global__ void __launch_bounds__(kPopThreads) k_finish_sample(QeDev q, const double2* __restrict__ partial, int nblocks, const int* stepp,
                                                               int stepv, SampleArgs<T> s) {
    if (static_cast<int>(blockIdx.x) < q.npop) pop_finish(q, partial, nblocks, 0, blockIdx.x, step_now(stepp, stepv));
    else sample_at<T>(s, (blockIdx.x - q.npop) * blockDim.x + threadIdx.x);
}

// Population detectors past the four the density kernel sums in LDS:
// on recording steps, block (b, jj - j0) sums entry (ri, cj) of the stored
// density matrices (the conjugate of (cj, ri) below the diagonal when
// packed) over a strided subset of the member/emitter columns, then a tree in
// LDS; k_ml_pop_finish adds the blocks' sums in a fixed order.
__global__ void __launch_bounds__(256) k_ml_pop_gather(QeDev q, int j0, double2* __restrict__ partial, const int* stepp, int stepv) {
    __shared__ double2 red[256];
    const int step = step_now(stepp, stepv);
    if (step % q.pop_interval != 0 || step / q.pop_interval >= q.pop_cap) return;
    const int k = q.pop_flat[j0 + blockIdx.y];
    const int N = q.N, ri = k % N, cj = k / N;
    long long si;
    bool conj = false;
    if (q.packed) {
        if (ri <= cj) si = cj * (cj + 1) / 2 + ri;
        else {
            si = ri * (ri + 1) / 2 + cj;
            conj = true;
        }
    } else {
        si = ri + static_cast<long long>(cj) * N;
    }
    const long long ld = static_cast<long long>(q.nmem) * q.nemit;
    double2 sum = make_double2(0.0, 0.0);
    for (long long col = blockIdx.x * 256LL + threadIdx.x; col < ld; col += gridDim.x * 256LL) {
        double2 v = q.rho[si * ld + col];
        if (conj) v.y = -v.y;
        sum = cadd(sum, v);
    }
    red[threadIdx.x] = sum;
    __syncthreads();
    for (int w = 128; w > 0; w >>= 1) {
        if (threadIdx.x < w) red[threadIdx.x] = cadd(red[threadIdx.x], red[threadIdx.x + w]);
        __syncthreads();
    }
    if (threadIdx.x == 0) partial[blockIdx.y * gridDim.x + blockIdx.x] = red[0];
}

// ----------------------------------------------------------------- TFSF ----
// Total-field / scattered-field surfaces (parallelTFSFBase,
// src/SOURCE/parallelTFSF.hpp:1058-1174).  Each surface owns twelve complex
// FP64 incident lines (six components, set 0 read by the surface adds, set 1
// the shorter pulse line whose values are recorded for the flux
// normalisation).  They are a few hundred to a few thousand points long, so
// one block steps all of them, between the H and E updates of the main grid,
// beside the blocks that add pf * Re(line) to the surface cells of H
// (k_tfsf_step); k_tfsf_add then adds to the cells of E.  256^3 FP32 with a
// 201^3 box: H adds 11.4 us and lines 16.2 us one after the other, 21.2 us
// together.  The adds are bound by the faces of constant x, where each point
// moves a cache line of its own; the sweeps, which hold those cells anyway,
// lost more to the search for them (k_h3_all 107 -> 167 us).
struct TfsfLineArgs {
    int len[2], present[6], margin, pulse_at, pulse_n, psi_n, rec_idx, rec_off[6];
    int nterm[6], tsrc[6][2], tpos[6][2], tneg[6][2];
    double tcoef[6][2];
    int nseg[6], ssrc[6][4], shigh[6][4], soff1[6][4], soff2[6][4];
    double sdb[6][4];
    const double* scoef;  // [6][4][psi_n][3]
    double2* line[2];     // set s: [6][len[s]]
    double2* psi;         // [2][6][4][psi_n]
    const double2* amp;   // [nsteps][6][pulse_n]
    double2* rec;         // [6][nrec]
    long long nrec;
    double2* snap[2];     // [6][len[0]] by step parity: the lines line[0] after the step, for the H adds of the next
};

// One line point: pulse, the derivative terms in the reference's order, then
// the CPML segments that cover it (updateIncdField*, parallelTFSF.cpp:11-45;
// addPsi / updatePsiField, src/PML/PML.cpp:12-29).  L: the set's lines, psi:
// the set's CPML fields [6][4][psi_n], co: coefficients [6][4][psi_n][3],
// amp: this step's pulse values [6][pulse_n].
__device__ void tfsf_point(const TfsfLineArgs& t, double2* L, double2* psi, const double* co, const double2* amp, int s, int c, int n) {
    const int len = t.len[s];
    double2 v = L[c * len + n];
    const int pr = n - t.pulse_at;
    if (pr >= 0 && pr < t.pulse_n) v = cadd(v, amp[c * t.pulse_n + pr]);
    if (n >= t.margin && n < len - t.margin)
        for (int k = 0; k < t.nterm[c]; ++k) {
            const double2* u = L + t.tsrc[c][k] * len;
            const double a = t.tcoef[c][k];
            v = cadd(v, cscale(u[n + t.tpos[c][k]], a));
            v = cadd(v, cscale(u[n + t.tneg[c][k]], -1.0 * a));
        }
    for (int g = 0; g < t.nseg[c]; ++g) {
        const int gl = t.shigh[c][g] ? len - 1 - t.psi_n - t.margin : t.margin;
        const int i = n - gl;
        if (i < 0 || i >= t.psi_n) continue;
        const double* q = co + ((c * 4 + g) * t.psi_n + i) * 3;
        const double2* u = L + t.ssrc[c][g] * len;
        double2& ps = psi[(c * 4 + g) * t.psi_n + i];
        double2 p = cscale(ps, q[0]);
        p = cadd(p, cscale(u[gl + t.soff1[c][g] + i], q[1]));
        p = cadd(p, cscale(u[gl + t.soff2[c][g] + i], q[2]));
        ps = p;
        v = cadd(v, cscale(p, t.sdb[c][g]));
    }
    L[c * len + n] = v;
}

// LDS bytes of the staged form of k_tfsf_step: both sets of lines, their
// CPML fields, the coefficients and one step of pulse values.
__host__ __device__ inline size_t tfsf_lds_bytes(const TfsfLineArgs& t) {
    return 16 * (6 * static_cast<size_t>(t.len[0] + t.len[1]) + 2 * 6 * 4 * static_cast<size_t>(t.psi_n) + 6 * static_cast<size_t>(t.pulse_n)) +
           8 * 6 * 4 * 3 * static_cast<size_t>(t.psi_n);
}

// parallelTFSFBase::step (parallelTFSF.hpp:1148-1174) for every line, with
// the incident H recorded before it and the incident E after it
// (parallelFDTDField.hpp:1240-1254).  One block.  The step is a chain of
// short dependent passes over small arrays that the field sweeps evict from
// the caches between steps, so with LDS every array the passes touch is
// staged in shared memory first (one batch of loads) and written back after;
// lines too long for it are stepped in global memory.
template <bool LDS>
__device__ __forceinline__ void tfsf_lines(const TfsfLineArgs& ta, unsigned char* tfsf_lds, int step) {
    // the parameter block is read by every pass: one copy into LDS, read in
    // parallel, instead of a chain of dependent argument loads per pass
    __shared__ TfsfLineArgs t;
    static_assert(sizeof(TfsfLineArgs) % 4 == 0, "parameter block is copied in 4-byte words");
    for (unsigned w = threadIdx.x; w < sizeof(TfsfLineArgs) / 4; w += blockDim.x)
        reinterpret_cast<int*>(&t)[w] = reinterpret_cast<const int*>(&ta)[w];
    __syncthreads();
    double2* L[2] = {t.line[0], t.line[1]};
    const int np = 6 * 4 * t.psi_n;
    double2* psi = t.psi;
    const double* co = t.scoef;
    const double2* amp = t.amp + static_cast<long long>(step) * 6 * t.pulse_n;
    if (LDS) {
        double2* sh = reinterpret_cast<double2*>(tfsf_lds);
        L[0] = sh;
        L[1] = L[0] + 6 * t.len[0];
        double2* sp = L[1] + 6 * t.len[1];
        double2* sa = sp + 2 * np;
        double* sc = reinterpret_cast<double*>(sa + 6 * t.pulse_n);
        for (int s = 0; s < 2; ++s)
            for (int q = threadIdx.x; q < 6 * t.len[s]; q += blockDim.x) L[s][q] = t.line[s][q];
        for (int q = threadIdx.x; q < 2 * np; q += blockDim.x) sp[q] = t.psi[q];
        for (int q = threadIdx.x; q < 3 * np; q += blockDim.x) sc[q] = t.scoef[q];
        for (int q = threadIdx.x; q < 6 * t.pulse_n; q += blockDim.x) sa[q] = amp[q];
        psi = sp;
        co = sc;
        amp = sa;
        __syncthreads();
    }
    auto record = [&](int c0) {
        const int c = c0 + static_cast<int>(threadIdx.x);
        if (threadIdx.x < 3 && t.present[c]) {
            const double2* P = L[1] + c * t.len[1];
            double2* r = t.rec + c * t.nrec + 2LL * step;
            r[0] = P[t.rec_idx];
            r[1] = P[t.rec_idx - t.rec_off[c]];
        }
    };
    record(3);
    __syncthreads();
    for (int ph = 0; ph < 2; ++ph) {  // H lines (3..5), then E lines (0..2)
        // the line is uniform across the block, so its parameters are scalar
        // loads; the lines of one phase are independent of each other
        for (int l = 0; l < 6; ++l) {
            const int s = l / 3, c = (ph == 0 ? 3 : 0) + l % 3;
            if (!t.present[c]) continue;
            for (int n = threadIdx.x; n < t.len[s]; n += blockDim.x) tfsf_point(t, L[s], psi + s * np, co, amp, s, c, n);
        }
        __syncthreads();
    }
    record(0);
    double2* const snap = t.snap[step & 1];
    for (int q = threadIdx.x; q < 6 * t.len[0]; q += blockDim.x) snap[q] = L[0][q];
    if (LDS) {
        for (int s = 0; s < 2; ++s)
            for (int q = threadIdx.x; q < 6 * t.len[s]; q += blockDim.x) t.line[s][q] = L[s][q];
        for (int q = threadIdx.x; q < 2 * np; q += blockDim.x) t.psi[q] = psi[q];
    }
}

struct TfsfSurfD {
    int comp, src;
    double pf;
    int o[3], a1, n1, a2, n2, incd0, s1, s2;
    long long start;  // first flat point of this surface in its launch
};

__device__ __forceinline__ bool tfsf_in(const TfsfSurfD& q, const int* x, int& i1, int& i2) {
    const int a3 = 3 - q.a1 - q.a2;
    i1 = x[q.a1] - q.o[q.a1];
    i2 = x[q.a2] - q.o[q.a2];
    return x[a3] == q.o[a3] && i1 >= 0 && i1 < q.n1 && i2 >= 0 && i2 < q.n2;
}

// U += pf * Re(line[src][incd0 + i1 s1 + i2 s2]) over the surfaces of one
// family (addIncdFields, parallelTFSF.cpp:78-84), for the 256 points from b0
// on (t: which of them).  Each surface starts on a multiple of 256, so the
// surface and the table reads are uniform; the points run along x where the
// surface contains x (coalesced).
// A cell on several surfaces of its component (an edge of the box) takes all
// their adds in order from the thread of its first surface, so the sums keep
// the reference's order.
template <typename T>
struct TfsfFields {
    T* F[6];
};
template <typename T>
__device__ __forceinline__ void tfsf_add(const TfsfSurfD* __restrict__ sf, int ns, long long b0, int t, const TfsfFields<T>& f,
                                         const double2* __restrict__ line, int len, int nx, int ny) {
    int s = 0;
    while (s + 1 < ns && sf[s + 1].start <= b0) ++s;
    const TfsfSurfD& q = sf[s];
    const long long pnt = b0 + t - q.start;
    const long long np = static_cast<long long>(q.n1) * q.n2;
    if (pnt >= np) return;
    int x[3] = {q.o[0], q.o[1], q.o[2]};
    // x fastest where the surface has rows along x
    const int fast = q.a2 == 0 ? q.a2 : q.a1, slow = q.a2 == 0 ? q.a1 : q.a2;
    const unsigned n = static_cast<unsigned>(q.a2 == 0 ? q.n2 : q.n1), up = static_cast<unsigned>(pnt), row = up / n;
    x[fast] += static_cast<int>(up - row * n);
    x[slow] += static_cast<int>(row);
    int i1, i2;
    for (int k = 0; k < s; ++k)
        if (sf[k].comp == q.comp && tfsf_in(sf[k], x, i1, i2)) return;
    T* F = f.F[q.comp];
    const long long idx = x[0] + static_cast<long long>(nx) * (x[1] + static_cast<long long>(ny) * x[2]);
    T v = F[idx];
    for (int k = s; k < ns; ++k) {
        const TfsfSurfD& r = sf[k];
        if (r.comp != q.comp || !tfsf_in(r, x, i1, i2)) continue;
        v += static_cast<T>(r.pf * line[r.src * len + r.incd0 + i1 * r.s1 + i2 * r.s2].x);
    }
    F[idx] = v;
}

template <typename T>
__global__ void __launch_bounds__(256) k_tfsf_add(const TfsfSurfD* __restrict__ sf, int ns, long long total, TfsfFields<T> f,
                                                  const double2* __restrict__ line, int len, int nx, int ny) {
    const long long b0 = blockIdx.x * 256LL;
    if (b0 < total) tfsf_add<T>(sf, ns, b0, threadIdx.x, f, line, len, nx, ny);
}

// Block 0: the lines; the others: the H adds, which read the lines as the step
// before left them, 1024 points a block.
template <typename T, bool LDS>
__global__ void __launch_bounds__(1024) k_tfsf_step(TfsfLineArgs ta, const TfsfSurfD* __restrict__ sf, int ns, long long total,
                                                    TfsfFields<T> f, int nx, int ny, const int* stepp, int stepv) {
    extern __shared__ __align__(16) unsigned char tfsf_lds[];
    const int step = step_now(stepp, stepv);
    if (blockIdx.x == 0) {
        tfsf_lines<LDS>(ta, tfsf_lds, step);
        return;
    }
    const long long b0 = ((blockIdx.x - 1) * 4LL + (threadIdx.x >> 8)) * 256;
    if (b0 < total) tfsf_add<T>(sf, ns, b0, threadIdx.x & 255, f, ta.snap[(step + 1) & 1], ta.len[0], nx, ny);
}

// Per-cell soft-source adds (oblique sources, parallelSourceOblique.cpp:17-23),
// between the H and the E update. The host sorts the cells by (component,
// point), keeping the sources' order within a point: the first thread of a
// run of equal keys adds the whole run, in order, so no two threads write
// one point.
template <typename T>
__global__ void __launch_bounds__(256) k_cell_src(const int* __restrict__ comp, const long long* __restrict__ idx,
                                                  const int* __restrict__ col, const T* __restrict__ amp, int n, int ncol,
                                                  const int* stepp, int stepv, T* F0, T* F1, T* F2, T* F3, T* F4, T* F5) {
    const int k = blockIdx.x * 256 + threadIdx.x;
    if (k >= n) return;
    const int c = comp[k];
    const long long i = idx[k];
    if (k > 0 && comp[k - 1] == c && idx[k - 1] == i) return;
    const long long row = static_cast<long long>(step_now(stepp, stepv)) * ncol;
    T* const Fs[6] = {F0, F1, F2, F3, F4, F5};
    T v = Fs[c][i];
    for (int j = k; j < n && comp[j] == c && idx[j] == i; ++j) v += amp[row + col[j]];
    Fs[c][i] = v;
}

// ------------------------------------------------------- batched launches ----
// One launch per kernel class covers many simulations (the serving loop's
// batches): slot k of a device-side descriptor table holds simulation k's
// parameter blocks, and a block finds its slot from the per-launch prefix
// table begin[] (blocks [begin[k], begin[k+1]) belong to slot k, each range
// starting on a multiple of 8 so that the XCD-aware block numbering of the
// sweeps holds within it).  The sweeps are the ones of the single
// simulation's launches, so each simulation's arithmetic is unchanged.
// Batched steps read the step number from each simulation's device counter
// (as captured graphs do), so the table is the same every step of a given
// counter parity.
template <typename T>
struct BatchSlot {
    StepArgs<T> a;
    SampleArgs<T> s;
    Box3 b;
    SlabMap m;
    int nib, nsbp, ade_bpc, fma;
    int nm[3];
    int nblk[5];  // blocks of each phase launch (unpadded)
};

enum { kPhH = 0, kPhHs = 1, kPhE = 2, kPhEs = 3, kPhS = 4, kPhases = 5 };

__device__ __forceinline__ int batch_slot(const int* __restrict__ begin, int n, int b) {
    int lo = 0, hi = n;  // begin[lo] <= b < begin[hi]
    while (hi - lo > 1) {
        const int mid = (lo + hi) >> 1;
        if (begin[mid] <= b) lo = mid;
        else hi = mid;
    }
    return lo;
}

template <typename T, int W>
__global__ void __launch_bounds__(256) k_bh2v(const BatchSlot<T>* __restrict__ sl, const int* __restrict__ begin, int n) {
    const int k = batch_slot(begin, n, blockIdx.x);
    const int bx = blockIdx.x - begin[k];
    const BatchSlot<T>& q = sl[k];
    if (bx >= q.nblk[kPhH]) return;
    h2v_sweep<T, W, true>(q.a, bx, q.nblk[kPhH]);
    advance_counter_at(q.a, bx);
}

template <typename T, int W>
__global__ void __launch_bounds__(256) k_be2v(const BatchSlot<T>* __restrict__ sl, const int* __restrict__ begin, int n) {
    __shared__ MatLds<T> mt[3][CHIML_MAX_MAT];
    const int k = batch_slot(begin, n, blockIdx.x);
    const int bx = blockIdx.x - begin[k];
    const BatchSlot<T>& q = sl[k];
    if (bx >= q.nblk[kPhE]) return;
    const int nm[3] = {0, 0, q.nm[2]};
    load_mat(q.a, mt, nm);
    if (q.fma) e2v_sweep<T, W, true, false, true>(q.a, q.s, mt, bx, q.nblk[kPhE]);
    else e2v_sweep<T, W, true, false, false>(q.a, q.s, mt, bx, q.nblk[kPhE]);
}

template <typename T, int W, bool NT>
__global__ void __launch_bounds__(256) k_bh3_all(const BatchSlot<T>* __restrict__ sl, const int* __restrict__ begin, int n) {
    const int k = batch_slot(begin, n, blockIdx.x);
    const int bx = blockIdx.x - begin[k];
    const BatchSlot<T>& q = sl[k];
    if (bx >= q.nblk[kPhH]) return;
    if (q.fma) h3_all_sweep<T, W, true, true, NT>(q.a, q.b, q.m, q.nib, q.nsbp, q.ade_bpc, bx);
    else h3_all_sweep<T, W, true, false, NT>(q.a, q.b, q.m, q.nib, q.nsbp, q.ade_bpc, bx);
    advance_counter_at(q.a, bx);
}

template <typename T, int W, bool NT>
__global__ void __launch_bounds__(256) k_be3_all(const BatchSlot<T>* __restrict__ sl, const int* __restrict__ begin, int n) {
    __shared__ MatLds<T> mt[3][CHIML_MAX_MAT];
    const int k = batch_slot(begin, n, blockIdx.x);
    const int bx = blockIdx.x - begin[k];
    const BatchSlot<T>& q = sl[k];
    if (bx >= q.nblk[kPhE]) return;
    load_mat(q.a, mt, q.nm);
    if (q.fma) e3_all_sweep<T, W, true, true, NT>(q.a, mt, q.b, q.m, q.nib, q.nsbp, bx);
    else e3_all_sweep<T, W, true, false, NT>(q.a, mt, q.b, q.m, q.nib, q.nsbp, bx);
}

template <typename T, int W, bool NT>
__global__ void __launch_bounds__(256) k_bh3_int(const BatchSlot<T>* __restrict__ sl, const int* __restrict__ begin, int n) {
    const int k = batch_slot(begin, n, blockIdx.x);
    const int bx = blockIdx.x - begin[k];
    const BatchSlot<T>& q = sl[k];
    if (bx >= q.nblk[kPhH]) return;
    h3_int_sweep<T, W, true, NT>(q.a, q.b, q.nib, q.ade_bpc, bx);
    advance_counter_at(q.a, bx);
}

template <typename T, int W, bool NT>
__global__ void __launch_bounds__(256) k_bh3_slab(const BatchSlot<T>* __restrict__ sl, const int* __restrict__ begin, int n) {
    const int k = batch_slot(begin, n, blockIdx.x);
    const int bx = blockIdx.x - begin[k];
    const BatchSlot<T>& q = sl[k];
    if (bx >= q.nblk[kPhHs]) return;
    h3_slab_sweep<T, W, true, NT>(q.a, q.m, bx, q.nblk[kPhHs]);
}

template <typename T, int W, bool NT>
__global__ void __launch_bounds__(256) k_be3_int(const BatchSlot<T>* __restrict__ sl, const int* __restrict__ begin, int n) {
    __shared__ MatLds<T> mt[3][CHIML_MAX_MAT];
    const int k = batch_slot(begin, n, blockIdx.x);
    const int bx = blockIdx.x - begin[k];
    const BatchSlot<T>& q = sl[k];
    if (bx >= q.nblk[kPhE]) return;
    load_mat(q.a, mt, q.nm);
    e3_int_sweep<T, W, true, NT>(q.a, mt, q.b, bx, q.nblk[kPhE]);
}

template <typename T, int W, bool NT>
__global__ void __launch_bounds__(256) k_be3_slab(const BatchSlot<T>* __restrict__ sl, const int* __restrict__ begin, int n) {
    __shared__ MatLds<T> mt[3][CHIML_MAX_MAT];
    const int k = batch_slot(begin, n, blockIdx.x);
    const int bx = blockIdx.x - begin[k];
    const BatchSlot<T>& q = sl[k];
    if (bx >= q.nblk[kPhEs]) return;
    load_mat(q.a, mt, q.nm);
    e3_slab_sweep<T, W, true, NT>(q.a, mt, q.m, bx, q.nblk[kPhEs]);
}

template <typename T>
__global__ void __launch_bounds__(256) k_bsample(const BatchSlot<T>* __restrict__ sl, const int* __restrict__ begin, int n) {
    const int k = batch_slot(begin, n, blockIdx.x);
    const int bx = blockIdx.x - begin[k];
    const BatchSlot<T>& q = sl[k];
    if (bx >= q.nblk[kPhS]) return;
    sample_at<T>(q.s, bx * blockDim.x + threadIdx.x);
}


__global__ void k_zero(double* p, long long n) {
    long long i = blockIdx.x * static_cast<long long>(blockDim.x) + threadIdx.x;
    if (i < n) p[i] = 0.0;
}

}  // namespace

// -------------------------------------------------------------- context -----
struct QeHost {
    QeDev dev;
    std::vector<std::unique_ptr<DevBuf>> bufs;
    int nblocks = 0;
    int N = 0;
    int npop_all = 0;             // population detectors; the density kernel sums the first 4
    int nb2 = 0;                  // blocks per extra population in k_ml_pop_gather
    double2* partial2 = nullptr;  // [npop_all - 4][nb2]
};

struct chiml_dev {
    std::string err;
    hipStream_t stream = nullptr;
    hipEvent_t ev = nullptr;  // joins this context's stream with a batch's stream
    int device = 0;
    int prec = 64;
    int nx = 0, ny = 0, nz = 0, dim = 3;
    int px = 0;         // cells per stored x row (StepArgs::px)
    bool vec = false;   // rows hold whole W-cell groups and the x psi regions are whole groups: the W-cell kernels apply
    int nsteps = 0, steps_done = 0;
    std::vector<std::unique_ptr<DevBuf>> bufs;
    DevBuf step_ctr;
    // parameter blocks for both precisions (only one used)
    StepArgs<float> a32{};
    StepArgs<double> a64{};
    SampleArgs<float> s32{};
    SampleArgs<double> s64{};
    bool hmap = false, has_src = false;
    int nmat[3] = {1, 1, 1};
    int enq_step = 0;    // step counter value after the step being enqueued
    int graph_steps = 0;  // > 0: replay captured graphs of this many steps (even)
    bool capturing = false;  // do_steps is being captured into a graph
    bool device_flush = false;  // launch the DFT flush every step; it decides on the device
    hipGraphExec_t gexec[2] = {nullptr, nullptr};  // captured graphs, by the tile buffer set they start on (0: no tiles)
    int graph_parity[2] = {0, 0};  // and the counter slot that a graph of sweeps starts on
    bool graph_tiles = false;      // the graphs are of tile launches
    bool split = false;  // 3D interior + CPML-slab kernels
    bool rows = false;   // split: whole-row interior, one launch per field
    double step_bytes = 0;     // fields and emitter state
    bool stream_hint = false;  // split: once-touched words go past the caches (streams_past_caches)
    bool cellwise = false;  // stepped alone with one thread per cell (GridLayout::cellwise)
    bool fma_curl = false;  // rows or x CPML no whole groups: curls as the per-cell kernels round them (curl_of)
    bool fused = false;  // 3D: one fused H + E launch per step on ping-pong buffers
    FuseMap fmap{};
    size_t fused_lds = 0;  // dynamic LDS of the fused launch (bytes)
    void* fbuf[2][6] = {};      // fused: the two field buffers (fbuf[0] is the build's F)
    void* fpsi[2][3][3] = {};   // fused: the two psi buffers of each H component and axis
    bool vec2d = false;  // 2D TMz W-cell group kernels
    // 2D: k_tile2 launches of up to kTileSteps steps on two sets of buffers;
    // tile_cur is the set (and the step counter's slot) that holds the present
    bool tile = false;
    int tile_shape = 0, tile_cur = 0, tile_nx = 0, tile_ny = 0;
    size_t tile_lds = 0;  // dynamic LDS (pole states)
    int tile_npole = 0;
    void* tbuf[2][9] = {};  // Ez, Hx, Hy, psi of Hx (y), Hy (x), Ez (x), Ez (y), P, J
    const int* tile_det_ofs = nullptr;
    const TileDet* tile_det = nullptr;
    int tile_nset = 0;
    bool fuse_sample = false;  // 2D: the E kernel takes the point detectors (no DFT, few single-cell points)
    bool det_single_field = true;  // every point detector reads one field (two cells) per point
    long long ade_groups = 0;  // largest pole-box group count over the E components (split path)
    Box3 ibox{};
    SlabMap slab{};
    int ndet = 0, totpts = 0, ndft = 0;
    std::vector<int> det_npts, det_cap, det_interval;
    std::vector<long long> det_out_off;
    double* det_out = nullptr;
    struct DftGroup {  // accumulators F[f][cell] of one DFT group, device memory
        int n = 0, nfreq = 0, interval = 1;
        double* F = nullptr;
        double* tmp = nullptr;
        void* stage = nullptr;
        const double* phasor = nullptr;
    };
    std::vector<DftGroup> dgs;
    struct FluxPlan {
        FluxPlanDev dev{};
        double2* partial = nullptr;  // [nfreq][blocks]
        int blocks = 0;
    };
    std::vector<FluxPlan> flux_plans;
    std::vector<QeHost> qes;
    const QeHost* finish_with_sample = nullptr;  // the group whose population finish rides on this step's sample launch
    struct TfsfHost {  // one TFSF surface: its lines and its surface table (H adds, then E adds)
        TfsfLineArgs line{};
        TfsfSurfD* surf = nullptr;
        int nsh = 0, nse = 0;
        long long toth = 0, tote = 0;
    };
    std::vector<TfsfHost> tfsf;
    struct CellSrc {  // per-cell source adds, sorted by (component, point)
        int n = 0, ncol = 0;
        int* comp = nullptr;
        long long* idx = nullptr;
        int* col = nullptr;
        void* amp = nullptr;  // T[nsteps][ncol]
    } cells;
    double2* incd_rec = nullptr;  // [6][nrec] incident records (E_incd_, H_incd_)
    long long nrec = 0;
    size_t footprint = 0;
    bool profile = false;
    std::string profile_only;  // non-empty: time only launches of this kernel
    std::map<std::string, std::pair<double, int>> prof;
    struct Span {  // an event pair around a launch, or around the launches of n steps
        std::string name;
        hipEvent_t e0, e1;
        int n;
    };
    std::vector<Span> pending;

    template <typename T>
    T* upload(const T* src, size_t n) {
        bufs.emplace_back(new DevBuf);
        bufs.back()->alloc(n * sizeof(T), stream, src == nullptr);
        footprint += n * sizeof(T);
        // a blocking copy: complete before any later launch on the stream
        if (src && n) HIP_TRY(hipMemcpy(bufs.back()->p, src, n * sizeof(T), hipMemcpyHostToDevice));
        return bufs.back()->as<T>();
    }
    template <typename T>
    T* zeros(size_t n) { return upload<T>(nullptr, n); }
};

// Does the emitter group keep rho Hermitian?  True when every member's H0 and
// the three dipole matrices are Hermitian and the Lindblad operator maps
// Hermitian to Hermitian: G[(a,b),(c,d)] = G[(b,a),(d,c)] for its real
// entries (column-major flat indices).  The density kernel then stores the
// upper triangle only.
static bool hermitian_preserving(const chiml_qe_t& qi) {
    const int N = qi.nlevel, S = N * N;
    auto herm = [&](const double* m) {
        for (int i = 0; i < N; ++i)
            for (int j = 0; j < N; ++j) {
                const double* a = m + 2 * (i + j * N);
                const double* b = m + 2 * (j + i * N);
                if (a[0] != b[0] || a[1] != -b[1]) return false;
            }
        return true;
    };
    for (int mm = 0; mm < qi.nmembers; ++mm)
        if (!herm(qi.h0 + 2 * static_cast<size_t>(mm) * S)) return false;
    for (int c = 0; c < 3; ++c)
        if (!herm(qi.mu + 2 * static_cast<size_t>(c) * S)) return false;
    std::map<std::pair<int, int>, double> g;
    for (int k = 0; k < qi.ngam; ++k) g[{qi.gam_row[k], qi.gam_col[k]}] += qi.gam_val[k];
    auto mirror = [&](int f) { return f / N + (f % N) * N; };
    for (const auto& kv : g) {
        auto it = g.find({mirror(kv.first.first), mirror(kv.first.second)});
        const double v = it == g.end() ? 0.0 : it->second;
        if (v != kv.second) return false;
    }
    return true;
}

bool chiml_qe_packed(const chiml_qe_t& qi) { return hermitian_preserving(qi) && std::getenv("CHIML_ML_UNPACKED") == nullptr; }

namespace {

template <typename T>
T* upload_cast(chiml_dev* c, const double* src, size_t n) {
    std::vector<T> tmp(n);
    for (size_t i = 0; i < n; ++i) tmp[i] = static_cast<T>(src[i]);
    return c->upload<T>(tmp.data(), n);
}

constexpr size_t kTfsfMaxLds = 160 * 1024 - 1024;  // dynamic LDS of k_tfsf_step: a gfx950 workgroup's 160 KB less its static parameter copy

// Per-cell source table: components, points and columns checked on the host.
template <typename T>
void build_cells(chiml_dev* c, const chiml_problem_t* p) {
    const int n = p->ncell_src;
    if (n < 0 || p->ncell_col < 0 || (n > 0 && (!p->cell_comp || !p->cell_xyz || !p->cell_col || !p->cell_amp || p->ncell_col == 0)))
        throw std::runtime_error("invalid per-cell source table");
    if (n == 0) return;
    const bool is3 = p->nz > 1;
    std::vector<std::pair<long long, int>> key(n);  // (component * points + point, position in the list)
    const long long npt = static_cast<long long>(c->px) * p->ny * p->nz;
    for (int k = 0; k < n; ++k) {
        const int cc = p->cell_comp[k], x = p->cell_xyz[3 * k], y = p->cell_xyz[3 * k + 1], z = p->cell_xyz[3 * k + 2];
        if (cc < 0 || cc > 5 || (!is3 && cc != 2 && cc != 3 && cc != 4)) throw std::runtime_error("per-cell source on a missing component");
        if (x < 0 || x >= p->nx || y < 0 || y >= p->ny || z < 0 || z >= p->nz) throw std::runtime_error("per-cell source outside the grid");
        if (p->cell_col[k] < 0 || p->cell_col[k] >= p->ncell_col) throw std::runtime_error("per-cell source column out of range");
        key[k] = {cc * npt + x + static_cast<long long>(c->px) * (y + static_cast<long long>(p->ny) * z), k};
    }
    std::stable_sort(key.begin(), key.end(), [](const auto& a, const auto& b) { return a.first < b.first; });
    std::vector<int> comp(n), col(n);
    std::vector<long long> idx(n);
    for (int k = 0; k < n; ++k) {
        const int o = key[k].second;
        comp[k] = static_cast<int>(key[k].first / npt);
        idx[k] = key[k].first % npt;
        col[k] = p->cell_col[o];
    }
    c->cells.n = n;
    c->cells.ncol = p->ncell_col;
    c->cells.comp = c->upload<int>(comp.data(), n);
    c->cells.idx = c->upload<long long>(idx.data(), n);
    c->cells.col = c->upload<int>(col.data(), n);
    c->cells.amp = upload_cast<T>(c, p->cell_amp, static_cast<size_t>(p->nsteps) * p->ncell_col);
}

// TFSF tables: every index a kernel will form is checked here, on the host.
template <typename T>
void build_tfsf(chiml_dev* c, const chiml_problem_t* p, const StepArgs<T>& a) {
    if (p->ntfsf < 0 || (p->ntfsf > 0 && !p->tfsf)) throw std::runtime_error("invalid TFSF table");
    if (p->ntfsf == 0) return;
    c->nrec = 2LL * (p->nsteps + 1) + 2;
    c->incd_rec = reinterpret_cast<double2*>(c->zeros<double>(2 * 6 * static_cast<size_t>(c->nrec)));
    HIP_TRY(hipFuncSetAttribute(reinterpret_cast<const void*>(k_tfsf_step<T, true>), hipFuncAttributeMaxDynamicSharedMemorySize,
                                static_cast<int>(kTfsfMaxLds)));
    auto need = [](bool ok, const char* what) {
        if (!ok) throw std::runtime_error(std::string("TFSF table: ") + what);
    };
    for (int k = 0; k < p->ntfsf; ++k) {
        const chiml_tfsf_t& tf = p->tfsf[k];
        chiml_dev::TfsfHost h;
        TfsfLineArgs& t = h.line;
        t.len[0] = tf.len0;
        t.len[1] = tf.len1;
        need(tf.len0 > 0 && tf.len1 > 0 && tf.margin >= 0 && tf.psi_n >= 0 && tf.pulse_n >= 0, "sizes");
        t.margin = tf.margin;
        t.pulse_at = tf.pulse_at;
        t.pulse_n = tf.pulse_n;
        t.psi_n = tf.psi_n;
        t.rec_idx = tf.rec_idx;
        need(tf.pulse_n == 0 || tf.amp, "pulse table");
        need(tf.psi_n == 0 || tf.seg_coef, "CPML coefficients");
        for (int cc = 0; cc < 6; ++cc) {
            t.present[cc] = tf.present[cc] ? 1 : 0;
            t.rec_off[cc] = tf.rec_off[cc];
            t.nterm[cc] = tf.nterm[cc];
            t.nseg[cc] = tf.nseg[cc];
            need(tf.nterm[cc] >= 0 && tf.nterm[cc] <= 2 && tf.nseg[cc] >= 0 && tf.nseg[cc] <= 4, "term or segment count");
            if (!t.present[cc]) {
                t.nterm[cc] = t.nseg[cc] = 0;
                continue;
            }
            for (int s = 0; s < 2; ++s) {
                const int len = t.len[s];
                need(tf.pulse_at >= 0 && tf.pulse_at + tf.pulse_n <= len, "pulse window");
                need(tf.rec_idx < tf.len1 && tf.rec_idx - tf.rec_off[cc] >= 0 && tf.rec_off[cc] >= 0, "record point");
                for (int j = 0; j < tf.nterm[cc]; ++j) {
                    const int lo = std::min(tf.term_pos[cc][j], tf.term_neg[cc][j]), hi = std::max(tf.term_pos[cc][j], tf.term_neg[cc][j]);
                    need(tf.term_src[cc][j] >= 0 && tf.term_src[cc][j] < 6 && tf.present[tf.term_src[cc][j]], "term line");
                    need(len - 2 * tf.margin <= 0 || (tf.margin + lo >= 0 && len - tf.margin - 1 + hi < len), "term offsets");
                }
                for (int g = 0; g < tf.nseg[cc]; ++g) {
                    const int gl = tf.seg_high[cc][g] ? len - 1 - tf.psi_n - tf.margin : tf.margin;
                    need(tf.seg_src[cc][g] >= 0 && tf.seg_src[cc][g] < 6 && tf.present[tf.seg_src[cc][g]], "segment line");
                    need(gl >= 0 && gl + tf.psi_n <= len, "segment position");
                    for (int off : {tf.seg_off1[cc][g], tf.seg_off2[cc][g]})
                        need(gl + off >= 0 && gl + off + tf.psi_n <= len, "segment offsets");
                }
            }
            for (int j = 0; j < 2; ++j) {
                t.tsrc[cc][j] = tf.term_src[cc][j];
                t.tpos[cc][j] = tf.term_pos[cc][j];
                t.tneg[cc][j] = tf.term_neg[cc][j];
                t.tcoef[cc][j] = tf.term_coef[cc][j];
            }
            for (int g = 0; g < 4; ++g) {
                t.ssrc[cc][g] = tf.seg_src[cc][g];
                t.shigh[cc][g] = tf.seg_high[cc][g];
                t.soff1[cc][g] = tf.seg_off1[cc][g];
                t.soff2[cc][g] = tf.seg_off2[cc][g];
                t.sdb[cc][g] = tf.seg_db[cc][g];
            }
        }
        t.line[0] = reinterpret_cast<double2*>(c->zeros<double>(2 * 6 * static_cast<size_t>(tf.len0)));
        t.line[1] = reinterpret_cast<double2*>(c->zeros<double>(2 * 6 * static_cast<size_t>(tf.len1)));
        t.psi = reinterpret_cast<double2*>(c->zeros<double>(2 * 2 * 6 * 4 * static_cast<size_t>(std::max(tf.psi_n, 1))));
        t.scoef = c->upload<double>(tf.seg_coef, 6 * 4 * static_cast<size_t>(tf.psi_n) * 3);
        t.amp = reinterpret_cast<const double2*>(c->upload<double>(tf.amp, 2 * static_cast<size_t>(p->nsteps) * 6 * tf.pulse_n));
        for (double2*& q : t.snap) q = reinterpret_cast<double2*>(c->zeros<double>(2 * 6 * static_cast<size_t>(tf.len0)));
        t.rec = c->incd_rec;
        t.nrec = c->nrec;
        // surfaces: H adds first, then E adds, each with flat point offsets
        need(tf.nsurf_h >= 0 && tf.nsurf_e >= 0 && (tf.nsurf_h + tf.nsurf_e == 0 || tf.surf), "surface table");
        std::vector<TfsfSurfD> sv;
        long long acc = 0;
        const int nn[3] = {p->nx, p->ny, p->nz};
        for (int i = 0; i < tf.nsurf_h + tf.nsurf_e; ++i) {
            if (i == tf.nsurf_h) {
                h.toth = acc;
                acc = 0;
            }
            const chiml_tfsf_surface_t& u = tf.surf[i];
            const bool hfam = i < tf.nsurf_h;
            need(u.comp >= (hfam ? 3 : 0) && u.comp < (hfam ? 6 : 3) && a.F[u.comp] != nullptr, "surface component");
            need(u.src >= 0 && u.src < 6 && tf.present[u.src], "surface line");
            need(u.a1 >= 0 && u.a1 < 3 && u.a2 >= 0 && u.a2 < 3 && u.a1 != u.a2 && u.n1 >= 0 && u.n2 >= 0, "surface axes");
            TfsfSurfD d{};
            d.comp = u.comp;
            d.src = u.src;
            d.pf = u.pf;
            d.o[0] = u.x0;
            d.o[1] = u.y0;
            d.o[2] = u.z0;
            d.a1 = u.a1;
            d.n1 = u.n1;
            d.a2 = u.a2;
            d.n2 = u.n2;
            d.incd0 = u.incd0;
            d.s1 = u.incd_s1;
            d.s2 = u.incd_s2;
            d.start = acc;  // a multiple of the add kernel's block size
            if (u.n1 > 0 && u.n2 > 0) {
                for (int ax = 0; ax < 3; ++ax) {
                    const int ext = ax == u.a1 ? u.n1 - 1 : (ax == u.a2 ? u.n2 - 1 : 0);
                    need(d.o[ax] >= 0 && d.o[ax] + ext < nn[ax], "surface cells");
                }
                for (int e1 : {0, u.n1 - 1})
                    for (int e2 : {0, u.n2 - 1}) {
                        const long long li = u.incd0 + static_cast<long long>(e1) * u.incd_s1 + static_cast<long long>(e2) * u.incd_s2;
                        need(li >= 0 && li < tf.len0, "surface line index");
                    }
            }
            acc += (static_cast<long long>(u.n1) * u.n2 + 255) / 256 * 256;
            sv.push_back(d);
        }
        if (tf.nsurf_e == 0) h.toth = acc;
        else h.tote = acc;
        h.nsh = tf.nsurf_h;
        h.nse = tf.nsurf_e;
        if (!sv.empty()) {
            h.surf = c->upload<TfsfSurfD>(sv.data(), sv.size());
        }
        c->tfsf.push_back(h);
    }
}

template <typename T>
void build(chiml_dev* c, const chiml_problem_t* p, StepArgs<T>& a, SampleArgs<T>& s) {
    const int nx = p->nx, ny = p->ny, nz = p->nz;
    a.nx = nx;
    a.ny = ny;
    a.nz = nz;
    {
        int lo = p->pml_T[0], hi = nx - p->pml_T[0];
        bool hmap = false;
        for (int comp = 0; comp < 6; ++comp) {
            if (p->pml_b[comp][0]) {
                lo = std::max(lo, p->psi_lo[comp][0]);
                hi = std::min(hi, p->psi_hi0[comp][0]);
            }
            if (comp < 3 && (nz > 1 || comp < 2) && p->mat_h[comp]) hmap = true;
        }
        const GridLayout gl = grid_layout(nx, ny, nz, p->pml_T, lo, hi, sizeof(T) == 4, hmap);
        c->vec = gl.vec;
        c->px = gl.px;
        c->split = gl.split;
        c->rows = gl.rows;
        c->cellwise = gl.cellwise && (nz > 1 || p->nsrc > 0);  // 2D groups without a search for sources keep up
        c->fma_curl = nx % gl.W != 0 || p->pml_T[0] % gl.W != 0;
    }
    const int px = c->px, rw = c->vec ? static_cast<int>(16 / sizeof(T)) : 1;
    a.px = px;
    const size_t N = static_cast<size_t>(px) * ny * nz;
    // a grid point's place in the padded rows (-1, the zero ghost, stays)
    auto padded = [&](long long i) { return i < 0 ? i : i / nx * px + i % nx; };
    auto padded_cells = [&](const long long* src, size_t n) {
        std::vector<long long> r(n);
        for (size_t i = 0; i < n; ++i) r[i] = padded(src[i]);
        return r;
    };
    // uploads a per-point array into padded rows
    auto upload_rows = [&](auto* src, auto fill) {
        using V = std::remove_const_t<std::remove_pointer_t<decltype(src)>>;
        if (px == nx) return c->upload<V>(src, N);
        std::vector<V> r(N, static_cast<V>(fill));
        const size_t nr = static_cast<size_t>(ny) * nz;
        for (size_t y = 0; y < nr; ++y) std::copy(src + y * nx, src + (y + 1) * nx, r.begin() + y * px);
        return c->upload<V>(r.data(), N);
    };
    for (int k = 0; k < 3; ++k) {
        a.inv_d[k] = static_cast<T>(1.0 / p->d[k]);
        a.Tp[k] = p->pml_T[k];
    }
    const bool is3 = nz > 1;
    {  // the present components in one allocation, x + px (y + ny z) each, in component order
        int nf = 0;
        for (int k = 0; k < 6; ++k) nf += (is3 || k == 2 || k == 3 || k == 4) ? 1 : 0;
        T* base = c->zeros<T>(N * nf);
        for (int k = 0; k < 6; ++k) {
            bool present = is3 || k == 2 || k == 3 || k == 4;
            a.F[k] = present ? base : nullptr;
            if (present) base += N;
        }
    }
    for (int k = 0; k < 3; ++k) {
        bool present = is3 || k == 2;
        a.mat_e[k] = (present && p->mat_e[k]) ? upload_rows(p->mat_e[k], 0) : nullptr;
        int nm = present ? p->nmat_e[k] : 1;
        if (present && (nm <= 0 || nm > CHIML_MAX_MAT)) throw std::runtime_error("material table size out of range");
        if (present) {
            a.ce[k] = upload_cast<T>(c, p->mat_e_ce[k], nm);
            a.inveps[k] = upload_cast<T>(c, p->mat_e_inveps[k], nm);
            a.flags[k] = c->upload<int>(p->mat_e_flags[k], nm);
            a.poleset[k] = c->upload<int>(p->mat_e_poleset[k], nm);
            c->nmat[k] = nm;
        }
        bool hpresent = is3 || k < 2;
        a.mat_h[k] = (hpresent && p->mat_h[k]) ? upload_rows(p->mat_h[k], 0) : nullptr;
        if (hpresent) {
            int nh = p->nmat_h[k] > 0 ? p->nmat_h[k] : 1;
            a.ch[k] = upload_cast<T>(c, p->mat_h_ch[k], nh);
            if (a.mat_h[k]) c->hmap = true;
        }
    }
    int nps = p->npoleset > 0 ? p->npoleset : 1;
    std::vector<int> pc(nps, 0);
    std::vector<double> pco(static_cast<size_t>(nps) * CHIML_MAX_POLES * 3, 0.0);
    for (int k = 0; k < p->npoleset; ++k) {
        pc[k] = p->pole_count[k];
        if (pc[k] > CHIML_MAX_POLES) throw std::runtime_error("too many poles");
        for (int j = 0; j < CHIML_MAX_POLES * 3; ++j) pco[k * CHIML_MAX_POLES * 3 + j] = p->pole_coef[k * CHIML_MAX_POLES * 3 + j];
    }
    a.pole_count = c->upload<int>(pc.data(), nps);
    a.pole_coef = upload_cast<T>(c, pco.data(), pco.size());
    int maxp = 0;
    for (int k = 0; k < p->npoleset; ++k) maxp = std::max(maxp, pc[k]);
    for (int k = 0; k < 3; ++k) {
        for (int j = 0; j < 6; ++j) a.box[k][j] = p->disp_box[k][j];
        // pole-state storage x-range aligned to 4 cells, so that a W-cell group
        // of the vector kernels is one aligned 16-byte access (the extra
        // storage belongs to cells without poles and is never changed)
        if (a.box[k][1] > a.box[k][0]) {
            a.box[k][0] = a.box[k][0] / 4 * 4;
            a.box[k][1] = std::min((a.box[k][1] + 3) / 4 * 4, px);
        }
        long long bn = 0;  // cells of the (aligned) pole-state box
        if (a.box[k][1] > a.box[k][0] && a.box[k][3] > a.box[k][2] && a.box[k][5] > a.box[k][4])
            bn = static_cast<long long>(a.box[k][1] - a.box[k][0]) * (a.box[k][3] - a.box[k][2]) * (a.box[k][5] - a.box[k][4]);
        a.boxn[k] = bn;
        a.P[k] = (bn > 0 && maxp > 0) ? c->zeros<T>(bn * maxp) : nullptr;
        a.J[k] = (bn > 0 && maxp > 0) ? c->zeros<T>(bn * maxp) : nullptr;
        a.jsum[k] = (bn > 0 && maxp > 0 && nz > 1) ? c->zeros<T>(bn) : nullptr;
    }
    const int nn[3] = {nx, ny, nz};
    for (int comp = 0; comp < 6; ++comp) {
        PmlDev<T>& pm = a.pml[comp];
        for (int ax = 0; ax < 3; ++ax) {
            pm.b[ax] = pm.cd[ax] = pm.kinv[ax] = nullptr;
            pm.psi[ax] = nullptr;
            if (!p->pml_b[comp][ax]) {
                pm.lo[ax] = 0;
                pm.hi0[ax] = pm.hi1[ax] = nn[ax];
                pm.S[ax] = 0;
                continue;
            }
            // Widen the psi region to whole slabs [0, T) and [n - T, n): the
            // added positions carry b = 0, c/d = 0, 1/kappa = 1, for which the
            // CPML term equals the plain dV/d bit for bit and psi stays 0.
            // Along x also to whole W-cell groups and over the row padding.
            const int n = nn[ax], T0 = p->pml_T[ax], ns = ax == 0 ? px : n, w = ax == 0 ? rw : 1;
            const int lo = p->psi_lo[comp][ax], hi0 = p->psi_hi0[comp][ax], hi1 = p->psi_hi1[comp][ax];
            pm.lo[ax] = round_up(std::max(lo, T0), w);
            pm.hi0[ax] = round_down(std::min(hi0, n - T0), w);
            pm.hi1[ax] = std::max(hi1, ns);
            pm.S[ax] = pm.lo[ax] + (pm.hi1[ax] - pm.hi0[ax]);
            std::vector<double> bb(p->pml_b[comp][ax], p->pml_b[comp][ax] + n), cc(p->pml_cd[comp][ax], p->pml_cd[comp][ax] + n),
                kk(p->pml_kinv[comp][ax], p->pml_kinv[comp][ax] + n);
            bb.resize(ns, 0.0);
            cc.resize(ns, 0.0);
            kk.resize(ns, 1.0);
            auto ident = [&](int q0, int q1) {
                for (int q = std::max(q0, 0); q < std::min(q1, ns); ++q) {
                    bb[q] = 0.0;
                    cc[q] = 0.0;
                    kk[q] = 1.0;
                }
            };
            ident(lo, pm.lo[ax]);
            ident(pm.hi0[ax], hi0);
            ident(hi1, pm.hi1[ax]);
            pm.b[ax] = upload_cast<T>(c, bb.data(), ns);
            pm.cd[ax] = upload_cast<T>(c, cc.data(), ns);
            pm.kinv[ax] = upload_cast<T>(c, kk.data(), ns);
            size_t ps = static_cast<size_t>(pm.S[ax]);
            for (int o = 0; o < 3; ++o)
                if (o != ax) ps *= o == 0 ? px : nn[o];
            pm.psi[ax] = ps ? c->zeros<T>(ps) : nullptr;
        }
    }
    a.nsrc = p->nsrc;
    c->has_src = p->nsrc > 0;
    if (p->nsrc > 0) {
        a.src_comp = c->upload<int>(p->src_comp, p->nsrc);
        a.src_box = c->upload<int>(p->src_box, static_cast<size_t>(p->nsrc) * 6);
        a.src_amp = upload_cast<T>(c, p->src_amp, static_cast<size_t>(p->nsteps) * p->nsrc);
    }
    for (int k = 0; k < 6; ++k) a.G[k] = a.F[k];
    for (int comp = 0; comp < 6; ++comp)
        for (int ax = 0; ax < 3; ++ax) a.pml[comp].psi_in[ax] = a.pml[comp].psi[ax];
    a.step = c->step_ctr.as<int>();
    a.stepv = -1;
    a.step_next = nullptr;
    // detectors and DFT
    for (int k = 0; k < 6; ++k) s.F[k] = a.F[k];
    s.step = a.step;
    s.stepv = -1;
    c->ndet = p->ndet;
    std::vector<int> off(p->ndet + 1, 0);
    std::vector<long long> ooff(p->ndet + 1, 0);
    c->det_npts.assign(p->det_npts, p->det_npts + p->ndet);
    c->det_interval.assign(p->det_interval, p->det_interval + p->ndet);
    c->det_cap.resize(p->ndet);
    std::vector<int> nf(p->ndet, 1);
    std::vector<long long> eoff(p->ndet + 1, 0);
    for (int d = 0; d < p->ndet; ++d) {
        if (p->det_interval[d] <= 0) throw std::runtime_error("detector interval must be positive");
        if (p->det_nfield) nf[d] = p->det_nfield[d];
        if (nf[d] < 1 || nf[d] > 3) throw std::runtime_error("detector fields per point must be 1..3");
        eoff[d + 1] = eoff[d] + static_cast<long long>(p->det_npts[d]) * nf[d];
        off[d + 1] = off[d] + p->det_npts[d];
        c->det_cap[d] = p->nsteps / p->det_interval[d] + 1;
        ooff[d + 1] = ooff[d] + static_cast<long long>(c->det_cap[d]) * p->det_npts[d];
    }
    c->det_out_off.assign(ooff.begin(), ooff.end());
    c->totpts = off[p->ndet];
    s.ndet = p->ndet;
    s.totpts = c->totpts;
    if (p->ndet > 0) {
        s.det_interval = c->upload<int>(p->det_interval, p->ndet);
        s.det_npts = c->upload<int>(p->det_npts, p->ndet);
        s.det_off = c->upload<int>(off.data(), p->ndet + 1);
        s.det_comp = c->upload<int>(p->det_comp, 2 * static_cast<size_t>(eoff[p->ndet]));
        s.det_cell = c->upload<long long>(padded_cells(p->det_cell, 2 * static_cast<size_t>(eoff[p->ndet])).data(), 2 * static_cast<size_t>(eoff[p->ndet]));
        s.det_nf = c->upload<int>(nf.data(), p->ndet);
        s.det_eoff = c->upload<long long>(eoff.data(), p->ndet + 1);
        c->det_single_field = std::all_of(nf.begin(), nf.end(), [](int v) { return v == 1; });
        s.det_all1 = c->det_single_field ? 1 : 0;
        s.det_conv = c->upload<double>(p->det_conv, p->ndet);
        s.det_pow = c->upload<int>(p->det_pow, p->ndet);
        c->det_out = c->zeros<double>(static_cast<size_t>(ooff[p->ndet]));
        s.det_out = c->det_out;
        s.det_out_off = c->upload<long long>(ooff.data(), p->ndet + 1);
        s.det_cap = c->upload<int>(c->det_cap.data(), p->ndet);
    }
    // DFT groups: 0 = the flux boxes (ndft / dft_*), then p->dftg[0..ndftg)
    if (p->ndftg < 0 || 1 + p->ndftg > kMaxDftGroups) throw std::runtime_error("too many DFT groups (at most 15 frequency detectors)");
    c->dgs.clear();
    c->ndft = 0;
    s.ndg = 1 + p->ndftg;
    s.gofs[0] = 0;
    for (int g = 0; g < s.ndg; ++g) {
        const int n = g == 0 ? p->ndft : p->dftg[g - 1].ncell;
        const int nf = g == 0 ? p->nfreq : p->dftg[g - 1].nfreq;
        const int iv = g == 0 ? p->dft_interval : p->dftg[g - 1].interval;
        const int* comp = g == 0 ? p->dft_comp : p->dftg[g - 1].comp;
        const long long* cell = g == 0 ? p->dft_cell : p->dftg[g - 1].cell;
        const double* ph = g == 0 ? p->dft_phasor : p->dftg[g - 1].phasor;
        if (n < 0 || (n > 0 && nf < 1)) throw std::runtime_error("invalid DFT group");
        chiml_dev::DftGroup d;
        d.n = n;
        d.nfreq = nf;
        d.interval = iv > 0 ? iv : 1;
        DftSample<T>& ds = s.dg[g];
        ds.n = n;
        ds.interval = d.interval;
        ds.comp = nullptr;
        ds.cell = nullptr;
        ds.stage = nullptr;
        if (n > 0) {
            ds.comp = c->upload<int>(comp, n);
            ds.cell = c->upload<long long>(padded_cells(cell, n).data(), n);
            T* st = c->zeros<T>(static_cast<size_t>(kDftBlock) * n);
            ds.stage = st;
            d.stage = st;
            d.F = c->zeros<double>(2 * static_cast<size_t>(n) * nf);
            d.tmp = c->zeros<double>(2 * static_cast<size_t>(n) * nf);
            d.phasor = c->upload<double>(ph, 2 * static_cast<size_t>(p->nsteps / d.interval + 1) * nf);
        }
        c->dgs.push_back(d);
        c->ndft += n;
        s.gofs[g + 1] = c->ndft;
    }
    s.ndft = c->ndft;
    // emitters
    const double* epsn = nullptr;
    if (p->nqe > 0) epsn = upload_rows(p->eps_node, 1.0);
    for (int g = 0; g < p->nqe; ++g) {
        const chiml_qe_t& qi = p->qe[g];
        QeHost qh;
        QeDev& q = qh.dev;
        if (qi.nlevel < 2 || qi.nlevel > kMaxLevels) throw std::runtime_error("emitter level count out of range (2..8)");
        q.N = qi.nlevel;
        qh.N = qi.nlevel;
        q.nmem = qi.nmembers;
        q.nemit = qi.nemit;
        const int S = q.N * q.N;
        q.xyz = c->upload<int>(qi.emit_xyz, 3 * static_cast<size_t>(qi.nemit));
        q.h0 = reinterpret_cast<const double2*>(c->upload<double>(qi.h0, 2 * static_cast<size_t>(qi.nmembers) * S));
        q.mu = reinterpret_cast<const double2*>(c->upload<double>(qi.mu, 2 * 3 * static_cast<size_t>(S)));
        q.ngam = qi.ngam;
        {
            // Lindblad entries by row (stable, so each row keeps its accumulation order)
            const int S = qi.nlevel * qi.nlevel;
            for (int g = 0; g < qi.ngam; ++g)
                if (qi.gam_row[g] < 0 || qi.gam_row[g] >= S || qi.gam_col[g] < 0 || qi.gam_col[g] >= S)
                    throw std::runtime_error("Lindblad entry index outside nlevel^2");
            std::vector<int> order(qi.ngam);
            for (int g = 0; g < qi.ngam; ++g) order[g] = g;
            std::stable_sort(order.begin(), order.end(), [&](int u, int v) { return qi.gam_row[u] < qi.gam_row[v]; });
            std::vector<int> gc(std::max(qi.ngam, 1)), ptr(S + 1, 0);
            std::vector<double> gv(std::max(qi.ngam, 1));
            for (int g = 0; g < qi.ngam; ++g) {
                gc[g] = qi.gam_col[order[g]];
                gv[g] = qi.gam_val[order[g]];
                ++ptr[qi.gam_row[order[g]] + 1];
            }
            for (int r = 0; r < S; ++r) ptr[r + 1] += ptr[r];
            q.gam_ptr = c->upload<int>(ptr.data(), ptr.size());
            q.gam_col = c->upload<int>(gc.data(), gc.size());
            q.gam_val = c->upload<double>(gv.data(), gv.size());
        }
        q.na = qi.na;
        q.ih = 1.0 / qi.hbar;
        const double wab[4] = {55.0, -59.0, 37.0, -9.0}, wam[4] = {9.0, 19.0, -5.0, 1.0};
        for (int k = 0; k < 4; ++k) {
            q.ab[k] = wab[k] * p->dt / 24.0;
            q.am[k] = wam[k] * p->dt / 24.0;
        }
        q.dim = is3 ? 3 : 2;
        q.fold_addp = (!is3 && std::getenv("CHIML_ML_ADDP") == nullptr) ? 1 : 0;
        for (int k = 0; k < 3; ++k) {
            q.bmin[k] = qi.box_min[k];
            q.bn[k] = qi.box_n[k];
        }
        if (!is3) q.bn[2] = 1;
        const size_t pb = static_cast<size_t>(q.bn[0] + 2) * (q.bn[1] + 2) * (q.bn[2] + 1 + (is3 ? 1 : 0));
        const size_t ab = static_cast<size_t>(q.bn[0] + 1) * (q.bn[1] + 1) * (is3 ? q.bn[2] + 1 : 1);
        for (int k = 0; k < 3; ++k) {
            q.Pbox[k] = c->zeros<double>(pb);
            q.Aprev[k] = c->zeros<double>(ab);
        }
        const size_t ld = static_cast<size_t>(q.nmem) * q.nemit;
        q.packed = chiml_qe_packed(qi) ? 1 : 0;
        const size_t SW = static_cast<size_t>(ml_store_words(q.N, q.packed != 0));
        std::vector<double> rho0(2 * SW * ld, 0.0);  // rho_00 = the member's weight (entry 0 in both layouts)
        for (int m = 0; m < q.nmem; ++m)
            for (int e = 0; e < q.nemit; ++e) rho0[2 * (0 * ld + static_cast<size_t>(m) * q.nemit + e)] = qi.weight[m];
        q.rho = reinterpret_cast<double2*>(c->upload<double>(rho0.data(), rho0.size()));
        q.hist = reinterpret_cast<double2*>(c->zeros<double>(2 * 4 * SW * ld));
        q.npop = std::min(qi.npop, 4);
        qh.npop_all = qi.npop;
        for (int k = 0; k < qi.npop; ++k)
            if (qi.pop_flat[k] < 0 || qi.pop_flat[k] >= qi.nlevel * qi.nlevel) throw std::runtime_error("population detector index out of range");
        q.pop_flat = c->upload<int>(qi.pop_flat, std::max(qi.npop, 1));
        q.pop_interval = qi.pop_interval > 0 ? qi.pop_interval : 1;
        const int per_block = ml_emitters(q.N, q.packed != 0);
        qh.nblocks = (q.nemit + per_block - 1) / per_block;
        q.pop_partial = reinterpret_cast<double2*>(c->zeros<double>(2 * 4 * static_cast<size_t>(qh.nblocks)));
        q.pop_cap = p->nsteps / q.pop_interval + 1;
        q.pop_out = reinterpret_cast<double2*>(c->zeros<double>(2 * std::max(qi.npop, 4) * static_cast<size_t>(q.pop_cap)));
        if (qi.npop > 4) {
            const long long ldc = static_cast<long long>(q.nmem) * q.nemit;
            qh.nb2 = static_cast<int>(std::min<long long>(1024, std::max<long long>(1, (ldc + 1023) / 1024)));
            qh.partial2 = reinterpret_cast<double2*>(c->zeros<double>(2 * static_cast<size_t>(qi.npop - 4) * qh.nb2));
        }
        q.eps_node = epsn;
        c->qes.push_back(std::move(qh));
    }
    build_tfsf(c, p, a);
    build_cells<T>(c, p);
    c->step_bytes = 6.0 * N * sizeof(T);
    for (const QeHost& qh : c->qes)
        c->step_bytes += 5.0 * 16 * ml_store_words(qh.N, qh.dev.packed != 0) * static_cast<double>(qh.dev.nmem) * qh.dev.nemit;
    c->stream_hint = streams_past_caches(c->step_bytes);
}

template <typename T>
StepArgs<T>& step_args(chiml_dev* c);
template <>
StepArgs<float>& step_args<float>(chiml_dev* c) { return c->a32; }
template <>
StepArgs<double>& step_args<double>(chiml_dev* c) { return c->a64; }

template <typename T>
void launch_sample(chiml_dev* c, SampleArgs<T>& s) {
    int tot = c->totpts + c->ndft;
    if (tot == 0) return;
    if (const QeHost* h = c->finish_with_sample) {
        c->finish_with_sample = nullptr;
        const StepArgs<T>& a = step_args<T>(c);
        hipLaunchKernelGGL(k_finish_sample<T>, dim3(h->dev.npop + (tot + kPopThreads - 1) / kPopThreads), dim3(kPopThreads), 0, c->stream,
                           h->dev, h->dev.pop_partial, h->nblocks, a.step, a.stepv, s);
        return;
    }
    hipLaunchKernelGGL(k_sample<T>, dim3((tot + 255) / 256), dim3(256), 0, c->stream, s);
}

// Is kernel n one of the comma-separated names in `list`?
bool in_name_list(const std::string& list, const char* n) {
    const size_t len = std::strlen(n);
    size_t p = 0;
    while (p <= list.size()) {
        size_t q = list.find(',', p);
        if (q == std::string::npos) q = list.size();
        if (q - p == len && list.compare(p, len, n) == 0) return true;
        p = q + 1;
    }
    return false;
}

struct Timed {
    chiml_dev* c;
    const char* name;
    hipEvent_t e0 = nullptr, e1 = nullptr;
    int count;
    bool on;
    Timed(chiml_dev* c_, const char* n, int count_ = 1)
        : c(c_), name(n), count(count_), on(c_->profile && !c_->device_flush && (c_->profile_only.empty() || in_name_list(c_->profile_only, n))) {
        if (on) {
            (void)hipEventCreate(&e0);
            (void)hipEventCreate(&e1);
            (void)hipEventRecord(e0, c->stream);
        }
    }
    ~Timed() {
        if (on) {
            (void)hipEventRecord(e1, c->stream);
            c->pending.push_back({name, e0, e1, count});
        }
    }
};

// step: the step number once the step being enqueued has advanced it (-1:
// read the device counter, inside captured graphs)
template <typename T>
void launch_flush(chiml_dev* c, int force, int step, const int* stepp) {
    // enq_step = the device step counter once the step being enqueued has advanced it
    const int st = c->enq_step;
    for (const chiml_dev::DftGroup& d : c->dgs) {
        if (d.n == 0) continue;
        if (!force && !c->device_flush && (st % d.interval != 0 || ((st / d.interval) % kDftBlock) != kDftBlock - 1)) continue;
        Timed t(c, "dft_flush");
        hipLaunchKernelGGL(k_dft_flush<T>, dim3((d.n + 255) / 256), dim3(256), 0, c->stream, static_cast<const T*>(d.stage), d.phasor,
                           d.F, stepp, d.n, d.nfreq, d.interval, force, step);
    }
}


template <typename T>
SampleArgs<T>& sample_args(chiml_dev* c);
template <>
SampleArgs<float>& sample_args<float>(chiml_dev* c) { return c->s32; }
template <>
SampleArgs<double>& sample_args<double>(chiml_dev* c) { return c->s64; }

// f(S, A) with S, A std::integral_constant<bool> for the two runtime flags
template <typename F>
void pick2(bool s, bool adv, F&& f) {
    using Y = std::true_type;
    using N = std::false_type;
    if (s) {
        if (adv) f(Y{}, Y{});
        else f(Y{}, N{});
    } else {
        if (adv) f(N{}, Y{});
        else f(N{}, N{});
    }
}

// The TFSF part of a step, between the H and E updates of the main grid:
// H surface adds, the incident lines, E surface adds (parallelFDTDField.hpp:1236-1256).
template <typename T>
void launch_tfsf(chiml_dev* c, StepArgs<T>& a) {
    TfsfFields<T> f;
    for (int k = 0; k < 6; ++k) f.F[k] = a.F[k];
    for (const auto& h : c->tfsf) {
        const TfsfLineArgs& t = h.line;
        const dim3 g(static_cast<unsigned>(1 + (h.toth + 1023) / 1024));
        const size_t lds = tfsf_lds_bytes(t);
        if (lds <= kTfsfMaxLds)
            hipLaunchKernelGGL((k_tfsf_step<T, true>), g, dim3(1024), lds, c->stream, t, h.surf, h.nsh, h.toth, f, c->px, c->ny, a.step, a.stepv);
        else
            hipLaunchKernelGGL((k_tfsf_step<T, false>), g, dim3(1024), 0, c->stream, t, h.surf, h.nsh, h.toth, f, c->px, c->ny, a.step, a.stepv);
        if (h.tote > 0)
            hipLaunchKernelGGL(k_tfsf_add<T>, dim3(static_cast<unsigned>((h.tote + 255) / 256)), dim3(256), 0, c->stream, h.surf + h.nsh,
                               h.nse, h.tote, f, t.line[0], t.len[0], c->px, c->ny);
    }
}

template <typename T>
void launch_cells(chiml_dev* c, StepArgs<T>& a) {
    const auto& q = c->cells;
    if (q.n == 0) return;
    hipLaunchKernelGGL(k_cell_src<T>, dim3(static_cast<unsigned>((q.n + 255) / 256)), dim3(256), 0, c->stream, q.comp, q.idx, q.col,
                       static_cast<const T*>(q.amp), q.n, q.ncol, a.step, a.stepv, a.F[0], a.F[1], a.F[2], a.F[3], a.F[4], a.F[5]);
}

template <typename T, int DIM>
void launch_fields(chiml_dev* c, StepArgs<T>& a) {
    const bool adv = a.step_next != nullptr;
    if (DIM == 3 && c->fused) {
        constexpr int W = 16 / sizeof(T);
        const int ade_bpc = static_cast<int>((c->ade_groups + 255) / 256);
        const bool pre = ade_bpc > 0;
        if (pre) {  // pole update from E before the step
            StepArgs<T> aa = a;
            for (int k = 0; k < 3; ++k) aa.F[k] = const_cast<T*>(a.G[k]);
            Timed t(c, "update_ade");
            if (c->has_src) hipLaunchKernelGGL((k_ade3<T, W, true>), dim3(3 * ade_bpc), dim3(256), 0, c->stream, aa, ade_bpc);
            else hipLaunchKernelGGL((k_ade3<T, W, false>), dim3(3 * ade_bpc), dim3(256), 0, c->stream, aa, ade_bpc);
        }
        const FuseMap& m = c->fmap;
        const dim3 g(static_cast<unsigned>(m.ntile * m.nseg)), blk(static_cast<unsigned>((m.nthr + 63) / 64 * 64));
        Timed t(c, "update_fused");
        auto go = [&](auto S, auto P, auto A) {
            hipLaunchKernelGGL((k_fused3<T, W, decltype(S)::value, decltype(P)::value, decltype(A)::value>), g, blk, c->fused_lds,
                               c->stream, a, m, c->nmat[0], c->nmat[1], c->nmat[2]);
        };
        using Y = std::true_type;
        using N = std::false_type;
        pick2(c->has_src, adv, [&](auto S, auto A) {
            if (pre) go(S, Y{}, A);
            else go(S, N{}, A);
        });
        return;
    }
    if (DIM == 3 && c->split && !c->cellwise) {
        constexpr int W = 16 / sizeof(T);
        const Box3 b = c->ibox;
        const int nyb = b.y1 - b.y0, by = b.by > 0 ? b.by : nyb;
        const long long ni = static_cast<long long>((b.x1 - b.x0) / W) * by * (b.z1 - b.z0) * ((nyb + by - 1) / by);
        const long long ns = static_cast<long long>(c->slab.nA) + c->slab.nB + c->slab.nC;
        const dim3 gi(static_cast<unsigned>((ni + 255) / 256)), gs(static_cast<unsigned>((ns + 255) / 256)), blk(256);
        const int nib = static_cast<int>(gi.x), ade_bpc = static_cast<int>((c->ade_groups + 255) / 256);
        if (c->rows) {  // one launch per field
            const int nsbp = static_cast<int>((gs.x + 7) / 8 * 8);
            const dim3 gh(static_cast<unsigned>(ade_blocks(ade_bpc) + nsbp + nib)), ge(static_cast<unsigned>(nsbp + nib));
            if (gh.x > 0) {
                Timed t(c, "update_h");
                pick2(c->has_src, adv, [&](auto S, auto A) {
                    auto go = [&](auto M) {
                        if (c->stream_hint)
                            hipLaunchKernelGGL((k_h3_all<T, W, decltype(S)::value, decltype(A)::value, decltype(M)::value, true>), gh, blk, 0, c->stream,
                                               a, b, c->slab, nib, nsbp, ade_bpc);
                        else
                            hipLaunchKernelGGL((k_h3_all<T, W, decltype(S)::value, decltype(A)::value, decltype(M)::value, false>), gh, blk, 0, c->stream,
                                               a, b, c->slab, nib, nsbp, ade_bpc);
                    };
                    if (c->fma_curl) go(std::true_type{});
                    else go(std::false_type{});
                });
            }
            launch_tfsf<T>(c, a);
            launch_cells<T>(c, a);
            if (ge.x > 0) {
                Timed t(c, "update_e");
                pick2(c->has_src, c->fma_curl, [&](auto S, auto M) {
                    if (c->stream_hint)
                        hipLaunchKernelGGL((k_e3_all<T, W, decltype(S)::value, decltype(M)::value, true>), ge, blk, 0, c->stream, a, b, c->slab, nib,
                                           nsbp, c->nmat[0], c->nmat[1], c->nmat[2]);
                    else
                        hipLaunchKernelGGL((k_e3_all<T, W, decltype(S)::value, decltype(M)::value, false>), ge, blk, 0, c->stream, a, b, c->slab, nib,
                                           nsbp, c->nmat[0], c->nmat[1], c->nmat[2]);
                });
            }
        } else if constexpr (W == 2) {  // FP64: the pole update rides on the H interior launch as its first blocks
            const dim3 gh(static_cast<unsigned>(nib + ade_blocks(ade_bpc)));
            if (gh.x > 0) {
                Timed t(c, "update_h");
                pick2(c->has_src, adv, [&](auto S, auto A) {
                    if (c->stream_hint)
                        hipLaunchKernelGGL((k_h3_int<T, W, decltype(S)::value, decltype(A)::value, true>), gh, blk, 0, c->stream, a, b, nib, ade_bpc);
                    else
                        hipLaunchKernelGGL((k_h3_int<T, W, decltype(S)::value, decltype(A)::value, false>), gh, blk, 0, c->stream, a, b, nib, ade_bpc);
                });
            }
            if (ns > 0) {
                Timed t(c, "update_h_pml");
                pick2(c->has_src, c->stream_hint, [&](auto S, auto H) {
                    hipLaunchKernelGGL((k_h3_slab<T, W, decltype(S)::value, decltype(H)::value>), gs, blk, 0, c->stream, a, c->slab);
                });
            }
            launch_tfsf<T>(c, a);
            launch_cells<T>(c, a);
            {
                Timed t(c, "update_e");
                pick2(c->has_src, c->stream_hint, [&](auto S, auto H) {
                    hipLaunchKernelGGL((k_e3_int<T, W, decltype(S)::value, decltype(H)::value>), gi, blk, 0, c->stream, a, b, c->nmat[0], c->nmat[1],
                                       c->nmat[2]);
                });
            }
            if (ns > 0) {
                Timed t(c, "update_e_pml");
                pick2(c->has_src, c->stream_hint, [&](auto S, auto H) {
                    hipLaunchKernelGGL((k_e3_slab<T, W, decltype(S)::value, decltype(H)::value>), gs, blk, 0, c->stream, a, c->slab, c->nmat[0],
                                       c->nmat[1], c->nmat[2]);
                });
            }
        }
        return;
    }
    if (DIM == 2 && c->vec2d && !c->cellwise) {
        constexpr int W = 16 / sizeof(T);
        const long long ng = static_cast<long long>(c->px / W) * c->ny;
        const dim3 g(static_cast<unsigned>((ng + 255) / 256)), blk(256);
        {
            Timed t(c, "update_h");
            pick2(c->has_src, adv, [&](auto S, auto A) {
                hipLaunchKernelGGL((k_h2v<T, W, decltype(S)::value, decltype(A)::value>), g, blk, 0, c->stream, a);
            });
        }
        launch_tfsf<T>(c, a);
        launch_cells<T>(c, a);
        {
            Timed t(c, "update_e");
            const SampleArgs<T>& sa = sample_args<T>(c);
            pick2(c->has_src, c->fuse_sample, [&](auto S, auto D) {
                if (c->fma_curl)
                    hipLaunchKernelGGL((k_e2v<T, W, decltype(S)::value, decltype(D)::value, true>), g, blk, 0, c->stream, a, sa, c->nmat[2]);
                else
                    hipLaunchKernelGGL((k_e2v<T, W, decltype(S)::value, decltype(D)::value, false>), g, blk, 0, c->stream, a, sa, c->nmat[2]);
            });
        }
        return;
    }
    dim3 blk(64, 4, 1);
    dim3 grd((c->nx + 63) / 64, (c->ny + 3) / 4, c->nz);
    {
        Timed t(c, "update_h");
        pick2(c->has_src, adv, [&](auto S, auto A) {
            if (c->hmap) hipLaunchKernelGGL((k_update_h<T, DIM, true, decltype(S)::value, decltype(A)::value>), grd, blk, 0, c->stream, a);
            else hipLaunchKernelGGL((k_update_h<T, DIM, false, decltype(S)::value, decltype(A)::value>), grd, blk, 0, c->stream, a);
        });
    }
    launch_tfsf<T>(c, a);
    launch_cells<T>(c, a);
    {
        Timed t(c, "update_e");
        if (c->has_src) hipLaunchKernelGGL((k_update_e<T, DIM, true>), grd, blk, 0, c->stream, a);
        else hipLaunchKernelGGL((k_update_e<T, DIM, false>), grd, blk, 0, c->stream, a);
    }
}

// sampled: the step's sample launch follows, and takes the last group's
// population finish with it
template <typename T>
void launch_ml(chiml_dev* c, StepArgs<T>& a, bool sampled) {
    for (auto& qh : c->qes) {
        QeDev& q = qh.dev;
        int ex = q.bn[0] + 1, ey = q.bn[1] + 1, ez = (q.dim == 3) ? q.bn[2] + 1 : 1;
        int n = ex * ey * ez;
        if (!q.fold_addp)
            hipLaunchKernelGGL(k_ml_addp<T>, dim3((n + 255) / 256, 3), dim3(256), 0, c->stream, q, a.F[0], a.F[1], a.F[2], c->px, c->ny,
                               c->nz);
        dim3 g(qh.nblocks);
        {
            Timed t(c, "ml_density");
            switch (qh.N) {
#define CHIML_ML_ENTRY(NN)                                                                                                       \
    case NN:                                                                                                                    \
        if (q.packed)                                                                                                           \
            hipLaunchKernelGGL((k_ml_entry<T, NN, true>), g, dim3(ml_threads(NN, true)), 0, c->stream, q, a.F[0], a.F[1], a.F[2], c->px, c->ny, \
                               c->nz, a.step, a.stepv);                                                                         \
        else                                                                                                                    \
            hipLaunchKernelGGL((k_ml_entry<T, NN, false>), g, dim3(ml_threads(NN, false)), 0, c->stream, q, a.F[0], a.F[1], a.F[2], c->px, c->ny, \
                               c->nz, a.step, a.stepv);                                                                         \
        break;
                CHIML_ML_ENTRY(2)
                CHIML_ML_ENTRY(3)
                CHIML_ML_ENTRY(4)
                CHIML_ML_ENTRY(5)
                CHIML_ML_ENTRY(6)
                CHIML_ML_ENTRY(7)
                CHIML_ML_ENTRY(8)
#undef CHIML_ML_ENTRY
            }
        }
        if (sampled && q.npop > 0 && &qh == &c->qes.back())
            c->finish_with_sample = &qh;
        else if (q.npop > 0)
            hipLaunchKernelGGL(k_ml_pop_finish, dim3(q.npop), dim3(kPopThreads), 0, c->stream, q, q.pop_partial, qh.nblocks, 0, a.step, a.stepv);
        if (qh.npop_all > 4) {
            hipLaunchKernelGGL(k_ml_pop_gather, dim3(static_cast<unsigned>(qh.nb2), static_cast<unsigned>(qh.npop_all - 4)), dim3(256), 0,
                               c->stream, q, 4, qh.partial2, a.step, a.stepv);
            hipLaunchKernelGGL(k_ml_pop_finish, dim3(static_cast<unsigned>(qh.npop_all - 4)), dim3(kPopThreads), 0, c->stream, q,
                               qh.partial2, qh.nb2, 4, a.step, a.stepv);
        }
    }
}

// Plain launches carry the step number from the host, so no counter work
// runs between steps, and the counter slot of the next step is set once at
// the end.  Steps being captured into a graph read the two-slot device
// counter instead (advance_counter), so that one graph serves every replay
// that starts on the same slot.
// Fused 3D step: step st reads the buffers of parity st & 1 and writes the
// other ones (fields and H psi); everything launched after the field update
// (emitters, detectors, DFT) and every read between steps sees the written
// ones.  The current buffers after k steps are those of parity k & 1.
template <typename T>
void set_fused_buffers(chiml_dev* c, StepArgs<T>& a, SampleArgs<T>& s, int st) {
    const int p = st & 1;
    for (int k = 0; k < 6; ++k) {
        a.G[k] = static_cast<const T*>(c->fbuf[p][k]);
        a.F[k] = static_cast<T*>(c->fbuf[p ^ 1][k]);
        s.F[k] = a.F[k];
    }
    for (int h = 0; h < 3; ++h)
        for (int ax = 0; ax < 3; ++ax) {
            a.pml[3 + h].psi_in[ax] = static_cast<const T*>(c->fpsi[p][h][ax]);
            a.pml[3 + h].psi[ax] = static_cast<T*>(c->fpsi[p ^ 1][h][ax]);
        }
}

template <typename T>
void do_steps(chiml_dev* c, StepArgs<T>& a, SampleArgs<T>& s, int n) {
    const bool host = !c->capturing;
    int* ctr = c->step_ctr.as<int>();
    for (int k = 0; k < n; ++k) {
        const int st = c->steps_done + k, p = st & 1;
        if (c->fused) set_fused_buffers<T>(c, a, s, st);
        a.stepv = host ? st : -1;
        s.stepv = host ? st + 1 : -1;
        a.step = ctr + p;
        a.step_next = host ? nullptr : ctr + (1 - p);
        s.step = ctr + (1 - p);
        {
            // one event pair around all field launches of the step ("field_step")
            Timed t(c, "field_step");
            if (c->dim == 3) launch_fields<T, 3>(c, a);
            else launch_fields<T, 2>(c, a);
        }
        if (!c->qes.empty()) launch_ml<T>(c, a, !c->fuse_sample && c->totpts + c->ndft > 0);
        c->enq_step = st + 1;
        if (!c->fuse_sample) launch_sample<T>(c, s);
        launch_flush<T>(c, 0, host ? st + 1 : -1, ctr + (1 - p));
        HIP_TRY(hipGetLastError());
    }
    if (host && n > 0) {
        const int end = c->steps_done + n;
        hipLaunchKernelGGL(k_set_step, dim3(1), dim3(1), 0, c->stream, ctr, end);
    }
    a.stepv = -1;
    s.stepv = -1;
    a.step_next = nullptr;
    c->steps_done += n;
    // between steps F (and the sample kernel's fields) are the current buffers
    if (c->fused) set_fused_buffers<T>(c, a, s, c->steps_done - 1);
}

// ------------------------------------------------------- 2D tile launches ----
template <typename T, typename F>
void pick_tile(int shape, F&& f) {
    if (shape == 0) f(TileS{});
    else if (sizeof(T) == 8 || shape == 1) f(TileM{});
    else f(std::conditional_t<sizeof(T) == 4, TileL, TileM>{});
}

// The pointers of the plain kernels and reads to buffer set k.
template <typename T>
void set_tile_buffers(chiml_dev* c, StepArgs<T>& a, SampleArgs<T>& s, int k) {
    void* const* b = c->tbuf[k];
    for (int j = 0; j < 3; ++j) {
        a.F[2 + j] = static_cast<T*>(b[j]);
        a.G[2 + j] = a.F[2 + j];
        s.F[2 + j] = a.F[2 + j];
    }
    T** psi[4] = {&a.pml[3].psi[1], &a.pml[4].psi[0], &a.pml[2].psi[0], &a.pml[2].psi[1]};
    for (int j = 0; j < 4; ++j) *psi[j] = static_cast<T*>(b[3 + j]);
    if (c->tile_npole > 0) {
        a.P[2] = static_cast<T*>(b[7]);
        a.J[2] = static_cast<T*>(b[8]);
    }
    c->tile_cur = k;
}

template <typename T>
TileArgs<T> tile_args(const chiml_dev* c, const StepArgs<T>& a, int cur) {
    TileArgs<T> t{};
    void* const* in = c->tbuf[cur];
    void* const* out = c->tbuf[1 - cur];
    t.ez = static_cast<const T*>(in[0]);
    t.hx = static_cast<const T*>(in[1]);
    t.hy = static_cast<const T*>(in[2]);
    t.ez_o = static_cast<T*>(out[0]);
    t.hx_o = static_cast<T*>(out[1]);
    t.hy_o = static_cast<T*>(out[2]);
    t.nx = a.nx;
    t.ny = a.ny;
    t.px = a.px;
    t.ntx = c->tile_nx;
    t.inv_dx = a.inv_d[0];
    t.inv_dy = a.inv_d[1];
    t.ch0 = a.ch[0];
    t.ch1 = a.ch[1];
    t.mat = a.mat_e[2];
    t.ce = a.ce[2];
    t.inveps = a.inveps[2];
    t.flags = a.flags[2];
    t.poleset = a.poleset[2];
    t.nmat = c->nmat[2];
    const int comp[4] = {3, 4, 2, 2}, ax[4] = {1, 0, 0, 1};
    for (int q = 0; q < 4; ++q) {
        const PmlDev<T>& p = a.pml[comp[q]];
        t.lo[q] = p.lo[ax[q]];
        t.hi0[q] = p.hi0[ax[q]];
        t.hi1[q] = p.hi1[ax[q]];
        t.S[q] = p.S[ax[q]];
        t.b[q] = p.b[ax[q]];
        t.cd[q] = p.cd[ax[q]];
        t.kinv[q] = p.kinv[ax[q]];
        t.psi[q] = static_cast<const T*>(in[3 + q]);
        t.psi_o[q] = static_cast<T*>(out[3 + q]);
    }
    t.npole = c->tile_npole;
    t.pole_count = a.pole_count;
    t.pole_coef = a.pole_coef;
    t.P = static_cast<const T*>(in[7]);
    t.J = static_cast<const T*>(in[8]);
    t.P_o = static_cast<T*>(out[7]);
    t.J_o = static_cast<T*>(out[8]);
    for (int j = 0; j < 4; ++j) t.box[j] = a.box[2][j];
    t.boxn = a.boxn[2];
    t.nsrc = a.nsrc;
    t.src_comp = a.src_comp;
    t.src_box = a.src_box;
    t.src_amp = a.src_amp;
    t.det_ofs = c->tile_det_ofs;
    t.det = c->tile_det;
    t.det_out = c->det_out;
    t.fma_curl = c->fma_curl;
    t.Tx = a.Tp[0];
    t.Ty = a.Tp[1];
    t.nset = c->tile_nset;
    return t;
}

// n steps in launches of up to kTileSteps.  Captured steps take an even
// number of launches, so that a graph ends on the buffer set it starts on.
int tile_launches(int n, bool captured) {
    const int l = (n + kTileSteps - 1) / kTileSteps;
    return captured ? l + l % 2 : l;
}

// Do tile launches beat the sweeps for n steps in one go?  A launch reads and
// writes its whole state with the halo (1.8-4x the cells) however few steps it
// takes, so one or two steps are faster swept, in place, on grids large enough
// for that to outweigh the launches saved.  us a call of 1, 2 and 3 steps that
// is waited for, sweeps / tiles: FP32 384^2 21.2/21.2, 30/22; 512^2 21.3/24.3,
// 31/26; 1024^2 25.7/32.7, 39/35; without the wait 2048^2 35/62, 68/71, 102/80;
// FP64 384^2 21.3/21.6, 31/23; 512^2 22.5/27.6, 33/29; 832^2 25.9/39.9, 40/44;
// 2048^2 59/125, 116/144, 174/164.  Replayed from graphs the sweeps cost no host
// launch and the second line lies lower (graphs of 4, us a step: FP32 896^2
// 13.1/11.4, 1280^2 14.9/16.0; FP64 576^2 11.8/9.8, 768^2 12.9/13.6).
bool tile_pays(const chiml_dev* c, int n) {
    const int l = tile_launches(n, c->capturing), k = (n + l - 1) / l;
    if (k > 2) return true;
    const double cells = static_cast<double>(c->nx) * c->ny;
    if (k == 1) return cells < 400.0 * 400;
    const double side = c->prec == 32 ? (c->capturing ? 1000.0 : 2000.0) : (c->capturing ? 620.0 : 800.0);
    return cells < side * side;
}

template <typename T>
void do_tile_steps(chiml_dev* c, StepArgs<T>& a, SampleArgs<T>& s, int n) {
    const bool host = !c->capturing;
    int* ctr = c->step_ctr.as<int>();
    const int launches = tile_launches(n, !host);
    int cur = c->tile_cur;
    for (int l = 0, done = 0; l < launches; ++l) {
        const int k = (n - done + launches - l - 1) / (launches - l);
        TileArgs<T> t = tile_args<T>(c, a, cur);
        t.step = ctr + cur;
        t.stepv = host ? c->steps_done + done : -1;
        t.step_next = host ? nullptr : ctr + (1 - cur);
        t.nstep = k;
        {
            Timed fs(c, "field_step", k);
            Timed tm(c, "update_tile");
            pick_tile<T>(c->tile_shape, [&](auto sh) {
                using SH = decltype(sh);
                hipLaunchKernelGGL((k_tile2<T, SH>), dim3(static_cast<unsigned>(c->tile_nx * c->tile_ny)), dim3(SH::threads), c->tile_lds,
                                   c->stream, t);
            });
        }
        HIP_TRY(hipGetLastError());
        done += k;
        cur = 1 - cur;
    }
    c->steps_done += n;
    c->enq_step = c->steps_done;
    if (host) hipLaunchKernelGGL(k_set_step, dim3(1), dim3(1), 0, c->stream, ctr, c->steps_done);
    set_tile_buffers<T>(c, a, s, cur);
}

// 2D decks whose whole step is the field update and point samples of single
// cells take k_tile2.  The tile shape is the one with the least estimated
// time: tiles per CU in rounds of 256, times the tile's cells at 30 issue
// slots each, plus the two barriers and exchanges of a step (about 400
// cycles); a shape whose pole states do not fit LDS is left out.
template <typename T>
void enable_tiles(chiml_dev* c, const chiml_problem_t* p, StepArgs<T>& a, SampleArgs<T>& s) {
    if (c->dim != 2 || c->hmap || !c->qes.empty() || !c->tfsf.empty() || c->cells.n > 0 || c->ndft > 0) return;
    if (!c->det_single_field) return;
    for (int t = 0; t < c->totpts; ++t) {
        const int cu = p->det_comp[2 * t];
        if (cu != p->det_comp[2 * t + 1] || p->det_cell[2 * t] != p->det_cell[2 * t + 1] || cu < 2 || cu > 4) return;
    }
    int npole = 0;
    if (a.boxn[2] > 0 && a.P[2])
        for (int k = 0; k < p->npoleset; ++k) npole = std::max(npole, p->pole_count[k]);
    if (npole > 0 && p->npoleset > kTileSets) return;
    int lds_max = 0;
    HIP_TRY(hipDeviceGetAttribute(&lds_max, hipDeviceAttributeMaxSharedMemoryPerBlock, c->device));
    int best = -1;
    double best_t = 0.0;
    size_t best_lds = 0, lds_limit = 0;
    for (int sh = 0; sh < (sizeof(T) == 4 ? 3 : 2); ++sh)
        pick_tile<T>(sh, [&](auto shape) {
            using SH = decltype(shape);
            const size_t dyn = static_cast<size_t>(npole) * 2 * sizeof(T) * SH::rx * SH::ry;
            hipFuncAttributes at{};
            const void* fn = reinterpret_cast<const void*>(k_tile2<T, SH>);
            HIP_TRY(hipFuncGetAttributes(&at, fn));
            if (dyn + at.sharedSizeBytes > static_cast<size_t>(lds_max)) return;
            const double nt = static_cast<double>((p->nx + SH::ux - 1) / SH::ux) * ((p->ny + SH::uy - 1) / SH::uy);
            const double est = std::ceil(nt / 256.0) * SH::rx * SH::ry * 0.47 + 400.0;
            if (best < 0 || est < best_t) {
                best = sh;
                best_t = est;
                best_lds = dyn;
                lds_limit = static_cast<size_t>(lds_max) - at.sharedSizeBytes;
            }
        });
    if (best < 0) return;
    int ux = 0, uy = 0, rx = 0, rows = 0;
    pick_tile<T>(best, [&](auto shape) {
        using SH = decltype(shape);
        ux = SH::ux;
        uy = SH::uy;
        rx = SH::rx;
        rows = SH::r;
        // the limit is the process's, not this context's: all that a block may
        // have, whatever this deck needs of it
        if (best_lds > 0)
            HIP_TRY(hipFuncSetAttribute(reinterpret_cast<const void*>(k_tile2<T, SH>), hipFuncAttributeMaxDynamicSharedMemorySize,
                                        static_cast<int>(lds_limit)));
    });
    const int ntx = (p->nx + ux - 1) / ux, nty = (p->ny + uy - 1) / uy;
    // the detector points of each tile (points outside the grid read the zero
    // ghost: their samples stay the zeros of the output buffer)
    std::vector<std::vector<TileDet>> of(static_cast<size_t>(ntx) * nty);
    for (int d = 0, t = 0; d < c->ndet; ++d)
        for (int k = 0; k < c->det_npts[d]; ++k, ++t) {
            const long long cell = p->det_cell[2 * t];
            if (cell < 0 || cell >= static_cast<long long>(p->nx) * p->ny) continue;
            const int x = static_cast<int>(cell % p->nx), y = static_cast<int>(cell / p->nx);
            const int lx = x % ux + kTileSteps, ly = y % uy + kTileSteps;
            TileDet q{};
            q.thr = ly / rows * rx + lx;
            q.row = ly % rows;
            q.comp = p->det_comp[2 * t];
            q.interval = c->det_interval[d];
            q.cap = c->det_cap[d];
            q.npts = c->det_npts[d];
            q.pow = p->det_pow[d];
            q.conv = p->det_conv[d];
            q.out = c->det_out_off[d] + k;
            of[static_cast<size_t>(y / uy) * ntx + x / ux].push_back(q);
        }
    std::vector<int> ofs(1, 0);
    std::vector<TileDet> pts;
    for (auto& v : of) {
        if (v.size() > static_cast<size_t>(kTileDet)) return;
        pts.insert(pts.end(), v.begin(), v.end());
        ofs.push_back(static_cast<int>(pts.size()));
    }
    if (pts.empty()) pts.emplace_back();
    const size_t N = static_cast<size_t>(c->px) * p->ny;
    T* const psi[4] = {a.pml[3].psi[1], a.pml[4].psi[0], a.pml[2].psi[0], a.pml[2].psi[1]};
    const size_t psin[4] = {static_cast<size_t>(a.pml[3].S[1]) * c->px, static_cast<size_t>(a.pml[4].S[0]) * p->ny,
                            static_cast<size_t>(a.pml[2].S[0]) * p->ny, static_cast<size_t>(a.pml[2].S[1]) * c->px};
    const size_t held = c->bufs.size(), footprint = c->footprint;
    try {
        c->tile_det_ofs = c->upload<int>(ofs.data(), ofs.size());
        c->tile_det = c->upload<TileDet>(pts.data(), pts.size());
        for (int j = 0; j < 3; ++j) c->tbuf[1][j] = c->zeros<T>(N);
        for (int j = 0; j < 4; ++j) c->tbuf[1][3 + j] = psi[j] ? c->zeros<T>(psin[j]) : nullptr;
        for (int j = 7; npole > 0 && j < 9; ++j) c->tbuf[1][j] = c->zeros<T>(static_cast<size_t>(a.boxn[2]) * npole);
    } catch (const std::exception&) {
        // no room for the second set: the sweeps need none
        (void)hipGetLastError();
        c->bufs.resize(held);
        c->footprint = footprint;
        return;
    }
    c->tile_nset = p->npoleset;
    for (int j = 0; j < 3; ++j) c->tbuf[0][j] = a.F[2 + j];
    for (int j = 0; j < 4; ++j) c->tbuf[0][3 + j] = psi[j];
    if (npole > 0) {
        c->tbuf[0][7] = a.P[2];
        c->tbuf[0][8] = a.J[2];
    }
    c->tile = true;
    c->tile_shape = best;
    c->tile_nx = ntx;
    c->tile_ny = nty;
    c->tile_lds = best_lds;
    c->tile_npole = npole;
    set_tile_buffers<T>(c, a, s, 0);
}

void collect_profile(chiml_dev* c) {
    for (auto& pe : c->pending) {
        float ms = 0.0f;
        (void)hipEventSynchronize(pe.e1);
        (void)hipEventElapsedTime(&ms, pe.e0, pe.e1);
        auto& slot = c->prof[pe.name];
        slot.first += ms;
        slot.second += pe.n;
        (void)hipEventDestroy(pe.e0);
        (void)hipEventDestroy(pe.e1);
    }
    c->pending.clear();
}

}  // namespace

// ----------------------------------------------------------- batched steps ----
// Scratch of the allocation-free batched step: the slot-descriptor tables
// and prefix tables of one call, at most kBatchMaxSlots simulations.  Each GPU
// holds its own copy; host code reaches it only through the address that
// hipGetSymbolAddress returns for the current device.
constexpr int kBatchMaxSlots = 64;
constexpr size_t kBatchScratchBytes = 2 * kBatchMaxSlots * sizeof(BatchSlot<double>) + kPhases * (kBatchMaxSlots + 1) * sizeof(int) + 4096;
static __device__ __align__(256) unsigned char scratch[kBatchScratchBytes];

namespace {
void enqueue_steps(chiml_dev* c, int n);
int fail(chiml_dev* c, int code, const std::string& msg);
constexpr int kMaxDevices = 64;
std::mutex g_scratch_mu;
void* g_scratch_ptr[kMaxDevices] = {};
unsigned char g_batch_host[kBatchScratchBytes];  // host image of one call's tables (under g_batch_mu)
std::mutex g_batch_mu;

// The scratch array's address on device dev (looked up once per device,
// with that device current).
void* scratch_on(int dev) {
    if (dev < 0 || dev >= kMaxDevices) throw std::runtime_error("device index out of range");
    std::lock_guard<std::mutex> lk(g_scratch_mu);
    if (!g_scratch_ptr[dev]) {
        int cur = 0;
        HIP_TRY(hipGetDevice(&cur));
        if (cur != dev) HIP_TRY(hipSetDevice(dev));
        void* p = nullptr;
        const hipError_t e = hipGetSymbolAddress(&p, HIP_SYMBOL(scratch));
        if (cur != dev) HIP_TRY(hipSetDevice(cur));
        HIP_TRY(e);
        g_scratch_ptr[dev] = p;
    }
    return g_scratch_ptr[dev];
}

// Kernel class of a context for batched launches: 1 = 2D W-cell kernels,
// 2 = 3D split sweeps; 0 = not batched (stepped on its own stream).
int batch_class(const chiml_dev* c) {
    if (c->fused || c->tile || c->capturing || !c->tfsf.empty() || c->cells.n > 0) return 0;  // TFSF and per-cell source steps stay on their own stream
    if (c->dim == 2 && c->vec2d) return 1;
    if (c->dim == 3 && c->split && c->rows == (c->prec == 32)) return 2;
    return 0;
}

// The slot of context c for the steps whose counter parity is p.
template <typename T>
BatchSlot<T> make_slot(chiml_dev* c, int p) {
    constexpr int W = 16 / sizeof(T);
    BatchSlot<T> q{};
    q.a = step_args<T>(c);
    q.s = sample_args<T>(c);
    int* ctr = c->step_ctr.as<int>();
    q.a.step = ctr + p;
    q.a.step_next = ctr + (1 - p);
    q.a.stepv = -1;
    q.s.step = ctr + (1 - p);
    q.s.stepv = -1;
    for (int k = 0; k < 3; ++k) q.nm[k] = c->nmat[k];
    q.fma = c->fma_curl ? 1 : 0;
    if (c->dim == 2) {
        const long long ng = static_cast<long long>(c->px / W) * c->ny;
        q.nblk[kPhH] = q.nblk[kPhE] = static_cast<int>((ng + 255) / 256);
    } else {
        const Box3 b = c->ibox;
        const int nyb = b.y1 - b.y0, by = b.by > 0 ? b.by : nyb;
        const long long ni = static_cast<long long>((b.x1 - b.x0) / W) * by * (b.z1 - b.z0) * ((nyb + by - 1) / by);
        const long long ns = static_cast<long long>(c->slab.nA) + c->slab.nB + c->slab.nC;
        q.b = b;
        q.m = c->slab;
        q.nib = static_cast<int>((ni + 255) / 256);
        q.ade_bpc = static_cast<int>((c->ade_groups + 255) / 256);
        const int gs = static_cast<int>((ns + 255) / 256);
        if (W == 4) {  // FP32: one launch per field, as launch_fields
            q.nsbp = (gs + 7) / 8 * 8;
            q.nblk[kPhH] = ade_blocks(q.ade_bpc) + q.nsbp + q.nib;
            q.nblk[kPhE] = q.nsbp + q.nib;
        } else {  // FP64: interior (+ pole update) and slab launches per field
            q.nblk[kPhH] = q.nib + ade_blocks(q.ade_bpc);
            q.nblk[kPhHs] = gs;
            q.nblk[kPhE] = q.nib;
            q.nblk[kPhEs] = gs;
        }
    }
    q.nblk[kPhS] = (c->totpts + c->ndft + 255) / 256;
    return q;
}

// Enqueues nsteps batched steps of the contexts g[0..n) (one class, type T)
// on stream bs, with their tables at device address dev (host image host).
template <typename T>
void batch_group(chiml_dev** g, int n, int nsteps, hipStream_t bs, unsigned char* dev, unsigned char* host) {
    constexpr int W = 16 / sizeof(T);
    BatchSlot<T>* hs = reinterpret_cast<BatchSlot<T>*>(host);
    int* hb = reinterpret_cast<int*>(host + 2 * n * sizeof(BatchSlot<T>));
    int total[kPhases] = {};
    for (int i = 0; i < n; ++i) {
        const int p = g[i]->steps_done & 1;
        hs[i] = make_slot<T>(g[i], p);
        hs[n + i] = make_slot<T>(g[i], 1 - p);
    }
    for (int ph = 0; ph < kPhases; ++ph) {
        int acc = 0;
        for (int i = 0; i < n; ++i) {
            hb[ph * (n + 1) + i] = acc;
            acc += (hs[i].nblk[ph] + 7) / 8 * 8;  // each simulation's range starts on a multiple of 8 blocks
        }
        hb[ph * (n + 1) + n] = acc;
        total[ph] = acc;
    }
    const size_t bytes = 2 * n * sizeof(BatchSlot<T>) + kPhases * (n + 1) * sizeof(int);
    HIP_TRY(hipMemcpyAsync(dev, host, bytes, hipMemcpyHostToDevice, bs));
    const BatchSlot<T>* ds = reinterpret_cast<const BatchSlot<T>*>(dev);
    const int* db = reinterpret_cast<const int*>(dev + 2 * n * sizeof(BatchSlot<T>));
    const dim3 blk(256);
    double state = 0;  // the batch's simulations share the caches
    for (int i = 0; i < n; ++i) state += g[i]->step_bytes;
    const bool stream_hint = streams_past_caches(state);
    for (int j = 0; j < nsteps; ++j) {
        const BatchSlot<T>* t = ds + (j & 1) * n;  // every slot's counter parity flips each step
        const int* bH = db + kPhH * (n + 1);
        const int* bHs = db + kPhHs * (n + 1);
        const int* bE = db + kPhE * (n + 1);
        const int* bEs = db + kPhEs * (n + 1);
        const int* bS = db + kPhS * (n + 1);
        if (g[0]->dim == 2) {
            if (total[kPhH]) hipLaunchKernelGGL((k_bh2v<T, W>), dim3(total[kPhH]), blk, 0, bs, t, bH, n);
            if (total[kPhE]) hipLaunchKernelGGL((k_be2v<T, W>), dim3(total[kPhE]), blk, 0, bs, t, bE, n);
        } else {
            auto go = [&](auto H) {
                constexpr bool NT = decltype(H)::value;
                if constexpr (W == 4) {
                    if (total[kPhH]) hipLaunchKernelGGL((k_bh3_all<T, W, NT>), dim3(total[kPhH]), blk, 0, bs, t, bH, n);
                    if (total[kPhE]) hipLaunchKernelGGL((k_be3_all<T, W, NT>), dim3(total[kPhE]), blk, 0, bs, t, bE, n);
                } else {
                    if (total[kPhH]) hipLaunchKernelGGL((k_bh3_int<T, W, NT>), dim3(total[kPhH]), blk, 0, bs, t, bH, n);
                    if (total[kPhHs]) hipLaunchKernelGGL((k_bh3_slab<T, W, NT>), dim3(total[kPhHs]), blk, 0, bs, t, bHs, n);
                    if (total[kPhE]) hipLaunchKernelGGL((k_be3_int<T, W, NT>), dim3(total[kPhE]), blk, 0, bs, t, bE, n);
                    if (total[kPhEs]) hipLaunchKernelGGL((k_be3_slab<T, W, NT>), dim3(total[kPhEs]), blk, 0, bs, t, bEs, n);
                }
            };
            if (stream_hint) go(std::true_type{});
            else go(std::false_type{});
        }
        // emitters per simulation, on the batch stream, between the E update and the sampling
        for (int i = 0; i < n; ++i) {
            chiml_dev* c = g[i];
            if (c->qes.empty()) continue;
            StepArgs<T>& a = step_args<T>(c);
            const int p = (c->steps_done + j) & 1;
            int* ctr = c->step_ctr.as<int>();
            a.step = ctr + p;
            a.stepv = -1;
            a.step_next = nullptr;
            const hipStream_t own = c->stream;
            c->stream = bs;
            launch_ml<T>(c, a, false);
            c->stream = own;
        }
        if (total[kPhS]) hipLaunchKernelGGL((k_bsample<T>), dim3(total[kPhS]), blk, 0, bs, t, bS, n);
        // DFT flushes decide on the device whether their block of samples is complete
        for (int i = 0; i < n; ++i) {
            chiml_dev* c = g[i];
            const int p = (c->steps_done + j) & 1;
            int* ctr = c->step_ctr.as<int>();
            for (const chiml_dev::DftGroup& d : c->dgs) {
                if (d.n == 0) continue;
                hipLaunchKernelGGL(k_dft_flush<T>, dim3((d.n + 255) / 256), blk, 0, bs, static_cast<const T*>(d.stage), d.phasor, d.F,
                                   ctr + (1 - p), d.n, d.nfreq, d.interval, 0, -1);
            }
        }
        HIP_TRY(hipGetLastError());
    }
    for (int i = 0; i < n; ++i) {
        StepArgs<T>& a = step_args<T>(g[i]);
        a.stepv = -1;
        a.step_next = nullptr;
        g[i]->steps_done += nsteps;
        g[i]->enq_step = g[i]->steps_done;
    }
}

// chiml_dev_step_batch(_noalloc): contexts of one kernel class and
// precision share every field and sample launch; the others step on their
// own streams.  The batch runs on the first batched context's stream, joined
// with the other contexts' streams by events before and after.
int step_batch(chiml_dev** ctxs, int n, int nsteps, bool noalloc) {
    if (!ctxs || n < 0 || nsteps < 0) return fail(nullptr, CHIML_E_INVALID, "invalid argument");
    if (noalloc && n > kBatchMaxSlots)
        return fail(nullptr, CHIML_E_INVALID, "chiml_dev_step_batch_noalloc: more than 64 simulations in one call");
    for (int i = 0; i < n; ++i) {
        if (!ctxs[i]) return fail(nullptr, CHIML_E_INVALID, "null context in batch");
        for (int k = 0; k < i; ++k)
            if (ctxs[k] == ctxs[i]) return fail(nullptr, CHIML_E_INVALID, "a context appears twice in one batch");
        if (ctxs[i]->steps_done + nsteps > ctxs[i]->nsteps) return fail(ctxs[i], CHIML_E_STATE, "step count exceeds the per-step tables built at create");
        if (ctxs[i]->device != ctxs[0]->device) return fail(nullptr, CHIML_E_INVALID, "a batch must share one device");
    }
    if (n == 0 || nsteps == 0) return CHIML_OK;
    try {
        chiml_dev* grp[4][kBatchMaxSlots];
        int ng[4] = {0, 0, 0, 0};
        size_t off = 0;  // the groups of one call take consecutive parts of the scratch and host image
        // the shared launches of one group (class x precision)
        auto run_group = [&](int gi) {
            const int m = ng[gi];
            ng[gi] = 0;
            if (m == 0) return;
            std::lock_guard<std::mutex> lk(g_batch_mu);
            chiml_dev** g = grp[gi];
            const hipStream_t bs = g[0]->stream;
            for (int i = 1; i < m; ++i) {
                HIP_TRY(hipEventRecord(g[i]->ev, g[i]->stream));
                HIP_TRY(hipStreamWaitEvent(bs, g[i]->ev, 0));
            }
            const bool fp32 = (gi & 1) == 0;
            const size_t bytes = 2 * m * (fp32 ? sizeof(BatchSlot<float>) : sizeof(BatchSlot<double>)) + kPhases * (m + 1) * sizeof(int);
            unsigned char* dev = nullptr;
            size_t at = (off + 255) / 256 * 256;
            if (at + bytes > kBatchScratchBytes) {
                // only the allocating form gets here (more than 64 per call): its
                // tables have their own device buffer, and the host image is
                // consumed by the copy before the call returns
                if (noalloc) throw std::runtime_error("batch tables exceed the scratch size");
                at = 0;
            }
            if (bytes > kBatchScratchBytes) throw std::runtime_error("batch tables exceed the host image size");
            off = at + bytes;
            if (noalloc) {
                dev = static_cast<unsigned char*>(scratch_on(g[0]->device)) + at;
            } else {
                HIP_TRY(hipMallocAsync(reinterpret_cast<void**>(&dev), bytes, bs));
            }
            if (fp32) batch_group<float>(g, m, nsteps, bs, dev, g_batch_host + at);
            else batch_group<double>(g, m, nsteps, bs, dev, g_batch_host + at);
            if (!noalloc) HIP_TRY(hipFreeAsync(dev, bs));
            HIP_TRY(hipEventRecord(g[0]->ev, bs));
            for (int i = 1; i < m; ++i) HIP_TRY(hipStreamWaitEvent(g[i]->stream, g[0]->ev, 0));
        };
        // groups: (class 1 or 2) x (FP32, FP64)
        for (int i = 0; i < n; ++i) {
            chiml_dev* c = ctxs[i];
            const int cls = batch_class(c);
            if (cls == 0) {  // stepped alone
                enqueue_steps(c, nsteps);
                continue;
            }
            const int gi = (cls - 1) * 2 + (c->prec == 32 ? 0 : 1);
            if (ng[gi] == kBatchMaxSlots) run_group(gi);  // a full group: step it and start another
            grp[gi][ng[gi]++] = c;
        }
        for (int gi = 0; gi < 4; ++gi) run_group(gi);
    } catch (std::exception& e) {
        return fail(nullptr, CHIML_E_HIP, e.what());
    }
    return CHIML_OK;
}
}  // namespace

namespace {
// Integer knob from the environment (tuning sweeps of the fused launch
// shape; 0 or unset keeps the default).
int env_int(const char* name) {
    const char* v = std::getenv(name);
    return v ? std::atoi(v) : 0;
}
}  // namespace

// Fused 3D step (k_fused3): tiles of ty whole x rows (plus the recomputed
// row below), segments of lz planes, one tile-segment per block; enough
// segments for about two blocks per CU.  Needs the whole x row of a tile
// plane in one block and a second buffer for every field and H psi array.
// It moves the compulsory bytes only (1.10x of them on the 256^3 deck) but
// runs at one 9-wave block per CU with a barrier per plane, and measured
// 0.39 ms per step against 0.29 ms for the split sweeps, so it is opt-in:
// CHIML_FUSED=1 selects it (both do the whole step);
// CHIML_FUSED_TY / CHIML_FUSED_LZ set the tile shape.
template <typename T>
void enable_fused(chiml_dev* c, const chiml_problem_t* p, StepArgs<T>& a, SampleArgs<T>& s) {
    constexpr int W = 16 / sizeof(T);
    const char* on = std::getenv("CHIML_FUSED");
    if (!on || std::atoi(on) != 1) return;
    if (!c->tfsf.empty() || c->cells.n > 0) return;  // TFSF and per-cell source adds sit between the H and E updates
    const int nx = p->nx, ny = p->ny, nz = p->nz;
    if (nx % W != 0 || p->pml_T[0] % W != 0 || c->hmap) return;
    FuseMap m{};
    m.gx = nx / W;
    int ty = env_int("CHIML_FUSED_TY");
    if (ty <= 0) ty = 8;
    ty = std::min(ty, kFusedMaxThreads / m.gx - 1);
    if (ty < 1) return;
    m.ty = ty;
    m.ntile = (ny + ty - 1) / ty;
    int lz = env_int("CHIML_FUSED_LZ");
    if (lz <= 0) {
        const int nseg = std::max(1, std::min(nz, (512 + m.ntile - 1) / m.ntile));
        lz = (nz + nseg - 1) / nseg;
    }
    m.lz = std::min(lz, nz);
    m.nseg = (nz + m.lz - 1) / m.lz;
    m.nthr = (ty + 1) * m.gx;
    // rows and planes inside every component's y / z psi-free range
    m.ys0 = 0; m.ys1 = ny; m.zs0 = 0; m.zs1 = nz;
    for (int comp = 0; comp < 6; ++comp) {
        const PmlDev<T>& pm = a.pml[comp];
        if (pm.psi[1]) { m.ys0 = std::max(m.ys0, pm.lo[1]); m.ys1 = std::min(m.ys1, pm.hi0[1]); }
        if (pm.psi[2]) { m.zs0 = std::max(m.zs0, pm.lo[2]); m.zs1 = std::min(m.zs1, pm.hi0[2]); }
    }
    for (int comp = 0; comp < 6; ++comp)
        for (int ax = 0; ax < 3; ++ax)
            if (a.pml[comp].psi[ax] && a.pml[comp].S[ax] > kFusedSlab) return;  // profiles must fit the LDS table
    const int nxp = (a.pml[4].psi[0] != nullptr) + (a.pml[5].psi[0] != nullptr) + (a.pml[1].psi[0] != nullptr) + (a.pml[2].psi[0] != nullptr);
    if (nxp != 0 && nxp != 4) return;
    m.xpsi = nxp == 4 ? 1 : 0;
    const size_t lds = 2ull * 3 * (ty + 1) * nx * sizeof(T);
    int lds_max = 0;
    HIP_TRY(hipDeviceGetAttribute(&lds_max, hipDeviceAttributeMaxSharedMemoryPerBlock, c->device));
    if (lds + sizeof(MatLds<T>) * 3 * CHIML_MAX_MAT + sizeof(SrcLds<T>) + sizeof(ProfLds<T>) > static_cast<size_t>(lds_max)) return;
    const size_t N = static_cast<size_t>(nx) * ny * nz;
    // byte offsets within a buffer of six components are 32-bit in the kernel
    if (6 * N * sizeof(T) >= (1ull << 32)) return;
    T* second = c->zeros<T>(6 * N);
    for (int k = 0; k < 6; ++k) {
        c->fbuf[0][k] = a.F[k];
        c->fbuf[1][k] = second + k * N;
    }
    m.cstride = static_cast<unsigned>(N * sizeof(T));
    const int nn[3] = {nx, ny, nz};
    for (int h = 0; h < 3; ++h)
        for (int ax = 0; ax < 3; ++ax) {
            const PmlDev<T>& pm = a.pml[3 + h];
            c->fpsi[0][h][ax] = pm.psi[ax];
            c->fpsi[1][h][ax] = nullptr;
            if (pm.psi[ax]) {
                size_t ps = static_cast<size_t>(pm.S[ax]);
                for (int o = 0; o < 3; ++o)
                    if (o != ax) ps *= nn[o];
                c->fpsi[1][h][ax] = c->zeros<T>(ps);
            }
        }
    c->fmap = m;
    c->fused_lds = lds;
    c->fused = true;
    set_fused_buffers<T>(c, a, s, -1);
}

namespace {
int fail(chiml_dev* c, int code, const std::string& msg) {
    if (c) c->err = msg;
    g_err = msg;
    return code;
}

}  // namespace

extern "C" {

int chiml_dev_create(const chiml_problem_t* p, chiml_dev_t** out) {
    if (!p || !out) return fail(nullptr, CHIML_E_INVALID, "null argument");
    *out = nullptr;
    if (p->nx < 2 || p->ny < 2 || p->nz < 1) return fail(nullptr, CHIML_E_INVALID, "grid too small");
    if (p->precision != 32 && p->precision != 64) return fail(nullptr, CHIML_E_INVALID, "precision must be 32 or 64");
    if (p->nsteps < 0) return fail(nullptr, CHIML_E_INVALID, "nsteps must be >= 0");
    if (p->nsrc > CHIML_MAX_SRC) return fail(nullptr, CHIML_E_INVALID, "too many sources");
    std::lock_guard<std::mutex> lk(g_capture_mu);
    auto c = std::make_unique<chiml_dev>();
    try {
        int ndev = 0;
        HIP_TRY(hipGetDeviceCount(&ndev));
        if (ndev < 1) throw std::runtime_error("no HIP device");
        HIP_TRY(hipGetDevice(&c->device));
        HIP_TRY(hipStreamCreateWithFlags(&c->stream, hipStreamNonBlocking));
        HIP_TRY(hipEventCreateWithFlags(&c->ev, hipEventDisableTiming));
        c->prec = p->precision;
        c->nx = p->nx;
        c->ny = p->ny;
        c->nz = p->nz;
        c->dim = p->nz > 1 ? 3 : 2;
        c->nsteps = p->nsteps;
        c->step_ctr.alloc(2 * sizeof(int), c->stream, true);
        if (c->prec == 32) build<float>(c.get(), p, c->a32, c->s32);
        else build<double>(c.get(), p, c->a64, c->s64);
        if (c->dim == 2) {
            const int W = c->prec == 32 ? 4 : 2;
            c->vec2d = c->vec;
            // the E kernel samples the point detectors when each point reads one
            // cell of Ez, Hx or Hy and there are few of them (every thread scans
            // the list), no flux box needs the sample launch anyway, no emitter
            // changes E after the E kernel (the back-coupling runs later), and
            // the grid is small enough for the saved launch to outweigh the scan
            // (256^2: 9.9 -> 8.6 us per step; 1024^2: 12.7 -> 13.5 us, so not there)
            bool single = c->det_single_field && c->totpts > 0 && c->totpts <= 32 && c->ndft == 0 && c->qes.empty() &&
                          static_cast<long long>(p->nx) * p->ny <= 512LL * 512;
            for (int t = 0; single && t < c->totpts; ++t) {
                const int cu = p->det_comp[2 * t];
                single = cu == p->det_comp[2 * t + 1] && p->det_cell[2 * t] == p->det_cell[2 * t + 1] && cu >= 2 && cu <= 4;
            }
            c->fuse_sample = c->vec2d && !c->cellwise && single;
            if (c->prec == 32) enable_tiles<float>(c.get(), p, c->a32, c->s32);
            else enable_tiles<double>(c.get(), p, c->a64, c->s64);
        }
        if (c->dim == 3) {
            const int Tx = p->pml_T[0], Ty = p->pml_T[1], Tz = p->pml_T[2];
            // rows: the interior walk takes whole x rows of the y/z interior
            // (the x slabs' CPML terms applied inline) and the slab region
            // covers the z and y slabs; else the x slabs stay in the slab region.
            Box3 b{c->rows ? 0 : Tx, c->rows ? c->px : p->nx - Tx, Ty, p->ny - Ty, Tz, p->nz - Tz, 0};
            b.by = (b.y1 - b.y0 + 7) / 8;  // one y band per XCD
            const int W = c->prec == 32 ? 4 : 2;
            if (c->split) {
                c->ibox = b;
                if (c->prec == 32) enable_fused<float>(c.get(), p, c->a32, c->s32);
                SlabMap& m = c->slab;
                m.nx = c->px; m.ny = p->ny; m.nz = p->nz;
                m.Tx = Tx; m.Ty = Ty; m.Tz = Tz;
                m.W = W;
                const long long gx = c->px / W;
                m.nA = static_cast<unsigned>(2LL * Tz * gx * p->ny);
                m.nB = static_cast<unsigned>(2LL * Ty * gx * (p->nz - 2 * Tz));
                m.nC = c->rows ? 0 : static_cast<unsigned>(2LL * (Tx / W) * (p->ny - 2 * Ty) * (p->nz - 2 * Tz));

                for (int k = 0; k < 3; ++k) {
                    const int* bx = c->prec == 32 ? c->a32.box[k] : c->a64.box[k];
                    const bool has = c->prec == 32 ? c->a32.jsum[k] != nullptr : c->a64.jsum[k] != nullptr;
                    if (has)
                        c->ade_groups = std::max(c->ade_groups, static_cast<long long>((bx[1] - bx[0]) / W) * (bx[3] - bx[2]) * (bx[5] - bx[4]));
                }
            }
        }
        // t = 0 samples (taken by the reference's constructor, parallelFDTDField.cpp:832-837)
        if (c->prec == 32) {
            launch_sample<float>(c.get(), c->s32);
        } else {
            launch_sample<double>(c.get(), c->s64);
        }
        HIP_TRY(hipGetLastError());
        HIP_TRY(hipStreamSynchronize(c->stream));
    } catch (std::exception& e) {
        return fail(nullptr, CHIML_E_HIP, e.what());
    }
    *out = c.release();
    return CHIML_OK;
}

namespace {
void sweep_steps(chiml_dev* c, int n) {
    if (c->prec == 32) do_steps<float>(c, c->a32, c->s32, n);
    else do_steps<double>(c, c->a64, c->s64, n);
}

void enqueue_steps(chiml_dev* c, int n) {
    if (n == 0) return;
    if (!c->tile || !tile_pays(c, n)) sweep_steps(c, n);
    else if (c->prec == 32) do_tile_steps<float>(c, c->a32, c->s32, n);
    else do_tile_steps<double>(c, c->a64, c->s64, n);
}

// Captures graph_steps steps of this context's launch sequence once; every
// launch reads the step number from the device counter, so one graph serves
// every chunk of the run that starts on the same buffers.
void ensure_graph(chiml_dev* c) {
    hipGraphExec_t& exec = c->gexec[c->tile_cur];
    if (exec) return;
    std::lock_guard<std::mutex> lk(g_capture_mu);
    hipGraph_t g = nullptr;
    const int saved = c->steps_done, saved_enq = c->enq_step;
    c->graph_parity[c->tile_cur] = c->steps_done & 1;
    HIP_TRY(hipStreamBeginCapture(c->stream, hipStreamCaptureModeThreadLocal));
    c->capturing = true;
    try {
        c->graph_tiles = c->tile && tile_pays(c, c->graph_steps);
        enqueue_steps(c, c->graph_steps);
    } catch (...) {
        c->capturing = false;
        (void)hipStreamEndCapture(c->stream, &g);
        if (g) (void)hipGraphDestroy(g);
        c->steps_done = saved;
        throw;
    }
    c->capturing = false;
    HIP_TRY(hipStreamEndCapture(c->stream, &g));
    c->steps_done = saved;  // capture enqueued nothing (and tile launches ended on the buffers they started on)
    c->enq_step = saved_enq;
    hipError_t e = hipGraphInstantiate(&exec, g, nullptr, nullptr, 0);
    (void)hipGraphDestroy(g);
    HIP_TRY(e);
}
}  // namespace

int chiml_dev_step(chiml_dev_t* c, int n) {
    if (!c || n < 0) return fail(c, CHIML_E_INVALID, "invalid argument");
    if (c->steps_done + n > c->nsteps) return fail(c, CHIML_E_STATE, "step count exceeds the per-step tables built at create");
    try {
        if (c->graph_steps > 0) {
            while (n >= c->graph_steps) {
                ensure_graph(c);
                if (!c->graph_tiles && (c->steps_done & 1) != c->graph_parity[c->tile_cur]) {
                    sweep_steps(c, 1);  // realign the counter slot with one plain step
                    --n;
                    continue;
                }
                HIP_TRY(hipGraphLaunch(c->gexec[c->tile_cur], c->stream));
                c->steps_done += c->graph_steps;
                n -= c->graph_steps;
            }
        }
        if (n > 0) enqueue_steps(c, n);
        if (c->profile) collect_profile(c);
    } catch (std::exception& e) {
        return fail(c, CHIML_E_HIP, e.what());
    }
    return CHIML_OK;
}

int chiml_dev_set_graph(chiml_dev_t* c, int steps_per_graph) {
    if (!c || steps_per_graph < 0) return fail(c, CHIML_E_INVALID, "invalid argument");
    for (hipGraphExec_t& e : c->gexec) {
        if (e) (void)hipGraphExecDestroy(e);
        e = nullptr;
    }
    // even, so that every replay starts on the counter slot the graph was captured on
    c->graph_steps = steps_per_graph + (steps_per_graph & 1);
    c->device_flush = steps_per_graph > 0;
    // graphs of tiles and of sweeps leave different slots current
    if (c->tile) hipLaunchKernelGGL(k_set_step, dim3(1), dim3(1), 0, c->stream, c->step_ctr.as<int>(), c->steps_done);
    return CHIML_OK;
}

int chiml_dev_query(chiml_dev_t* c, int* idle) {
    if (!c || !idle) return fail(c, CHIML_E_INVALID, "invalid argument");
    hipError_t e = hipStreamQuery(c->stream);
    if (e == hipSuccess) *idle = 1;
    else if (e == hipErrorNotReady) *idle = 0;
    else return fail(c, CHIML_E_HIP, hipGetErrorString(e));
    return CHIML_OK;
}

int chiml_dev_step_batch(chiml_dev_t** ctxs, int n, int nsteps) { return step_batch(ctxs, n, nsteps, false); }

int chiml_dev_step_batch_noalloc(chiml_dev_t** ctxs, int n, int nsteps) { return step_batch(ctxs, n, nsteps, true); }

int chiml_dev_sync(chiml_dev_t* c) {
    if (!c) return fail(nullptr, CHIML_E_INVALID, "null context");
    hipError_t e = hipStreamSynchronize(c->stream);
    if (e != hipSuccess) return fail(c, CHIML_E_HIP, hipGetErrorString(e));
    return CHIML_OK;
}

int chiml_dev_read_field(chiml_dev_t* c, int comp, double* host) {
    if (!c || !host || comp < 0 || comp > 5) return fail(c, CHIML_E_INVALID, "invalid argument");
    const size_t nr = static_cast<size_t>(c->ny) * c->nz, N = static_cast<size_t>(c->nx) * nr, Np = static_cast<size_t>(c->px) * nr;
    std::lock_guard<std::mutex> lk(g_capture_mu);
    try {
        HIP_TRY(hipStreamSynchronize(c->stream));
        if (!(c->prec == 32 ? static_cast<void*>(c->a32.F[comp]) : static_cast<void*>(c->a64.F[comp]))) {
            std::memset(host, 0, N * sizeof(double));
            return CHIML_OK;
        }
        // rows leave their padding behind
        if (c->prec == 32) {
            std::vector<float> tmp(Np);
            HIP_TRY(hipMemcpy(tmp.data(), c->a32.F[comp], Np * sizeof(float), hipMemcpyDeviceToHost));
            for (size_t r = 0; r < nr; ++r)
                for (int x = 0; x < c->nx; ++x) host[r * c->nx + x] = tmp[r * c->px + x];
        } else if (c->px == c->nx) {
            HIP_TRY(hipMemcpy(host, c->a64.F[comp], N * sizeof(double), hipMemcpyDeviceToHost));
        } else {
            std::vector<double> tmp(Np);
            HIP_TRY(hipMemcpy(tmp.data(), c->a64.F[comp], Np * sizeof(double), hipMemcpyDeviceToHost));
            for (size_t r = 0; r < nr; ++r) std::copy(tmp.data() + r * c->px, tmp.data() + r * c->px + c->nx, host + r * c->nx);
        }
    } catch (std::exception& e) {
        return fail(c, CHIML_E_HIP, e.what());
    }
    return CHIML_OK;
}

int chiml_dev_read_points(chiml_dev_t* c, int d, double* values, size_t cap, size_t* nsamples) {
    if (!c || d < 0 || d >= c->ndet || !nsamples) return fail(c, CHIML_E_INVALID, "invalid argument");
    int ns = c->steps_done / c->det_interval[d] + 1;
    if (ns > c->det_cap[d]) ns = c->det_cap[d];
    *nsamples = static_cast<size_t>(ns);
    size_t n = static_cast<size_t>(ns) * c->det_npts[d];
    if (!values) return CHIML_OK;
    if (cap < n) return fail(c, CHIML_E_INVALID, "buffer too small");
    std::lock_guard<std::mutex> lk(g_capture_mu);
    try {
        HIP_TRY(hipStreamSynchronize(c->stream));
        HIP_TRY(hipMemcpy(values, c->det_out + c->det_out_off[d], n * sizeof(double), hipMemcpyDeviceToHost));
    } catch (std::exception& e) {
        return fail(c, CHIML_E_HIP, e.what());
    }
    return CHIML_OK;
}

}  // extern "C"
namespace {
// The accumulators of group d with the samples of the open block added (in
// d.tmp, leaving F as it is), enqueued on the context's stream.
const double* dft_with_open_block(chiml_dev* c, const chiml_dev::DftGroup& d) {
    const int kmax = c->steps_done / d.interval;
    if ((kmax % kDftBlock) == kDftBlock - 1) return d.F;  // no open block
    const size_t n = 2 * static_cast<size_t>(d.n) * d.nfreq;
    HIP_TRY(hipMemcpyAsync(d.tmp, d.F, n * sizeof(double), hipMemcpyDeviceToDevice, c->stream));
    const int last = kmax * d.interval;
    if (c->prec == 32)
        hipLaunchKernelGGL(k_dft_flush<float>, dim3((d.n + 255) / 256), dim3(256), 0, c->stream, static_cast<const float*>(d.stage),
                           d.phasor, d.tmp, c->step_ctr.as<int>(), d.n, d.nfreq, d.interval, 1, last);
    else
        hipLaunchKernelGGL(k_dft_flush<double>, dim3((d.n + 255) / 256), dim3(256), 0, c->stream, static_cast<const double*>(d.stage),
                           d.phasor, d.tmp, c->step_ctr.as<int>(), d.n, d.nfreq, d.interval, 1, last);
    HIP_TRY(hipGetLastError());
    return d.tmp;
}
}  // namespace
extern "C" {

int chiml_dev_read_dft_group(chiml_dev_t* c, int g, double* reim, size_t cap) {
    if (!c) return fail(nullptr, CHIML_E_INVALID, "null context");
    if (g < 0 || g >= static_cast<int>(c->dgs.size())) return fail(c, CHIML_E_INVALID, "DFT group index out of range");
    const chiml_dev::DftGroup& d = c->dgs[g];
    size_t n = 2 * static_cast<size_t>(d.n) * d.nfreq;
    if (n == 0) return CHIML_OK;
    if (!reim || cap < n) return fail(c, CHIML_E_INVALID, "buffer too small");
    std::lock_guard<std::mutex> lk(g_capture_mu);
    try {
        std::vector<double> host(n);
        const double* F = dft_with_open_block(c, d);
        HIP_TRY(hipStreamSynchronize(c->stream));
        HIP_TRY(hipMemcpy(host.data(), F, n * sizeof(double), hipMemcpyDeviceToHost));
        // device layout [f][s] -> ABI layout [s][f]
        for (int f = 0; f < d.nfreq; ++f)
            for (int sm = 0; sm < d.n; ++sm) {
                reim[2 * (static_cast<size_t>(sm) * d.nfreq + f)] = host[2 * (static_cast<size_t>(f) * d.n + sm)];
                reim[2 * (static_cast<size_t>(sm) * d.nfreq + f) + 1] = host[2 * (static_cast<size_t>(f) * d.n + sm) + 1];
            }
    } catch (std::exception& e) {
        return fail(c, CHIML_E_HIP, e.what());
    }
    return CHIML_OK;
}

int chiml_dev_flux_plan(chiml_dev_t* c, int nface, const int* npt, const int* const* ids, const double* cw, const double* const* sw, int* plan) {
    if (!c) return fail(nullptr, CHIML_E_INVALID, "null context");
    if (nface < 1 || nface > kFluxFaces || !npt || !ids || !cw || !sw || !plan) return fail(c, CHIML_E_INVALID, "invalid argument");
    if (c->dgs.empty() || c->dgs[0].n == 0) return fail(c, CHIML_E_INVALID, "no flux samples");
    std::lock_guard<std::mutex> lk(g_capture_mu);
    const size_t held = c->bufs.size(), footprint = c->footprint;
    try {
        chiml_dev::FluxPlan pl;
        FluxPlanDev& d = pl.dev;
        d.nface = nface;
        for (int f = 0; f < nface; ++f) {
            if (npt[f] < 0) throw std::invalid_argument("flux plan: point count");
            d.npt[f] = npt[f];
            d.start[f + 1] = d.start[f] + (npt[f] + 255) / 256 * 256;
            for (int k = 0; k < 4; ++k) d.cw[f][k] = cw[4 * f + k];
        }
        const size_t total = d.start[nface];
        std::vector<int> hi(16 * std::max<size_t>(total, 1), -1);
        std::vector<double> hw(std::max<size_t>(total, 1), 0.0);
        for (int f = 0; f < nface; ++f)
            for (int p = 0; p < npt[f]; ++p) {
                hw[d.start[f] + p] = sw[f][p];
                for (int k = 0; k < 16; ++k) {
                    const int id = ids[f][static_cast<size_t>(k) * npt[f] + p];
                    if (id >= c->dgs[0].n) throw std::invalid_argument("flux plan: sample index out of range");
                    hi[k * total + d.start[f] + p] = id;
                }
            }
        d.ids = c->upload<int>(hi.data(), hi.size());
        d.sw = c->upload<double>(hw.data(), hw.size());
        pl.blocks = static_cast<int>(total / 256);
        pl.partial = reinterpret_cast<double2*>(c->zeros<double>(2 * static_cast<size_t>(std::max(pl.blocks, 1)) * c->dgs[0].nfreq));
        *plan = static_cast<int>(c->flux_plans.size());
        c->flux_plans.push_back(pl);
    } catch (std::invalid_argument& e) {
        return fail(c, CHIML_E_INVALID, e.what());
    } catch (std::exception& e) {
        (void)hipGetLastError();
        c->bufs.resize(held);
        c->footprint = footprint;
        return fail(c, CHIML_E_HIP, e.what());
    }
    return CHIML_OK;
}

int chiml_dev_flux(chiml_dev_t* c, int plan, double nt, double* reim) {
    if (!c) return fail(nullptr, CHIML_E_INVALID, "null context");
    if (plan < 0 || plan >= static_cast<int>(c->flux_plans.size()) || !reim) return fail(c, CHIML_E_INVALID, "invalid argument");
    const chiml_dev::FluxPlan& pl = c->flux_plans[plan];
    const chiml_dev::DftGroup& d = c->dgs[0];
    const int nf = d.nfreq, nb = pl.blocks;
    std::fill(reim, reim + 2 * static_cast<size_t>(pl.dev.nface) * nf, 0.0);
    if (nb == 0) return CHIML_OK;
    std::lock_guard<std::mutex> lk(g_capture_mu);
    try {
        const double* F = dft_with_open_block(c, d);
        hipLaunchKernelGGL(k_flux_faces, dim3(nb, nf), dim3(256), 0, c->stream, pl.dev, reinterpret_cast<const double2*>(F), d.n, 1.0 / (nt * nt),
                           pl.partial);
        HIP_TRY(hipGetLastError());
        HIP_TRY(hipStreamSynchronize(c->stream));
        std::vector<double2> part(static_cast<size_t>(nb) * nf);
        HIP_TRY(hipMemcpy(part.data(), pl.partial, part.size() * sizeof(double2), hipMemcpyDeviceToHost));
        for (int fc = 0; fc < pl.dev.nface; ++fc)
            for (int f = 0; f < nf; ++f)
                for (int b = pl.dev.start[fc] / 256; b < pl.dev.start[fc + 1] / 256; ++b) {
                    reim[2 * (static_cast<size_t>(fc) * nf + f)] += part[static_cast<size_t>(f) * nb + b].x;
                    reim[2 * (static_cast<size_t>(fc) * nf + f) + 1] += part[static_cast<size_t>(f) * nb + b].y;
                }
    } catch (std::exception& e) {
        return fail(c, CHIML_E_HIP, e.what());
    }
    return CHIML_OK;
}

int chiml_dev_read_dft(chiml_dev_t* c, double* reim, size_t cap) { return chiml_dev_read_dft_group(c, 0, reim, cap); }

int chiml_dev_read_incd(chiml_dev_t* c, int comp, double* reim, size_t cap, size_t* n) {
    if (!c || comp < 0 || comp > 5 || !n) return fail(c, CHIML_E_INVALID, "invalid argument");
    const long long nrec = c->incd_rec ? c->nrec : 2LL * (c->nsteps + 1) + 2;
    *n = static_cast<size_t>(nrec);
    if (!reim) return CHIML_OK;
    if (cap < 2 * static_cast<size_t>(nrec)) return fail(c, CHIML_E_INVALID, "buffer too small");
    if (!c->incd_rec) {
        std::fill(reim, reim + 2 * nrec, 0.0);
        return CHIML_OK;
    }
    std::lock_guard<std::mutex> lk(g_capture_mu);
    try {
        HIP_TRY(hipStreamSynchronize(c->stream));
        HIP_TRY(hipMemcpy(reim, c->incd_rec + static_cast<size_t>(comp) * nrec, 2 * nrec * sizeof(double), hipMemcpyDeviceToHost));
    } catch (std::exception& e) {
        return fail(c, CHIML_E_HIP, e.what());
    }
    return CHIML_OK;
}

int chiml_dev_read_pops(chiml_dev_t* c, int q, int j, double* reim, size_t cap, size_t* nsamples) {
    if (!c || q < 0 || q >= static_cast<int>(c->qes.size()) || !nsamples) return fail(c, CHIML_E_INVALID, "invalid argument");
    QeDev& d = c->qes[q].dev;
    if (j < 0 || j >= c->qes[q].npop_all) return fail(c, CHIML_E_INVALID, "population detector index out of range");
    int ns = (c->steps_done - 1) / d.pop_interval + 1;
    if (c->steps_done == 0) ns = 0;
    if (ns > d.pop_cap) ns = d.pop_cap;
    *nsamples = static_cast<size_t>(ns);
    if (!reim) return CHIML_OK;
    if (cap < 2 * static_cast<size_t>(ns)) return fail(c, CHIML_E_INVALID, "buffer too small");
    std::lock_guard<std::mutex> lk(g_capture_mu);
    try {
        HIP_TRY(hipStreamSynchronize(c->stream));
        HIP_TRY(hipMemcpy(reim, d.pop_out + static_cast<size_t>(j) * d.pop_cap, 2 * ns * sizeof(double), hipMemcpyDeviceToHost));
    } catch (std::exception& e) {
        return fail(c, CHIML_E_HIP, e.what());
    }
    return CHIML_OK;
}

int chiml_dev_read_density(chiml_dev_t* c, int q, int m, int e, double* reim) {
    if (!c || q < 0 || q >= static_cast<int>(c->qes.size()) || !reim) return fail(c, CHIML_E_INVALID, "invalid argument");
    QeDev& d = c->qes[q].dev;
    if (m < 0 || m >= d.nmem || e < 0 || e >= d.nemit) return fail(c, CHIML_E_INVALID, "index out of range");
    const int S = d.N * d.N;
    const size_t ld = static_cast<size_t>(d.nmem) * d.nemit;
    std::lock_guard<std::mutex> lk(g_capture_mu);
    try {
        HIP_TRY(hipStreamSynchronize(c->stream));
        for (int k = 0; k < S; ++k) {
            const int i = k % d.N, j = k / d.N;
            // packed: entry (i, j) stored for i <= j; below the diagonal the conjugate of (j, i)
            const int ks = !d.packed ? k : (i <= j ? j * (j + 1) / 2 + i : i * (i + 1) / 2 + j);
            HIP_TRY(hipMemcpy(reim + 2 * k, d.rho + ks * ld + static_cast<size_t>(m) * d.nemit + e, sizeof(double2), hipMemcpyDeviceToHost));
            if (d.packed && i > j) reim[2 * k + 1] = -reim[2 * k + 1];
        }
    } catch (std::exception& ex) {
        return fail(c, CHIML_E_HIP, ex.what());
    }
    return d.N;
}

int chiml_dev_steps_done(chiml_dev_t* c, int* steps) {
    if (!c || !steps) return fail(c, CHIML_E_INVALID, "invalid argument");
    *steps = c->steps_done;
    return CHIML_OK;
}

int chiml_dev_profile(chiml_dev_t* c, int enable) {
    if (!c) return fail(nullptr, CHIML_E_INVALID, "null context");
    collect_profile(c);
    c->profile = enable != 0;
    c->profile_only.clear();
    c->prof.clear();
    return CHIML_OK;
}

int chiml_dev_profile_only(chiml_dev_t* c, const char* kernel) {
    if (!c || !kernel) return fail(c, CHIML_E_INVALID, "invalid argument");
    collect_profile(c);
    c->profile = true;
    c->profile_only = kernel;
    c->prof.clear();
    return CHIML_OK;
}

int chiml_dev_profile_read(chiml_dev_t* c, const char* kernel, double* total_ms, int* launches) {
    if (!c || !kernel || !total_ms || !launches) return fail(c, CHIML_E_INVALID, "invalid argument");
    collect_profile(c);
    auto it = c->prof.find(kernel);
    *total_ms = it == c->prof.end() ? 0.0 : it->second.first;
    *launches = it == c->prof.end() ? 0 : it->second.second;
    return CHIML_OK;
}

int chiml_dev_footprint(chiml_dev_t* c, size_t* bytes) {
    if (!c || !bytes) return fail(c, CHIML_E_INVALID, "invalid argument");
    *bytes = c->footprint;
    return CHIML_OK;
}

const char* chiml_dev_last_error(const chiml_dev_t* c) { return c ? c->err.c_str() : g_err.c_str(); }
const char* chiml_dev_global_error(void) { return g_err.c_str(); }

void chiml_dev_destroy(chiml_dev_t* c) {
    if (!c) return;
    std::lock_guard<std::mutex> lk(g_capture_mu);
    (void)hipStreamSynchronize(c->stream);
    for (hipGraphExec_t e : c->gexec)
        if (e) (void)hipGraphExecDestroy(e);
    for (auto& pe : c->pending) {
        (void)hipEventDestroy(pe.e0);
        (void)hipEventDestroy(pe.e1);
    }
    c->bufs.clear();
    c->qes.clear();
    if (c->ev) (void)hipEventDestroy(c->ev);
    if (c->stream) (void)hipStreamDestroy(c->stream);
    delete c;
}

}  // extern "C"
