// afd_launch.hpp -- host-side launchers of the gfx950 kernels (one per kernel family).
#pragma once
#include <hip/hip_runtime.h>

#include "afd_kernels.hpp"

namespace afd {

// Arguments of a face-kernel launch in precision-neutral form.
struct FaceLaunch {
    const double *P;
    void *F, *Fcar, *zs;  // flux type: double (plain) or float (mixed)
    double *aux;
    Grid g;
    Phys<double> phd;
    Phys<float> phf;
    double p_max, v_max;
    int lim, recon, riemann, dir, diss;
    bool mixed;
    bool shared_edges;  // FP32 RMHD WENO5: the shared-edge kernels (afd_params.face_path == 0)
    float *D;           // FP32 RMHD WENO5 with shared edges: the flux-divergence accumulator (else null)
    bool dfirst;        // ... written by this launch (the stage's first face kernel), not added to
    float idn;          // 1 / spacing along dir
};

template <typename T> inline FaceArgs<T> face_args(const FaceLaunch &l) {
    FaceArgs<T> a;
    a.P = l.P;
    a.F = (T *)l.F;
    a.Fcar = (T *)l.Fcar;
    a.zs = (T *)l.zs;
    a.aux = l.aux;
    a.g = l.g;
    a.p_max = l.p_max;
    a.v_max = l.v_max;
    a.lim = l.lim;
    a.diss = l.diss;
    a.D = l.D;
    a.idn = l.idn;
    if constexpr (sizeof(T) == 8) a.ph = l.phd;
    else a.ph = l.phf;
    const int *r0 = l.g.r0, *r1 = l.g.r1;
    a.dk = make_udiv((unsigned)(r1[2] - r0[2] + (l.dir == 2 ? 1 : 0)));
    a.dn = make_udiv((unsigned)(l.dir == 0 ? r1[0] - r0[0] + 1 : r1[1] - r0[1] + (l.dir == 1 ? 1 : 0)));
    return a;
}

// Number of faces (threads) of the face box of direction dir.
inline long face_count(const Grid &g, int dir) {
    long n = 1;
    for (int a = 0; a < 3; ++a) n *= (long)(g.r1[a] - g.r0[a] + (a == dir ? 1 : 0));
    return n;
}

// SRHD MUSCL x and y faces go by runs (afd_srhd.hip) from RUN_FACES faces on, in one launch of one thread a face
// below.  Step (SSPRK2, HLLC) by runs over the merged launch, FP64 and mixed: 96^3 1.08 and 1.12, 128^3 (2.1 million
// faces) 1.00 and 1.01, 90 x 90 x 300 (2.5) 1.02 and 1.01, 144^3 (3.0) 1.01 and 0.99, 150^3 (3.4) 0.98 and 0.97,
// 152^3 (3.5) 0.96 and 0.95, 192^3 (7.1) 0.95 and 0.92; HLLE FP64 1.02 at 128^3, 1.00 at 144^3, 0.99 at 152^3.
constexpr long RUN_FACES = 3l << 20;

// The other schemes' directions share a launch below this many x faces.  Step (SSPRK2) merged over a launch each:
// RMHD FP64 MUSCL 0.82 at 64^3, 0.98 at 128^3, 0.987 at 150^3 (3.4 million faces), 0.992 at 168^3 (4.8), 0.994 to
// 0.998 above; PPM, where z stays by itself, 0.91, 0.987, 0.995 and 0.994, 1.00 at 224^3; WENO5 0.93, 0.987, 0.998
// and 0.999, 1.00 above; mixed PPM 0.89, 0.985, 0.997 and 0.996, above 0.995 to 1.00.  Mixed RMHD MUSCL loses from
// four million on: 0.87, 0.98, 0.98, 1.007 at 160^3 and 168^3, 1.02 at 176^3.  SRHD FP64 PPM 0.89 at 64^3, 0.97 at 152^3
// (3.5), 1.01 at 168^3 and 176^3, 1.00 at 256^3; WENO5 0.90, 0.98, 0.995 and 0.99, 1.00; mixed 0.89 to 0.90, 0.97 to 0.98,
// 0.97 to 0.99, 1.00.  (Medians of paired bursts, quartiles within 0.01.)
inline long merge_faces(bool rmhd, int recon, bool mixed) {
    if (recon == 0 && !rmhd) return RUN_FACES;
    return recon == 0 && mixed ? 7l << 19 : 9l << 19;
}

// The faces of one direction; y, z not null: l's (x) faces with those in one launch (k_faces_srhd, k_faces_rmhd).
hipError_t launch_face_srhd(const FaceLaunch &l, const FaceLaunch *y, hipStream_t s);
hipError_t launch_face_rmhd(const FaceLaunch &l, const FaceLaunch *y, const FaceLaunch *z, hipStream_t s);

// RMHD stage update / rhs-only launch.  flux pointers typed by `mixed`.
struct UpdLaunch {
    UpdArgs<double> a;  // flux pointers reinterpreted as float when mixed
    bool mixed;
};
hipError_t launch_update(const UpdLaunch &l, bool rhs_only, hipStream_t s);

// SRHD: the stage update with the z faces in it (l: the z faces), or with rhs_only the right-hand side
// into u.a.Pout.
hipError_t launch_update_srhd(const FaceLaunch &l, const UpdLaunch &u, bool rhs_only, hipStream_t s);

// The passives of a stage into a.out (contexts with passive fluxes: RMHD MUSCL, SRHD MUSCL and PPM).
hipError_t launch_passives(const PassiveArgs &a, bool rmhd, int recon, hipStream_t s);

// Mixed RMHD WENO5 on the flux-divergence path: the y faces fused with the stage update
// (k_face_march_update), the ghost shell's update and the learned start's fallback queue.
hipError_t launch_stage_fused(const FaceLaunch &l, const UpdLaunch &u, hipStream_t s);
// ... and the FP64 repair of the cells whose FP32 right-hand side was not finite (k_repair_weno;
// l: the stage's faces, its primitives)
hipError_t launch_repair(const FaceLaunch &l, const UpdLaunch &u, hipStream_t s);
long shell_cells(const Grid &g);
long fused_blocks(const Grid &g);


}  // namespace afd
