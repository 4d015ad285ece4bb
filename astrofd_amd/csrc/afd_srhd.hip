// afd_srhd.hip -- SRHD face kernels (MUSCL/PPM/WENO x HLLE/HLLC x x,y x FP64/mixed) and the update with the
// z faces.
#include <algorithm>

#include "afd_launch.hpp"

namespace afd {

// MUSCL faces go by runs from RUN_FACES faces on; SLOTS waves of them run at a time (four on each of the
// 1024 SIMDs), and the length is the one whose rounds of waves take the fewest face times, a run's start
// counted as START of them (RUN_MAX: longer runs gain nothing and leave the L2s).
constexpr long RUN_MAX = 32, SLOTS = 4096;
constexpr double START = 1.5;

static int run_length(long npos, int faces) {
    int best = 1;
    double least = 0.0;
    for (int m = 1; m <= std::min<long>(faces, RUN_MAX); ++m) {
        const long waves = (npos + 63) / 64 * ((faces + m - 1) / m);
        const double t = (double)((waves + SLOTS - 1) / SLOTS) * (m + START);
        if (m == 1 || t < least) {
            least = t;
            best = m;
        }
    }
    return best;
}

template <int RECON, int RIEM, typename T> static void go(const FaceLaunch &l, const FaceLaunch *y, hipStream_t s) {
    FaceArgs<T> a = face_args<T>(l);
    const Grid &g = l.g;
    const long count = face_count(g, l.dir);
    if (y) {  // l: the x faces
        const unsigned nx = grid1d(count).x, ny = grid1d(face_count(g, 1)).x;
        hipLaunchKernelGGL((k_faces_srhd<RECON, RIEM, T>), dim3(nx + ny), dim3(BLOCK), 0, s, a, face_args<T>(*y), nx);
        return;
    }
    if constexpr (RECON == 0) {
        if (count >= RUN_FACES) {
            const int faces = g.r1[l.dir] - g.r0[l.dir] + 1;
            const long npos = count / faces, nb = (npos + BLOCK - 1) / BLOCK;
            const int run = run_length(npos, faces);
            a.dn = make_udiv((unsigned)nb);
            const dim3 grid((unsigned)(nb * ((faces + run - 1) / run)));
            if (l.dir == 0) k_face_srhd<RECON, RIEM, 0, T><<<grid, dim3(BLOCK), 0, s>>>(a, run);
            else k_face_srhd<RECON, RIEM, 1, T><<<grid, dim3(BLOCK), 0, s>>>(a, run);
            return;
        }
    }
    const dim3 grid = grid1d(count);
    if (l.dir == 0) k_face_srhd<RECON, RIEM, 0, T><<<grid, dim3(BLOCK), 0, s>>>(a);
    else k_face_srhd<RECON, RIEM, 1, T><<<grid, dim3(BLOCK), 0, s>>>(a);
}

template <typename T> static void go_t(const FaceLaunch &l, const FaceLaunch *y, hipStream_t s) {
    int key = l.recon * 2 + (l.riemann == 1 ? 1 : 0);
    switch (key) {
        case 0: go<0, 0, T>(l, y, s); break;
        case 1: go<0, 1, T>(l, y, s); break;
        case 2: go<1, 0, T>(l, y, s); break;
        case 3: go<1, 1, T>(l, y, s); break;
        case 4: go<2, 0, T>(l, y, s); break;
        default: go<2, 1, T>(l, y, s); break;
    }
}

hipError_t launch_face_srhd(const FaceLaunch &l, const FaceLaunch *y, hipStream_t s) {
    if (l.mixed) go_t<float>(l, y, s);
    else go_t<double>(l, y, s);
    return hipGetLastError();
}

static dim3 update_grid(const Grid &g) {
    constexpr int cells = ZCELLS * (BLOCK / 64);
    return dim3((unsigned)((g.ncell + cells - 1) / cells));
}

template <int RECON, int RIEM>
static void go_update(const FaceLaunch &l, const UpdLaunch &u, bool rhs_only, hipStream_t s) {
    hipLaunchKernelGGL((k_update_faces_z<RECON, RIEM>), update_grid(l.g), dim3(BLOCK), 0, s, face_args<double>(l), u.a,
                       rhs_only);
}

hipError_t launch_update_srhd(const FaceLaunch &l, const UpdLaunch &u, bool rhs_only, hipStream_t s) {
    if (l.mixed) {
        UpdArgs<float> ua;
        static_assert(sizeof(UpdArgs<float>) == sizeof(UpdArgs<double>), "layout");
        memcpy((void *)&ua, (const void *)&u.a, sizeof(ua));
        k_update<5, float, false><<<update_grid(l.g), dim3(BLOCK), 0, s>>>(face_args<float>(l), ua, l.recon,
                                                                           l.riemann, rhs_only);
        return hipGetLastError();
    }
    switch (l.recon * 2 + (l.riemann == 1 ? 1 : 0)) {
        case 0: go_update<0, 0>(l, u, rhs_only, s); break;
        case 1: go_update<0, 1>(l, u, rhs_only, s); break;
        case 2: go_update<1, 0>(l, u, rhs_only, s); break;
        case 3: go_update<1, 1>(l, u, rhs_only, s); break;
        case 4: go_update<2, 0>(l, u, rhs_only, s); break;
        default: go_update<2, 1>(l, u, rhs_only, s); break;
    }
    return hipGetLastError();
}

}  // namespace afd
