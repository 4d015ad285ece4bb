// afd_srhd.hip -- SRHD face kernels (MUSCL/PPM/WENO x HLLE/HLLC x x,y x FP64/mixed) and the update with the
// z faces.
#include "afd_launch.hpp"

namespace afd {

template <int RECON, int RIEM, typename T> static void go(const FaceLaunch &l, hipStream_t s) {
    FaceArgs<T> a = face_args<T>(l);
    dim3 grid = grid1d(face_count(l.g, l.dir));
    if (l.dir == 0) hipLaunchKernelGGL((k_face_srhd<RECON, RIEM, 0, T>), grid, dim3(BLOCK), 0, s, a);
    else hipLaunchKernelGGL((k_face_srhd<RECON, RIEM, 1, T>), grid, dim3(BLOCK), 0, s, a);
}

template <typename T> static void go_t(const FaceLaunch &l, hipStream_t s) {
    int key = l.recon * 2 + (l.riemann == 1 ? 1 : 0);
    switch (key) {
        case 0: go<0, 0, T>(l, s); break;
        case 1: go<0, 1, T>(l, s); break;
        case 2: go<1, 0, T>(l, s); break;
        case 3: go<1, 1, T>(l, s); break;
        case 4: go<2, 0, T>(l, s); break;
        default: go<2, 1, T>(l, s); break;
    }
}

hipError_t launch_face_srhd(const FaceLaunch &l, hipStream_t s) {
    if (l.mixed) go_t<float>(l, s);
    else go_t<double>(l, s);
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
