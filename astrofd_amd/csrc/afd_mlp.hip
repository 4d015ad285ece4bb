// afd_mlp.hip -- kernels of the learned con2prim guess: weight packing, dataset preparation,
// inference (BF16 MFMA, FP32 accumulation) and the con2prim batch with the learned initial guess.
// Training is in afd_mlp_train.hip.
#include <cstring>
#include <vector>

#include "afd_mlp.hpp"

namespace afd {

int mlp_alloc(MlpDevice &m, const std::function<int(void **, size_t)> &alloc) {
    int rc;
    if ((rc = alloc((void **)&m.master, MLP_NPARAM * 4))) return rc;
    if ((rc = alloc(&m.w, MLP_DEV_BYTES))) return rc;
    if ((rc = alloc((void **)&m.adam_m, MLP_NPARAM * 4))) return rc;
    if ((rc = alloc((void **)&m.adam_v, MLP_NPARAM * 4))) return rc;
    if ((rc = alloc((void **)&m.grad, MLP_NPARAM * 4))) return rc;
    return alloc((void **)&m.loss, 8 * 65536);
}

// Master FP32 weights -> BF16 A-operand blocks (lane order, afd_mlp_device.hpp) + FP32 biases.
__global__ __launch_bounds__(BLOCK) void k_mlp_pack(const float *master, void *wout) {
    const int t = blockIdx.x * BLOCK + threadIdx.x;
    __bf16 *blk = (__bf16 *)wout;
    float *bias = (float *)((char *)wout + (size_t)MLP_NBLK * 64 * 16);
    if (t < MLP_NBLK * 64 * 8) {
        const int e = t % 8, lane = (t / 8) % 64, b = t / 512;
        const int m = lane % 32, k = 8 * (lane / 32) + e;
        float v = 0.0f;
        if (b >= BLK_B2) {  // b2 as the split pair hi + lo in K columns 0, 1
            const float bb = master[MLP_OFF_B2 + 32 * (b - BLK_B2) + m];
            if (k < 2) v = bias_part(bb, k);
        } else if (b < BLK_W2) {
            int mt = b - BLK_W1;
            if (k < MLP_IN) v = master[MLP_OFF_W1 + (32 * mt + m) * MLP_IN + k];
            else if (k < MLP_IN + 2) v = bias_part(master[MLP_OFF_B1 + 32 * mt + m], k - MLP_IN);
        } else if (b < BLK_W3) {
            int idx = b - BLK_W2, mt = idx / 4, kb = idx % 4;
            v = master[MLP_OFF_W2 + (32 * mt + m) * 64 + 16 * kb + k];
        } else if (b < BLK_W3T) {
            int kb = b - BLK_W3;
            if (m < MLP_OUT) v = master[MLP_OFF_W3 + m * 64 + 16 * kb + k];
        } else if (b < BLK_W2T) {
            int mt = b - BLK_W3T;
            if (k < MLP_OUT) v = master[MLP_OFF_W3 + k * 64 + 32 * mt + m];
        } else {
            int idx = b - BLK_W2T, mt = idx / 4, kb = idx % 4;
            v = master[MLP_OFF_W2 + (16 * kb + k) * 64 + 32 * mt + m];
        }
        blk[t] = (__bf16)v;
    }
    if (t < MLP_BIAS_FLOATS) {
        if (t < 64) bias[t] = master[MLP_OFF_B1 + t];
        else if (t < 128) bias[t] = master[MLP_OFF_B2 + t - 64];
        else bias[t] = master[MLP_OFF_B3 + t - 128];
    }
}

hipError_t mlp_pack(const float *master, void *w, hipStream_t s) {
    hipLaunchKernelGGL(k_mlp_pack, dim3((MLP_NBLK * 64 * 8 + BLOCK - 1) / BLOCK), dim3(BLOCK), 0, s, master, w);
    return hipGetLastError();
}

hipError_t mlp_upload(MlpDevice &m, const float *w, hipStream_t s) {
    hipError_t e = hipMemcpyAsync(m.master, w, MLP_NPARAM * 4, hipMemcpyHostToDevice, s);
    if (e == hipSuccess) e = hipMemsetAsync(m.adam_m, 0, MLP_NPARAM * 4, s);
    if (e == hipSuccess) e = hipMemsetAsync(m.adam_v, 0, MLP_NPARAM * 4, s);
    if (e == hipSuccess) e = mlp_pack(m.master, m.w, s);
    m.adam_t = 0;
    return e;
}

// ------------------------------------------------------------------ dataset
// (conserved -> primitive) pairs of the solver's own con2prim: p2c of the sampled primitives,
// the FP64 RMHD con2prim, features of the conserved state and scaled targets (log p/D, log W).
__global__ __launch_bounds__(BLOCK) void k_mlp_dataset(MlpDataArgs a) {
    long m = (long)blockIdx.x * BLOCK + threadIdx.x;
    if (m >= a.n) return;
    double q[9], U[9], out[9];
    for (int v = 0; v < 9; ++v) q[v] = a.prim[9 * m + v];
    rmhd_p2c_cell(a.gfac, a.p_max, a.v_max, q, U);
    RmhdC2PParams cp = {a.gamma, a.gfac, a.p_max, a.v_max};
    C2PStats st = {0, 0, 0};
    rmhd_c2p(cp, U, out, st, false);
    float x[5];
    bool ok = mlp_features(U, x);
    double v2 = out[1] * out[1] + out[2] * out[2] + out[3] * out[3];
    double W = 1.0 / sqrt(1.0 - (v2 < 1.0 ? v2 : 1.0 - 1e-14));
    float y0 = (float)(log10(out[4] / U[0]) * 0.25), y1 = (float)log10(W);
    // only pairs where the con2prim converged by Newton to a valid state: elsewhere it returns the
    // bisection result or the hydro guess, which no initial guess changes
    ok = ok && isfinite(y0) && isfinite(y1) && (st.flags & 6) == 0;
    for (int f = 0; f < 5; ++f) a.X[5 * m + f] = ok ? x[f] : 0.0f;
    a.Y[2 * m] = ok ? y0 : 0.0f;
    a.Y[2 * m + 1] = ok ? y1 : 0.0f;
    a.valid[m] = ok ? 1 : 0;
}

hipError_t mlp_prepare_dataset(const MlpDataArgs &a, hipStream_t s) {
    hipLaunchKernelGGL(k_mlp_dataset, grid1d(a.n), dim3(BLOCK), 0, s, a);
    return hipGetLastError();
}

// ------------------------------------------------------------------ inference (test hook)
__global__ __launch_bounds__(BLOCK) void k_mlp_forward(const void *w, const float *X, long n, float *Y) {
    long sidx = (long)blockIdx.x * BLOCK + threadIdx.x;
    float x[5] = {0.f, 0.f, 0.f, 0.f, 0.f}, y[2];
    if (sidx < n)
        for (int f = 0; f < 5; ++f) x[f] = X[5 * sidx + f];
    mlp_infer_wave(MlpGlobal{mlp_view(w)}, x, y);  // every lane of the wave participates
    if (sidx < n) {
        Y[2 * sidx] = y[0];
        Y[2 * sidx + 1] = y[1];
    }
}

hipError_t mlp_forward(const void *w, const float *X, long n, float *Y, hipStream_t s) {
    hipLaunchKernelGGL(k_mlp_forward, grid1d(n), dim3(BLOCK), 0, s, w, X, n, Y);
    return hipGetLastError();
}

// ------------------------------------------------------------------ con2prim batch
__global__ __launch_bounds__(BLOCK) void k_c2p_batch_learned(BatchArgs a, const void *mlp) {
    long m = (long)blockIdx.x * BLOCK + threadIdx.x;
    const bool live = m < a.n;
    double U[9], q[9];
    for (int v = 0; v < 9; ++v) U[v] = live ? a.in[9 * m + v] : 0.0;
    C2PStats st = {0, 0, 0};
    RmhdC2PParams cp = {a.gamma, a.gfac, a.p_max, a.v_max};
    float x[5], y[2];
    bool fok = mlp_features(U, x) && live;
    mlp_infer_wave(MlpGlobal{mlp_view(mlp)}, x, y);
    bool done = fok && rmhd_c2p_from_guess(cp, U, mlp_guess_Z(U[0], a.gfac, y), q, st);
    if (live && !done) rmhd_c2p(cp, U, q, st, a.iters || a.stats);
    if (live) {
        for (int v = 0; v < 9; ++v) a.out[9 * m + v] = q[v];
        if (a.iters) a.iters[m] = st.hydro_iters + st.newton_iters;
    }
    if (a.stats) wave_add_stats(a.stats, st);
}

void launch_c2p_batch(const BatchArgs &a, const C2PBatchExtra &x, hipStream_t s) {
    if (x.mlp && a.physics == 1)
        hipLaunchKernelGGL(k_c2p_batch_learned, grid1d(a.n), dim3(BLOCK), 0, s, a, x.mlp);
    else
        hipLaunchKernelGGL(k_c2p_batch, grid1d(a.n), dim3(BLOCK), 0, s, a);
}

}  // namespace afd
