// afd_mlp_train.hip -- training of the learned con2prim guess: the fused forward/backward gradient
// kernel (BF16 MFMA, FP32 accumulation), the reduction with Adam and the repacking of the operands.
// Compiled without -amdgpu-mfma-vgpr-form: the weight gradients' accumulators (128 registers a lane)
// live across the kernel and belong in the accumulation registers.
#include "afd_mlp.hpp"

namespace afd {

// ------------------------------------------------------------------ forward + backward
// One wavefront per 32-sample tile and round: forward (MFMA), output error, backprop of the
// activations through W3^T and W2^T (MFMA), then the weight gradients as GEMMs over the sample
// dimension (MFMA) from BF16 tiles staged in LDS as [feature][sample].  A workgroup of TRAIN_WAVES
// waves sums its waves' gradients through LDS and stores one partial gradient and loss to the
// workspace; k_mlp_reduce adds the partials.  (The partials used to be added by float atomics: 4674
// addresses taking one from each of 512 waves held a 32768-sample step at 134 us; with them gone the
// gradient takes 21 us and the reduction 5 us.)  A minibatch of 32768 is one round of 256 workgroups, one wave
// per SIMD: what bounds the kernel is the chain of one tile (four dependent layers of MFMAs, exp and
// rcp, two LDS transposes), so the samples are spread as widely as tiles of 32 allow.
constexpr int LDS_S = 40;  // row stride in BF16 elements (32 samples + pad, 80 bytes)
constexpr int TRAIN_WAVES = 4, TRAIN_BLOCKS = 256;
constexpr int PARTIAL = MLP_NPARAM + 2;  // a partial gradient, then the partial loss as a double's two words
static_assert(PARTIAL % 2 == 0, "the loss is 8-byte aligned");

static_assert(128 * 33 * sizeof(float) <= (4 * 64 + 2 * 32) * LDS_S * sizeof(__bf16), "bias rows fit a tile");

struct TrainTile {  // one wave's staged BF16 tiles (X and DO adjacent: cleared together)
    __bf16 H1[64 * LDS_S], H2[64 * LDS_S], DZ1[64 * LDS_S], DZ2[64 * LDS_S], X[32 * LDS_S], DO[32 * LDS_S];
};

// h = silu(z) and d = silu'(z), from one sigmoid (silu, dsilu)
AFD_D void silu_pair(float z, float &h, float &d) {
    const float s = __builtin_amdgcn_rcpf(1.0f + __expf(-z));
    h = z * s;
    d = s * (1.0f + z * (1.0f - s));
}

__global__ __launch_bounds__(64 * TRAIN_WAVES) void k_mlp_train_grad(const void *wp, const float *X, const float *Yt,
                                                                    long n, float inv_n, float *partial) {
    __shared__ union {
        __attribute__((aligned(16))) TrainTile tile[TRAIN_WAVES];
        float grad[TRAIN_WAVES][MLP_NPARAM];
    } sh;
    __shared__ double sloss[TRAIN_WAVES];
    const MlpDevW w = mlp_view(wp);
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    const bool upper = lane >= 32;
    const int col = lane & 31;
    TrainTile &S = sh.tile[wave];
    // rows of X beyond the 5 features and of dO beyond the 2 outputs stay 0
    for (int v = lane; v < 2 * 32 * LDS_S / 8; v += 64) ((bf16x8 *)S.X)[v] = pack8(0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f);
    floatx16 gW2[2][2], gW1[2], gW3[2];
    for (int a = 0; a < 2; ++a) {
        gW1[a] = zero16();
        gW3[a] = zero16();
        for (int b = 0; b < 2; ++b) gW2[a][b] = zero16();
    }
    float gb1[2][16], gb2[2][16], gb3[2] = {0.f, 0.f};
    for (int a = 0; a < 2; ++a)
        for (int i = 0; i < 16; ++i) gb1[a][i] = gb2[a][i] = 0.f;
    double lsum = 0.0;
    __syncthreads();
    // every wave runs the same number of rounds (the barriers below); tiles past the end contribute 0
    const long step = (long)gridDim.x * TRAIN_WAVES * 32, first = (long)blockIdx.x * TRAIN_WAVES * 32;
    for (long base = first; base < n; base += step) {
        const long sidx = base + 32 * wave + col;
        const bool tlive = sidx < n;
        float x[5] = {0.f, 0.f, 0.f, 0.f, 0.f}, y[2] = {0.f, 0.f};
        if (tlive) {
            for (int f = 0; f < 5; ++f) x[f] = X[5 * sidx + f];
            y[0] = Yt[2 * sidx];
            y[1] = Yt[2 * sidx + 1];
        }
        // the forward pass of mlp_tile_forward, keeping h and silu'(z) of both layers
        const MlpGlobal wf{w};
        floatx16 h1[2], h2[2], ds1[2], ds2[2];
        bf16x8 hb[4];
        const bf16x8 xb = input_operand(x, upper);
        for (int mt = 0; mt < 2; ++mt) {
            const floatx16 z = mfma_bf16(wf.blk(BLK_W1 + mt, lane), xb, zero16());
            for (int i = 0; i < 16; ++i) {
                float h, d;
                silu_pair(z[i], h, d);
                h1[mt][i] = h;
                ds1[mt][i] = d;
                S.H1[(32 * mt + drow(i, lane)) * LDS_S + col] = (__bf16)h;
            }
        }
        d_to_b(h1, lane, hb);
        for (int mt = 0; mt < 2; ++mt) {
            floatx16 z = mfma_bf16(wf.blk(BLK_B2 + mt, lane), ones_operand(upper), zero16());
            for (int kb = 0; kb < 4; ++kb) z = mfma_bf16(wf.blk(BLK_W2 + 4 * mt + kb, lane), hb[kb], z);
            for (int i = 0; i < 16; ++i) {
                float h, d;
                silu_pair(z[i], h, d);
                h2[mt][i] = h;
                ds2[mt][i] = d;
                S.H2[(32 * mt + drow(i, lane)) * LDS_S + col] = (__bf16)h;
            }
        }
        d_to_b(h2, lane, hb);
        floatx16 o = zero16();
        o[0] = wf.b3(0);
        o[1] = wf.b3(1);
        for (int kb = 0; kb < 4; ++kb) o = mfma_bf16(wf.blk(BLK_W3 + kb, lane), hb[kb], o);
        float d0 = 0.f, d1 = 0.f;
        if (!upper && tlive) {
            const float e0 = o[0] - y[0], e1 = o[1] - y[1];
            d0 = 2.0f * inv_n * e0;
            d1 = 2.0f * inv_n * e1;
            lsum += (double)(e0 * e0 + e1 * e1) * inv_n;
            gb3[0] += d0;
            gb3[1] += d1;
        }
        const bf16x8 dob = upper ? pack8(0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f) : pack8(d0, d1, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f);
        floatx16 dz2[2], dz1[2];
        for (int mt = 0; mt < 2; ++mt) {
            dz2[mt] = mfma_bf16(w.blk[(BLK_W3T + mt) * 64 + lane], dob, zero16());
            for (int i = 0; i < 16; ++i) dz2[mt][i] *= ds2[mt][i];
        }
        bf16x8 dz2b[4];
        d_to_b(dz2, lane, dz2b);
        for (int mt = 0; mt < 2; ++mt) {
            floatx16 acc = zero16();
            for (int kb = 0; kb < 4; ++kb) acc = mfma_bf16(w.blk[(BLK_W2T + 4 * mt + kb) * 64 + lane], dz2b[kb], acc);
            for (int i = 0; i < 16; ++i) acc[i] *= ds1[mt][i];
            dz1[mt] = acc;
        }
        for (int mt = 0; mt < 2; ++mt)
            for (int i = 0; i < 16; ++i) {
                const int row = 32 * mt + drow(i, lane);
                gb2[mt][i] += dz2[mt][i];
                gb1[mt][i] += dz1[mt][i];
                S.DZ2[row * LDS_S + col] = (__bf16)dz2[mt][i];
                S.DZ1[row * LDS_S + col] = (__bf16)dz1[mt][i];
            }
        if (!upper) {
            for (int f = 0; f < 5; ++f) S.X[f * LDS_S + col] = (__bf16)x[f];
            S.DO[0 * LDS_S + col] = (__bf16)d0;
            S.DO[1 * LDS_S + col] = (__bf16)d1;
        }
        __syncthreads();
        for (int kb = 0; kb < 2; ++kb) {
            const int cb = 16 * kb + 8 * (lane >> 5);
            bf16x8 aDZ2[2], aDZ1[2], bH1[2], bH2[2];
            for (int mt = 0; mt < 2; ++mt) {
                aDZ2[mt] = *(const bf16x8 *)&S.DZ2[(32 * mt + col) * LDS_S + cb];
                aDZ1[mt] = *(const bf16x8 *)&S.DZ1[(32 * mt + col) * LDS_S + cb];
                bH1[mt] = *(const bf16x8 *)&S.H1[(32 * mt + col) * LDS_S + cb];
                bH2[mt] = *(const bf16x8 *)&S.H2[(32 * mt + col) * LDS_S + cb];
            }
            const bf16x8 aDO = *(const bf16x8 *)&S.DO[col * LDS_S + cb];
            const bf16x8 bX = *(const bf16x8 *)&S.X[col * LDS_S + cb];
            for (int mt = 0; mt < 2; ++mt) {
                for (int nt = 0; nt < 2; ++nt) gW2[mt][nt] = mfma_bf16(aDZ2[mt], bH1[nt], gW2[mt][nt]);
                gW1[mt] = mfma_bf16(aDZ1[mt], bX, gW1[mt]);
            }
            for (int nt = 0; nt < 2; ++nt) gW3[nt] = mfma_bf16(aDO, bH2[nt], gW3[nt]);
        }
        __syncthreads();  // the last one also ends every wave's use of the tiles
    }
    // bias gradients: each lane holds 64 rows of its sample column; through the wave's tile as
    // [row][33], then two rows a lane (shuffles took 640 of the kernel's 4000 instructions)
    float *gb = (float *)&S;
    for (int mt = 0; mt < 2; ++mt)
        for (int i = 0; i < 16; ++i) {
            const int row = 32 * mt + drow(i, lane);
            gb[row * 33 + col] = gb1[mt][i];
            gb[(64 + row) * 33 + col] = gb2[mt][i];
        }
    __syncthreads();
    float b1 = 0.f, b2 = 0.f;
    for (int k = 0; k < 32; ++k) {
        b1 += gb[lane * 33 + k];
        b2 += gb[(64 + lane) * 33 + k];
    }
    __syncthreads();
    float *g = sh.grad[wave];  // over the tiles
    g[MLP_OFF_B1 + lane] = b1;
    g[MLP_OFF_B2 + lane] = b2;
    for (int mt = 0; mt < 2; ++mt)
        for (int i = 0; i < 16; ++i) {
            const int row = 32 * mt + drow(i, lane);
            for (int nt = 0; nt < 2; ++nt) g[MLP_OFF_W2 + row * 64 + 32 * nt + col] = gW2[mt][nt][i];
            if (col < MLP_IN) g[MLP_OFF_W1 + row * MLP_IN + col] = gW1[mt][i];
        }
    for (int nt = 0; nt < 2; ++nt)
        for (int i = 0; i < 16; ++i) {
            const int row = drow(i, lane);
            if (row < MLP_OUT) g[MLP_OFF_W3 + row * 64 + 32 * nt + col] = gW3[nt][i];
        }
    for (int j = 0; j < 2; ++j) {
        float v = gb3[j];
        for (int off = 32; off > 0; off >>= 1) v += __shfl_xor(v, off);
        if (lane == 0) g[MLP_OFF_B3 + j] = v;
    }
    for (int off = 32; off > 0; off >>= 1) lsum += __shfl_xor(lsum, off);
    if (lane == 0) sloss[wave] = lsum;
    __syncthreads();
    float *out = partial + (size_t)blockIdx.x * PARTIAL;
    for (int i = threadIdx.x; i < MLP_NPARAM; i += 64 * TRAIN_WAVES) {
        float v = sh.grad[0][i];
        for (int k = 1; k < TRAIN_WAVES; ++k) v += sh.grad[k][i];
        out[i] = v;
    }
    if (threadIdx.x == 0) {
        double v = sloss[0];
        for (int k = 1; k < TRAIN_WAVES; ++k) v += sloss[k];
        *(double *)(out + MLP_NPARAM) = v;
    }
}

// ------------------------------------------------------------------ reduction, Adam (Kingma & Ba 2015), packing
// The BF16 operand entries of master weight i (k_mlp_pack's layout; the entries no weight maps to
// stay the zeros k_mlp_pack wrote when the weights were set).
AFD_D void pack_one(int i, float v, void *wout) {
    __bf16 *blk = (__bf16 *)wout;
    float *bias = (float *)((char *)wout + (size_t)MLP_NBLK * 64 * 16);
    // entry (m, k) of operand block b
    auto put = [&](int b, int m, int k, float x) { blk[((size_t)b * 64 + 32 * (k / 8) + m) * 8 + k % 8] = (__bf16)x; };
    if (i < MLP_OFF_B1) {
        const int r = i / MLP_IN, c = i % MLP_IN;
        put(BLK_W1 + r / 32, r % 32, c, v);
    } else if (i < MLP_OFF_W2) {
        const int r = i - MLP_OFF_B1;
        for (int h = 0; h < 2; ++h) put(BLK_W1 + r / 32, r % 32, MLP_IN + h, bias_part(v, h));
        bias[r] = v;
    } else if (i < MLP_OFF_B2) {
        const int r = (i - MLP_OFF_W2) / 64, c = (i - MLP_OFF_W2) % 64;
        put(BLK_W2 + 4 * (r / 32) + c / 16, r % 32, c % 16, v);
        put(BLK_W2T + 4 * (c / 32) + r / 16, c % 32, r % 16, v);
    } else if (i < MLP_OFF_W3) {
        const int r = i - MLP_OFF_B2;
        for (int h = 0; h < 2; ++h) put(BLK_B2 + r / 32, r % 32, h, bias_part(v, h));
        bias[64 + r] = v;
    } else if (i < MLP_OFF_B3) {
        const int r = (i - MLP_OFF_W3) / 64, c = (i - MLP_OFF_W3) % 64;
        put(BLK_W3 + c / 16, r, c % 16, v);
        put(BLK_W3T + c / 32, c % 32, r, v);
    } else {
        bias[128 + i - MLP_OFF_B3] = v;
    }
}

// Sums the nb partial gradients of 64 weights per workgroup (RED_WAVES waves, each over its share of
// the partials, in a fixed order and in FP64) and, with `master`, applies one Adam step to them and writes their
// packed operands, so that a training step is two launches and nothing is cleared between steps.
// Otherwise the gradient goes to `grad`.  The loss goes to `loss`.
constexpr int RED_WAVES = 16;
__global__ __launch_bounds__(64 * RED_WAVES) void k_mlp_reduce(const float *partial, int nb, float *grad, double *loss,
                                                              float *master, float *m, float *v, void *wpack, float lr,
                                                              float bc1, float bc2) {
    __shared__ double red[RED_WAVES][64];
    __shared__ double lred[RED_WAVES];
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6, i = blockIdx.x * 64 + lane;
    double s = 0.0;
    if (i < MLP_NPARAM) {
#pragma unroll 4
        for (int b = wave; b < nb; b += RED_WAVES) s += (double)partial[(size_t)b * PARTIAL + i];
    }
    red[wave][lane] = s;
    if (blockIdx.x == 0) {
        double l = 0.0;
        for (int b = threadIdx.x; b < nb; b += 64 * RED_WAVES) l += *(const double *)(partial + (size_t)b * PARTIAL + MLP_NPARAM);
        for (int off = 32; off > 0; off >>= 1) l += __shfl_xor(l, off);
        if (lane == 0) lred[wave] = l;
    }
    __syncthreads();
    if (threadIdx.x == 0 && blockIdx.x == 0) {
        double l = 0.0;
        for (int k = 0; k < RED_WAVES; ++k) l += lred[k];
        *loss = l;
    }
    if (wave != 0 || i >= MLP_NPARAM) return;
    double sum = 0.0;
    for (int k = 0; k < RED_WAVES; ++k) sum += red[k][lane];
    const float gi = (float)sum;
    if (!master) {
        grad[i] = gi;
        return;
    }
    const float mi = 0.9f * m[i] + 0.1f * gi;
    const float vi = 0.999f * v[i] + 0.001f * gi * gi;
    m[i] = mi;
    v[i] = vi;
    const float p = master[i] - lr * (mi / bc1) / (sqrtf(vi / bc2) + 1e-8f);
    master[i] = p;
    pack_one(i, p, wpack);
}

size_t mlp_partial_bytes() { return sizeof(float) * PARTIAL * TRAIN_BLOCKS; }

// Partial gradients of n samples; returns the number of partials.
static int launch_grad(const void *w, const float *X, const float *Y, long n, float *partial, hipStream_t s) {
    const long wg = (n + 32 * TRAIN_WAVES - 1) / (32 * TRAIN_WAVES);
    const int blocks = (int)(wg < TRAIN_BLOCKS ? wg : TRAIN_BLOCKS);
    hipLaunchKernelGGL(k_mlp_train_grad, dim3(blocks), dim3(64 * TRAIN_WAVES), 0, s, w, X, Y, n, 1.0f / (float)n, partial);
    return blocks;
}

hipError_t mlp_loss_grad(const MlpDevice &d, const float *X, const float *Y, long n, hipStream_t s) {
    const int nb = launch_grad(d.w, X, Y, n, d.partial, s);
    hipLaunchKernelGGL(k_mlp_reduce, dim3((MLP_NPARAM + 63) / 64), dim3(64 * RED_WAVES), 0, s, (const float *)d.partial, nb,
                       d.grad, d.loss, (float *)nullptr, (float *)nullptr, (float *)nullptr, (void *)nullptr, 0.0f, 1.0f,
                       1.0f);
    return hipGetLastError();
}

hipError_t mlp_train_step(MlpDevice &d, const float *X, const float *Y, long n, float lr, double *loss, hipStream_t s) {
    const int nb = launch_grad(d.w, X, Y, n, d.partial, s);
    const long t = ++d.adam_t;
    const float bc1 = 1.0f - powf(0.9f, (float)t), bc2 = 1.0f - powf(0.999f, (float)t);
    hipLaunchKernelGGL(k_mlp_reduce, dim3((MLP_NPARAM + 63) / 64), dim3(64 * RED_WAVES), 0, s, (const float *)d.partial, nb,
                       (float *)nullptr, loss, d.master, d.adam_m, d.adam_v, d.w, lr, bc1, bc2);
    return hipGetLastError();
}

}  // namespace afd
