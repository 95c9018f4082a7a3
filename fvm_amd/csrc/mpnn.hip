// Learned correction for the AMG preconditioner: a 3-layer message-passing
// network over the graph of a CRMatrix (no counterpart in the reference).
//
// Graph of a system A (self rows, symmetric pattern): edge weight of entry p of
// row i c_p = -off_p / d_i, node feature l_i = (log|d_i| - mean) / std.
// For a residual r (delta form, A e = -r):
//   u = -r / d, s = rms(u), v = u / s, h0 = [v, C v, l, 0 x 13]      (16 features)
//   layer k: a = C h ; h' = relu(Ws_k h + Wn_k a + b_k)                 (64 features)
//   e = s (wo . h3 + bo)
// Weights are held as FP32 masters and used as bf16 copies: every dense layer
// runs on the matrix cores (v_mfma_f32_16x16x32_bf16, FP32 accumulation);
// activations are stored in bf16. Training (residual loss ||r + A e||^2 / ||r||^2,
// A symmetric) uses FP32 backward kernels with deterministic reductions and Adam.
#include "amg.hpp"

#include <cmath>

namespace fvm {
namespace {

constexpr int MH = 64;       // hidden features
constexpr int MF0 = 16;      // input features (3 used)
constexpr int MLAYERS = 3;
constexpr int BSZ = 256;

typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef float f32x4 __attribute__((ext_vector_type(4)));

__device__ __forceinline__ float bf2f(uint16_t h) { return __uint_as_float(((unsigned)h) << 16); }
__device__ __forceinline__ uint16_t f2bf(float f) {
    unsigned u = __float_as_uint(f);
    if ((u & 0x7f800000u) == 0x7f800000u) return (uint16_t)((u >> 16) | ((u & 0xffffu) ? 0x40u : 0u));
    u += 0x7fffu + ((u >> 16) & 1u);
    return (uint16_t)(u >> 16);
}

constexpr int fin_of(int k) { return k == 0 ? MF0 : MH; }
// packed parameter offsets: per layer Ws (64 x fin), Wn (64 x fin), b (64); then wo (64), bo (1)
constexpr int layer_off(int k) { return k == 0 ? 0 : (k == 1 ? 2 * MH * MF0 + MH : 2 * MH * MF0 + MH + (k - 1) * (2 * MH * MH + MH)); }
constexpr int WO_OFF = layer_off(MLAYERS);
constexpr int NPARAM = WO_OFF + MH + 1;

template <int B>
__device__ double bsum(double v) {
    __shared__ double sh[B / 64];
    for (int o = 32; o > 0; o >>= 1) v += __shfl_down(v, o, 64);
    if ((threadIdx.x & 63) == 0) sh[threadIdx.x >> 6] = v;
    __syncthreads();
    double t = 0;
    if (threadIdx.x == 0)
        for (int k = 0; k < B / 64; k++) t += sh[k];
    __syncthreads();
    return t;
}

// ------------------------------------------------------------------ graph preparation
__global__ void k_mp_weights(int n, const int *row, const int *col, const double *off, const double *diag,
                             float *c) {
    for (int i = blockIdx.x * blockDim.x + threadIdx.x; i < n; i += gridDim.x * blockDim.x) {
        const double d = diag[i];
        for (int p = row[i]; p < row[i + 1]; p++) c[p] = (float)(-off[p] / d);
    }
}

// ct[q] for entry q = (j, i) of row j: the weight of entry (i, j) of row i; flag if absent
__global__ void k_mp_weights_t(int n, const int *row, const int *col, const float *c, float *ct, int *flag) {
    for (int j = blockIdx.x * blockDim.x + threadIdx.x; j < n; j += gridDim.x * blockDim.x)
        for (int q = row[j]; q < row[j + 1]; q++) {
            const int i = col[q];
            float w = 0.f;
            bool found = false;
            for (int p = row[i]; p < row[i + 1]; p++)
                if (col[p] == j) { w = c[p]; found = true; break; }
            if (!found) atomicOr(flag, 1);
            ct[q] = w;
        }
}

__global__ void __launch_bounds__(BSZ) k_mp_logd_partial(int n, const double *diag, double *part) {
    double s = 0, s2 = 0;
    for (int i = blockIdx.x * BSZ + threadIdx.x; i < n; i += gridDim.x * BSZ) {
        const double l = log(fabs(diag[i]));
        s += l;
        s2 += l * l;
    }
    s = bsum<BSZ>(s);
    s2 = bsum<BSZ>(s2);
    if (threadIdx.x == 0) { part[2 * blockIdx.x] = s; part[2 * blockIdx.x + 1] = s2; }
}

__global__ void __launch_bounds__(BSZ) k_mp_logd(int n, int nb, const double *diag, const double *part, float *l) {
    __shared__ double mean, sd;
    double s = 0, s2 = 0;
    for (int b = threadIdx.x; b < nb; b += BSZ) { s += part[2 * b]; s2 += part[2 * b + 1]; }
    s = bsum<BSZ>(s);
    s2 = bsum<BSZ>(s2);
    if (threadIdx.x == 0) {
        mean = s / n;
        double var = s2 / n - mean * mean;
        sd = sqrt(var > 0 ? var : 0.0) + 1e-12;
    }
    __syncthreads();
    for (int i = blockIdx.x * blockDim.x + threadIdx.x; i < n; i += gridDim.x * blockDim.x)
        l[i] = (float)((log(fabs(diag[i])) - mean) / sd);
}

// ------------------------------------------------------------------ forward
// partial sums of u^2, u = -r / d
__global__ void __launch_bounds__(BSZ) k_mp_u(int n, const double *r, const double *diag, double *part) {
    double s = 0;
    for (int i = blockIdx.x * BSZ + threadIdx.x; i < n; i += gridDim.x * BSZ) {
        const double ui = -r[i] / diag[i];
        s += ui * ui;
    }
    s = bsum<BSZ>(s);
    if (threadIdx.x == 0) part[blockIdx.x] = s;
}

// one block: the partial sums side by side (one thread adding 1,024 of them took 51 us)
__device__ double mp_total(int nb, const double *part) {
    double s = 0;
    for (int b = threadIdx.x; b < nb; b += BSZ) s += part[b];
    return bsum<BSZ>(s);
}
__global__ void __launch_bounds__(BSZ) k_mp_scale(int n, int nb, const double *part, double *s_out) {
    const double s = mp_total(nb, part);
    if (threadIdx.x == 0) *s_out = sqrt(s / (n > 0 ? n : 1)) + 1e-300;
}

__global__ void __launch_bounds__(BSZ) k_mp_sum2(int nb, const double *part, double *out) {
    const double s0 = mp_total(nb, part), s1 = mp_total(nb, part + nb);
    if (threadIdx.x == 0) { out[0] = s0; out[1] = s1; }
}

__global__ void k_mp_v(int n, const double *r, const double *diag, const double *s, float *v) {
    const double inv = 1.0 / *s;
    for (int i = blockIdx.x * blockDim.x + threadIdx.x; i < n; i += gridDim.x * blockDim.x)
        v[i] = (float)((-r[i] / diag[i]) * inv);
}

// The input features that are not zero, packed: h0 = {v, C v, l, 0} in bf16 (8 bytes).
typedef float f32x2 __attribute__((ext_vector_type(2)));
typedef __bf16 bf16x2 __attribute__((ext_vector_type(2)));
// two values to bf16, nearest even: one v_cvt_pk_bf16_f32 (14 instructions as integers)
__device__ __forceinline__ unsigned pack2(float a, float b) {
    return __builtin_bit_cast(unsigned, __builtin_convertvector(f32x2{a, b}, bf16x2));
}
__global__ void k_mp_h0(int n, const int *__restrict__ row, const int *__restrict__ col, const float *__restrict__ c,
                        const float *__restrict__ v, const float *__restrict__ l, uint2 *__restrict__ h0) {
    for (int i = blockIdx.x * blockDim.x + threadIdx.x; i < n; i += gridDim.x * blockDim.x) {
        const int rb = row[i], re = row[i + 1];
        float a = 0.f;
        for (int p = rb; p < re; p += 8) {   // eight entries in flight, added in order
            int j[8];
            float w[8], x[8];
#pragma unroll
            for (int u = 0; u < 8; u++) {
                j[u] = p + u < re ? col[p + u] : -1;
                w[u] = p + u < re ? c[p + u] : 0.f;
            }
#pragma unroll
            for (int u = 0; u < 8; u++) x[u] = j[u] >= 0 ? v[j[u]] : 0.f;
#pragma unroll
            for (int u = 0; u < 8; u++)
                if (p + u < re) a += w[u] * x[u];
        }
        h0[i] = make_uint2(pack2(v[i], a), pack2(l[i], 0.f));
    }
}

typedef unsigned u32x4 __attribute__((ext_vector_type(4)));
__device__ __forceinline__ float lo16(unsigned u) { return __uint_as_float(u << 16); }
__device__ __forceinline__ float hi16(unsigned u) { return __uint_as_float(u & 0xffff0000u); }
__device__ __forceinline__ void add8(float *acc, float w, u32x4 q) {
#pragma unroll
    for (int k = 0; k < 4; k++) {
        acc[2 * k] += w * lo16(q[k]);
        acc[2 * k + 1] += w * hi16(q[k]);
    }
}
__device__ __forceinline__ u32x4 pack8(const float *a) {
    u32x4 q;
#pragma unroll
    for (int k = 0; k < 4; k++) q[k] = pack2(a[2 * k], a[2 * k + 1]);
    return q;
}
__device__ __forceinline__ bf16x8 frag(u32x4 q) { return __builtin_bit_cast(bf16x8, q); }

// Aggregate of the input features, one node per thread (in the layer the four lanes of a node
// would each gather all of it: 763,560 nodes 63 us, against 35 us and 17 us for this launch).
__global__ void k_mp_a0(int n, const int *__restrict__ row, const int *__restrict__ col, const float *__restrict__ c,
                        const uint2 *__restrict__ h0, uint2 *__restrict__ a0) {
    for (int i = blockIdx.x * blockDim.x + threadIdx.x; i < n; i += gridDim.x * blockDim.x) {
        const int rb = row[i], re = row[i + 1];
        float s0 = 0.f, s1 = 0.f, s2 = 0.f;
        for (int p = rb; p < re; p += 4) {   // four entries in flight, added in order
            uint2 g[4];
            float w[4];
#pragma unroll
            for (int u = 0; u < 4; u++) {
                g[u] = h0[p + u < re ? col[p + u] : i];
                w[u] = p + u < re ? c[p + u] : 0.f;
            }
#pragma unroll
            for (int u = 0; u < 4; u++)
                if (p + u < re) {
                    s0 += w[u] * lo16(g[u].x);
                    s1 += w[u] * hi16(g[u].x);
                    s2 += w[u] * lo16(g[u].y);
                }
        }
        a0[i] = make_uint2(pack2(s0, s1), pack2(s2, 0.f));
    }
}

// Tiles of 16 nodes, one per wavefront and step. Blocks are handed to the 8 XCDs in turn,
// so block b works on eighth b % 8 of the tiles, and its blocks walk through that eighth
// side by side: the nodes of a step are consecutive and the neighbours they gather stay in
// that XCD's L2. At most 1,536 blocks (6 per CU stay resident); each loads its weights once.
__host__ __device__ constexpr int mp_tiles(int n) { return (n + 15) / 16; }
unsigned mp_grid(int n) { return std::min((unsigned)(mp_tiles(n) + 31) / 32, 192u) * 8u; }
struct MpTiles {
    int t, end, step;
    __device__ explicit MpTiles(int n) {
        const int T = mp_tiles(n), x = blockIdx.x & 7;
        t = (int)((long long)T * x / 8) + (blockIdx.x >> 3) * 4 + (threadIdx.x >> 6);
        end = (int)((long long)T * (x + 1) / 8);
        step = (gridDim.x >> 3) * 4;
    }
};

// One layer:  a_i = sum_p c_p h_col(p)  (FP32 sums, then bf16; kept for the backward pass)
//             h'_i = relu([h_i | a_i] W^T + b), W row o = [Ws(o,:) | Wn(o,:)] (bf16)
// Every value that is rounded to bf16 is summed in this order, entries ascending and the bias
// last: another order moves some over a rounding boundary (1e-5 of a loss).
// The products run as v_mfma_f32_16x16x32_bf16 with the weights as the first operand (lane l:
// output l%16, k = 8(l/16)..+8) and the nodes as the second (node l%16, same k), so lane l
// gathers for node l%16 exactly the features that it feeds to the matrix cores, and ends
// with four consecutive outputs of its node per output block (rows 4(l/16)..+4). The
// weights lie in LDS in lane order (16 KB a block), which leaves registers for six
// wavefronts per SIMD. LAST: the readout e = s (wo . h' + bo) is taken from the registers;
// h' is stored only for a backward pass. What bounds it: the gathers, 128 bytes per entry.
// 763,560 nodes (7-point rows): layer 64 -> 64 165 -> 129 us, the last one with its readout
// 260 -> 120 us (296 and 218 MB from memory, 10 and 7 million L2 accesses), layer 0 68 -> 35 us
// (and k_mp_a0 17 us).
// Weights in registers over several tiles: 142 us (3 wavefronts per SIMD). Stores and
// column reads that bypass the caches, or 96 blocks instead of 192 per XCD: slower.
template <int FIN, bool LAST>
__global__ void __launch_bounds__(BSZ, 6)
k_mp_layer(int n, const int *__restrict__ row, const int *__restrict__ col, const float *__restrict__ c,
           const void *__restrict__ Hv, const uint16_t *__restrict__ W, const float *__restrict__ bias, void *Aout,
           uint16_t *Hn, const float *__restrict__ wo, const double *__restrict__ sc, double *e, int accumulate,
           int *bad) {
    constexpr int K2 = 2 * FIN, NK = K2 / 32;
    const int lane = threadIdx.x & 63, r16 = lane & 15, q = lane >> 4;
    __shared__ u32x4 ws[4 * NK * 64];
    __shared__ f32x4 bs[16], wos[16];
    for (int t = threadIdx.x; t < 4 * NK * 64; t += BSZ) {
        const int l = t & 63, ob = (t >> 6) / NK, kk = (t >> 6) % NK;
        ws[t] = *reinterpret_cast<const u32x4 *>(W + (size_t)(ob * 16 + (l & 15)) * K2 + kk * 32 + (l >> 4) * 8);
    }
    if (threadIdx.x < MH) {
        ((float *)bs)[threadIdx.x] = bias[threadIdx.x];
        if (LAST) ((float *)wos)[threadIdx.x] = wo[threadIdx.x];
    }
    __syncthreads();
    for (MpTiles T(n); T.t < T.end; T.t += T.step) {
        asm volatile("" ::: "memory");   // the weights are read from LDS in each step, not kept in registers
        const int node0 = T.t * 16;
        const int i = node0 + r16, ic = min(i, n - 1);
        const int rb = row[ic], re = row[ic + 1];
        bf16x8 x[NK];
        if constexpr (FIN == MF0) {
            // three features: k 0..7 (lanes q = 0) hold h, k 16..23 (q = 2) hold a (k_mp_a0)
            const uint2 hi = ((const uint2 *)Hv)[ic], ai = ((const uint2 *)Aout)[ic];
            const u32x4 z = {q == 0 ? hi.x : q == 2 ? ai.x : 0u, q == 0 ? hi.y : q == 2 ? ai.y : 0u, 0u, 0u};
            x[0] = frag(z);
        } else {
            const u32x4 *H = (const u32x4 *)Hv;   // eight features; node i holds 8 i .. 8 i + 7
            float a[16];
#pragma unroll
            for (int k = 0; k < 16; k++) a[k] = 0.f;
            for (int p = rb; p < re; p += 4) {   // four entries in flight, added in order
                int j[4];
                float wt[4];
                u32x4 g[4][2];
#pragma unroll
                for (int u = 0; u < 4; u++) {
                    j[u] = p + u < re ? col[p + u] : ic;
                    wt[u] = p + u < re ? c[p + u] : 0.f;
                }
#pragma unroll
                for (int u = 0; u < 4; u++) {
                    g[u][0] = H[(size_t)j[u] * 8 + q];
                    g[u][1] = H[(size_t)j[u] * 8 + 4 + q];
                }
#pragma unroll
                for (int u = 0; u < 4; u++)
                    if (p + u < re) {
                        add8(a, wt[u], g[u][0]);
                        add8(a + 8, wt[u], g[u][1]);
                    }
            }
            const u32x4 b0 = pack8(a), b1 = pack8(a + 8);
            if (Aout && i < n) {
                ((u32x4 *)Aout)[(size_t)i * 8 + q] = b0;
                ((u32x4 *)Aout)[(size_t)i * 8 + 4 + q] = b1;
            }
            x[0] = frag(H[(size_t)ic * 8 + q]);
            x[1] = frag(H[(size_t)ic * 8 + 4 + q]);
            x[2] = frag(b0);
            x[3] = frag(b1);
        }
        float y = 0.f;
#pragma unroll
        for (int ob = 0; ob < 4; ob++) {
            f32x4 d = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
            for (int kk = 0; kk < NK; kk++)
                d = __builtin_amdgcn_mfma_f32_16x16x32_bf16(frag(ws[(ob * NK + kk) * 64 + lane]), x[kk], d, 0, 0, 0);
            const f32x4 bias4 = bs[ob * 4 + q];
            float h[4];
#pragma unroll
            for (int t = 0; t < 4; t++) {
                const float z = d[t] + bias4[t];
                h[t] = z > 0.f ? z : 0.f;
            }
            const uint2 st = make_uint2(pack2(h[0], h[1]), pack2(h[2], h[3]));
            if (Hn && i < n) *reinterpret_cast<uint2 *>(Hn + (size_t)i * MH + ob * 16 + 4 * q) = st;
            if (LAST) {
                const f32x4 wr = wos[ob * 4 + q];
                y += wr[0] * lo16(st.x) + wr[1] * hi16(st.x) + wr[2] * lo16(st.y) + wr[3] * hi16(st.y);
            }
        }
        if (LAST) {
            y += __shfl_xor(y, 16, 64);
            y += __shfl_xor(y, 32, 64);
            if (q == 0 && i < n) {
                const double ei = *sc * (double)(y + wo[MH]);
                if (!isfinite(ei)) atomicOr(bad, 1);
                e[i] = accumulate ? e[i] + ei : ei;
            }
        }
    }
}

// ------------------------------------------------------------------ loss and backward
// y = A x
__global__ void k_mp_spmv(int n, const int *row, const int *col, const double *off, const double *diag,
                          const double *x, double *y) {
    for (int i = blockIdx.x * blockDim.x + threadIdx.x; i < n; i += gridDim.x * blockDim.x) {
        double s = diag[i] * x[i];
        for (int p = row[i]; p < row[i + 1]; p++) s += off[p] * x[col[p]];
        y[i] = s;
    }
}

// The loss against a known correction et, in one pass: t = e - et, At = -A t and the partial
// sums of et^T (-A et) (part[b]) and t^T (-A t) (part[nb + b])
__global__ void __launch_bounds__(BSZ) k_mp_loss_pair(int n, const int *__restrict__ row, const int *__restrict__ col,
                                                      const double *__restrict__ off, const double *__restrict__ diag,
                                                      const double *__restrict__ e, const double *__restrict__ et,
                                                      double *__restrict__ At, double *__restrict__ part) {
    double den = 0, num = 0;
    for (int i = blockIdx.x * BSZ + threadIdx.x; i < n; i += gridDim.x * BSZ) {
        const double xi = et[i], ti = e[i] - xi, d = diag[i];
        double s = d * ti, x = d * xi;
        for (int p = row[i]; p < row[i + 1]; p++) {
            const int j = col[p];
            const double w = off[p], xj = et[j];
            s += w * (e[j] - xj);
            x += w * xj;
        }
        At[i] = -s;
        den += xi * -x;
        num += ti * -s;
    }
    den = bsum<BSZ>(den);
    num = bsum<BSZ>(num);
    if (threadIdx.x == 0) { part[blockIdx.x] = den; part[gridDim.x + blockIdx.x] = num; }
}

// The residual loss: t = r + A e and the partial sums of r^2 and t^2
__global__ void __launch_bounds__(BSZ) k_mp_loss_res(int n, const int *__restrict__ row, const int *__restrict__ col,
                                                     const double *__restrict__ off, const double *__restrict__ diag,
                                                     const double *__restrict__ e, const double *__restrict__ r,
                                                     double *__restrict__ t, double *__restrict__ part) {
    double den = 0, num = 0;
    for (int i = blockIdx.x * BSZ + threadIdx.x; i < n; i += gridDim.x * BSZ) {
        double s = diag[i] * e[i];
        for (int p = row[i]; p < row[i + 1]; p++) s += off[p] * e[col[p]];
        const double ri = r[i], ti = ri + s;
        t[i] = ti;
        den += ri * ri;
        num += ti * ti;
    }
    den = bsum<BSZ>(den);
    num = bsum<BSZ>(num);
    if (threadIdx.x == 0) { part[blockIdx.x] = den; part[gridDim.x + blockIdx.x] = num; }
}

// dy_i = s * 2 (A t)_i / ||r||^2
__global__ void k_mp_dy(int n, const double *At, const double *s, const double *rr, float *dy) {
    const double f = 2.0 * (*s) / (*rr);
    for (int i = blockIdx.x * blockDim.x + threadIdx.x; i < n; i += gridDim.x * blockDim.x) dy[i] = (float)(f * At[i]);
}

// Backward through layer k (k > 0), with delta_k+1 = dL/dh_k+1 * [h_k+1 > 0]:
//   g_i = sum over entries q of row i of ct_q delta_k+1(col q)
//   delta_k(i) = (delta_k+1(i) Ws + g_i Wn) * [h_k(i) > 0]
// (aggregating delta and not delta Wn: one pass, nothing between). All in FP32: the products
// are v_mfma_f32_16x16x4f32 with the weights' columns as the first operand and the nodes as
// the second; step 4v + u of lane l is feature 16 v + 4 (l/16) + u of node l%16, so the four
// lanes of a node read 64 consecutive bytes at a time. The weights lie in LDS as FP32 in
// lane order (32 KB a block). TOP: delta_3(j) = dy_j wo [h_3(j) > 0] is formed from dy and
// the bf16 h_3 where it is gathered. What bounds it: the gathers, and at 34,720 nodes its
// 8 wavefronts per CU.
// 34,720 nodes: 98 -> 22 us per layer (products per node and feature on the vector units and
// an aggregation of delta Wn, 390 MB a layer at 763,560 nodes, before).
template <bool TOP>
__global__ void __launch_bounds__(BSZ, 4)
k_mp_bwd(int n, const int *__restrict__ row, const int *__restrict__ col, const float *__restrict__ ct,
         const float *__restrict__ D, const uint16_t *__restrict__ Hn, const float *__restrict__ wo,
         const uint16_t *__restrict__ W, const uint16_t *__restrict__ H, float *__restrict__ Dk) {
    const int lane = threadIdx.x & 63, r16 = lane & 15, q = lane >> 4;
    __shared__ f32x4 ws[2 * 4 * 4 * 64];   // [part][output block][v][lane], component u
    for (int t = threadIdx.x; t < 2 * 4 * 4 * 64; t += BSZ) {
        const int l = t & 63, v = (t >> 6) & 3, fb = (t >> 8) & 3, part = t >> 10;
        f32x4 w;
#pragma unroll
        for (int u = 0; u < 4; u++)
            w[u] = bf2f(W[(size_t)(16 * v + 4 * (l >> 4) + u) * (2 * MH) + part * MH + 16 * fb + (l & 15)]);
        ws[t] = w;
    }
    __syncthreads();
    for (MpTiles T(n); T.t < T.end; T.t += T.step) {
        asm volatile("" ::: "memory");   // the weights are read from LDS in each step, not kept in registers
        const int i = T.t * 16 + r16, ic = min(i, n - 1);
        const int rb = row[ic], re = row[ic + 1];
        f32x4 x[2][4];
        // features of node j as multiples of wt (TOP: without the factor wo)
        auto gather = [&](f32x4 *acc, int j, float wt) {
            if constexpr (TOP) {
                const uint2 *h = (const uint2 *)(Hn + (size_t)j * MH) + q;
#pragma unroll
                for (int v = 0; v < 4; v++) {
                    const uint2 hv = h[4 * v];
                    acc[v][0] += lo16(hv.x) > 0.f ? wt : 0.f;
                    acc[v][1] += hi16(hv.x) > 0.f ? wt : 0.f;
                    acc[v][2] += lo16(hv.y) > 0.f ? wt : 0.f;
                    acc[v][3] += hi16(hv.y) > 0.f ? wt : 0.f;
                }
            } else {
                const f32x4 *d = (const f32x4 *)(D + (size_t)j * MH) + q;
#pragma unroll
                for (int v = 0; v < 4; v++) {
                    const f32x4 dv = d[4 * v];
#pragma unroll
                    for (int u = 0; u < 4; u++) acc[v][u] = fmaf(wt, dv[u], acc[v][u]);
                }
            }
        };
#pragma unroll
        for (int v = 0; v < 4; v++) x[0][v] = x[1][v] = f32x4{0.f, 0.f, 0.f, 0.f};
        gather(x[0], ic, TOP ? D[ic] : 1.f);
        for (int p = rb; p < re; p += 2) {
            const bool two = p + 1 < re;
            const int j0 = col[p], j1 = two ? col[p + 1] : j0;
            float w0 = ct[p], w1 = two ? ct[p + 1] : 0.f;
            if (TOP) {
                w0 *= D[j0];
                w1 *= D[j1];
            }
            gather(x[1], j0, w0);
            if (two) gather(x[1], j1, w1);
        }
        if constexpr (TOP) {
#pragma unroll
            for (int v = 0; v < 4; v++)
#pragma unroll
                for (int u = 0; u < 4; u++) {
                    const float w = wo[16 * v + 4 * q + u];
                    x[0][v][u] *= w;
                    x[1][v][u] *= w;
                }
        }
        f32x4 d[4];
#pragma unroll
        for (int fb = 0; fb < 4; fb++) d[fb] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
        for (int part = 0; part < 2; part++)
#pragma unroll
            for (int v = 0; v < 4; v++)
#pragma unroll
                for (int fb = 0; fb < 4; fb++) {   // four independent sums in turn
                    const f32x4 w = ws[((part * 4 + fb) * 4 + v) * 64 + lane];
#pragma unroll
                    for (int u = 0; u < 4; u++)
                        d[fb] = __builtin_amdgcn_mfma_f32_16x16x4f32(w[u], x[part][v][u], d[fb], 0, 0, 0);
                }
        if (i < n) {
#pragma unroll
            for (int fb = 0; fb < 4; fb++) {
                const uint2 h = *reinterpret_cast<const uint2 *>(H + (size_t)i * MH + 16 * fb + 4 * q);
                f32x4 o;
                o[0] = lo16(h.x) > 0.f ? d[fb][0] : 0.f;
                o[1] = hi16(h.x) > 0.f ? d[fb][1] : 0.f;
                o[2] = lo16(h.y) > 0.f ? d[fb][2] : 0.f;
                o[3] = hi16(h.y) > 0.f ? d[fb][3] : 0.f;
                *reinterpret_cast<f32x4 *>(Dk + (size_t)i * MH + 16 * fb + 4 * q) = o;
            }
        }
    }
}

// Weight gradients of all layers and of the readout, one launch: blockIdx.y = layer,
// blockIdx.x = a run of consecutive nodes, whose sums go to part[blockIdx.x].
//   dW_k[o][f] = sum_i delta_k+1(i)[o] x_i[f], x_i = [h_k(i) | a_k(i)];  db_k[o] = sum_i delta_k+1(i)[o]
//   dwo[o] = sum_i dy_i h_3(i)[o];  dbo = sum_i dy_i
// FP32 v_mfma_f32_16x16x4f32, four nodes per step (node l/16 of lane l). Row r of the output
// tile of wavefront w is o = 4 r + w, column r of tile fb is feature 4 r + fb of h (fb < 4) or
// of a, so that each lane reads 16 bytes of delta and 8 bytes each of h and a, whole rows
// across 16 lanes. A run's sums stay in registers and are written as they lie there.
// What bounds it: the matrix cores' FP32 rate.
// 34,720 nodes, three layers and readout: 147 us -> 33 us, and their reduction 422 -> 7 us
// (543 partial blocks of 33 KB per layer, added by one thread per value, before). Both the
// runs' sums (n / 256 terms) and their total in FP64 are shorter chains than 64 + n / 64.
constexpr int WG_W = 4 * 8 * 4 * 64, WG_W0 = 4 * 1 * 4 * 64;   // values of a layer, of layer 0
constexpr int WG_L = WG_W + MH;
constexpr int WG_O0 = 2 * WG_L, WG_OWO = WG_O0 + WG_W0 + MH, WG_S = WG_OWO + MH + 1;
constexpr int WG_MAX = 256;     // runs per layer: 3 x 256 blocks, 18 MB of partial sums
unsigned mp_runs(int n) { return (unsigned)std::min((n + 127) / 128, WG_MAX); }

template <int K>
__device__ void mp_wgrad_run(int n, int w, const float *__restrict__ dy, const float *__restrict__ D,
                             const uint16_t *__restrict__ Hn, const float *__restrict__ wo,
                             const uint16_t *__restrict__ H, const uint16_t *__restrict__ A, float *__restrict__ pw,
                             float *__restrict__ pb, float *__restrict__ po) {
    constexpr bool TOP = K == MLAYERS - 1;
    constexpr int NF = K == 0 ? 1 : 8;
    const int lane = threadIdx.x & 63, r16 = lane & 15, q = lane >> 4;
    const int steps = (n + 3) / 4;
    const int s0 = (int)((long long)steps * blockIdx.x / gridDim.x);
    const int s1 = (int)((long long)steps * (blockIdx.x + 1) / gridDim.x);
    f32x4 acc[NF];
#pragma unroll
    for (int f = 0; f < NF; f++) acc[f] = f32x4{0.f, 0.f, 0.f, 0.f};
    float db = 0.f, dwo = 0.f, dbo = 0.f;
    const float wow = TOP ? wo[4 * r16 + w] : 0.f;
    for (int s = s0; s < s1; s += 4) {
        float d[4], hn[4], y[4];
        uint2 h[4], a[4];
        uint16_t x0[4];
#pragma unroll
        for (int u = 0; u < 4; u++) {   // clamped loads; a node outside the run gets delta = 0
            const int i = min(4 * (s + u) + q, n - 1);
            const bool in = s + u < s1 && 4 * (s + u) + q < n;
            if constexpr (TOP) {
                y[u] = in ? dy[i] : 0.f;
                hn[u] = bf2f(Hn[(size_t)i * MH + 4 * r16 + w]);
                d[u] = hn[u] > 0.f ? y[u] * wow : 0.f;
            } else {
                d[u] = D[(size_t)i * MH + 4 * r16 + w];
                d[u] = in ? d[u] : 0.f;
            }
            if constexpr (K == 0) {
                x0[u] = (r16 & 4 ? A : H)[(size_t)i * 4 + (r16 & 3)];
            } else {
                h[u] = *reinterpret_cast<const uint2 *>(H + (size_t)i * MH + 4 * r16);
                a[u] = *reinterpret_cast<const uint2 *>(A + (size_t)i * MH + 4 * r16);
            }
        }
#pragma unroll
        for (int u = 0; u < 4; u++) {
            db += d[u];
            if constexpr (TOP) {
                dwo = fmaf(y[u], hn[u], dwo);
                dbo += y[u];
            }
            if constexpr (K == 0) {
                const float x = r16 < 8 ? bf2f(x0[u]) : 0.f;
                acc[0] = __builtin_amdgcn_mfma_f32_16x16x4f32(d[u], x, acc[0], 0, 0, 0);
            } else {
                const float x[8] = {lo16(h[u].x), hi16(h[u].x), lo16(h[u].y), hi16(h[u].y),
                                    lo16(a[u].x), hi16(a[u].x), lo16(a[u].y), hi16(a[u].y)};
#pragma unroll
                for (int f = 0; f < 8; f++) acc[f] = __builtin_amdgcn_mfma_f32_16x16x4f32(d[u], x[f], acc[f], 0, 0, 0);
            }
        }
    }
#pragma unroll
    for (int f = 0; f < NF; f++)
#pragma unroll
        for (int t = 0; t < 4; t++) pw[((w * NF + f) * 4 + t) * 64 + lane] = acc[f][t];
    for (int o = 16; o < 64; o <<= 1) {
        db += __shfl_xor(db, o, 64);
        if constexpr (TOP) {
            dwo += __shfl_xor(dwo, o, 64);
            dbo += __shfl_xor(dbo, o, 64);
        }
    }
    if (q == 0) {
        pb[4 * r16 + w] = db;
        if constexpr (TOP) {
            po[4 * r16 + w] = dwo;
            if (r16 == 0 && w == 0) po[MH] = dbo;
        }
    }
}

__global__ void __launch_bounds__(BSZ)
k_mp_wgrad(int n, const float *dy, const float *D2, const float *D1, const uint16_t *H3, const uint16_t *H2,
           const uint16_t *H1, const uint16_t *H0, const uint16_t *A2, const uint16_t *A1, const uint16_t *A0,
           const float *wo, float *part) {
    const int w = threadIdx.x >> 6;
    float *p = part + (size_t)blockIdx.x * WG_S;
    if (blockIdx.y == 0)
        mp_wgrad_run<2>(n, w, dy, nullptr, H3, wo, H2, A2, p, p + WG_W, p + WG_OWO);
    else if (blockIdx.y == 1)
        mp_wgrad_run<1>(n, w, nullptr, D2, nullptr, nullptr, H1, A1, p + WG_L, p + WG_L + WG_W, nullptr);
    else
        mp_wgrad_run<0>(n, w, nullptr, D1, nullptr, nullptr, H0, A0, p + WG_O0, p + WG_O0 + WG_W0, nullptr);
}

// grad += the runs' sums, added in FP64: 64 values by 4 threads each in a block
__global__ void __launch_bounds__(BSZ) k_mp_reduce(int nrun, const float *__restrict__ part, float *grad) {
    __shared__ double sh[4][64];
    const int g = threadIdx.x >> 6, v = threadIdx.x & 63, j = blockIdx.x * 64 + v;
    double s = 0;
    if (j < WG_S) {
#pragma unroll 8
        for (int b = g; b < nrun; b += 4) s += part[(size_t)b * WG_S + j];
    }
    sh[g][v] = s;
    __syncthreads();
    if (g != 0 || j >= WG_S) return;
    int dst = -1;
    if (j >= WG_OWO) {
        dst = WO_OFF + j - WG_OWO;
    } else {
        const int k = j < WG_L ? 2 : j < WG_O0 ? 1 : 0;
        const int jj = j - (k == 2 ? 0 : k == 1 ? WG_L : WG_O0), nw = k ? WG_W : WG_W0;
        const int fin = k ? MH : MF0, nf = k ? 8 : 1;
        if (jj >= nw) {
            dst = layer_off(k) + 2 * MH * fin + jj - nw;
        } else {
            const int lane = jj & 63, t = (jj >> 6) & 3, fb = (jj >> 8) % nf, w = (jj >> 8) / nf;
            const int o = 4 * (4 * (lane >> 4) + t) + w, r = lane & 15;
            if (k) dst = layer_off(k) + (fb < 4 ? 0 : MH * MH) + o * MH + 4 * r + (fb & 3);
            else if (r < 8) dst = layer_off(0) + (r < 4 ? 0 : MH * MF0) + o * MF0 + (r & 3);
        }
    }
    if (dst >= 0) grad[dst] += (float)((sh[0][v] + sh[1][v]) + (sh[2][v] + sh[3][v]));
}

__global__ void k_mp_adam(int np, float *theta, float *grad, float *m, float *v, float lr, float b1, float b2,
                          float eps, float inv_count, float c1, float c2) {
    for (int j = blockIdx.x * blockDim.x + threadIdx.x; j < np; j += gridDim.x * blockDim.x) {
        const float g = grad[j] * inv_count;
        const float mj = b1 * m[j] + (1.f - b1) * g;
        const float vj = b2 * v[j] + (1.f - b2) * g * g;
        m[j] = mj;
        v[j] = vj;
        theta[j] -= lr * (mj / c1) / (sqrtf(vj / c2) + eps);
        grad[j] = 0.f;
    }
}

// bf16 copies of the layer matrices: row o = [Ws(o,:) | Wn(o,:)]
__global__ void k_mp_quantize(const float *theta, uint16_t *w0, uint16_t *w1, uint16_t *w2) {
    for (int k = 0; k < MLAYERS; k++) {
        const int fin = fin_of(k), off = layer_off(k);
        uint16_t *w = k == 0 ? w0 : (k == 1 ? w1 : w2);
        for (int t = blockIdx.x * blockDim.x + threadIdx.x; t < MH * 2 * fin; t += gridDim.x * blockDim.x) {
            const int o = t / (2 * fin), f = t % (2 * fin);
            w[t] = f2bf(f < fin ? theta[off + o * fin + f] : theta[off + MH * fin + o * fin + (f - fin)]);
        }
    }
}

__global__ void k_mp_gather(int n, const int *perm, const double *src, double *dst) {
    for (int p = blockIdx.x * blockDim.x + threadIdx.x; p < n; p += gridDim.x * blockDim.x) dst[p] = src[perm[p]];
}
__global__ void k_mp_scatter_sub(int n, const int *perm, const double *a, const double *b, double *dst) {
    for (int p = blockIdx.x * blockDim.x + threadIdx.x; p < n; p += gridDim.x * blockDim.x)
        dst[perm ? perm[p] : p] = a[p] - b[p];
}
__global__ void k_mp_add_gathered(int n, const int *perm, const double *e, double *z) {
    for (int p = blockIdx.x * blockDim.x + threadIdx.x; p < n; p += gridDim.x * blockDim.x)
        z[p] += e[perm ? perm[p] : p];
}

}  // namespace
}  // namespace fvm

using fvm::DArr;

extern "C" int fvm_mpnn_set_graph(fvm_mpnn *m, int n, const int32_t *d_row, const int32_t *d_col,
                                  const double *d_off, const double *d_diag);
extern "C" const char *fvm_last_error(void);

struct fvm_mpnn {
    int device = 0;
    hipStream_t stream = nullptr;
    fvm::Pool pool;
    DArr<float> theta, grad, adam_m, adam_v;
    DArr<uint16_t> wbf[fvm::MLAYERS];
    int adam_t = 0;
    int grad_count = 0;
    // graph (borrowed CSR)
    int n = 0;
    const int *row = nullptr, *col = nullptr;
    const double *off = nullptr, *diag = nullptr;
    unsigned long long bound = 0;   // hierarchy whose finest level it is (0: set by fvm_mpnn_set_graph)
    DArr<float> c, ct, l;
    // activations and work
    // layer inputs and aggregates; those of layer 0 hold its four packed features per node
    DArr<uint16_t> H[fvm::MLAYERS + 1], A[fvm::MLAYERS];
    DArr<float> v, dy, D1, D2, part;
    DArr<double> s, rr, e, t, At, dpart, tmp_b;
    DArr<int> flag;
};

namespace fvm {
namespace {

struct MpScope {
    int prev = -1;
    PoolScope ps;
    explicit MpScope(fvm_mpnn *m) : ps(&m->pool) {
        if (hipGetDevice(&prev) != hipSuccess) prev = -1;
        FVM_HIP(hipSetDevice(m->device));
    }
    ~MpScope() { if (prev >= 0) (void)hipSetDevice(prev); }
};

void mp_alloc_acts(fvm_mpnn *m) {
    const size_t n = std::max(m->n, 1);
    const size_t nb = (n + BSZ - 1) / BSZ;
    m->H[0].ensure(n * 4);
    for (int k = 1; k <= MLAYERS; k++) m->H[k].ensure(n * MH);
    m->A[0].ensure(n * 4);
    for (int k = 1; k < MLAYERS; k++) m->A[k].ensure(n * MH);
    m->v.ensure(n);
    m->s.ensure(4);
    m->rr.ensure(4);
    m->dpart.ensure(2 * std::max<size_t>(nb, 1) + 8);
    m->flag.ensure(1);
}

// forward pass of the current graph on residual r (device, n); result in e_out or added to it;
// keep: store the aggregates for a backward pass
void mp_forward(fvm_mpnn *m, const double *r, double *e_out, int accumulate, bool keep = false) {
    hipStream_t st = m->stream;
    const int n = m->n;
    mp_alloc_acts(m);
    const unsigned nb = grid_for(n, BSZ, 1024);
    k_mp_u<<<nb, BSZ, 0, st>>>(n, r, m->diag, m->dpart.p);
    k_mp_scale<<<1, BSZ, 0, st>>>(n, (int)nb, m->dpart.p, m->s.p);
    k_mp_v<<<grid_for(n, BSZ), BSZ, 0, st>>>(n, r, m->diag, m->s.p, m->v.p);
    k_mp_h0<<<grid_for(n, BSZ), BSZ, 0, st>>>(n, m->row, m->col, m->c.p, m->v.p, m->l.p, (uint2 *)m->H[0].p);
    k_mp_a0<<<grid_for(n, BSZ), BSZ, 0, st>>>(n, m->row, m->col, m->c.p, (const uint2 *)m->H[0].p, (uint2 *)m->A[0].p);
    FVM_HIP(hipMemsetAsync(m->flag.p, 0, sizeof(int), st));
    const unsigned gl = mp_grid(n);
    for (int k = 0; k < MLAYERS; k++) {
        const float *bias = m->theta.p + layer_off(k) + 2 * MH * fin_of(k);
        const bool last = k == MLAYERS - 1;
        auto launch = [&](auto kern) {
            kern<<<gl, BSZ, 0, st>>>(n, m->row, m->col, m->c.p, m->H[k].p, m->wbf[k].p, bias,
                                     k == 0 || keep ? m->A[k].p : nullptr, (!last || keep) ? m->H[k + 1].p : nullptr,
                                     m->theta.p + WO_OFF, m->s.p, e_out, accumulate, m->flag.p);
        };
        if (k == 0) launch(k_mp_layer<MF0, false>);
        else if (!last) launch(k_mp_layer<MH, false>);
        else launch(k_mp_layer<MH, true>);
    }
    FVM_HIP(hipGetLastError());
}

// forward + backward on one residual; gradient added to m->grad; returns the loss:
// et null: ||r + A e||^2 / ||r||^2; else (e - et)^T (-A) (e - et) / et^T (-A) et
double mp_loss_grad(fvm_mpnn *m, const double *r, const double *et) {
    hipStream_t st = m->stream;
    const int n = m->n;
    mp_alloc_acts(m);
    const size_t nn = std::max(n, 1);
    m->e.ensure(nn); m->t.ensure(nn); m->At.ensure(nn);
    const unsigned runs = mp_runs(n);
    m->dy.ensure(nn); m->D1.ensure(nn * MH); m->D2.ensure(nn * MH);
    m->part.ensure((size_t)runs * WG_S);
    mp_forward(m, r, m->e.p, 0, true);
    const unsigned gs = grid_for(n, BSZ);
    const unsigned nb = grid_for(n, BSZ, 1024);
    // rr[0] = denominator, rr[1] = numerator; At = d(numerator)/de / 2
    if (!et) {   // t = r + A e ; At = A t (A symmetric)
        k_mp_loss_res<<<nb, BSZ, 0, st>>>(n, m->row, m->col, m->off, m->diag, m->e.p, r, m->t.p, m->dpart.p);
        k_mp_spmv<<<gs, BSZ, 0, st>>>(n, m->row, m->col, m->off, m->diag, m->t.p, m->At.p);
    } else {
        k_mp_loss_pair<<<nb, BSZ, 0, st>>>(n, m->row, m->col, m->off, m->diag, m->e.p, et, m->At.p, m->dpart.p);
    }
    k_mp_sum2<<<1, BSZ, 0, st>>>((int)nb, m->dpart.p, m->rr.p);
    k_mp_dy<<<gs, BSZ, 0, st>>>(n, m->At.p, m->s.p, m->rr.p, m->dy.p);
    const float *wo = m->theta.p + WO_OFF;
    const unsigned gl = mp_grid(n);
    k_mp_bwd<true><<<gl, BSZ, 0, st>>>(n, m->row, m->col, m->ct.p, m->dy.p, m->H[3].p, wo, m->wbf[2].p, m->H[2].p,
                                       m->D2.p);
    k_mp_bwd<false><<<gl, BSZ, 0, st>>>(n, m->row, m->col, m->ct.p, m->D2.p, nullptr, nullptr, m->wbf[1].p, m->H[1].p,
                                        m->D1.p);
    k_mp_wgrad<<<dim3(runs, MLAYERS), BSZ, 0, st>>>(n, m->dy.p, m->D2.p, m->D1.p, m->H[3].p, m->H[2].p, m->H[1].p,
                                                    m->H[0].p, m->A[2].p, m->A[1].p, m->A[0].p, wo, m->part.p);
    k_mp_reduce<<<(WG_S + 63) / 64, BSZ, 0, st>>>((int)runs, m->part.p, m->grad.p);
    FVM_HIP(hipGetLastError());
    m->grad_count++;
    double h_rr[2];
    FVM_HIP(hipMemcpyAsync(h_rr, m->rr.p, sizeof(double) * 2, hipMemcpyDeviceToHost, st));
    FVM_HIP(hipStreamSynchronize(st));
    return h_rr[1] / h_rr[0];
}

void mp_quantize(fvm_mpnn *m) {
    k_mp_quantize<<<64, BSZ, 0, m->stream>>>(m->theta.p, m->wbf[0].p, m->wbf[1].p, m->wbf[2].p);
    FVM_HIP(hipGetLastError());
}

}  // namespace

// Preconditioner correction inside FGMRES: z += NN(A z - v) on the finest level.
// v, z in the AMG handle's layout (perm: coloured position -> row, or null).
void mpnn_correct(fvm_mpnn *m, hipStream_t st, const int *perm, const double *Az, const double *v, double *z,
                  int n, int *bad_out) {
    MpScope g(m);
    FVM_CHECK(n == m->n, FVM_E_INVALID, "learned correction: graph and system sizes differ");
    const hipStream_t keep = m->stream;
    m->stream = st;
    m->tmp_b.ensure((size_t)std::max(n, 1) * 2);
    double *rn = m->tmp_b.p, *en = m->tmp_b.p + std::max(n, 1);
    k_mp_scatter_sub<<<grid_for(n, BSZ), BSZ, 0, st>>>(n, perm, Az, v, rn);
    mp_forward(m, rn, en, 0);
    k_mp_add_gathered<<<grid_for(n, BSZ), BSZ, 0, st>>>(n, perm, en, z);
    FVM_HIP(hipGetLastError());
    m->stream = keep;
    if (bad_out) *bad_out = read_scalar(m->flag.p, st);
}

// (the arrays' addresses do not tell: the next setup of a handle may get the same ones)
void mpnn_bind(fvm_mpnn *m, unsigned long long hierarchy_id, int n, const int *row, const int *col, const double *off,
               const double *diag) {
    if (m->bound == hierarchy_id) return;
    const int rc = fvm_mpnn_set_graph(m, n, row, col, off, diag);
    if (rc) throw Error(rc, std::string("learned correction: ") + fvm_last_error());
    m->bound = hierarchy_id;
}

}  // namespace fvm

#define FVM_API_BEGIN try {
#define FVM_API_END                                  \
    }                                                \
    catch (const fvm::Error &e) {                    \
        fvm::set_last_error(e.what());               \
        return e.code;                               \
    }                                                \
    catch (const std::exception &e) {                \
        fvm::set_last_error(e.what());               \
        return FVM_E_INVALID;                        \
    }

extern "C" {

int fvm_mpnn_num_params(void) { return fvm::NPARAM; }

int fvm_mpnn_create(fvm_mpnn **out, int device, uint64_t seed) {
    FVM_API_BEGIN
    FVM_CHECK(out, FVM_E_INVALID, "null output handle");
    int ndev = 0;
    FVM_HIP(hipGetDeviceCount(&ndev));
    FVM_CHECK(device >= 0 && device < ndev, FVM_E_INVALID, "device ordinal out of range");
    fvm_mpnn *m = new fvm_mpnn();
    m->device = device;
    try {
        fvm::MpScope g(m);
        FVM_HIP(hipStreamCreateWithFlags(&m->stream, hipStreamDefault));
        const int np = fvm::NPARAM;
        m->theta.alloc(np); m->grad.alloc(np); m->adam_m.alloc(np); m->adam_v.alloc(np);
        for (int k = 0; k < fvm::MLAYERS; k++) m->wbf[k].alloc((size_t)fvm::MH * 2 * fvm::fin_of(k));
        // He-style initialization from a seeded generator (host side, once)
        std::vector<float> th(np, 0.f);
        uint64_t x = seed * 0x9E3779B97F4A7C15ull + 0x2545F4914F6CDD1Dull;
        auto gauss = [&]() {
            auto u01 = [&]() {
                x ^= x << 13; x ^= x >> 7; x ^= x << 17;
                return ((x >> 11) + 0.5) * (1.0 / 9007199254740992.0);
            };
            const double a = u01(), b = u01();
            return std::sqrt(-2.0 * std::log(a)) * std::cos(6.283185307179586 * b);
        };
        for (int k = 0; k < fvm::MLAYERS; k++) {
            const int fin = fvm::fin_of(k), off = fvm::layer_off(k);
            for (int j = 0; j < 2 * fvm::MH * fin; j++) th[off + j] = (float)(gauss() * std::sqrt(1.0 / fin));
        }
        for (int j = 0; j < fvm::MH; j++) th[fvm::WO_OFF + j] = (float)(gauss() * std::sqrt(1.0 / fvm::MH) * 0.1);
        FVM_HIP(hipMemcpyAsync(m->theta.p, th.data(), sizeof(float) * np, hipMemcpyHostToDevice, m->stream));
        FVM_HIP(hipMemsetAsync(m->grad.p, 0, sizeof(float) * np, m->stream));
        FVM_HIP(hipMemsetAsync(m->adam_m.p, 0, sizeof(float) * np, m->stream));
        FVM_HIP(hipMemsetAsync(m->adam_v.p, 0, sizeof(float) * np, m->stream));
        fvm::mp_quantize(m);
        FVM_HIP(hipStreamSynchronize(m->stream));
    } catch (...) {
        delete m;
        throw;
    }
    *out = m;
    return FVM_OK;
    FVM_API_END
}

int fvm_mpnn_destroy(fvm_mpnn *m) {
    FVM_API_BEGIN
    if (!m) return FVM_OK;
    {
        int prev = -1;
        (void)hipGetDevice(&prev);
        (void)hipSetDevice(m->device);
        hipStream_t st = m->stream;
        delete m;
        if (st) (void)hipStreamDestroy(st);
        if (prev >= 0) (void)hipSetDevice(prev);
    }
    return FVM_OK;
    FVM_API_END
}

int fvm_mpnn_set_params(fvm_mpnn *m, const float *theta) {
    FVM_API_BEGIN
    FVM_CHECK(m && theta, FVM_E_INVALID, "null argument");
    fvm::MpScope g(m);
    FVM_HIP(hipMemcpyAsync(m->theta.p, theta, sizeof(float) * fvm::NPARAM, hipMemcpyHostToDevice, m->stream));
    fvm::mp_quantize(m);
    FVM_HIP(hipStreamSynchronize(m->stream));
    return FVM_OK;
    FVM_API_END
}

int fvm_mpnn_get_params(const fvm_mpnn *m, float *theta) {
    FVM_API_BEGIN
    FVM_CHECK(m && theta, FVM_E_INVALID, "null argument");
    int prev = -1;
    (void)hipGetDevice(&prev);
    FVM_HIP(hipSetDevice(m->device));
    FVM_HIP(hipMemcpyAsync(theta, m->theta.p, sizeof(float) * fvm::NPARAM, hipMemcpyDeviceToHost, m->stream));
    FVM_HIP(hipStreamSynchronize(m->stream));
    if (prev >= 0) (void)hipSetDevice(prev);
    return FVM_OK;
    FVM_API_END
}

int fvm_mpnn_set_graph(fvm_mpnn *m, int n, const int32_t *d_row, const int32_t *d_col, const double *d_off,
                       const double *d_diag) {
    FVM_API_BEGIN
    FVM_CHECK(m && n >= 0 && d_row && (n == 0 || d_diag), FVM_E_INVALID, "null argument");
    fvm::MpScope g(m);
    hipStream_t st = m->stream;
    const long long nnz = n > 0 ? fvm::read_scalar(d_row + n, st) : 0;
    FVM_CHECK(nnz == 0 || (d_col && d_off), FVM_E_INVALID, "null col/off arrays");
    m->bound = 0;
    m->n = n; m->row = d_row; m->col = d_col; m->off = d_off; m->diag = d_diag;
    m->c.alloc(std::max<long long>(nnz, 1));
    m->ct.alloc(std::max<long long>(nnz, 1));
    m->l.alloc(std::max(n, 1));
    fvm::mp_alloc_acts(m);
    if (n > 0) {
        FVM_HIP(hipMemsetAsync(m->flag.p, 0, sizeof(int), st));
        fvm::k_mp_weights<<<fvm::grid_for(n, fvm::BSZ), fvm::BSZ, 0, st>>>(n, d_row, d_col, d_off, d_diag, m->c.p);
        fvm::k_mp_weights_t<<<fvm::grid_for(n, fvm::BSZ), fvm::BSZ, 0, st>>>(n, d_row, d_col, m->c.p, m->ct.p,
                                                                             m->flag.p);
        const unsigned nb = fvm::grid_for(n, fvm::BSZ, 1024);
        fvm::k_mp_logd_partial<<<nb, fvm::BSZ, 0, st>>>(n, d_diag, m->dpart.p);
        fvm::k_mp_logd<<<fvm::grid_for(n, fvm::BSZ), fvm::BSZ, 0, st>>>(n, (int)nb, d_diag, m->dpart.p, m->l.p);
        FVM_HIP(hipGetLastError());
        FVM_CHECK(fvm::read_scalar(m->flag.p, st) == 0, FVM_E_INVALID,
                  "learned correction needs a structurally symmetric pattern");
    }
    FVM_HIP(hipStreamSynchronize(st));
    return FVM_OK;
    FVM_API_END
}

int fvm_mpnn_forward(fvm_mpnn *m, const double *d_r, double *d_e, int accumulate) {
    FVM_API_BEGIN
    FVM_CHECK(m && d_r && d_e, FVM_E_INVALID, "null argument");
    fvm::MpScope g(m);
    if (m->n > 0) fvm::mp_forward(m, d_r, d_e, accumulate);
    FVM_HIP(hipStreamSynchronize(m->stream));
    return FVM_OK;
    FVM_API_END
}

int fvm_mpnn_loss_grad(fvm_mpnn *m, const double *d_r, double *loss) {
    FVM_API_BEGIN
    FVM_CHECK(m && d_r, FVM_E_INVALID, "null argument");
    FVM_CHECK(m->n > 0, FVM_E_NOT_SETUP, "no graph");
    fvm::MpScope g(m);
    const double L = fvm::mp_loss_grad(m, d_r, nullptr);
    FVM_HIP(hipStreamSynchronize(m->stream));
    if (loss) *loss = L;
    return FVM_OK;
    FVM_API_END
}

int fvm_mpnn_loss_grad_pair(fvm_mpnn *m, const double *d_r, const double *d_e, double *loss) {
    FVM_API_BEGIN
    FVM_CHECK(m && d_r && d_e, FVM_E_INVALID, "null argument");
    FVM_CHECK(m->n > 0, FVM_E_NOT_SETUP, "no graph");
    fvm::MpScope g(m);
    const double L = fvm::mp_loss_grad(m, d_r, d_e);
    FVM_HIP(hipStreamSynchronize(m->stream));
    if (loss) *loss = L;
    return FVM_OK;
    FVM_API_END
}

int fvm_mpnn_get_grad(fvm_mpnn *m, float *grad, int reset) {
    FVM_API_BEGIN
    FVM_CHECK(m, FVM_E_INVALID, "null handle");
    fvm::MpScope g(m);
    if (grad)
        FVM_HIP(hipMemcpyAsync(grad, m->grad.p, sizeof(float) * fvm::NPARAM, hipMemcpyDeviceToHost, m->stream));
    if (reset) {
        FVM_HIP(hipMemsetAsync(m->grad.p, 0, sizeof(float) * fvm::NPARAM, m->stream));
        m->grad_count = 0;
    }
    FVM_HIP(hipStreamSynchronize(m->stream));
    return FVM_OK;
    FVM_API_END
}

int fvm_mpnn_adam_step(fvm_mpnn *m, float lr) {
    FVM_API_BEGIN
    FVM_CHECK(m, FVM_E_INVALID, "null handle");
    FVM_CHECK(m->grad_count > 0, FVM_E_INVALID, "no accumulated gradient");
    fvm::MpScope g(m);
    const float b1 = 0.9f, b2 = 0.999f, eps = 1e-8f;
    m->adam_t++;
    const float c1 = 1.f - std::pow(b1, (float)m->adam_t), c2 = 1.f - std::pow(b2, (float)m->adam_t);
    fvm::k_mp_adam<<<fvm::grid_for(fvm::NPARAM, fvm::BSZ), fvm::BSZ, 0, m->stream>>>(
        fvm::NPARAM, m->theta.p, m->grad.p, m->adam_m.p, m->adam_v.p, lr, b1, b2, eps, 1.f / m->grad_count, c1, c2);
    fvm::mp_quantize(m);
    m->grad_count = 0;
    FVM_HIP(hipStreamSynchronize(m->stream));
    return FVM_OK;
    FVM_API_END
}

}  // extern "C"
