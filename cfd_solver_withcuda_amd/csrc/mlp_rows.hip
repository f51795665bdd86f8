// Training step and prediction of the surrogate MLP for networks of up to 256 (padded) features a
// layer (and 32 outputs, the most that a network may have), in three launches a step:
//   rows    a workgroup takes 32 samples through the whole network and, in training, back again:
//           activations and gradients stay in LDS from layer to layer, weights stream from L2 (one
//           layer ahead, in registers, laid out as the matrix instructions take them). Layer by layer
//           (mlp_kernels.hip) every result goes through memory three times (pre-activations, rows,
//           columns) and each layer is a launch. Prediction writes the outputs alone.
//   wgrad   the weight gradients of all layers, split over row ranges (128 x 128 tiles);
//   update  sums the row ranges, and the bias gradients over the rows, and applies Adam, writing the
//           master weights and both bf16 copies.
// Products, rounding points and orders of accumulation are mlp_kernels.hip's, so training and
// predictions have the same bits.
//
// Measured on MI355X, 6 x 256 network, layer by layer -> here: ten steps of 16384 rows with their host
// copies 3.68 -> 1.59 ms (a step: rows 72 us, wgrad 25, update 20); 200,000 predictions with theirs
// 3.87 -> 0.77 ms (kernels 0.36 ms).
#include <hip/hip_runtime.h>
#include <stdint.h>

#include <algorithm>

#include "mlp_device.h"
#include "mlp_kernels.h"

namespace cfd {
namespace {

constexpr int NT = 2;             // row tiles of 16 samples of a workgroup
constexpr int kRows = 16 * NT;    // its samples
constexpr int kRowThreads = 512;  // eight waves, 32 outputs of a layer each
constexpr int kSlices = kMlpRowsWidth / 32;
constexpr int kAct = kMlpRowsWidth + 8;  // bf16 per row in LDS: 16-byte reads of 16 rows hit all banks

// The part of a layer that wave w computes: 32 outputs from c0 on, of the row tiles [i0, i1).
struct WavePart {
    int c0, i0, i1;
};
__device__ __forceinline__ WavePart wave_part(int w, int outputs) {
    const int nb = outputs / 32;                          // blocks of 32 outputs
    const int rs = min(NT, nb > 4 ? 1 : nb > 2 ? 2 : 4);  // waves that share a block's rows
    const int part = w / nb;
    WavePart p;
    p.c0 = 32 * (w - part * nb);
    p.i0 = part < rs ? part * (NT / rs) : NT;
    p.i1 = part < rs ? p.i0 + NT / rs : NT;
    return p;
}

// The wave's weights of one layer: rows c0 .. c0 + 31 of W [outputs x K], in MFMA operand order.
// Slices beyond K repeat the last one and stay unused: no branch parts the loads.
__device__ __forceinline__ void load_weights(const uint16_t *W, int K, const WavePart &p, int l,
                                             bf16x8 (&w)[kSlices][2]) {
    const uint16_t *base = W + (size_t)p.c0 * K;
#pragma unroll
    for (int s = 0; s < kSlices; s++)
#pragma unroll
        for (int j = 0; j < 2; j++) w[s][j] = load8(base + 16 * j * K + 16 * min(32 * s, K - 32) + 8 * l);
}

// acc[i][j][v]: output c0 + 16 j + 4 (l / 16) + v of row 16 i + l % 16.
__device__ __forceinline__ void layer_product(const uint16_t *act, int K, const WavePart &p, int l,
                                              const bf16x8 (&w)[kSlices][2], f32x4 (&acc)[NT][2]) {
    const uint16_t *x0 = act + (l % 16) * kAct + 8 * (l / 16);
#pragma unroll
    for (int i = 0; i < NT; i++)
        for (int j = 0; j < 2; j++) acc[i][j] = f32x4{0.f, 0.f, 0.f, 0.f};
    if (K == 32 * kSlices) {  // widest layers: straight through; rows of other waves' parts go unused
#pragma unroll
        for (int s = 0; s < kSlices; s++)
#pragma unroll
            for (int i = 0; i < NT; i++) {
                const bf16x8 x = *reinterpret_cast<const bf16x8 *>(x0 + 16 * i * kAct + 32 * s);
                acc[i][0] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(w[s][0], x, acc[i][0], 0, 0, 0);
                acc[i][1] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(w[s][1], x, acc[i][1], 0, 0, 0);
            }
        return;
    }
#pragma unroll
    for (int s = 0; s < kSlices; s++)
        if (32 * s < K) {
#pragma unroll
            for (int i = 0; i < NT; i++) {
                const bf16x8 x = *reinterpret_cast<const bf16x8 *>(x0 + 16 * i * kAct + 32 * s);
                acc[i][0] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(w[s][0], x, acc[i][0], 0, 0, 0);
                acc[i][1] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(w[s][1], x, acc[i][1], 0, 0, 0);
            }
        }
}

// The first `cols` columns of 32 rows in LDS as block `blk` of out: [rows / 32][cols][32], so that a
// workgroup writes, and a weight gradient reads, whole runs of memory. A thread takes eight rows of two
// columns.
__device__ __forceinline__ void store_columns(const uint16_t *act, int cols, uint16_t *out, int blk, int t) {
    out += (size_t)blk * cols * 32;
#pragma unroll 1
    for (int e = t; e < cols * 2; e += kRowThreads) {
        const int g = e & 3, cp = e >> 2;
        uint32_t v[8];
        for (int q = 0; q < 8; q++) v[q] = *reinterpret_cast<const uint32_t *>(act + (8 * g + q) * kAct + 2 * cp);
        uint32_t lo[4], hi[4];
        for (int q = 0; q < 4; q++) {
            lo[q] = (v[2 * q] & 0xffffu) | (v[2 * q + 1] << 16);
            hi[q] = (v[2 * q] >> 16) | (v[2 * q + 1] & 0xffff0000u);
        }
        uint16_t *o = out + 64 * cp + 8 * g;
        *reinterpret_cast<uint4 *>(o) = make_uint4(lo[0], lo[1], lo[2], lo[3]);
        *reinterpret_cast<uint4 *>(o + 32) = make_uint4(hi[0], hi[1], hi[2], hi[3]);
    }
}

// Bound by the matrix and activation instructions of a layer following each other and by the weights'
// way from L2. Two workgroups share a compute unit (32 samples: 128 registers and 38 KB of LDS each),
// one in its products while the other is in its activations. 64 samples read half as many weights and
// take as long (200,000 predictions: 340 us against 360). With row-major weights, whose operand loads
// touch 16 runs of 64 bytes, a minibatch of 16384 took 118 us instead of 72.
template <bool TRAIN>
__global__ void __launch_bounds__(kRowThreads) __attribute__((amdgpu_waves_per_eu(4))) rows_kernel(MlpLayers T, MlpRows a) {
    __shared__ __attribute__((aligned(16))) uint16_t act[2][kRows * kAct];
    __shared__ float zl[kRows * 33];  // the output layer's results
    __shared__ int sample[kRows];
    const int t = threadIdx.x, w = __builtin_amdgcn_readfirstlane(t / 64), l = t % 64;
    const int R0 = blockIdx.x * kRows;
    const int L = T.L;
    bf16x8 wt[kSlices][2];
    WavePart p = wave_part(w, T.Mp[0]);
    load_weights(T.Wb[0], T.Kp[0], p, l, wt);
    if (t < kRows) {
        const int r = R0 + t;
        int s = r < a.n ? r : a.n - 1;
        if (TRAIN && a.draw) s = sample_index(a.seed, a.d_step ? *a.d_step : a.step, a.rows, r, a.n);
        sample[t] = s;
    }
    __syncthreads();
    // normalised features, four columns of a row per thread
#pragma unroll 1
    for (int e = t; e < kRows * (T.Kp[0] / 4); e += kRowThreads) {
        const int r = e / (T.Kp[0] / 4), c = 4 * (e % (T.Kp[0] / 4));
        float h[4];
        for (int q = 0; q < 4; q++) {
            const int k = c + q;
            h[q] = k < a.n_in ? (a.feat[(size_t)sample[r] * a.n_in + k] - a.norm[k]) * a.norm[a.n_in + k] : 0.f;
        }
        *reinterpret_cast<uint2 *>(&act[0][r * kAct + c]) = f2bf4(h);
    }
    __syncthreads();
    if (TRAIN) store_columns(act[0], T.Kp[0], T.Xt[0], blockIdx.x, t);
    int cur = 0;
    f32x4 acc[NT][2];
    // ---- forward ---------------------------------------------------------------------------
    for (int k = 0; k < L; k++) {
        const bool last = k == L - 1;
        const int valid = T.M[k];
        float bv[2][4];  // the biases of this lane's outputs
        for (int j = 0; j < 2; j++)
            for (int q = 0; q < 4; q++) {
                const int c = p.c0 + 16 * j + 4 * (l / 16) + q;
                bv[j][q] = a.b[T.boff[k] + (c < valid ? c : 0)];
            }
        layer_product(act[cur], T.Kp[k], p, l, wt, acc);
        // the next weights travel during the activations
        WavePart pn = p;
        if (!last) {
            pn = wave_part(w, T.Mp[k + 1]);
            load_weights(T.Wb[k + 1], T.Kp[k + 1], pn, l, wt);
        } else if (TRAIN) {
            pn = wave_part(w, T.Kp[k]);
            load_weights(T.Wt[k], T.Mp[k], pn, l, wt);
        }
#pragma unroll
        for (int i = 0; i < NT; i++)
            if (i >= p.i0 && i < p.i1) {
                const int row = 16 * i + l % 16;
                uint2 zp[2];
#pragma unroll
                for (int j = 0; j < 2; j++) {
                    const int c = p.c0 + 16 * j + 4 * (l / 16);
                    float z[4], y[4];
#pragma unroll
                    for (int q = 0; q < 4; q++) z[q] = c + q < valid ? acc[i][j][q] + bv[j][q] : 0.f;
                    if (last) {
                        for (int q = 0; q < 4; q++) zl[row * 33 + c + q] = z[q];
                    } else {
                        sigmoid4(z, y);
#pragma unroll
                        for (int q = 0; q < 4; q++) y[q] = c + q < valid ? z[q] * y[q] : 0.f;
                        *reinterpret_cast<uint2 *>(&act[cur ^ 1][row * kAct + c]) = f2bf4(y);
                        zp[j] = f2bf4(z);
                    }
                }
                // bf16 pre-activations for the way back, in the order this lane reads them
                if (TRAIN && !last)
                    reinterpret_cast<uint4 *>(a.Z)[((((size_t)k * gridDim.x + blockIdx.x) * 8 + w) * NT + i) * 64 + l] =
                        make_uint4(zp[0].x, zp[0].y, zp[1].x, zp[1].y);
            }
        __syncthreads();
        if (!last) {
            cur ^= 1;
            if (TRAIN) store_columns(act[cur], T.Mp[k], T.Xt[k + 1], blockIdx.x, t);
        }
        p = pn;
    }
    // ---- outputs, or the loss and its gradient: one row per thread --------------------------
    const float *om = a.norm + 2 * a.n_in, *os = om + a.n_out;
    if (!TRAIN) {
#pragma unroll 1
        for (int e = t; e < kRows * a.n_out; e += kRowThreads) {
            const int r = e / a.n_out, c = e % a.n_out;
            if (R0 + r < a.n) a.out[(size_t)(R0 + r) * a.n_out + c] = zl[r * 33 + c] / os[c] + om[c];
        }
        return;
    }
    cur ^= 1;
    if (t < kRows) {
        const float inv = 2.0f / (float)(a.rows * a.n_out);
        float loss = 0.f;
#pragma unroll 1
        for (int c = 0; c < T.Mp[L - 1]; c += 4) {
            float h[4];
            for (int q = 0; q < 4; q++) {
                float d = 0.f;
                if (c + q < a.n_out) {
                    const float tg = (a.targ[(size_t)sample[t] * a.n_out + c + q] - om[c + q]) * os[c + q];
                    const float e = zl[t * 33 + c + q] - tg;
                    loss += e * e;
                    d = inv * e;
                }
                h[q] = d;
            }
            *reinterpret_cast<uint2 *>(&act[cur][t * kAct + c]) = f2bf4(h);
        }
        a.lrow[R0 + t] = loss / (float)a.n_out;
    }
    __syncthreads();
    store_columns(act[cur], T.Mp[L - 1], T.dZt[L - 1], blockIdx.x, t);
    // ---- backward: gradients of the pre-activations ------------------------------------------
    for (int k = L - 1; k > 0; k--) {
        const int valid = T.M[k - 1];
        uint4 zq[NT];
#pragma unroll
        for (int i = 0; i < NT; i++)
            if (i >= p.i0 && i < p.i1)
                zq[i] = reinterpret_cast<const uint4 *>(a.Z)[((((size_t)(k - 1) * gridDim.x + blockIdx.x) * 8 + w) * NT + i) * 64 + l];
        layer_product(act[cur], T.Mp[k], p, l, wt, acc);
        WavePart pn = p;
        if (k > 1) {
            pn = wave_part(w, T.Kp[k - 1]);
            load_weights(T.Wt[k - 1], T.Mp[k - 1], pn, l, wt);
        }
#pragma unroll
        for (int i = 0; i < NT; i++)
            if (i >= p.i0 && i < p.i1) {
                const int row = 16 * i + l % 16;
                const uint32_t zz[4] = {zq[i].x, zq[i].y, zq[i].z, zq[i].w};
#pragma unroll
                for (int j = 0; j < 2; j++) {
                    const int c = p.c0 + 16 * j + 4 * (l / 16);
                    float z[4], s[4], h[4];
#pragma unroll
                    for (int q = 0; q < 4; q++) z[q] = bf2f((uint16_t)(zz[2 * j + q / 2] >> (16 * (q % 2))));
                    sigmoid4(z, s);
#pragma unroll
                    for (int q = 0; q < 4; q++)
                        h[q] = c + q < valid ? acc[i][j][q] * (s[q] * (1.0f + z[q] * (1.0f - s[q]))) : 0.f;
                    *reinterpret_cast<uint2 *>(&act[cur ^ 1][row * kAct + c]) = f2bf4(h);
                }
            }
        __syncthreads();
        cur ^= 1;
        store_columns(act[cur], T.Kp[k], T.dZt[k - 1], blockIdx.x, t);
        p = pn;
    }
}

// ---- weight gradients ------------------------------------------------------------------------
// Layer by layer, 128 x 128 tiles of dZ^T X over one of `split` row ranges: four waves of 64 x 64,
// the operands' 32-row slices through LDS, double-buffered. Workgroups go round the eight XCDs in turn,
// so the tiles of a row range are dealt to one XCD, whose L2 then reads the range once: 36 -> 25 us for
// 16384 rows of the 6 x 256 network.
constexpr int kTile = 128;
constexpr int kLd = 40;  // bf16 per staged row: 32 + 8 of padding (conflict-free 16-byte reads)

__global__ void __launch_bounds__(256) wgrad_kernel(MlpLayers T, int rows, int split, float *P, int *d_step) {
    __shared__ __attribute__((aligned(16))) uint16_t sA[2][kTile * kLd], sB[2][kTile * kLd];
    // the step that a captured launch sequence is in advances here: the rows kernel has read it, and
    // the update reads the previous one
    if (d_step && blockIdx.x == 0 && threadIdx.x == 0) *d_step += 1;
    const int tiles = gridDim.x / split, turn = blockIdx.x / 8;  // split is a multiple of 8
    const int range = blockIdx.x % 8 + 8 * (turn / tiles);
    int k = 0, tile = turn % tiles;
    for (;; k++) {
        const int n = ((T.Mp[k] + kTile - 1) / kTile) * ((T.Kp[k] + kTile - 1) / kTile);
        if (tile < n) break;
        tile -= n;
    }
    const int Mp = T.Mp[k], Kp = T.Kp[k];
    const int tc = (Kp + kTile - 1) / kTile;
    const int R0 = (tile / tc) * kTile, C0 = (tile % tc) * kTile;
    const int nr = min(kTile, Mp - R0), ncol = min(kTile, Kp - C0);
    const int t = threadIdx.x, w = t / 64, l = t % 64;
    const int per = rows / split, kb = range * per;
    // staging: thread t moves 16 bf16 of row t / 2 of each operand's 128 x 32 slice
    const int sr = t / 2, sc = 16 * (t % 2);
    const bool ra = sr < nr, rb = sr < ncol;
    const uint16_t *ga = T.dZt[k] + (size_t)kb * Mp + (R0 + (ra ? sr : 0)) * 32 + sc;
    const uint16_t *gb = T.Xt[k] + (size_t)kb * Kp + (C0 + (rb ? sr : 0)) * 32 + sc;
    const int so = sr * kLd + sc;
    auto put = [&](int b, const bf16x8 *va, const bf16x8 *vb) {
        for (int q = 0; q < 2; q++) {
            *reinterpret_cast<bf16x8 *>(&sA[b][so + 8 * q]) = va[q];
            *reinterpret_cast<bf16x8 *>(&sB[b][so + 8 * q]) = vb[q];
        }
    };
    // the slices of the next two iterations travel in registers
    bf16x8 va[2][2], vb[2][2];
    auto get = [&](int u, int r) {
        if (r < per)
            for (int q = 0; q < 2; q++) {
                va[u][q] = load8(ga + r * Mp + 8 * q);
                vb[u][q] = load8(gb + r * Kp + 8 * q);
            }
    };
    get(0, 0);
    put(0, va[0], vb[0]);
    get(0, 32);
    get(1, 64);
    __syncthreads();
    const int wr = 64 * (w / 2), wc = 64 * (w % 2);
    const bool on = wr < nr && wc < ncol;  // this wave's block holds results
    const int fa = (wr + l % 16) * kLd + 8 * (l / 16), fb = (wc + l % 16) * kLd + 8 * (l / 16);
    f32x4 acc[4][4];
    for (int i = 0; i < 4; i++)
        for (int j = 0; j < 4; j++) acc[i][j] = f32x4{0.f, 0.f, 0.f, 0.f};
    auto slice = [&](int buf, int u, int r) {
        if (on) {
            bf16x8 xa[4], xb[4];
#pragma unroll
            for (int i = 0; i < 4; i++) {
                xa[i] = *reinterpret_cast<const bf16x8 *>(&sA[buf][fa + 16 * i * kLd]);
                xb[i] = *reinterpret_cast<const bf16x8 *>(&sB[buf][fb + 16 * i * kLd]);
            }
#pragma unroll
            for (int i = 0; i < 4; i++)
#pragma unroll
                for (int j = 0; j < 4; j++)
                    acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(xa[i], xb[j], acc[i][j], 0, 0, 0);
        }
        if (r + 32 < per) put(buf ^ 1, va[u], vb[u]);  // last read before the previous barrier
        get(u, r + 96);
        __syncthreads();
    };
    for (int r = 0; r < per; r += 64) {
        slice(0, 0, r);
        if (r + 32 < per) slice(1, 1, r + 32);
    }
    if (!on) return;
    float *out = P + T.poff[k] + (size_t)range * Mp * Kp;
    for (int i = 0; i < 4; i++)
        for (int q = 0; q < 4; q++) {
            const int m = wr + 16 * i + 4 * (l / 16) + q;
            if (m >= nr) continue;
            for (int j = 0; j < 4; j++) {
                const int c = wc + 16 * j + l % 16;
                if (c < ncol) out[(size_t)(R0 + m) * Kp + C0 + c] = acc[i][j][q];
            }
        }
}

// ---- sums of the row ranges, then Adam -------------------------------------------------------
// A workgroup takes a 32 x 32 tile of a layer's weights (four in a row per thread), or eight
// biases, whose gradients it sums over the rows (row_sum_layers_kernel's parts and order). Bound by the
// reads of P and dZt, 44 and 52 MB at 16384 rows of 6 x 256: 20 us, with one bias a workgroup 26 us.
template <bool ADAM>
__global__ void __launch_bounds__(256) update_kernel(MlpLayers T, const float *P, int split, int rows, int biases, MlpAdam a,
                                                     float *gW, float *gb) {
    constexpr int kRed = 260;  // columns two banks apart
    __shared__ uint16_t tr[32 * 34];
    __shared__ float red[8 * kRed];
    const int t = threadIdx.x;
    float lr = a.lr, c1 = a.c1, c2 = a.c2;
    if (ADAM && a.d_step) {
        const int step = *a.d_step - 1;
        lr = a.sched[3 * step];
        c1 = a.sched[3 * step + 1];
        c2 = a.sched[3 * step + 2];
    }
    int tile = blockIdx.x;
    if (tile < biases) {  // the longest chains: first
        int layer = 0;
        while (tile >= (T.M[layer] + 7) / 8) tile -= (T.M[layer++] + 7) / 8;
        // a wave reads 8 x 64 bytes of two blocks of 32 rows at a time; parts tt of eight columns
        const int g = t & 3, c = (t >> 2) & 7, b0 = ((t >> 5) & 1) + 2 * (t / 64);
        const size_t run = 32 * (size_t)T.Mp[layer];
        const uint16_t *col = T.dZt[layer] + (8 * tile + c) * 32;
        auto at = [&](int j) { return col + (j / 32) * run + j % 32; };
        for (int i0 = 0; i0 < 8; i0 += 4) {
            int tt[4], j = 0;
            float s4[4][4] = {};
            for (int i = 0; i < 4; i++) tt[i] = 4 * (b0 + 8 * (i0 + i)) + g;
            for (; j + 8192 <= rows; j += 8192) {
                uint4 v[4][4];
#pragma unroll
                for (int i = 0; i < 4; i++)
#pragma unroll
                    for (int u = 0; u < 4; u++) v[i][u] = *reinterpret_cast<const uint4 *>(at(j + 8 * tt[i] + 2048 * u));
#pragma unroll
                for (int i = 0; i < 4; i++)
#pragma unroll
                    for (int u = 0; u < 4; u++) s4[i][u] = add8(s4[i][u], v[i][u]);
            }
#pragma unroll
            for (int i = 0; i < 4; i++) red[c * kRed + tt[i]] = row_part(at, j + 8 * tt[i], rows, s4[i]);
        }
        __syncthreads();
        for (int h = 128; h > 0; h >>= 1) {  // 32 threads a column
            float *r = red + (t / 32) * kRed;
            for (int q = t % 32; q < h; q += 32) r[q] += r[q + h];
            __syncthreads();
        }
        const int m = 8 * tile + t;
        if (t < 8 && m < T.M[layer]) {
            const float g = red[t * kRed];
            const long long i = T.boff[layer] + m;
            if constexpr (ADAM) adam_one(a.b[i], a.mb[i], a.vb[i], g, lr, a.b1, a.b2, a.eps, c1, c2);
            else gb[i] = g;
        }
        return;
    }
    tile -= biases;
    int k = 0;
    while (tile >= (T.Mp[k] / 32) * (T.Kp[k] / 32)) {
        tile -= (T.Mp[k] / 32) * (T.Kp[k] / 32);
        k++;
    }
    const int Mp = T.Mp[k], Kp = T.Kp[k], M = T.M[k], K = T.K[k];
    const int m0 = (tile / (Kp / 32)) * 32, k0 = (tile % (Kp / 32)) * 32;
    const int m = m0 + t / 8, kk = k0 + 4 * (t % 8);
    const float4 *src = reinterpret_cast<const float4 *>(P + T.poff[k] + (size_t)m * Kp + kk);
    const size_t step4 = (size_t)Mp * Kp / 4;
    const long long o = T.woff[k] + (long long)m * K + kk;
    float W[4], m1[4], m2[4];  // on their way during the sums
    if constexpr (ADAM)
        for (int q = 0; q < 4; q++)
            if (m < M && kk + q < K) {
                W[q] = a.W[o + q];
                m1[q] = a.mW[o + q];
                m2[q] = a.vW[o + q];
            }
    float g[4] = {0.f, 0.f, 0.f, 0.f};
    for (int q = 0; q < split; q += 16) {  // split is 16 or 32
        float4 v[16];
#pragma unroll
        for (int u = 0; u < 16; u++) v[u] = src[(size_t)(q + u) * step4];
#pragma unroll
        for (int u = 0; u < 16; u++) {
            g[0] += v[u].x;
            g[1] += v[u].y;
            g[2] += v[u].z;
            g[3] += v[u].w;
        }
    }
    uint16_t h[4] = {0, 0, 0, 0};
    for (int q = 0; q < 4; q++)
        if (m < M && kk + q < K) {
            if constexpr (ADAM) {
                adam_one(W[q], m1[q], m2[q], g[q], lr, a.b1, a.b2, a.eps, c1, c2);
                a.W[o + q] = W[q];
                a.mW[o + q] = m1[q];
                a.vW[o + q] = m2[q];
                h[q] = f2bf(W[q]);
            } else {
                gW[o + q] = g[q];
            }
        }
    if constexpr (!ADAM) return;
    *reinterpret_cast<uint2 *>(T.Wb[k] + operand_at(m, kk, Kp)) =
        make_uint2((uint32_t)h[0] | ((uint32_t)h[1] << 16), (uint32_t)h[2] | ((uint32_t)h[3] << 16));
    for (int q = 0; q < 4; q++) tr[(4 * (t % 8) + q) * 34 + t / 8] = h[q];
    __syncthreads();
    // transposed copy: four outputs m of one input per thread
    const uint16_t *s = tr + (t / 8) * 34 + 4 * (t % 8);
    *reinterpret_cast<uint2 *>(T.Wt[k] + operand_at(k0 + t / 8, m0 + 4 * (t % 8), Mp)) =
        make_uint2((uint32_t)s[0] | ((uint32_t)s[1] << 16), (uint32_t)s[2] | ((uint32_t)s[3] << 16));
}

}  // namespace

bool mlp_rows_fits(const MlpLayers &t) {
    for (int k = 0; k < t.L; k++)
        if (t.Mp[k] > kMlpRowsWidth || t.Kp[k] > kMlpRowsWidth) return false;
    return t.Mp[t.L - 1] <= 32;
}

hipError_t mlp_rows(const MlpLayers &t, const MlpRows &a, bool train, hipStream_t s) {
    if (train && a.rows % kRows) return hipErrorInvalidValue;
    if (train) hipLaunchKernelGGL((rows_kernel<true>), dim3(a.rows / kRows), dim3(kRowThreads), 0, s, t, a);
    else hipLaunchKernelGGL((rows_kernel<false>), dim3((a.n + kRows - 1) / kRows), dim3(kRowThreads), 0, s, t, a);
    return hipGetLastError();
}

hipError_t mlp_wgrad(const MlpLayers &t, int rows, int split, float *P, int *d_step, hipStream_t s) {
    if (split % 8 || rows % (32 * split)) return hipErrorInvalidValue;
    int tiles = 0;
    for (int k = 0; k < t.L; k++) tiles += ((t.Mp[k] + kTile - 1) / kTile) * ((t.Kp[k] + kTile - 1) / kTile);
    hipLaunchKernelGGL(wgrad_kernel, dim3(tiles * split), dim3(256), 0, s, t, rows, split, P, d_step);
    return hipGetLastError();
}

hipError_t mlp_update(const MlpLayers &t, const float *P, int split, int rows, const MlpAdam *a, float *gW, float *gb,
                      hipStream_t s) {
    if (split % 16 || rows % 512) return hipErrorInvalidValue;
    int weights = 0, biases = 0;
    for (int k = 0; k < t.L; k++) {
        weights += (t.Mp[k] / 32) * (t.Kp[k] / 32);
        biases += (t.M[k] + 7) / 8;
    }
    const dim3 grid(weights + biases);
    if (a) hipLaunchKernelGGL(update_kernel<true>, grid, dim3(256), 0, s, t, P, split, rows, biases, *a, gW, gb);
    else hipLaunchKernelGGL(update_kernel<false>, grid, dim3(256), 0, s, t, P, split, rows, biases, MlpAdam{}, gW, gb);
    return hipGetLastError();
}

}  // namespace cfd
