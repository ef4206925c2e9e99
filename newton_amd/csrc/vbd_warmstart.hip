// libvbd_ws.so -- learned warm start of the VBD iteration: 1-ring features and
// a BF16 MLP (48 -> 128 -> 128 -> 128 -> 3, SiLU) with forward, backward and
// Adam, written for gfx950's MFMA units.  C ABI in include/vbd_warmstart.h.
//
// Matrix products use v_mfma_f32_16x16x16_bf16 (16x16 output tile, K = 16,
// FP32 accumulation).  Operand layout per 64-lane wave, with li = lane % 16 and
// lq = lane / 16:
//   A (16 x 16, M x K): lane holds A[li][4*lq + 0..3]
//   B (16 x 16, K x N): lane holds B[4*lq + 0..3][li]
//   D (16 x 16, M x N): lane holds D[4*lq + 0..3][li]
// Each wave owns 16 rows (particles); a workgroup of 4 waves owns 64 rows.
// Hidden activations of a wave live in LDS as BF16 rows, so the next layer's
// A operand is one aligned 8-byte LDS read per lane.  Weights are read from
// global memory (L2-resident, 160 KB) in pre-packed layouts whose per-lane
// operand is one aligned 8-byte load: W^T for the forward pass, W for dH = dZ W^T.
//
// BF16 rounding points (restated by the CPU oracle, oracle/mlp_oracle.py):
// features; H_l = bf16(silu(Z_l)); dZ_l = bf16(dH_l * silu'(Z_l)); dZ_4 =
// bf16(dY).  Z, the output, dH (accumulators), bias sums and all gradients
// are FP32.
#include <hip/hip_runtime.h>

#include <cmath>
#include <cstdint>
#include <cstdio>
#include <algorithm>
#include <string>

#include "vbd_scalar.h"
#include "vbd_warmstart.h"

namespace {

constexpr int kIn = VBD_WS_IN;          // 48
constexpr int kHid = VBD_WS_HIDDEN;     // 128
constexpr int kOut = VBD_WS_OUT;        // 3
constexpr int kOutP = 16;               // last layer padded to one MFMA tile
constexpr int kWaveRows = 16;
constexpr int kWaves = 4;
constexpr int kBlock = 64 * kWaves;
constexpr int kRowsWG = kWaveRows * kWaves;  // 64 rows per workgroup
constexpr int kStride = kHid + 8;            // BF16 elements per LDS activation row (bank skew)
constexpr int kStrideIn = kIn + 8;
constexpr int kStrideOut = kOutP + 8;

// FP32 parameter offsets
constexpr int oW1 = 0;
constexpr int ob1 = oW1 + kIn * kHid;
constexpr int oW2 = ob1 + kHid;
constexpr int ob2 = oW2 + kHid * kHid;
constexpr int oW3 = ob2 + kHid;
constexpr int ob3 = oW3 + kHid * kHid;
constexpr int oW4 = ob3 + kHid;
constexpr int ob4 = oW4 + kHid * kOut;
constexpr int kParams = ob4 + kOut;  // 39683

// packed BF16 offsets (elements)
constexpr int pWt1 = 0;                       // [128][48]
constexpr int pW1 = pWt1 + kHid * kIn;        // [48][128]
constexpr int pWt2 = pW1 + kIn * kHid;        // [128][128]
constexpr int pW2 = pWt2 + kHid * kHid;
constexpr int pWt3 = pW2 + kHid * kHid;
constexpr int pW3 = pWt3 + kHid * kHid;
constexpr int pWt4 = pW3 + kHid * kHid;       // [16][128], rows >= 3 zero
constexpr int pW4 = pWt4 + kOutP * kHid;      // [128][16], cols >= 3 zero
constexpr int kPacked = pW4 + kHid * kOutP;   // 81920

constexpr int kFeatBlock = 256;

thread_local std::string g_err;

int32_t fail(int32_t code, const std::string& msg) {
    g_err = msg;
    return code;
}

#define WS_LAUNCH_CHECK(what)                                                                     \
    do {                                                                                          \
        hipError_t e_ = hipGetLastError();                                                        \
        if (e_ != hipSuccess) return fail(-2, std::string(what) + ": " + hipGetErrorString(e_)); \
    } while (0)

typedef short bf16x4 __attribute__((ext_vector_type(4)));
typedef float floatx4 __attribute__((ext_vector_type(4)));

__device__ __host__ inline uint16_t f2bf(float f) {
    uint32_t u;
    __builtin_memcpy(&u, &f, 4);
    if ((u & 0x7fffffffu) > 0x7f800000u) return (uint16_t)((u >> 16) | 0x40);  // quiet NaN
    u += 0x7fffu + ((u >> 16) & 1u);
    return (uint16_t)(u >> 16);
}

__device__ inline float bf2f(uint16_t h) {
    uint32_t u = (uint32_t)h << 16;
    float f;
    __builtin_memcpy(&f, &u, 4);
    return f;
}

__device__ inline float sigmoid(float z) { return 1.0f / (1.0f + expf(-z)); }

__device__ inline floatx4 mfma(bf16x4 a, bf16x4 b, floatx4 c) {
    return __builtin_amdgcn_mfma_f32_16x16x16bf16_1k(a, b, c, 0, 0, 0);
}

__device__ inline bf16x4 ld4(const uint16_t* p) { return *reinterpret_cast<const bf16x4*>(p); }

__device__ inline bf16x4 ld4_strided(const uint16_t* p, int stride) {
    bf16x4 r;
    r[0] = (short)p[0];
    r[1] = (short)p[stride];
    r[2] = (short)p[2 * stride];
    r[3] = (short)p[3 * stride];
    return r;
}

__device__ inline floatx4 zero4() { return floatx4{0.0f, 0.0f, 0.0f, 0.0f}; }

typedef float floatx2 __attribute__((ext_vector_type(2)));
typedef __bf16 bf16x2 __attribute__((ext_vector_type(2)));

// two floats -> two BF16 (round to nearest even) in one v_cvt_pk_bf16_f32
__device__ inline uint32_t pack_bf16x2(float a, float b) {
    const bf16x2 p = __builtin_convertvector((floatx2){a, b}, bf16x2);
    uint32_t u;
    __builtin_memcpy(&u, &p, 4);
    return u;
}

// Work-group -> block of particles such that each XCD (work-group i runs on XCD i % 8) takes one contiguous run of
// blocks: its L2 then holds the neighbours its particles share, instead of every L2 reading the whole field.
__device__ inline int xcd_block(int bid, int nb) {
    const int xcd = bid & 7, q = nb >> 3, r = nb & 7;
    return xcd * q + (xcd < r ? xcd : r) + (bid >> 3);
}


// neighbours whose indexes, and then values, are loaded together (a triangle mesh has six)
constexpr int kRing = 6;

// ---- features ----------------------------------------------------------------
// Columns (a = (y - x0) / s_disp, c = corr / s_corr, over 1-ring neighbours j):
//  0-2 a          3-5 c          6-8 mean(a_j) - a    9-11 mean(c_j) - c
//  12-14 max(a_j) - a            15-17 min(a_j) - a   18-20 max(c_j) - c   21-23 min(c_j) - c
//  24-26 mean(x0_j - x0_i) / s_len   27-29 mean, max, min |x0_j - x0_i| / s_len
//  30-32 acc * dt^2 / s_disp     33 |a|  34 |c|  35 mean |c_j|  36 max |c_j|
//  37 mass / mean mass   38 area / mean area   39 pinned fraction of neighbours   40 degree / 6
//  41-43 mean(y_j - y_i) / s_len   44-46 sum over pinned j of (x0_j - x0_i) / (degree * s_len)   47 1
// A particle without neighbours gets its own values for the neighbour statistics.
// Bound: gathers and vector instructions (8 divisions and square roots a neighbour): 1,048,576 particles 78 us
// (116 us with one neighbour's loads at a time and rows stored by their lanes).
__global__ __launch_bounds__(kFeatBlock) void k_features(int n, const int* __restrict__ nbr_off,
                                                        const int* __restrict__ nbr, const float* __restrict__ x0,
                                                        const float* __restrict__ y, const float* __restrict__ corr,
                                                        const float* __restrict__ acc, const float* __restrict__ mass,
                                                        const float* __restrict__ area, float dt,
                                                        const float* __restrict__ scales, uint16_t* __restrict__ out) {
    __shared__ uint2 s_rows[kFeatBlock * (kIn / 4)];
    const int i = xcd_block(blockIdx.x, gridDim.x) * kFeatBlock + threadIdx.x;
    if (i >= n) return;
    const float sd = scales[0], sc = scales[1], sl = scales[2], mm = scales[3], ma = scales[4];
    float xi[3], yi[3], a[3], c[3];
    for (int k = 0; k < 3; ++k) {
        xi[k] = x0[3 * i + k];
        yi[k] = y[3 * i + k];
        a[k] = (yi[k] - xi[k]) / sd;
        c[k] = corr ? corr[3 * i + k] / sc : 0.0f;
    }
    float sa[3] = {0, 0, 0}, sc3[3] = {0, 0, 0}, mxa[3], mna[3], mxc[3], mnc[3];
    float sdx[3] = {0, 0, 0}, sdy[3] = {0, 0, 0}, spin[3] = {0, 0, 0};
    float slen = 0.0f, mxl = 0.0f, mnl = 0.0f, sabsc = 0.0f, mxabsc = 0.0f;
    int npin = 0;
    const int j0 = nbr_off[i], j1 = nbr_off[i + 1], deg = j1 - j0;
    for (int k = 0; k < 3; ++k) {
        mxa[k] = mna[k] = a[k];
        mxc[k] = mnc[k] = c[k];
    }
    for (int jc = j0; jc < j1; jc += kRing / 2) {
        // three neighbours' values are loaded together
        int js[kRing / 2];
        float xs[kRing / 2][3], ys[kRing / 2][3], cs[kRing / 2][3] = {}, ms[kRing / 2];
#pragma unroll
        for (int u = 0; u < kRing / 2; ++u) js[u] = nbr[min(jc + u, j1 - 1)];
#pragma unroll
        for (int u = 0; u < kRing / 2; ++u) {
            ms[u] = mass[js[u]];
#pragma unroll
            for (int k = 0; k < 3; ++k) {
                xs[u][k] = x0[3 * js[u] + k];
                ys[u][k] = y[3 * js[u] + k];
                if (corr) cs[u][k] = corr[3 * js[u] + k];
            }
        }
#pragma unroll
        for (int u = 0; u < kRing / 2; ++u) {
            const int jj = jc + u;
            if (jj >= j1) break;
            float aj[3], cj[3], dx[3];
            for (int k = 0; k < 3; ++k) {
                float xj = xs[u][k];
                aj[k] = (ys[u][k] - xj) / sd;
                cj[k] = corr ? cs[u][k] / sc : 0.0f;
                dx[k] = xj - xi[k];
                sdy[k] += ys[u][k] - yi[k];
            }
            float len = sqrtf(dx[0] * dx[0] + dx[1] * dx[1] + dx[2] * dx[2]) / sl;
            float ac = sqrtf(cj[0] * cj[0] + cj[1] * cj[1] + cj[2] * cj[2]);
            if (jj == j0) {
                for (int k = 0; k < 3; ++k) {
                    mxa[k] = mna[k] = aj[k];
                    mxc[k] = mnc[k] = cj[k];
                }
                mxl = mnl = len;
                mxabsc = ac;
            } else {
                for (int k = 0; k < 3; ++k) {
                    mxa[k] = fmaxf(mxa[k], aj[k]);
                    mna[k] = fminf(mna[k], aj[k]);
                    mxc[k] = fmaxf(mxc[k], cj[k]);
                    mnc[k] = fminf(mnc[k], cj[k]);
                }
                mxl = fmaxf(mxl, len);
                mnl = fminf(mnl, len);
                mxabsc = fmaxf(mxabsc, ac);
            }
            for (int k = 0; k < 3; ++k) {
                sa[k] += aj[k];
                sc3[k] += cj[k];
                sdx[k] += dx[k];
            }
            slen += len;
            sabsc += ac;
            if (ms[u] == 0.0f) {
                ++npin;
                for (int k = 0; k < 3; ++k) spin[k] += dx[k];
            }
        }
    }
    float f[kIn];
    const float inv = deg > 0 ? 1.0f / (float)deg : 0.0f;
    const float absa = sqrtf(a[0] * a[0] + a[1] * a[1] + a[2] * a[2]);
    const float absc = sqrtf(c[0] * c[0] + c[1] * c[1] + c[2] * c[2]);
    for (int k = 0; k < 3; ++k) {
        f[0 + k] = a[k];
        f[3 + k] = c[k];
        f[6 + k] = deg > 0 ? sa[k] * inv - a[k] : 0.0f;
        f[9 + k] = deg > 0 ? sc3[k] * inv - c[k] : 0.0f;
        f[12 + k] = mxa[k] - a[k];
        f[15 + k] = mna[k] - a[k];
        f[18 + k] = mxc[k] - c[k];
        f[21 + k] = mnc[k] - c[k];
        f[24 + k] = sdx[k] * inv / sl;
        f[30 + k] = acc ? acc[3 * i + k] * dt * dt / sd : 0.0f;
        f[41 + k] = sdy[k] * inv / sl;
        f[44 + k] = spin[k] * inv / sl;
    }
    f[27] = slen * inv;
    f[28] = mxl;
    f[29] = mnl;
    f[33] = absa;
    f[34] = absc;
    f[35] = deg > 0 ? sabsc * inv : absc;
    f[36] = deg > 0 ? mxabsc : absc;
    f[37] = mass[i] / mm;
    f[38] = area[i] / ma;
    f[39] = (float)npin * inv;
    f[40] = (float)deg / 6.0f;
    f[47] = 1.0f;
    // rows leave through LDS: a lane's 96 bytes would be twelve 8-byte stores 96 bytes from the next lane's, the
    // wave's rows together are contiguous
    constexpr int kRowWords = kIn / 4;  // 8 bytes each
    uint2* const rows = s_rows + (threadIdx.x >> 6) * 64 * kRowWords;
#pragma unroll
    for (int k = 0; k < kIn; k += 4)
        rows[(threadIdx.x & 63) * kRowWords + k / 4] = make_uint2(pack_bf16x2(f[k], f[k + 1]),
                                                                  pack_bf16x2(f[k + 2], f[k + 3]));
    __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
    __builtin_amdgcn_wave_barrier();
    const int first = i - (int)(threadIdx.x & 63), count = min(64, n - first);  // the wave's rows, one a lane
    uint2* const dst = reinterpret_cast<uint2*>(out + (size_t)first * kIn);
    for (int e = threadIdx.x & 63; e < count * kRowWords; e += count) dst[e] = rows[e];
}

// ---- weight packing ------------------------------------------------------------
// ---- low-pass of correction fields --------------------------------------------
// One sweep of the 1-ring mean with the particle itself, for `width` floats per particle (e.g. two
// [n,3] fields side by side): out_i = (v_i + sum_j v_j) / (1 + degree_i) over solved particles
// (inactive ones read and write 0).  Repeated sweeps damp rough, neighbour-to-neighbour components
// of a predicted correction fast and its smooth ones slowly.
constexpr int kSmoothMaxWidth = 12;

// W > 0: the width at compile time (3 and 6: one and two fields; 1: a scalar, for which the run-time width's selects
// cost more than its loads, eight sweeps of 144 particles 23.1 -> 15.2 us); 0: width at run time.
// Bound: memory.  Six index loads and then six gathers are in flight at a time (one dependent pair after another
// before), and an XCD's particles share its L2: 1,048,576 particles of width 3 13.5 us a sweep, 4.7 TB/s (26.4 us).
template <int W>
__global__ __launch_bounds__(256) void k_smooth(int n, int width, const int* __restrict__ nbr_off,
                                                const int* __restrict__ nbr, const float* __restrict__ active,
                                                const float* __restrict__ in, float* __restrict__ out) {
    const int i = xcd_block(blockIdx.x, gridDim.x) * 256 + threadIdx.x;
    if (i >= n) return;
    constexpr int MAX = W > 0 ? W : kSmoothMaxWidth;
    if (W > 0) width = W;
    const int b = nbr_off[i], e = nbr_off[i + 1];
    const float act = active[i];
    float acc[MAX];
    const float* vi = in + (size_t)width * i;
#pragma unroll
    for (int c = 0; c < MAX; ++c)
        if (W > 0 || c < width) acc[c] = vi[c];
    float* o = out + (size_t)width * i;
    if (act == 0.0f) {
#pragma unroll
        for (int c = 0; c < MAX; ++c)
            if (W > 0 || c < width) o[c] = 0.0f;
        return;
    }
    if constexpr (W > 0) {
        for (int k = b; k < e; k += kRing) {
            int j[kRing];
            float w[kRing], v[kRing][MAX];
#pragma unroll
            for (int u = 0; u < kRing; ++u) j[u] = nbr[min(k + u, e - 1)];
#pragma unroll
            for (int u = 0; u < kRing; ++u) {
                w[u] = active[j[u]];
#pragma unroll
                for (int c = 0; c < MAX; ++c) v[u][c] = in[(size_t)W * j[u] + c];
            }
#pragma unroll
            for (int u = 0; u < kRing; ++u)
                if (k + u < e)
#pragma unroll
                    for (int c = 0; c < MAX; ++c) acc[c] += w[u] * v[u][c];
        }
    } else {
        for (int k = b; k < e; ++k) {
            const int j = nbr[k];
            const float w = active[j];
            const float* vj = in + (size_t)width * j;
#pragma unroll
            for (int c = 0; c < MAX; ++c)
                if (c < width) acc[c] += w * vj[c];
        }
    }
    const float inv = 1.0f / (float)(1 + e - b);
#pragma unroll
    for (int c = 0; c < MAX; ++c)
        if (W > 0 || c < width) o[c] = acc[c] * inv;
}

__global__ void k_pack(const float* __restrict__ prm, uint16_t* __restrict__ pk) {
    int e = blockIdx.x * blockDim.x + threadIdx.x;
    if (e >= kPacked) return;
    float v = 0.0f;
    if (e < pW1) {  // Wt1[j][k] = W1[k][j]
        int j = (e - pWt1) / kIn, k = (e - pWt1) % kIn;
        v = prm[oW1 + k * kHid + j];
    } else if (e < pWt2) {
        v = prm[oW1 + (e - pW1)];
    } else if (e < pW2) {
        int j = (e - pWt2) / kHid, k = (e - pWt2) % kHid;
        v = prm[oW2 + k * kHid + j];
    } else if (e < pWt3) {
        v = prm[oW2 + (e - pW2)];
    } else if (e < pW3) {
        int j = (e - pWt3) / kHid, k = (e - pWt3) % kHid;
        v = prm[oW3 + k * kHid + j];
    } else if (e < pWt4) {
        v = prm[oW3 + (e - pW3)];
    } else if (e < pW4) {  // Wt4[j][k] = W4[k][j], j < 3
        int j = (e - pWt4) / kHid, k = (e - pWt4) % kHid;
        v = j < kOut ? prm[oW4 + k * kOut + j] : 0.0f;
    } else {  // W4p[k][j], j < 3
        int k = (e - pW4) / kOutP, j = (e - pW4) % kOutP;
        v = j < kOut ? prm[oW4 + k * kOut + j] : 0.0f;
    }
    pk[e] = f2bf(v);
}

// ---- forward of the separate training pieces (the tests' reference; training takes k_gradient) ----
// One hidden layer for the wave's 16 rows: acc = A (16 x K) * Wt^T, A read from
// LDS rows (stride kStride) or, for the first layer, from the feature rows.
template <int K>
__device__ inline void layer_mm(const uint16_t* a_base, int a_stride, const uint16_t* __restrict__ wt, int li, int lq,
                                floatx4 (&acc)[8], bool a_valid) {
#pragma unroll
    for (int nt = 0; nt < 8; ++nt) acc[nt] = zero4();
#pragma unroll
    for (int kt = 0; kt < K / 16; ++kt) {
        bf16x4 a = a_valid ? ld4(a_base + li * a_stride + kt * 16 + lq * 4) : bf16x4{0, 0, 0, 0};
#pragma unroll
        for (int nt = 0; nt < 8; ++nt) {
            bf16x4 b = ld4(wt + (nt * 16 + li) * K + kt * 16 + lq * 4);
            acc[nt] = mfma(a, b, acc[nt]);
        }
    }
}

// bias + SiLU; writes the BF16 activations to the wave's LDS rows and, when
// saving, Z (FP32) and H (BF16) of layer l to global memory.
__device__ inline void layer_epilogue(floatx4 (&acc)[8], const float* __restrict__ bias, uint16_t* h_lds, int li,
                                      int lq, int row0, int n, int l, uint16_t* __restrict__ h_save,
                                      float* __restrict__ z_save) {
#pragma unroll
    for (int nt = 0; nt < 8; ++nt) {
        int j = nt * 16 + li;
        float bj = bias[j];
#pragma unroll
        for (int it = 0; it < 4; ++it) {
            int i = lq * 4 + it;
            float z = acc[nt][it] + bj;
            uint16_t hb = f2bf(z * sigmoid(z));
            h_lds[i * kStride + j] = hb;
            int r = row0 + i;
            if (h_save && r < n) {
                size_t o = ((size_t)r * 3 + l) * kHid + j;
                z_save[o] = z;
                h_save[o] = hb;
            }
        }
    }
}

__global__ __launch_bounds__(kBlock) void k_forward(int n, const uint16_t* __restrict__ feat,
                                                   const uint16_t* __restrict__ pk, const float* __restrict__ prm,
                                                   float* __restrict__ out, uint16_t* __restrict__ h_save,
                                                   float* __restrict__ z_save) {
    __shared__ __align__(16) uint16_t s_h[kWaves][kWaveRows * kStride];
    const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63, li = lane & 15, lq = lane >> 4;
    const int row0 = (blockIdx.x * kWaves + wave) * kWaveRows;
    uint16_t* H = s_h[wave];
    floatx4 acc[8];
    const bool valid = row0 + li < n;
    layer_mm<kIn>(feat + (size_t)row0 * kIn, kIn, pk + pWt1, li, lq, acc, valid);
    layer_epilogue(acc, prm + ob1, H, li, lq, row0, n, 0, h_save, z_save);
    __syncthreads();
    layer_mm<kHid>(H, kStride, pk + pWt2, li, lq, acc, true);
    __syncthreads();
    layer_epilogue(acc, prm + ob2, H, li, lq, row0, n, 1, h_save, z_save);
    __syncthreads();
    layer_mm<kHid>(H, kStride, pk + pWt3, li, lq, acc, true);
    __syncthreads();
    layer_epilogue(acc, prm + ob3, H, li, lq, row0, n, 2, h_save, z_save);
    __syncthreads();
    floatx4 o = zero4();
#pragma unroll
    for (int kt = 0; kt < kHid / 16; ++kt) {
        bf16x4 a = ld4(H + li * kStride + kt * 16 + lq * 4);
        bf16x4 b = ld4(pk + pWt4 + li * kHid + kt * 16 + lq * 4);
        o = mfma(a, b, o);
    }
    if (li < kOut) {
        float b4 = prm[ob4 + li];
#pragma unroll
        for (int it = 0; it < 4; ++it) {
            int r = row0 + lq * 4 + it;
            if (r < n) out[(size_t)r * kOut + li] = o[it] + b4;
        }
    }
}

// ---- inference: weights resident in LDS, activations in registers, 16x16x32 BF16 MFMA ---------
// k_forward re-reads every weight tile from L2 for each 16 rows (about 6 KB per row), which bounds
// it far below the matrix cores.  The inference kernel keeps all four BF16 weight matrices in LDS
// (84 KB, loaded once per work-group) and uses gfx950's v_mfma_f32_16x16x32_bf16 (A: lane = row l % 16,
// k = 8 (l / 16) .. + 7 of the 32-wide k step; B: lane = column l % 16, same k; C: lane holds rows
// 4 (l / 16) .. + 3 of column l % 16).  Each layer is computed transposed, Z^T = W^T H^T: the weight
// tile is the A operand and the activation rows the B operand, so a lane ends with four consecutive
// output columns of one row in each of eight tiles.  The sum over k may take k in any order, as long as
// both operands take the same: with lane (li, lq) carrying k = 32 kt + 4 lq .. + 3 and 32 kt + 16 + 4 lq
// .. + 3, a lane's own columns of tiles 2 kt and 2 kt + 1 are its B operand of the next layer.  So the
// activations never leave their lane -- no LDS, no shuffle, no barrier -- and the weights lie in LDS in
// that order, one 16-byte read per lane and tile, without bank conflicts.  A wave carries one or two
// groups of 16 rows.  SiLU uses the hardware exp2 and reciprocal (the
// activations are rounded to BF16 right after); the biases are the accumulators' first values.
// Bound: the 384 SiLUs a row, two quarter-rate instructions each (about 85 us per million rows, 120 with the
// multiplies); without the barriers of an LDS exchange the other waves' products fill in beside them:
// 1,048,576 rows 127 us, 650 TFLOP/s (223 us with activations exchanged through LDS; 137 to 144 us on other cards and
// under a kernel trace), 16,384 rows 9.2 us (17.7).
typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));

constexpr int kFrag1 = 0;                      // layer 1: k to 64 (zero past 48), then eight tiles of 16 columns
constexpr int kFrag2 = kFrag1 + 2 * 8 * 64;    // layers 2 and 3: four k steps
constexpr int kFrag3 = kFrag2 + 4 * 8 * 64;
constexpr int kFrag4 = kFrag3 + 4 * 8 * 64;    // layer 4: one tile
constexpr int kFrags = kFrag4 + 4 * 64;        // 16-byte fragments, (k step, tile, lane)

__device__ inline floatx4 mfma32(bf16x8 a, bf16x8 b, floatx4 c) {
    return __builtin_amdgcn_mfma_f32_16x16x32_bf16(a, b, c, 0, 0, 0);
}

__device__ inline bf16x8 ld8(const uint16_t* p) { return *reinterpret_cast<const bf16x8*>(p); }

__device__ inline float silu_fast(float z) {
    return z * __builtin_amdgcn_rcpf(1.0f + __builtin_amdgcn_exp2f(-1.4426950408889634f * z));
}

// fragment f of the weights: lane (li, lq) of tile nt and k step kt of its layer
__device__ inline uint4 weight_fragment(const uint16_t* __restrict__ pk, int f) {
    const int lane = f & 63, li = lane & 15, lq = lane >> 4;
    if (f < kFrag2) {
        const int nt = (f >> 6) & 7, k = ((f >> 9) & 1) * 32 + lq * 8;
        if (k >= kIn) return make_uint4(0u, 0u, 0u, 0u);
        return *reinterpret_cast<const uint4*>(pk + pWt1 + (nt * 16 + li) * kIn + k);
    }
    const bool last = f >= kFrag4;
    const int at = f - (last ? kFrag4 : (f >= kFrag3 ? kFrag3 : kFrag2));
    const int nt = last ? 0 : (at >> 6) & 7, kt = last ? at >> 6 : at >> 9;
    const uint16_t* row = pk + (last ? pWt4 : (f >= kFrag3 ? pWt3 : pWt2)) + (nt * 16 + li) * kHid + kt * 32 + lq * 4;
    const uint2 lo = *reinterpret_cast<const uint2*>(row), hi = *reinterpret_cast<const uint2*>(row + 16);
    return make_uint4(lo.x, lo.y, hi.x, hi.y);
}

// one layer of the wave's S row groups: accumulators from the biases, then the k steps
template <int S, int KSTEPS>
__device__ inline void infer_layer(const uint4* w, const float4* bias, const bf16x8 (&b)[S][KSTEPS], int lane,
                                   floatx4 (&acc)[S][8]) {
    asm volatile("" ::: "memory");  // the weights stay in LDS: hoisted out of the row loop they would fill every register
#pragma unroll
    for (int nt = 0; nt < 8; ++nt) {
        const float4 v = bias[nt * 4 + (lane >> 4)];
#pragma unroll
        for (int s = 0; s < S; ++s) acc[s][nt] = floatx4{v.x, v.y, v.z, v.w};
    }
#pragma unroll
    for (int kt = 0; kt < KSTEPS; ++kt)
#pragma unroll
        for (int nt = 0; nt < 8; ++nt) {
            const bf16x8 a = __builtin_bit_cast(bf16x8, w[(kt * 8 + nt) * 64 + lane]);
#pragma unroll
            for (int s = 0; s < S; ++s) acc[s][nt] = mfma32(a, b[s][kt], acc[s][nt]);
        }
}

// SiLU of the accumulators into the next layer's operands, lane by lane
template <int S>
__device__ inline void infer_silu(const floatx4 (&acc)[S][8], bf16x8 (&b)[S][4]) {
#pragma unroll
    for (int s = 0; s < S; ++s)
#pragma unroll
        for (int kt = 0; kt < 4; ++kt) {
            const floatx4 lo = acc[s][2 * kt], hi = acc[s][2 * kt + 1];
            const uint4 u = make_uint4(pack_bf16x2(silu_fast(lo[0]), silu_fast(lo[1])),
                                       pack_bf16x2(silu_fast(lo[2]), silu_fast(lo[3])),
                                       pack_bf16x2(silu_fast(hi[0]), silu_fast(hi[1])),
                                       pack_bf16x2(silu_fast(hi[2]), silu_fast(hi[3])));
            b[s][kt] = __builtin_bit_cast(bf16x8, u);
        }
}

// WAVES a work-group, S groups of 16 rows a wave
template <int WAVES, int S>
__global__ __launch_bounds__(64 * WAVES) void k_infer(int n, const uint16_t* __restrict__ feat,
                                                      const uint16_t* __restrict__ pk, const float* __restrict__ prm,
                                                      float* __restrict__ out) {
    __shared__ uint4 s_w[kFrags];
    __shared__ float4 s_b[3][kHid / 4];
    for (int f = threadIdx.x; f < kFrags; f += 64 * WAVES) s_w[f] = weight_fragment(pk, f);
    for (int e = threadIdx.x; e < 3 * kHid; e += 64 * WAVES)
        reinterpret_cast<float*>(s_b)[e] = prm[(e < kHid ? ob1 : (e < 2 * kHid ? ob2 - kHid : ob3 - 2 * kHid)) + e];
    __syncthreads();
    const int lane = threadIdx.x & 63, li = lane & 15, lq = lane >> 4;
    const float b40 = prm[ob4], b41 = prm[ob4 + 1], b42 = prm[ob4 + 2];
    constexpr int ROWS = 16 * S;
    const long groups = ((long)n + ROWS - 1) / ROWS;
    for (long g = (long)blockIdx.x * WAVES + (threadIdx.x >> 6); g < groups; g += (long)gridDim.x * WAVES) {
        floatx4 acc[S][8];
        bf16x8 b[S][4];
        {
            // layer 1: the B operand straight from the feature rows (48 BF16 each); k >= 48 and rows >= n
            // read as 0
            bf16x8 f[S][2] = {};
#pragma unroll
            for (int s = 0; s < S; ++s) {
                const long r = g * ROWS + s * 16 + li;
                if (r < n) {
                    f[s][0] = ld8(feat + r * kIn + lq * 8);
                    if (lq < 2) f[s][1] = ld8(feat + r * kIn + 32 + lq * 8);
                }
            }
            infer_layer<S, 2>(s_w + kFrag1, s_b[0], f, lane, acc);
        }
        infer_silu<S>(acc, b);
        infer_layer<S, 4>(s_w + kFrag2, s_b[1], b, lane, acc);
        infer_silu<S>(acc, b);
        infer_layer<S, 4>(s_w + kFrag3, s_b[2], b, lane, acc);
        infer_silu<S>(acc, b);
        floatx4 o[S];
#pragma unroll
        for (int s = 0; s < S; ++s) o[s] = zero4();
#pragma unroll
        for (int kt = 0; kt < 4; ++kt) {
            const bf16x8 a = __builtin_bit_cast(bf16x8, s_w[kFrag4 + kt * 64 + lane]);
#pragma unroll
            for (int s = 0; s < S; ++s) o[s] = mfma32(a, b[s][kt], o[s]);
        }
        // lane (li, lq = 0) holds outputs 0..3 of its row; the first three are the network's
        if (lq == 0)
#pragma unroll
            for (int s = 0; s < S; ++s) {
                const long r = g * ROWS + s * 16 + li;
                if (r < n) {
                    out[r * kOut] = o[s][0] + b40;
                    out[r * kOut + 1] = o[s][1] + b41;
                    out[r * kOut + 2] = o[s][2] + b42;
                }
            }
    }
}

// ---- backward --------------------------------------------------------------------
// dA (16 x Kout) of the wave's rows times W^T: dH[r][j] = sum_k dZ[r][k] W[j][k];
// B operand B[k][j] = W[j][k] read from the natural W layout [in][out] (stride KO).
template <int KO>
__device__ inline void back_mm(const uint16_t* dz_lds, int dz_stride, const uint16_t* __restrict__ w, int li, int lq,
                               floatx4 (&acc)[8]) {
#pragma unroll
    for (int nt = 0; nt < 8; ++nt) acc[nt] = zero4();
#pragma unroll
    for (int kt = 0; kt < KO / 16; ++kt) {
        bf16x4 a = ld4(dz_lds + li * dz_stride + kt * 16 + lq * 4);
#pragma unroll
        for (int nt = 0; nt < 8; ++nt) {
            bf16x4 b = ld4(w + (nt * 16 + li) * KO + kt * 16 + lq * 4);
            acc[nt] = mfma(a, b, acc[nt]);
        }
    }
}

// dZ = bf16(dH * silu'(Z)) for the wave's rows into LDS (rows past n get 0).
__device__ inline void back_epilogue(floatx4 (&acc)[8], const float* __restrict__ z_save, int l, uint16_t* dz_lds,
                                     int li, int lq, int row0, int n) {
#pragma unroll
    for (int nt = 0; nt < 8; ++nt) {
        int j = nt * 16 + li;
#pragma unroll
        for (int it = 0; it < 4; ++it) {
            int i = lq * 4 + it;
            int r = row0 + i;
            float d = 0.0f;
            if (r < n) {
                float z = z_save[((size_t)r * 3 + l) * kHid + j];
                float s = sigmoid(z);
                d = acc[nt][it] * (s * (1.0f + z * (1.0f - s)));
            }
            dz_lds[i * kStride + j] = f2bf(d);
        }
    }
}

// Partial weight gradient dW[i][j] = sum_rows A[r][i] * dZ[r][j] over the
// workgroup's 64 rows, for output tiles (it_i, it_j) assigned to this wave.
// a: [64][a_stride] BF16 rows, dz: [64][dz_stride] BF16 rows.
template <int MI, int NJ>
__device__ inline void weight_grad(const uint16_t* a, int a_stride, const uint16_t* dz, int dz_stride, int wave,
                                   int li, int lq, float* __restrict__ gw, int ld_out, int ncols) {
    constexpr int tiles = (MI / 16) * (NJ / 16);
    for (int t = wave; t < tiles; t += kWaves) {
        int ti = t / (NJ / 16), tj = t % (NJ / 16);
        floatx4 acc = zero4();
#pragma unroll
        for (int kt = 0; kt < kRowsWG / 16; ++kt) {
            int r = kt * 16 + lq * 4;
            bf16x4 av = ld4_strided(a + r * a_stride + ti * 16 + li, a_stride);
            bf16x4 bv = ld4_strided(dz + r * dz_stride + tj * 16 + li, dz_stride);
            acc = mfma(av, bv, acc);
        }
        int j = tj * 16 + li;
        if (j < ncols) {
#pragma unroll
            for (int it = 0; it < 4; ++it) {
                int i = ti * 16 + lq * 4 + it;
                gw[i * ld_out + j] = acc[it];
            }
        }
    }
}

// column sums of dZ (BF16 rows) over the workgroup's rows, in row order
__device__ inline void bias_grad(const uint16_t* dz, int dz_stride, int ncols, float* __restrict__ gb) {
    for (int j = threadIdx.x; j < ncols; j += kBlock) {
        float s = 0.0f;
        for (int r = 0; r < kRowsWG; ++r) s += bf2f(dz[r * dz_stride + j]);
        gb[j] = s;
    }
}

// stage a [64][K] BF16 block of global rows (row stride ld, first column col0) into LDS
template <int K>
__device__ inline void stage_rows(const uint16_t* __restrict__ src, size_t ld, int col0, int row0, int n,
                                  uint16_t* dst, int dst_stride) {
    for (int e = threadIdx.x; e < kRowsWG * (K / 4); e += kBlock) {
        int r = e / (K / 4), c = (e % (K / 4)) * 4;
        bf16x4 v = bf16x4{0, 0, 0, 0};
        if (row0 + r < n) v = ld4(src + (size_t)(row0 + r) * ld + col0 + c);
        *reinterpret_cast<bf16x4*>(dst + r * dst_stride + c) = v;
    }
}

// LDS: dZ4 (64 x 16) and three 64 x 128 BF16 row blocks A, B, C (~55 KB), reused as
//   A: dZ3, later dZ1     B: staged H3, H2, H1, X     C: dZ2
__global__ __launch_bounds__(kBlock) void k_backward(int n, const uint16_t* __restrict__ feat,
                                                    const float* __restrict__ target, const float* __restrict__ roww,
                                                    const uint16_t* __restrict__ pk, const float* __restrict__ out,
                                                    const uint16_t* __restrict__ h_save,
                                                    const float* __restrict__ z_save, float* __restrict__ pgrad,
                                                    float* __restrict__ ploss, float inv_count) {
    __shared__ __align__(16) uint16_t s_dz4[kRowsWG * kStrideOut];
    __shared__ __align__(16) uint16_t s_a[kRowsWG * kStride];
    __shared__ __align__(16) uint16_t s_b[kRowsWG * kStride];
    __shared__ __align__(16) uint16_t s_c[kRowsWG * kStride];
    __shared__ float s_loss[kBlock];
    const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63, li = lane & 15, lq = lane >> 4;
    const int wg_row0 = blockIdx.x * kRowsWG;
    const int wr = wave * kWaveRows;
    const int row0 = wg_row0 + wr;
    float* g = pgrad + (size_t)blockIdx.x * kParams;

    // dY = 2 w (out - target) / (3 n); dZ4 = bf16(dY), padded to 16 columns
    float lsum = 0.0f;
    for (int e = threadIdx.x; e < kRowsWG * kOutP; e += kBlock) {
        int r = e / kOutP, j = e % kOutP, gr = wg_row0 + r;
        float d = 0.0f;
        if (j < kOut && gr < n) {
            float w = roww ? roww[gr] : 1.0f;
            float diff = out[(size_t)gr * kOut + j] - target[(size_t)gr * kOut + j];
            lsum += w * diff * diff;
            d = 2.0f * w * diff * inv_count;
        }
        s_dz4[r * kStrideOut + j] = f2bf(d);
    }
    s_loss[threadIdx.x] = lsum;
    __syncthreads();
    if (threadIdx.x == 0) {
        float s = 0.0f;
        for (int t = 0; t < kBlock; ++t) s += s_loss[t];
        ploss[blockIdx.x] = s * inv_count;
    }

    floatx4 acc[8];
    // dZ3 (wave rows) -> A; H3 -> B
    back_mm<kOutP>(s_dz4 + wr * kStrideOut, kStrideOut, pk + pW4, li, lq, acc);
    back_epilogue(acc, z_save, 2, s_a + wr * kStride, li, lq, row0, n);
    stage_rows<kHid>(h_save, (size_t)3 * kHid, 2 * kHid, wg_row0, n, s_b, kStride);
    __syncthreads();
    // dW4 = H3^T dZ4, db4; dZ2 (wave rows) -> C
    weight_grad<kHid, kOutP>(s_b, kStride, s_dz4, kStrideOut, wave, li, lq, g + oW4, kOut, kOut);
    bias_grad(s_dz4, kStrideOut, kOut, g + ob4);
    back_mm<kHid>(s_a + wr * kStride, kStride, pk + pW3, li, lq, acc);
    back_epilogue(acc, z_save, 1, s_c + wr * kStride, li, lq, row0, n);
    __syncthreads();
    // H2 -> B; dW3 = H2^T dZ3, db3
    stage_rows<kHid>(h_save, (size_t)3 * kHid, kHid, wg_row0, n, s_b, kStride);
    __syncthreads();
    weight_grad<kHid, kHid>(s_b, kStride, s_a, kStride, wave, li, lq, g + oW3, kHid, kHid);
    bias_grad(s_a, kStride, kHid, g + ob3);
    __syncthreads();
    // dZ1 (wave rows) -> A; H1 -> B
    back_mm<kHid>(s_c + wr * kStride, kStride, pk + pW2, li, lq, acc);
    back_epilogue(acc, z_save, 0, s_a + wr * kStride, li, lq, row0, n);
    stage_rows<kHid>(h_save, (size_t)3 * kHid, 0, wg_row0, n, s_b, kStride);
    __syncthreads();
    // dW2 = H1^T dZ2, db2
    weight_grad<kHid, kHid>(s_b, kStride, s_c, kStride, wave, li, lq, g + oW2, kHid, kHid);
    bias_grad(s_c, kStride, kHid, g + ob2);
    __syncthreads();
    // X -> B; dW1 = X^T dZ1, db1
    stage_rows<kIn>(feat, (size_t)kIn, 0, wg_row0, n, s_b, kStrideIn);
    __syncthreads();
    weight_grad<kIn, kHid>(s_b, kStrideIn, s_a, kStride, wave, li, lq, g + oW1, kHid, kHid);
    bias_grad(s_a, kStride, kHid, g + ob1);
}

__global__ void k_reduce(int nparts, const float* __restrict__ pgrad, const float* __restrict__ ploss,
                         float* __restrict__ grad, float* __restrict__ loss) {
    int p = blockIdx.x * blockDim.x + threadIdx.x;
    if (p < kParams) {
        float s = 0.0f;
        for (int w = 0; w < nparts; ++w) s += pgrad[(size_t)w * kParams + p];
        grad[p] = s;
    }
    if (p == 0 && loss) {
        float s = 0.0f;
        for (int w = 0; w < nparts; ++w) s += ploss[w];
        loss[0] = s;
    }
}

// ---- gradient in one kernel ----------------------------------------------------------
// vbd_ws_forward_train + vbd_ws_backward write H and Z of every row to memory and read them back (2.3 KB a row), and
// one partial gradient (159 KB) per 64 rows.  Here a work-group of four waves keeps everything of its 64 rows on the
// CU and the weight gradients of all its row blocks in registers, and writes one partial gradient.
// Forward and backward run in the transposed form of k_infer (a lane holds four columns of one row in each of eight
// tiles, which are its operand of the next product), so both chains stay in registers, with silu'(Z) in FP32 where
// the forward pass had Z.  The weight gradients contract over rows: H_l and dZ_l go to LDS once, column by column
// (64 rows of one column are 144 bytes), where 16 bytes are the eight rows a lane needs; wave w owns the tiles of
// rows 32 w .. 32 w + 31 of W2 and W3 (and a quarter of the others), 160 registers of sums.  Bias gradients are
// products with ones.  Rounding points as listed at the top; the order of the FP32 sums over rows is fixed.
// The hidden layers' weights are loaded a layer ahead and pass through LDS (read from L2 fragment by fragment they
// were half the kernel: 82 -> 41 us).  Bound: a block's chain of products on one wave per SIMD (18 us), and 159 KB of
// partial gradients a CU.  Training step: 16,384 rows 52 us (190 us in five kernels), 150,000 rows 218 us (1,739).
constexpr int kTS = kRowsWG + 8;                     // BF16 elements per LDS column (conflict-free 16-byte reads)
constexpr int kTrainTiles = 3 * 2 * kHid + kIn + kOutP;  // columns in LDS: H1-3, dZ1-3, X, dZ4

__device__ inline bf16x8 frag_perm(const uint16_t* __restrict__ row, int kt, int lq) {
    const uint16_t* p = row + kt * 32 + lq * 4;
    const uint2 lo = *reinterpret_cast<const uint2*>(p), hi = *reinterpret_cast<const uint2*>(p + 16);
    return __builtin_bit_cast(bf16x8, make_uint4(lo.x, lo.y, hi.x, hi.y));
}

// A 128 x 128 weight matrix on its way to LDS: eight 16-byte loads a thread, issued a layer ahead, then stored in
// the order the products read it (fragments of one k step and tile, lane by lane).
struct WeightStage {
    uint4 u[8];
    __device__ inline void load(const uint16_t* __restrict__ w) {
#pragma unroll
        for (int i = 0; i < 8; ++i) u[i] = reinterpret_cast<const uint4*>(w)[i * kBlock + threadIdx.x];
    }
    __device__ inline void store(uint4* s) const {
#pragma unroll
        for (int i = 0; i < 8; ++i) {
            const int e = i * kBlock + threadIdx.x, r = e >> 4, k = (e & 15) * 8;
            uint2* f = reinterpret_cast<uint2*>(s + ((k >> 5) * 8 + (r >> 4)) * 64 + (r & 15));
            const int lq = (k >> 2) & 3, half = (k >> 4) & 1;  // k .. k + 3 and k + 4 .. k + 7
            f[lq * 32 + half] = make_uint2(u[i].x, u[i].y);
            f[lq * 32 + 32 + half] = make_uint2(u[i].z, u[i].w);
        }
    }
};

// products of the staged matrix with the wave's operand
__device__ inline void train_mm(const uint4* w, const bf16x8 (&b)[4], int lane, floatx4 (&acc)[8]) {
#pragma unroll
    for (int kt = 0; kt < 4; ++kt)
#pragma unroll
        for (int nt = 0; nt < 8; ++nt)
            acc[nt] = mfma32(__builtin_bit_cast(bf16x8, w[(kt * 8 + nt) * 64 + lane]), b[kt], acc[nt]);
}

// column `col` of the lane's row (block row `row`) <- four BF16 values of consecutive columns
__device__ inline void put_columns(uint16_t* t, int col, int row, uint32_t lo, uint32_t hi) {
    t[col * kTS + row] = (uint16_t)lo;
    t[(col + 1) * kTS + row] = (uint16_t)(lo >> 16);
    t[(col + 2) * kTS + row] = (uint16_t)hi;
    t[(col + 3) * kTS + row] = (uint16_t)(hi >> 16);
}

// SiLU of the accumulators: the next operand, its columns in LDS, and silu'(z)
__device__ inline void train_silu(const floatx4 (&acc)[8], bf16x8 (&b)[4], floatx4 (&dsilu)[8], uint16_t* t, int lq,
                                  int row) {
    uint32_t u[8][2];
#pragma unroll
    for (int nt = 0; nt < 8; ++nt) {
        float h[4];
#pragma unroll
        for (int c = 0; c < 4; ++c) {
            const float z = acc[nt][c], s = vbd_scalar::sigmoid_short(z);
            h[c] = z * s;
            dsilu[nt][c] = s * (1.0f + z * (1.0f - s));
        }
        u[nt][0] = pack_bf16x2(h[0], h[1]);
        u[nt][1] = pack_bf16x2(h[2], h[3]);
        put_columns(t, nt * 16 + lq * 4, row, u[nt][0], u[nt][1]);
    }
#pragma unroll
    for (int kt = 0; kt < 4; ++kt)
        b[kt] = __builtin_bit_cast(bf16x8, make_uint4(u[2 * kt][0], u[2 * kt][1], u[2 * kt + 1][0], u[2 * kt + 1][1]));
}

// dZ = bf16(dH silu'(Z)): the next operand and its columns in LDS
__device__ inline void train_dz(const floatx4 (&acc)[8], const floatx4 (&dsilu)[8], bf16x8 (&b)[4], uint16_t* t,
                                int lq, int row) {
    uint32_t u[8][2];
#pragma unroll
    for (int nt = 0; nt < 8; ++nt) {
        u[nt][0] = pack_bf16x2(acc[nt][0] * dsilu[nt][0], acc[nt][1] * dsilu[nt][1]);
        u[nt][1] = pack_bf16x2(acc[nt][2] * dsilu[nt][2], acc[nt][3] * dsilu[nt][3]);
        put_columns(t, nt * 16 + lq * 4, row, u[nt][0], u[nt][1]);
    }
#pragma unroll
    for (int kt = 0; kt < 4; ++kt)
        b[kt] = __builtin_bit_cast(bf16x8, make_uint4(u[2 * kt][0], u[2 * kt][1], u[2 * kt + 1][0], u[2 * kt + 1][1]));
}

__device__ inline void bias_init(const float* __restrict__ bias, int lq, floatx4 (&acc)[8]) {
#pragma unroll
    for (int nt = 0; nt < 8; ++nt)
#pragma unroll
        for (int c = 0; c < 4; ++c) acc[nt][c] = bias[nt * 16 + lq * 4 + c];
}

// rows of tile ti x columns of tile tj of sum_rows A[row][i] B[row][j], 64 rows
__device__ inline floatx4 rows_mm(const uint16_t* a, int ti, const uint16_t* b, int tj, int li, int lq, floatx4 acc) {
#pragma unroll
    for (int ks = 0; ks < 2; ++ks)
        acc = mfma32(ld8(a + (ti * 16 + li) * kTS + ks * 32 + lq * 8), ld8(b + (tj * 16 + li) * kTS + ks * 32 + lq * 8),
                     acc);
    return acc;
}

__device__ inline void put_tile(float* __restrict__ g, int ld, int ti, int tj, int cols, int li, int lq, floatx4 v) {
    const int j = tj * 16 + li;
    if (j < cols)
#pragma unroll
        for (int it = 0; it < 4; ++it) g[(ti * 16 + lq * 4 + it) * ld + j] = v[it];
}

__global__ __launch_bounds__(kBlock) __attribute__((amdgpu_waves_per_eu(1, 1))) void k_gradient(
    int n, const uint16_t* __restrict__ feat, const float* __restrict__ target, const float* __restrict__ roww,
    const uint16_t* __restrict__ pk, const float* __restrict__ prm, float* __restrict__ pgrad,
    float* __restrict__ ploss, float inv_count) {
    __shared__ __align__(16) uint16_t s_t[kTrainTiles * kTS];
    __shared__ uint4 s_w[4 * 8 * 64];
    __shared__ float s_loss[kBlock];
    uint16_t* const tH[3] = {s_t, s_t + kHid * kTS, s_t + 2 * kHid * kTS};
    uint16_t* const tD[3] = {s_t + 3 * kHid * kTS, s_t + 4 * kHid * kTS, s_t + 5 * kHid * kTS};
    uint16_t* const tX = s_t + 6 * kHid * kTS;
    uint16_t* const tD4 = tX + kIn * kTS;
    const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63, li = lane & 15, lq = lane >> 4;
    const int row = wave * kWaveRows + li;  // the block row this lane carries
    for (int e = threadIdx.x; e < kOutP * kTS; e += kBlock) tD4[e] = 0;  // columns 3 .. 15 stay zero
    __syncthreads();

    floatx4 w1[3][2], w2[2][8], w3[2][8], w4[2], gb[3][2], gb4 = zero4();
#pragma unroll
    for (int a = 0; a < 2; ++a) {
        w4[a] = zero4();
#pragma unroll
        for (int b = 0; b < 3; ++b) w1[b][a] = gb[b][a] = zero4();
#pragma unroll
        for (int b = 0; b < 8; ++b) w2[a][b] = w3[a][b] = zero4();
    }
    float lsum = 0.0f;
    const bf16x8 ones = {(__bf16)1.0f, (__bf16)1.0f, (__bf16)1.0f, (__bf16)1.0f,
                         (__bf16)1.0f, (__bf16)1.0f, (__bf16)1.0f, (__bf16)1.0f};
    const int blocks = (n + kRowsWG - 1) / kRowsWG;
    for (int blk = blockIdx.x; blk < blocks; blk += gridDim.x) {
        const long r = (long)blk * kRowsWG + row;
        const bool valid = r < n;
        // the weights are read anew for every block: hoisted out of the loop they would fill every register
        asm volatile("" : "+s"(pk), "+s"(prm));
        floatx4 acc[8], d1[8], d2[8], d3[8];
        bf16x8 b[4];
        WeightStage stage;
        stage.load(pk + pWt2);
        // layer 1: k in natural order (rows >= n and k >= 48 read as 0)
        {
            uint4 f0 = make_uint4(0u, 0u, 0u, 0u), f1 = f0;
            if (valid) {
                f0 = *reinterpret_cast<const uint4*>(feat + r * kIn + lq * 8);
                if (lq < 2) f1 = *reinterpret_cast<const uint4*>(feat + r * kIn + 32 + lq * 8);
            }
            put_columns(tX, lq * 8, row, f0.x, f0.y);
            put_columns(tX, lq * 8 + 4, row, f0.z, f0.w);
            if (lq < 2) {
                put_columns(tX, 32 + lq * 8, row, f1.x, f1.y);
                put_columns(tX, 32 + lq * 8 + 4, row, f1.z, f1.w);
            }
            bias_init(prm + ob1, lq, acc);
#pragma unroll
            for (int nt = 0; nt < 8; ++nt) {
                const uint16_t* w = pk + pWt1 + (nt * 16 + li) * kIn;
                acc[nt] = mfma32(ld8(w + lq * 8), __builtin_bit_cast(bf16x8, f0), acc[nt]);
                bf16x8 a1 = {};
                if (lq < 2) a1 = ld8(w + 32 + lq * 8);
                acc[nt] = mfma32(a1, __builtin_bit_cast(bf16x8, f1), acc[nt]);
            }
        }
        train_silu(acc, b, d1, tH[0], lq, row);
        stage.store(s_w);
        stage.load(pk + pWt3);
        __syncthreads();
        bias_init(prm + ob2, lq, acc);
        train_mm(s_w, b, lane, acc);
        __syncthreads();
        stage.store(s_w);
        stage.load(pk + pW3);
        train_silu(acc, b, d2, tH[1], lq, row);
        __syncthreads();
        bias_init(prm + ob3, lq, acc);
        train_mm(s_w, b, lane, acc);
        __syncthreads();
        stage.store(s_w);
        stage.load(pk + pW2);
        train_silu(acc, b, d3, tH[2], lq, row);
        floatx4 o = zero4();
#pragma unroll
        for (int kt = 0; kt < 4; ++kt) o = mfma32(frag_perm(pk + pWt4 + li * kHid, kt, lq), b[kt], o);
        // dY = 2 w (out - target) / (3 n); the lanes with lq = 0 hold the row's outputs
        uint32_t dz_lo = 0u, dz_hi = 0u;
        if (lq == 0) {
            float d[3] = {0.0f, 0.0f, 0.0f};
            if (valid) {
                const float w = roww ? roww[r] : 1.0f;
#pragma unroll
                for (int j = 0; j < kOut; ++j) {
                    const float diff = o[j] + prm[ob4 + j] - target[r * kOut + j];
                    lsum += w * diff * diff;
                    d[j] = 2.0f * w * diff * inv_count;
                }
            }
            dz_lo = pack_bf16x2(d[0], d[1]);
            dz_hi = pack_bf16x2(d[2], 0.0f);
            put_columns(tD4, 0, row, dz_lo, dz_hi);
        }
        // backward chain
        const bf16x8 dz4 = __builtin_bit_cast(bf16x8, make_uint4(dz_lo, dz_hi, 0u, 0u));
#pragma unroll
        for (int nt = 0; nt < 8; ++nt) {
            uint2 w = make_uint2(0u, 0u);
            if (lq == 0) w = *reinterpret_cast<const uint2*>(pk + pW4 + (nt * 16 + li) * kOutP);
            acc[nt] = mfma32(__builtin_bit_cast(bf16x8, make_uint4(w.x, w.y, 0u, 0u)), dz4, zero4());
        }
        train_dz(acc, d3, b, tD[2], lq, row);
#pragma unroll
        for (int nt = 0; nt < 8; ++nt) acc[nt] = zero4();
        __syncthreads();
        train_mm(s_w, b, lane, acc);
        __syncthreads();
        stage.store(s_w);
        train_dz(acc, d2, b, tD[1], lq, row);
        __syncthreads();
#pragma unroll
        for (int nt = 0; nt < 8; ++nt) acc[nt] = zero4();
        train_mm(s_w, b, lane, acc);
        train_dz(acc, d1, b, tD[0], lq, row);
        __syncthreads();
        // weight gradients over the block's 64 rows
#pragma unroll
        for (int a = 0; a < 2; ++a) {
            const int t = 2 * wave + a;
#pragma unroll
            for (int tj = 0; tj < 8; ++tj) {
                w2[a][tj] = rows_mm(tH[0], t, tD[1], tj, li, lq, w2[a][tj]);
                w3[a][tj] = rows_mm(tH[1], t, tD[2], tj, li, lq, w3[a][tj]);
            }
            w4[a] = rows_mm(tH[2], t, tD4, 0, li, lq, w4[a]);
#pragma unroll
            for (int ti = 0; ti < 3; ++ti) w1[ti][a] = rows_mm(tX, ti, tD[0], t, li, lq, w1[ti][a]);
#pragma unroll
            for (int l = 0; l < 3; ++l)
#pragma unroll
                for (int ks = 0; ks < 2; ++ks)
                    gb[l][a] = mfma32(ones, ld8(tD[l] + (t * 16 + li) * kTS + ks * 32 + lq * 8), gb[l][a]);
        }
#pragma unroll
        for (int ks = 0; ks < 2; ++ks) gb4 = mfma32(ones, ld8(tD4 + li * kTS + ks * 32 + lq * 8), gb4);
        __syncthreads();
    }
    float* g = pgrad + (size_t)blockIdx.x * kParams;
#pragma unroll
    for (int a = 0; a < 2; ++a) {
        const int t = 2 * wave + a;
#pragma unroll
        for (int tj = 0; tj < 8; ++tj) {
            put_tile(g + oW2, kHid, t, tj, kHid, li, lq, w2[a][tj]);
            put_tile(g + oW3, kHid, t, tj, kHid, li, lq, w3[a][tj]);
        }
        put_tile(g + oW4, kOut, t, 0, kOut, li, lq, w4[a]);
#pragma unroll
        for (int ti = 0; ti < 3; ++ti) put_tile(g + oW1, kHid, ti, t, kHid, li, lq, w1[ti][a]);
        if (lq == 0) {  // every row of a product with ones is the column sums
            g[ob1 + t * 16 + li] = gb[0][a][0];
            g[ob2 + t * 16 + li] = gb[1][a][0];
            g[ob3 + t * 16 + li] = gb[2][a][0];
        }
    }
    if (wave == 0 && lq == 0 && li < kOut) g[ob4 + li] = gb4[0];
    s_loss[threadIdx.x] = lsum;
    __syncthreads();
    if (threadIdx.x == 0) {
        float s = 0.0f;
        for (int t = 0; t < kBlock; ++t) s += s_loss[t];
        ploss[blockIdx.x] = s * inv_count;
    }
}

// packed places of parameter p (k_pack's layouts)
__device__ inline void pack_param(int p, float v, uint16_t* __restrict__ pk) {
    const uint16_t h = f2bf(v);
    auto both = [&](int at, int cols, int t, int w) {  // W [rows][cols] -> W^T and W
        const int k = (p - at) / cols, j = (p - at) % cols;
        const int in = at == oW1 ? kIn : kHid;
        pk[t + j * in + k] = h;
        pk[w + (p - at)] = h;
    };
    if (p < ob1)
        both(oW1, kHid, pWt1, pW1);
    else if (p >= oW2 && p < ob2)
        both(oW2, kHid, pWt2, pW2);
    else if (p >= oW3 && p < ob3)
        both(oW3, kHid, pWt3, pW3);
    else if (p >= oW4 && p < ob4) {
        const int k = (p - oW4) / kOut, j = (p - oW4) % kOut;
        pk[pWt4 + j * kHid + k] = h;
        pk[pW4 + k * kOutP + j] = h;
    }
}

struct AdamStep {
    float *prm, *m, *v;  // prm null: only the gradient
    uint16_t* pk;
    float lr, b1, b2, eps, c1, c2;
};

__device__ inline float adam_update(const AdamStep& A, int p, float gp) {
    const float mp = A.b1 * A.m[p] + (1.0f - A.b1) * gp;
    const float vp = A.b2 * A.v[p] + (1.0f - A.b2) * gp * gp;
    A.m[p] = mp;
    A.v[p] = vp;
    const float w = A.prm[p] - A.lr * (mp / A.c1) / (sqrtf(vp / A.c2) + A.eps);
    A.prm[p] = w;
    return w;
}

__global__ void k_adam(const float* __restrict__ grad, AdamStep A) {
    int p = blockIdx.x * blockDim.x + threadIdx.x;
    if (p < kParams) adam_update(A, p, grad[p]);
}

// Sum of the partial gradients in a fixed order -- 64 parameters a work-group, 16 waves that each add a run of
// partials (one thread per parameter walked 256 partials alone: 71 us for 41 MB, 10.9 now) -- and, in a training
// step, Adam and the packed weights of the new parameters.
constexpr int kSumWaves = 16;
__global__ __launch_bounds__(64 * kSumWaves) void k_gradient_sum(int nparts, const float* __restrict__ pgrad,
                                                                const float* __restrict__ ploss,
                                                                float* __restrict__ grad, float* __restrict__ loss,
                                                                AdamStep A) {
    __shared__ float s_sum[kSumWaves][64];
    const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63;
    const int p = blockIdx.x * 64 + lane;
    const int q0 = (int)((long)nparts * wave / kSumWaves), q1 = (int)((long)nparts * (wave + 1) / kSumWaves);
    float s = 0.0f;
    if (p < kParams) {
        const float* g = pgrad + p;
        int q = q0;
        for (; q + 8 <= q1; q += 8) {
            float a[8];
#pragma unroll
            for (int k = 0; k < 8; ++k) a[k] = g[(size_t)(q + k) * kParams];
#pragma unroll
            for (int k = 0; k < 8; ++k) s += a[k];
        }
        for (; q < q1; ++q) s += g[(size_t)q * kParams];
    }
    s_sum[wave][lane] = s;
    __syncthreads();
    if (wave == 0 && p < kParams) {
        float t = s_sum[0][lane];
#pragma unroll
        for (int w = 1; w < kSumWaves; ++w) t += s_sum[w][lane];
        grad[p] = t;
        if (A.prm) pack_param(p, adam_update(A, p, t), A.pk);
    }
    if (blockIdx.x == 0 && loss) {
        if (wave == 1) {
            float l = 0.0f;
            for (int q = lane; q < nparts; q += 64) l += ploss[q];
            for (int o = 32; o > 0; o >>= 1) l += __shfl_down(l, o, 64);
            if (lane == 0) loss[0] = l;
        }
    }
}

inline int blocks_for(long n, int bs) { return (int)((n + bs - 1) / bs); }

int compute_units() {
    int dev = 0, cus = 0;
    if (hipGetDevice(&dev) != hipSuccess ||
        hipDeviceGetAttribute(&cus, hipDeviceAttributeMultiprocessorCount, dev) != hipSuccess || cus <= 0)
        cus = 256;
    return cus;
}

int gradient_parts(int32_t n) { return std::min(blocks_for(n, kRowsWG), compute_units()); }

int32_t launch_gradient(void* stream, int32_t n, const uint16_t* feat, const float* target, const float* row_weight,
                        const uint16_t* packed, const float* params, float* partial_grad, float* partial_loss,
                        float* grad, float* loss, const AdamStep& A) {
    hipStream_t s = (hipStream_t)stream;
    const int parts = gradient_parts(n);
    hipLaunchKernelGGL(k_gradient, dim3(parts), dim3(kBlock), 0, s, n, feat, target, row_weight, packed, params,
                       partial_grad, partial_loss, 1.0f / (3.0f * (float)n));
    WS_LAUNCH_CHECK("k_gradient");
    hipLaunchKernelGGL(k_gradient_sum, dim3(blocks_for(kParams, 64)), dim3(64 * kSumWaves), 0, s, parts, partial_grad,
                       partial_loss, grad, loss, A);
    WS_LAUNCH_CHECK("k_gradient_sum");
    return 0;
}

}  // namespace

extern "C" {

const char* vbd_ws_last_error(void) { return g_err.c_str(); }

int32_t vbd_ws_sizes(int64_t* out3) {
    if (!out3) return fail(-1, "vbd_ws_sizes: null argument");
    out3[0] = kParams;
    out3[1] = kPacked;
    out3[2] = kRowsWG;
    return 0;
}

int32_t vbd_ws_features(void* stream, int32_t n, const int32_t* nbr_off, const int32_t* nbr, const float* x0,
                        const float* y, const float* corr, const float* acc, const float* mass, const float* area,
                        float dt, const float* scales, uint16_t* feat_out) {
    if (n < 0 || (n > 0 && (!nbr_off || !x0 || !y || !mass || !area || !scales || !feat_out)))
        return fail(-1, "vbd_ws_features: bad argument");
    if (n == 0) return 0;
    hipLaunchKernelGGL(k_features, dim3(blocks_for(n, kFeatBlock)), dim3(kFeatBlock), 0, (hipStream_t)stream, n,
                       nbr_off, nbr, x0, y, corr, acc, mass, area, dt, scales, feat_out);
    WS_LAUNCH_CHECK("k_features");
    return 0;
}

int32_t vbd_ws_smooth(void* stream, int32_t n, int32_t width, const int32_t* nbr_off, const int32_t* nbr,
                      const float* active, int32_t sweeps, float* v, float* tmp) {
    if (n < 0 || sweeps < 0 || width < 1 || width > kSmoothMaxWidth ||
        (n > 0 && (!nbr_off || !active || !v || (sweeps > 0 && !tmp))))
        return fail(-1, "vbd_ws_smooth: bad argument (width 1..12)");
    if (n == 0 || sweeps == 0) return 0;
    hipStream_t s = (hipStream_t)stream;
    float* src = v;
    float* dst = tmp;
    for (int k = 0; k < sweeps; ++k) {
        const dim3 grid(blocks_for(n, 256)), block(256);
        if (width == 1)
            hipLaunchKernelGGL(k_smooth<1>, grid, block, 0, s, n, width, nbr_off, nbr, active, src, dst);
        else if (width == 3)
            hipLaunchKernelGGL(k_smooth<3>, grid, block, 0, s, n, width, nbr_off, nbr, active, src, dst);
        else if (width == 6)
            hipLaunchKernelGGL(k_smooth<6>, grid, block, 0, s, n, width, nbr_off, nbr, active, src, dst);
        else
            hipLaunchKernelGGL(k_smooth<0>, grid, block, 0, s, n, width, nbr_off, nbr, active, src, dst);
        WS_LAUNCH_CHECK("k_smooth");
        float* t = src;
        src = dst;
        dst = t;
    }
    if (src != v) {
        hipError_t e = hipMemcpyAsync(v, src, sizeof(float) * (size_t)width * (size_t)n, hipMemcpyDeviceToDevice, s);
        if (e != hipSuccess) return fail(-2, std::string("vbd_ws_smooth: ") + hipGetErrorString(e));
    }
    return 0;
}

int32_t vbd_ws_pack(void* stream, const float* params, uint16_t* packed) {
    if (!params || !packed) return fail(-1, "vbd_ws_pack: null argument");
    hipLaunchKernelGGL(k_pack, dim3(blocks_for(kPacked, 256)), dim3(256), 0, (hipStream_t)stream, params, packed);
    WS_LAUNCH_CHECK("k_pack");
    return 0;
}

int32_t vbd_ws_forward(void* stream, int32_t n, const uint16_t* feat, const uint16_t* packed, const float* params,
                       float* out) {
    if (n < 0 || (n > 0 && (!feat || !packed || !params || !out))) return fail(-1, "vbd_ws_forward: bad argument");
    if (n == 0) return 0;
    const int cus = compute_units();
    // One work-group per CU (its weights fill half the LDS), with as few waves as give every group of 16 rows its
    // own: a short call pays for loading the weights and one chain of layers (16,384 rows: 4 waves 9.2 us, 8 waves
    // 9.7, 16 waves 12.3).  32 rows a wave read the weights half as often but leave more of the last round idle: they
    // win from about four rounds on (16 and 32 rows a wave timed in turn: 400,000 rows 56.3 and 61.9 us, 1,048,576 rows
    // 122.8 and 118.5 us).
    hipStream_t s = (hipStream_t)stream;
    const int g16 = blocks_for(n, 16), g32 = blocks_for(n, 32);
    if (g16 <= 4 * cus)
        hipLaunchKernelGGL((k_infer<4, 1>), dim3(blocks_for(g16, 4)), dim3(256), 0, s, n, feat, packed, params, out);
    else if (g16 <= 8 * cus)
        hipLaunchKernelGGL((k_infer<8, 1>), dim3(blocks_for(g16, 8)), dim3(512), 0, s, n, feat, packed, params, out);
    else if (g32 < 4 * 16 * cus)
        hipLaunchKernelGGL((k_infer<16, 1>), dim3(std::min(blocks_for(g16, 16), cus)), dim3(1024), 0, s, n, feat,
                           packed, params, out);
    else
        hipLaunchKernelGGL((k_infer<16, 2>), dim3(cus), dim3(1024), 0, s, n, feat, packed, params, out);
    WS_LAUNCH_CHECK("k_infer");
    return 0;
}

int32_t vbd_ws_forward_train(void* stream, int32_t n, const uint16_t* feat, const uint16_t* packed,
                             const float* params, float* out, uint16_t* h_save, float* z_save) {
    if (n < 0 || (n > 0 && (!feat || !packed || !params || !out || !h_save || !z_save)))
        return fail(-1, "vbd_ws_forward_train: bad argument");
    if (n == 0) return 0;
    hipLaunchKernelGGL(k_forward, dim3(blocks_for(n, kRowsWG)), dim3(kBlock), 0, (hipStream_t)stream, n, feat, packed,
                       params, out, h_save, z_save);
    WS_LAUNCH_CHECK("k_forward(train)");
    return 0;
}

int32_t vbd_ws_backward(void* stream, int32_t n, const uint16_t* feat, const float* target, const float* row_weight,
                        const uint16_t* packed, const float* out, const uint16_t* h_save, const float* z_save,
                        float* partial_grad, float* partial_loss) {
    if (n <= 0 || !feat || !target || !packed || !out || !h_save || !z_save || !partial_grad || !partial_loss)
        return fail(-1, "vbd_ws_backward: bad argument");
    float inv_count = 1.0f / (3.0f * (float)n);
    hipLaunchKernelGGL(k_backward, dim3(blocks_for(n, kRowsWG)), dim3(kBlock), 0, (hipStream_t)stream, n, feat, target,
                       row_weight, packed, out, h_save, z_save, partial_grad, partial_loss, inv_count);
    WS_LAUNCH_CHECK("k_backward");
    return 0;
}

int32_t vbd_ws_reduce(void* stream, int32_t n, const float* partial_grad, const float* partial_loss, float* grad,
                      float* loss) {
    if (n <= 0 || !partial_grad || !partial_loss || !grad) return fail(-1, "vbd_ws_reduce: bad argument");
    hipLaunchKernelGGL(k_reduce, dim3(blocks_for(kParams, 256)), dim3(256), 0, (hipStream_t)stream,
                       blocks_for(n, kRowsWG), partial_grad, partial_loss, grad, loss);
    WS_LAUNCH_CHECK("k_reduce");
    return 0;
}

int32_t vbd_ws_gradient_parts(int32_t n) { return n > 0 ? gradient_parts(n) : 0; }

int32_t vbd_ws_gradient(void* stream, int32_t n, const uint16_t* feat, const float* target, const float* row_weight,
                        const uint16_t* packed, const float* params, float* partial_grad, float* partial_loss,
                        float* grad, float* loss) {
    if (n <= 0 || !feat || !target || !packed || !params || !partial_grad || !partial_loss || !grad)
        return fail(-1, "vbd_ws_gradient: bad argument");
    return launch_gradient(stream, n, feat, target, row_weight, packed, params, partial_grad, partial_loss, grad, loss,
                           AdamStep{});
}

int32_t vbd_ws_train_step(void* stream, int32_t n, const uint16_t* feat, const float* target, const float* row_weight,
                          uint16_t* packed, float* params, float* partial_grad, float* partial_loss, float* grad,
                          float* loss, float* m, float* v, float lr, float beta1, float beta2, float eps,
                          int32_t step) {
    if (n <= 0 || !feat || !target || !packed || !params || !partial_grad || !partial_loss || !grad || !m || !v ||
        step < 1)
        return fail(-1, "vbd_ws_train_step: bad argument");
    const float c1 = 1.0f - powf(beta1, (float)step), c2 = 1.0f - powf(beta2, (float)step);
    return launch_gradient(stream, n, feat, target, row_weight, packed, params, partial_grad, partial_loss, grad, loss,
                           AdamStep{params, m, v, packed, lr, beta1, beta2, eps, c1, c2});
}

int32_t vbd_ws_adam(void* stream, float* params, const float* grad, float* m, float* v, float lr, float beta1,
                    float beta2, float eps, int32_t step) {
    if (!params || !grad || !m || !v || step < 1) return fail(-1, "vbd_ws_adam: bad argument");
    float c1 = 1.0f - powf(beta1, (float)step), c2 = 1.0f - powf(beta2, (float)step);
    const AdamStep A{params, m, v, nullptr, lr, beta1, beta2, eps, c1, c2};
    hipLaunchKernelGGL(k_adam, dim3(blocks_for(kParams, 256)), dim3(256), 0, (hipStream_t)stream, grad, A);
    WS_LAUNCH_CHECK("k_adam");
    return 0;
}

}  // extern "C"
