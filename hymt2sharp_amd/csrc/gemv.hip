// gemv.hip -- y (+)= W x for the reference's quantized weight formats, one
// token (decode): the weight GEMVs of a decode step (HunyuanDenseModel.Decode.cs
// DecodeQkv / DecodeLinear / DecodeGateUp; Vulkan dec_gemvadd_*.comp).
//
// Weights sit in HBM in the device layout of hymt_weight_upload (weights.cpp):
// every format is cut into 32-value units whose bytes are 8- or 16-byte
// aligned, so a lane reads its units with plain vector loads.  HBM-bound: a
// decode GEMV moves 1-15 MB, so the kernel is as much about memory latency as
// bandwidth: a lane issues the loads of all its units before it touches x.
//
// Work split of every type but Q4_K, Q6_K and Q8_0, which run on the matrix cores
// (gemv_kq_kernel): 256 threads (4 waves).  A row takes a group of LPR lanes (8..64,
// a power of two); lane j of the group handles units j + LPR k (k < K =
// UPR / LPR, UPR = cols / 32 units per row), so neighbouring lanes read
// neighbouring bytes and a row costs one reduction over its group (DPP).  x
// is staged in LDS with the sums of its 8-value runs (the formats' offset
// and min terms need sums of x, not per-value products).
#include <hip/hip_runtime.h>

#include <cstdint>
#include <type_traits>

#include "ktimer.hpp"
#include "weights.hpp"

namespace hymt {
namespace {


// Sum over aligned groups of `lanes` lanes (8, 16, 32 or 64); every lane of
// a group receives it.  DPP within a row of 16 (quad_perm xor 1, xor 2,
// half-row mirror, row mirror), lane shuffles across rows.
__device__ __forceinline__ float group_sum(float v, int lanes) {
    v += __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(v), 0xB1, 0xF, 0xF, false));
    v += __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(v), 0x4E, 0xF, 0xF, false));
    v += __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(v), 0x141, 0xF, 0xF, false));
    if (lanes >= 16) v += __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(v), 0x140, 0xF, 0xF, false));
    if (lanes >= 32) v += __shfl_xor(v, 16, 64);
    if (lanes >= 64) v += __shfl_xor(v, 32, 64);
    return v;
}

__device__ __forceinline__ float h2f(uint32_t h) { return (float)__builtin_bit_cast(_Float16, (uint16_t)h); }

// bytes 0..3 of w as floats (v_cvt_f32_ubyte0..3)
__device__ __forceinline__ void bytes4(uint32_t w, float *o) {
    o[0] = (float)(w & 0xFFu);
    o[1] = (float)((w >> 8) & 0xFFu);
    o[2] = (float)((w >> 16) & 0xFFu);
    o[3] = (float)(w >> 24);
}

// x is staged in LDS with 4 floats of padding after every 64, so that the
// 16-byte reads of the lanes of a wave (every row of the wave reads the same
// 8 or 16 addresses, 64 floats apart) fall in different banks
__device__ __forceinline__ int xpad(int f) { return f + ((f >> 6) << 2); }

__device__ __forceinline__ float dot4(const float *a, float4 b, float acc) {
    acc = fmaf(a[0], b.x, acc);
    acc = fmaf(a[1], b.y, acc);
    acc = fmaf(a[2], b.z, acc);
    return fmaf(a[3], b.w, acc);
}

// ---- per-format units: load() issues the loads of unit u of row r, dot()
// returns its contribution given x (LDS) and the 8-value sums xs (LDS) ----

struct UnitF32 {
    static constexpr int kMax = 4;  // units in flight per lane
    uint4 v[8];
    __device__ void load(const WeightDev &w, int r, int u) {
        const uint4 *p = (const uint4 *)((const float *)w.q + (size_t)r * w.cols + 32 * u);
#pragma unroll
        for (int i = 0; i < 8; i++) v[i] = p[i];
    }
    __device__ float dot(const WeightDev &, int, int u, const float *x, const float *) const {
        const float4 *xv = (const float4 *)(x + xpad(32 * u));
        float a = 0.f;
#pragma unroll
        for (int i = 0; i < 8; i++) {
            const float wv[4] = {__uint_as_float(v[i].x), __uint_as_float(v[i].y), __uint_as_float(v[i].z),
                                 __uint_as_float(v[i].w)};
            a = dot4(wv, xv[i], a);
        }
        return a;
    }
    __device__ void store(int u, float dsc, float *o) const {
#pragma unroll
        for (int i = 0; i < 8; i++)
            *(float4 *)(o + 32 * u + 4 * i) = make_float4(__uint_as_float(v[i].x), __uint_as_float(v[i].y),
                                                          __uint_as_float(v[i].z), __uint_as_float(v[i].w));
    }
};

struct UnitF16 {
    static constexpr int kMax = 4;  // units in flight per lane
    uint4 v[4];
    __device__ void load(const WeightDev &w, int r, int u) {
        const uint4 *p = (const uint4 *)((const uint16_t *)w.q + (size_t)r * w.cols + 32 * u);
#pragma unroll
        for (int i = 0; i < 4; i++) v[i] = p[i];
    }
    __device__ float dot(const WeightDev &, int, int u, const float *x, const float *) const {
        const float4 *xv = (const float4 *)(x + xpad(32 * u));
        float a = 0.f;
#pragma unroll
        for (int i = 0; i < 4; i++) {
            const uint32_t h[4] = {v[i].x, v[i].y, v[i].z, v[i].w};
            const float w0[4] = {h2f(h[0] & 0xFFFF), h2f(h[0] >> 16), h2f(h[1] & 0xFFFF), h2f(h[1] >> 16)};
            const float w1[4] = {h2f(h[2] & 0xFFFF), h2f(h[2] >> 16), h2f(h[3] & 0xFFFF), h2f(h[3] >> 16)};
            a = dot4(w0, xv[2 * i], a);
            a = dot4(w1, xv[2 * i + 1], a);
        }
        return a;
    }
    __device__ void store(int u, float, float *o) const {
#pragma unroll
        for (int i = 0; i < 4; i++) {
            const uint32_t h[4] = {v[i].x, v[i].y, v[i].z, v[i].w};
#pragma unroll
            for (int e = 0; e < 4; e++) {
                o[32 * u + 8 * i + 2 * e] = h2f(h[e] & 0xFFFF);
                o[32 * u + 8 * i + 2 * e + 1] = h2f(h[e] >> 16);
            }
        }
    }
};

// Q8_0 (Q8_0.cs:16-35) in the tiles of weights.hpp, dequantized.  Unit u is
// block u%8 of 256 columns: g = (u%8)/2, its 16-value halves m = 2 (u%2) and the
// next.
struct UnitQ8_0 {
    uint4 v[2];
    float d;
    __device__ void load(const WeightDev &w, int r, int u) {
        const int sub = u & 7, lane = (sub >> 1) * 16 + (r & 15);
        const uint8_t *b = (const uint8_t *)w.q + ((size_t)(r >> 4) * (w.cols / 256) + (u >> 3)) * kQ8Tile;
        v[0] = *(const uint4 *)(b + 2048 * (sub & 1) + 16 * lane);
        v[1] = *(const uint4 *)(b + 2048 * (sub & 1) + 1024 + 16 * lane);
        d = h2f(*(const uint16_t *)(b + kQ8D + 16 * (r & 15) + 2 * sub));
    }
    __device__ void store(int u, float, float *o) const {
        const uint32_t wd[8] = {v[0].x, v[0].y, v[0].z, v[0].w, v[1].x, v[1].y, v[1].z, v[1].w};
#pragma unroll
        for (int i = 0; i < 8; i++)
#pragma unroll
            for (int e = 0; e < 4; e++) o[32 * u + 4 * i + e] = d * (float)(int8_t)(wd[i] >> (8 * e));
    }
};

// Q4_K (Q4K.cs:8-19, 36-61) in the tiles of weights.hpp, dequantized (the
// embedding and the dense copies; the GEMV is gemv_kq_kernel).  Unit u is
// super-block u/8, sub = u%8 -> g = sub/2, h = sub%2: qs bytes
// 32 g + 16 h + [0,16), their low nibbles at 64 g + 16 h + i (sub-block 2 g),
// high nibbles at 64 g + 32 + 16 h + i (sub-block 2 g + 1).
struct UnitQ4_K {
    uint4 qs;
    uint32_t sm, dd;
    __device__ void load(const WeightDev &w, int r, int u) {
        const int sub = u & 7, lane = (sub >> 1) * 16 + (r & 15);
        const uint8_t *b = (const uint8_t *)w.q + ((size_t)(r >> 4) * (w.cols / 256) + (u >> 3)) * kQ4Tile;
        qs = *(const uint4 *)(b + 1024 * (sub & 1) + 16 * lane);
        sm = *(const uint32_t *)(b + kQ4Scales + 16 * (r & 15) + 4 * (sub >> 1));
        dd = *(const uint32_t *)(b + kQ4D + 4 * (r & 15));
    }
    __device__ void store(int u, float, float *o) const {
        const int g = (u & 7) >> 1, h = (u & 1);
        const int base = 256 * (u >> 3) + 64 * g + 16 * h;
        const float d = h2f(dd & 0xFFFF), dmin = h2f(dd >> 16);
        const float d1 = d * (int)(sm & 0xFF), d2 = d * (int)((sm >> 8) & 0xFF);
        const float m1 = dmin * (int)((sm >> 16) & 0xFF), m2 = dmin * (int)(sm >> 24);
        const uint32_t wd[4] = {qs.x, qs.y, qs.z, qs.w};
#pragma unroll
        for (int i = 0; i < 4; i++) {
            float lo[4], hi[4];
            bytes4(wd[i] & 0x0F0F0F0Fu, lo);
            bytes4((wd[i] >> 4) & 0x0F0F0F0Fu, hi);
#pragma unroll
            for (int e = 0; e < 4; e++) {
                o[base + 4 * i + e] = d1 * lo[e] - m1;
                o[base + 32 + 4 * i + e] = d2 * hi[e] - m2;
            }
        }
    }
};

// Q6_K (Q6K.cs:37-66) in the tiles of weights.hpp, dequantized.  Unit u is
// super-block u/8, sub = u%8 -> g = sub/2: its sub-blocks of 16 values 4 g + m,
// m = 2 (sub%2) (low nibbles) and the next (high nibbles).
struct UnitQ6_K {
    uint4 q, hi;
    uint32_t sc;
    float d;
    __device__ void load(const WeightDev &w, int r, int u) {
        const int sub = u & 7, lane = (sub >> 1) * 16 + (r & 15);
        const uint8_t *b = (const uint8_t *)w.q + ((size_t)(r >> 4) * (w.cols / 256) + (u >> 3)) * kQ6Tile;
        q = *(const uint4 *)(b + 1024 * (sub & 1) + 16 * lane);
        hi = *(const uint4 *)(b + kQ6Hi + 16 * lane);
        sc = *(const uint32_t *)(b + kQ6Scales + 16 * (r & 15) + 4 * (sub >> 1));
        d = h2f(*(const uint16_t *)(b + kQ6D + 2 * (r & 15)));
    }
    __device__ void store(int u, float, float *o) const {
        const int s16 = 16 * (u & 1);  // bits of sc, 4 (u & 1) bits of the high ones
        const float d0 = d * (float)(int8_t)(sc >> s16), d1 = d * (float)(int8_t)(sc >> (s16 + 8));
        const uint32_t lo[4] = {q.x, q.y, q.z, q.w}, h[4] = {hi.x, hi.y, hi.z, hi.w};
#pragma unroll
        for (int i = 0; i < 4; i++) {
            const uint32_t t = h[i] << (4 * (u & 1));
            const uint32_t c0 = (t & 0xC0C0C0C0u) | ((lo[i] << 2) & 0x3C3C3C3Cu);
            const uint32_t c1 = ((t << 2) & 0xC0C0C0C0u) | ((lo[i] >> 2) & 0x3C3C3C3Cu);
#pragma unroll
            for (int e = 0; e < 4; e++) {
                o[32 * u + 4 * i + e] = d0 * (float)((int8_t)(c0 >> (8 * e)) >> 2);
                o[32 * u + 16 + 4 * i + e] = d1 * (float)((int8_t)(c1 >> (8 * e)) >> 2);
            }
        }
    }
};

// Q2_0C (Q2_0C.cs:13-26): codes [rows][cols/4] bytes, d fp32 [rows][cols/512];
// unit u = 8 bytes = values 32 u + [0, 32), value (2 c - 3) d.
struct UnitQ2_0C {
    static constexpr int kMax = 8;  // units in flight per lane
    uint2 q;
    float d;
    __device__ void load(const WeightDev &w, int r, int u) {
        q = *(const uint2 *)((const uint8_t *)w.q + (size_t)r * (w.cols / 4) + 8 * u);
        d = w.d[(size_t)r * (w.cols / 512) + u / 16];
    }
    __device__ float dot(const WeightDev &, int, int u, const float *x, const float *xs) const {
        const float4 *xv = (const float4 *)(x + xpad(32 * u));
        float a = 0.f;
#pragma unroll
        for (int i = 0; i < 2; i++) {
            const uint32_t wd = i ? q.y : q.x;  // 16 codes: byte b holds values 4b + [0,4)
#pragma unroll
            for (int s = 0; s < 4; s++) {
                // value 4 b + s of byte b is bits 2 s of byte b
                float f[4];
                bytes4((wd >> (2 * s)) & 0x03030303u, f);  // codes (4b + s) for b = 0..3
                const float4 x0 = xv[4 * i], x1 = xv[4 * i + 1], x2 = xv[4 * i + 2], x3 = xv[4 * i + 3];
                const float xsel[4] = {(&x0.x)[s], (&x1.x)[s], (&x2.x)[s], (&x3.x)[s]};
                a = fmaf(f[0], xsel[0], a);
                a = fmaf(f[1], xsel[1], a);
                a = fmaf(f[2], xsel[2], a);
                a = fmaf(f[3], xsel[3], a);
            }
        }
        const float sx = xs[4 * u] + xs[4 * u + 1] + xs[4 * u + 2] + xs[4 * u + 3];
        return d * (2.f * a - 3.f * sx);
    }
    __device__ void store(int u, float, float *o) const {
#pragma unroll
        for (int i = 0; i < 2; i++) {
            const uint32_t wd = i ? q.y : q.x;
#pragma unroll
            for (int b = 0; b < 4; b++)
#pragma unroll
                for (int t = 0; t < 4; t++)
                    o[32 * u + 16 * i + 4 * b + t] = (float)((int)((wd >> (8 * b + 2 * t)) & 3u) * 2 - 3) * d;
        }
    }
};

// STQ1_0 (STQ1_0.cs:57-101): slots [rows][cols/8] bytes (two per byte), signs
// [rows][cols/32] bytes, d fp32 [rows][cols/256].  Unit u: block u/8, chunk
// c = (u%8)/2, groups 16 c + 8 hg + [0, 8) (hg = u%2): 4 slot bytes, 1 sign
// byte; group gi's lanes are values 64 c + 8 hg + gi + 16 lane.
struct UnitSTQ1_0 {
    static constexpr int kMax = 8;  // units in flight per lane
    uint32_t slots;
    uint32_t signs;
    float d;
    __device__ void load(const WeightDev &w, int r, int u) {
        slots = *(const uint32_t *)((const uint8_t *)w.q + (size_t)r * (w.cols / 8) + 4 * u);
        signs = ((const uint8_t *)w.q2)[(size_t)r * (w.cols / 32) + u];
        d = w.d[(size_t)r * (w.cols / 256) + (u >> 3)];
    }
    __device__ float dot(const WeightDev &, int, int u, const float *x, const float *xs, const uint8_t *book) const {
        const int c = (u & 7) >> 1, hg = (u & 1);
        const int base = 256 * (u >> 3) + 64 * c + 8 * hg;
        uint32_t pk[8];
#pragma unroll
        for (int gi = 0; gi < 8; gi++) pk[gi] = book[(((signs >> gi) & 1) << 4) | ((slots >> (4 * gi)) & 0xF)];
        float a = 0.f;
#pragma unroll
        for (int ln = 0; ln < 4; ln++) {
            const float4 xa = *(const float4 *)(x + xpad(base + 16 * ln)), xb = *(const float4 *)(x + xpad(base + 16 * ln + 4));
            const float xv[8] = {xa.x, xa.y, xa.z, xa.w, xb.x, xb.y, xb.z, xb.w};
#pragma unroll
            for (int gi = 0; gi < 8; gi++) a = fmaf((float)((pk[gi] >> (2 * ln)) & 3), xv[gi], a);
        }
        const float sx = xs[base / 8] + xs[base / 8 + 2] + xs[base / 8 + 4] + xs[base / 8 + 6];
        return d * (a - sx);
    }
    __device__ void store(int u, const uint8_t *book, float *o) const {
        const int c = (u & 7) >> 1, hg = (u & 1);
        const int base = 256 * (u >> 3) + 64 * c + 8 * hg;
#pragma unroll
        for (int gi = 0; gi < 8; gi++) {
            const uint32_t pk = book[(((signs >> gi) & 1) << 4) | ((slots >> (4 * gi)) & 0xF)];
#pragma unroll
            for (int ln = 0; ln < 4; ln++) o[base + gi + 16 * ln] = (float)((int)((pk >> (2 * ln)) & 3u) - 1) * d;
        }
    }
};

// STQ1_0.Codebook (STQ1_0.cs:57-63)
__constant__ uint8_t kStqBook[32] = {
    0xA9, 0x89, 0x29, 0x09, 0xA6, 0x86, 0x26, 0x06, 0x9A, 0x92, 0x1A, 0x12, 0x6A, 0x62, 0x4A, 0x42,
    0x01, 0x21, 0x81, 0xA1, 0x04, 0x24, 0x84, 0xA4, 0x10, 0x18, 0x90, 0x98, 0x40, 0x48, 0x60, 0x68,
};

// K = cols / 32 / lpr units per lane and the input mode are template
// arguments: the loads then sit in straight-line code, so the wait before the
// activations' arithmetic counts only the activation loads (a run-time loop
// bound and mode made the compiler wait for every weight load there too, and
// the RMSNorm, the LDS staging and its barriers ran after the weights had
// landed: 0.7 us on the 12288 x 2048 gate/up GEMV).
// MODE is the input mode: 0 x as given, 1 RMSNorm (kGemvInRmsNorm), 2
// SwiGLU (kGemvInSwiGLU); each loads only the vectors it needs.
template <typename Unit, bool STQ, int NJ, int K, int MODE>
__global__ __launch_bounds__(256) void gemv_kernel(WeightDev w, const float *__restrict__ xg, float *__restrict__ y,
                                                   int lpr, int flags, const float *__restrict__ nw, float eps) {
    extern __shared__ __attribute__((aligned(16))) float smem[];
    float *x = smem;                        // [cols + cols / 16] (xpad)
    float *xs = smem + w.cols + w.cols / 16;  // [cols / 8]
    __shared__ uint8_t book[32];
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    // lane group gi computes row gi; with kGemvOutSwiGLU (W = [gate; up], F
    // rows each) the groups alternate gate row gi/2 and up row F + gi/2, so
    // that a row pair sits in neighbouring groups
    const int gi = (blockIdx.x * 4 + wave) * (64 / lpr) + lane / lpr;
    const bool out_swiglu = flags & kGemvOutSwiGLU;
    const int row = out_swiglu ? (gi & 1) * (w.rows >> 1) + (gi >> 1) : gi;
    const int sub = lane % lpr;
    // unit sub + lpr k, written with lpr = 8 lpr8 (lpr is 8, 16, 32 or 64) so
    // that the compiler sees u & 7 = sub & 7: the unit's place inside its
    // 256-value block (and the scale bytes it needs) is a lane constant
    const int lpr8 = lpr >> 3;

    // 1. the activations first (small, from L2: their data returns while the
    // weight loads below are still in flight), then this lane's weight loads,
    // all issued before anything waits.  Thread tid holds the 8 values
    // [8i, 8i+8) for i = tid + 256j, j < NJ = cols / 2048.
    constexpr int nj = NJ;
    constexpr bool swiglu = MODE == 2, rms = MODE == 1;
    float4 xa[NJ], xb[NJ], ua[NJ], ub[NJ], ga[NJ], gb[NJ];
#pragma unroll
    for (int j = 0; j < NJ; j++) {
        const int i = tid + 256 * j;
        xa[j] = ((const float4 *)xg)[2 * i];
        xb[j] = ((const float4 *)xg)[2 * i + 1];
        if constexpr (swiglu) {
            ua[j] = ((const float4 *)(xg + w.cols))[2 * i];
            ub[j] = ((const float4 *)(xg + w.cols))[2 * i + 1];
        }
        if constexpr (rms) {
            ga[j] = ((const float4 *)nw)[2 * i];
            gb[j] = ((const float4 *)nw)[2 * i + 1];
        }
    }
    Unit un[K];
    const int rl = gi < w.rows ? row : w.rows - 1;
#pragma unroll
    for (int k = 0; k < K; k++) un[k].load(w, rl, sub + 8 * (lpr8 * k));
    // nothing moves across: left free, the scheduler put the RMSNorm's sum
    // of squares (and with it a wait for x) before the weight loads
    __builtin_amdgcn_sched_barrier(0);
    if (STQ && tid < 32) book[tid] = kStqBook[tid];
    // 2. x as the input mode makes it, into LDS with its 8-value sums
    auto silu_mul = [](float4 g, float4 u) {
        // Ops.SiLUMulRange (Ops.cs:1016-1052): g / (1 + exp(-g)) * u
        return make_float4(g.x / (1.f + expf(-g.x)) * u.x, g.y / (1.f + expf(-g.y)) * u.y,
                           g.z / (1.f + expf(-g.z)) * u.z, g.w / (1.f + expf(-g.w)) * u.w);
    };
    if constexpr (swiglu) {
#pragma unroll
        for (int j = 0; j < NJ; j++)
            if (j < nj) {
                xa[j] = silu_mul(xa[j], ua[j]);
                xb[j] = silu_mul(xb[j], ub[j]);
            }
    }
    if constexpr (rms) {
        // x / sqrt(mean(x^2) + eps) * nw (Ops.RmsNorm, Ops.cs:12-90)
        __shared__ float red[4];
        float ss = 0.f;
#pragma unroll
        for (int j = 0; j < NJ; j++)
            if (j < nj) {
                const float4 a = xa[j], b = xb[j];
                ss += ((a.x * a.x + a.y * a.y) + (a.z * a.z + a.w * a.w)) +
                      ((b.x * b.x + b.y * b.y) + (b.z * b.z + b.w * b.w));
            }
        ss = group_sum(ss, 64);
        if (lane == 0) red[wave] = ss;
        __syncthreads();
        const float rr = 1.0f / sqrtf(((red[0] + red[1]) + (red[2] + red[3])) / (float)w.cols + eps);
#pragma unroll
        for (int j = 0; j < NJ; j++)
            if (j < nj) {
                const float4 a = xa[j], b = xb[j], g = ga[j], h = gb[j];
                xa[j] = make_float4(a.x * rr * g.x, a.y * rr * g.y, a.z * rr * g.z, a.w * rr * g.w);
                xb[j] = make_float4(b.x * rr * h.x, b.y * rr * h.y, b.z * rr * h.z, b.w * rr * h.w);
            }
    }
#pragma unroll
    for (int j = 0; j < NJ; j++)
        if (j < nj) {
            const int i = tid + 256 * j;
            const float4 a = xa[j], b = xb[j];
            float4 *xd = (float4 *)(x + xpad(8 * i));
            xd[0] = a;
            xd[1] = b;
            xs[i] = ((a.x + a.y) + (a.z + a.w)) + ((b.x + b.y) + (b.z + b.w));
        }
    __syncthreads();
    // 3. dot products, then the row's sum over its lane group
    float part = 0.f;
#pragma unroll
    for (int k = 0; k < K; k++) {
        if constexpr (STQ) part += un[k].dot(w, 0, sub + 8 * (lpr8 * k), x, xs, book);
        else part += un[k].dot(w, 0, sub + 8 * (lpr8 * k), x, xs);
    }
    const float s = group_sum(part, lpr);
    if (out_swiglu) {
        // y[gi/2] = silu(gate) * up (Ops.SiLUMul, Ops.cs:1016-1052; the
        // reference's fused decode gate/up, dec_ffngu.comp:9-11, 292-301): the
        // up sum comes from the neighbouring group, in this wave for lpr < 64,
        // else from the neighbouring wave through LDS
        float u;
        if (lpr < 64) {
            u = __shfl_xor(s, lpr, 64);
        } else {
            __shared__ float pair[4];
            if (lane == 0) pair[wave] = s;
            __syncthreads();
            u = pair[wave ^ 1];
        }
        if (sub == 0 && !(gi & 1) && gi < w.rows) y[gi >> 1] = s / (1.f + expf(-s)) * u;
        return;
    }
    if (sub == 0 && gi < w.rows) y[row] = (flags & kGemvAccumulate) ? y[row] + s : s;
}

// One row of the matrix, dequantized (the embedding lookup,
// HunyuanDenseModel.Embed, HunyuanDenseModel.cs:494-557): a workgroup of 256
// threads, one unit per thread and pass.
template <typename Unit, bool STQ>
__global__ __launch_bounds__(256) void embed_kernel(WeightDev w, int row, float *__restrict__ out) {
    __shared__ uint8_t book[32];
    if (STQ && threadIdx.x < 32) book[threadIdx.x] = kStqBook[threadIdx.x];
    __syncthreads();
    for (int u = threadIdx.x; u < w.cols / 32; u += 256) {
        Unit un;
        un.load(w, row, u);
        if constexpr (STQ) un.store(u, book, out);
        else un.store(u, 0.f, out);
    }
}

// ---- Q4_K, Q6_K and Q8_0 on the matrix cores --------------------------------------
// y = W x' for Q4_K, in integers.  The VALU form of the other types spends a
// convert and an fma per weight, the scales' bit fields, and x and its sums
// staged by every workgroup behind two barriers: on 120818 x 2048 rows 74 us
// where the bytes take 25.  Here a super-block's 256 products run on
// v_mfma_i32_16x16x64_i8, exactly:
//  - the codes enter as they are, bytes of 0..15 (one mask per four weights);
//  - x' enters as a 61-bit fixed-point number, x' s = h + l 2^-30, h and l in
//    four signed bytes each, sum_p d_p 256^p; s is the power of two that brings
//    the super-block's largest |x'| to [2^29, 2^30).  That holds every fp32
//    value down to 2^-36 of the largest exactly.  A super-block with smaller
//    ones (but 0), one of 2^74, an infinity or NaN takes fp32 products instead
//    (plain_dot), which take several times as long.
//    h alone lost what lay 2^-30 below the largest: beside a value 3000 times
//    the others, at weight 0, the error was 2.1e-6 (under 1e-7 with l); l costs
//    a second set of products, 1-4 % of eight layers' GEMVs;
//  - the A operand's 16 rows are (digit p, sub-block pair g): row 4 p + g holds
//    digit p of h (or l) in the k range of lane group g and zeros elsewhere, its 16
//    columns are weight rows.  So a lane (p, c) receives digit p's sums of row
//    c over the four low-code sub-blocks 2 g and, from the other two MFMAs, the
//    high-code ones 2 g + 1, and weighs them by the 6-bit scales in integers
//    (below 2^25 together).
// The minima take sums of x' per sub-block, in fp64, and a wave's products and
// minima are summed in fp64, because they cancel: with weights spread about 0 and
// x of one sign each is some 30 times what is left, and the error of a sum of x is
// the same in every row.  In fp32 that left 9e-7 to 13e-7 of y (the VALU form, which
// cancels them per 32 columns, 5e-7 to 6e-7); fp64 costs 3-4 % of a call.  rms error
// against 64 bits over 2048 rows, in 1e-7 of the rms of y, here and in the VALU
// form, for two kinds of weights and 2048 to 8192 columns: normal x 0.5-0.7
// (1.0-2.6), one value per super-block 100 to 30000 times the others 0.5-0.7
// (1.1-2.5), log-normal magnitudes with sigma 3 0.5-0.6 (0.9-1.9), all x positive
// 0.4-0.6 (0.4-5.8).
//
// Q6_K the same way: the codes enter as signed bytes 4 (q - 32) (the high two
// bits stored with 32's flipped, so that two masks and an or make four), each
// MFMA's lane groups hold one 16-value sub-block each, so a lane (p, c) receives
// digit p's sums of row c over four of them and weighs them by their signed
// scales (below 2^29 together).  There are no minima, and fp32 sums do.  rms
// error as above: normal x 0.6-0.7 (1.5-2.0), outliers 0.6-0.7 (1.1-1.9), log-normal
// 0.6-0.7 (1.3-1.9), all positive 0.5-0.7 (1.1-2.6).
//
// Q8_0's codes are the B operand's bytes as they are; a lane (p, c) receives the
// sums over blocks 2 g and 2 g + 1 as with Q4_K, below 2^20 and so exact in
// fp32, where the blocks' fp16 scales meet them.  rms error: normal x 0.8-0.9
// (1.3), outliers 0.6-0.8 (1.4-1.5), log-normal 0.6-0.7 (0.8-1.4), all positive 0.8
// (1.1-1.3).
//
// Work split: a workgroup of NW waves takes RT tiles of 16 rows; wave v takes
// super-blocks [v NSB, (v + 1) NSB) of all of them, whose x' it prepares for
// itself in LDS, so nothing waits for another wave until the partial sums of a
// row meet at the end (where the RMSNorm's factor, a scalar of x, is applied
// too).  Every load is issued before the first use.
typedef int i32x4 __attribute__((ext_vector_type(4)));

template <int CTRL> __device__ __forceinline__ float dpp(float v) {
    return __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(v), CTRL, 0xF, 0xF, false));
}
template <int CTRL> __device__ __forceinline__ uint32_t dpp(uint32_t v) {
    return (uint32_t)__builtin_amdgcn_update_dpp(0, (int)v, CTRL, 0xF, 0xF, false);
}
// over the 4 rows of 16 lanes, every lane receiving the result
__device__ __forceinline__ float rows_sum(float v) {
    auto a = __builtin_amdgcn_permlane16_swap(__float_as_uint(v), __float_as_uint(v), false, false);
    v = __uint_as_float(a[0]) + __uint_as_float(a[1]);
    auto b = __builtin_amdgcn_permlane32_swap(__float_as_uint(v), __float_as_uint(v), false, false);
    return __uint_as_float(b[0]) + __uint_as_float(b[1]);
}
template <int CTRL> __device__ __forceinline__ double dpp(double v) {
    return __hiloint2double((int)dpp<CTRL>((uint32_t)__double2hiint(v)), (int)dpp<CTRL>((uint32_t)__double2loint(v)));
}
__device__ __forceinline__ double rows_sum(double v) {
    auto h = __builtin_amdgcn_permlane16_swap(__double2hiint(v), __double2hiint(v), false, false);
    auto l = __builtin_amdgcn_permlane16_swap(__double2loint(v), __double2loint(v), false, false);
    v = __hiloint2double(h[0], l[0]) + __hiloint2double(h[1], l[1]);
    h = __builtin_amdgcn_permlane32_swap(__double2hiint(v), __double2hiint(v), false, false);
    l = __builtin_amdgcn_permlane32_swap(__double2loint(v), __double2loint(v), false, false);
    return __hiloint2double(h[0], l[0]) + __hiloint2double(h[1], l[1]);
}
__device__ __forceinline__ uint32_t rows_max(uint32_t v) {
    auto a = __builtin_amdgcn_permlane16_swap(v, v, false, false);
    v = max((uint32_t)a[0], (uint32_t)a[1]);
    auto b = __builtin_amdgcn_permlane32_swap(v, v, false, false);
    return max((uint32_t)b[0], (uint32_t)b[1]);
}
// Keeps a wave's LDS accesses in program order (the LDS unit serves them so).
__device__ __forceinline__ void wave_order() {
    asm volatile("" ::: "memory");
    __builtin_amdgcn_wave_barrier();
}

// Columns 64 grp + [0, 64) of a tile's row r times x, in fp32, a code and a
// value at a time as the VALU form has them: the way of super-blocks whose x'
// has no digits.  16 columns at a time, so that the rare path takes no more
// registers than the kernel around it.
template <int T> __device__ __forceinline__ float plain_dot(const uint8_t *tile, int r, int grp, const float *x) {
    const int at = 16 * (16 * grp + r);
    float y = 0.f;
#pragma unroll 1
    for (int m = 0; m < 4; m++) {  // columns 16 m + [0, 16)
        const uint4 c4 = *(const uint4 *)(tile + 1024 * (T == kW_Q8_0 ? m : T == kW_Q6_K ? m >> 1 : m & 1) + at);
        const uint32_t c[4] = {c4.x, c4.y, c4.z, c4.w};
        uint4 h4 = make_uint4(0, 0, 0, 0);
        if constexpr (T == kW_Q6_K) h4 = *(const uint4 *)(tile + kQ6Hi + at);
        const uint32_t h[4] = {h4.x, h4.y, h4.z, h4.w};
        float a = 0.f, sx = 0.f;
#pragma unroll
        for (int j = 0; j < 4; j++) {
            const float4 xv = *(const float4 *)(x + 16 * m + 4 * j);
            const float v[4] = {xv.x, xv.y, xv.z, xv.w};
#pragma unroll
            for (int e = 0; e < 4; e++) {
                if constexpr (T == kW_Q8_0) {
                    a = fmaf((float)(int8_t)(c[j] >> (8 * e)), v[e], a);
                } else if constexpr (T == kW_Q6_K) {  // the stored upper bit is flipped
                    const uint32_t lo = c[j] >> (4 * (m & 1)), hb = h[j] >> (6 - 2 * m);
                    a = fmaf((float)((int)(((lo >> (8 * e)) & 0xFu) | ((((hb >> (8 * e)) & 3u) ^ 2u) << 4)) - 32), v[e], a);
                } else {
                    a = fmaf((float)((c[j] >> (8 * e + 4 * (m >> 1))) & 0xFu), v[e], a);
                }
                sx += v[e];
            }
        }
        if constexpr (T == kW_Q8_0) {
            y += h2f(*(const uint16_t *)(tile + kQ8D + 16 * r + 4 * grp + 2 * (m >> 1))) * a;
        } else if constexpr (T == kW_Q6_K) {
            // with the offset taken off afterwards (code v less 32 v) an
            // infinity of x' is NaN whatever the code: 0 sx keeps that
            y += (float)*(const int8_t *)(tile + kQ6Scales + 16 * r + 4 * grp + m) * fmaf(0.f, sx, a);
        } else {  // low codes, then high ones: sub-blocks 2 grp and 2 grp + 1
            const uint8_t *sm = tile + kQ4Scales + 16 * r + 4 * grp + (m >> 1);
            const uint32_t dd = *(const uint32_t *)(tile + kQ4D + 4 * r);
            y += h2f(dd & 0xFFFF) * ((float)sm[0] * a) - h2f(dd >> 16) * ((float)sm[2] * sx);
        }
    }
    return T == kW_Q6_K ? y * h2f(*(const uint16_t *)(tile + kQ6D + 2 * r)) : y;
}

template <int T, int RT, int NW, int NSB, int MODE, bool MANY>
__global__ __launch_bounds__(64 * NW, T != kW_Q8_0 && MANY && RT == 2 && NSB == 1 ? 6 : 1) void gemv_kq_kernel(WeightDev w, const float *__restrict__ xg,
                                                          float *__restrict__ y, int flags,
                                                          const float *__restrict__ nw, float eps) {
    constexpr bool Q6 = T == kW_Q6_K, Q8 = T == kW_Q8_0, kLean = RT == 2 && !Q8 && (MANY || NW * NSB > 8);
    constexpr int kTile = Q8 ? kQ8Tile : Q6 ? kQ6Tile : kQ4Tile;
    // a wave's super-blocks as digits, [first, second][group][digit][64
    // columns], or as they are (the bits of `plain`), and zeros
    __shared__ __attribute__((aligned(16))) uint8_t s_x[NW][NSB][2][1024];
    __shared__ __attribute__((aligned(16))) uint8_t s_zero[NW][64];
    __shared__ float s_p[NW][RT][16];
    __shared__ float s_ss[NW];
    const int tid = threadIdx.x, lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int grp = lane >> 4, c = lane & 15;
    const bool out_swiglu = flags & kGemvOutSwiGLU;
    const int F = w.rows >> 1, nsb = NW * NSB, sb0 = wave * NSB;

    // the lane's columns of super-block s: 4 lane + [0, 4)
    float4 xv[NSB], gv[NSB];
#pragma unroll
    for (int s = 0; s < NSB; s++) {
        xv[s] = ((const float4 *)xg)[(sb0 + s) * 64 + lane];
        if constexpr (MODE == 1) gv[s] = ((const float4 *)nw)[(sb0 + s) * 64 + lane];
        if constexpr (MODE == 2) gv[s] = ((const float4 *)(xg + w.cols))[(sb0 + s) * 64 + lane];
    }
    // tile i's row of this lane; with SwiGLU the tiles alternate between gate
    // rows and the same rows of up, or (RT = 1) a tile is 8 of each
    uint4 q0[RT][NSB], q1[RT][NSB], q2[RT][NSB], q3[RT][NSB], sm[RT][NSB];
    uint32_t dd[RT][NSB];
    auto row_of = [&](int i) {
        return min(out_swiglu && RT == 1 ? (c >> 3) * F + 8 * (int)blockIdx.x + (c & 7)
                   : out_swiglu          ? (i & 1) * F + 16 * ((int)(blockIdx.x * RT + i) >> 1) + c
                                         : 16 * (int)(blockIdx.x * RT + i) + c,
                   w.rows - 1);
    };
#pragma unroll
    for (int i = 0; i < RT; i++) {
        const int row = row_of(i);
        const int r = row & 15, li = grp * 16 + r;
        const uint8_t *b = (const uint8_t *)w.q + ((size_t)(row >> 4) * nsb + sb0) * kTile;
#pragma unroll
        for (int s = 0; s < NSB; s++) {
            q0[i][s] = *(const uint4 *)(b + s * kTile + 16 * li);
            q1[i][s] = *(const uint4 *)(b + s * kTile + 1024 + 16 * li);
            if constexpr (Q8) {
                q2[i][s] = *(const uint4 *)(b + s * kTile + 2048 + 16 * li);
                q3[i][s] = *(const uint4 *)(b + s * kTile + 3072 + 16 * li);
                sm[i][s] = *(const uint4 *)(b + s * kTile + kQ8D + 16 * r);
            } else if constexpr (Q6) {
                q2[i][s] = *(const uint4 *)(b + s * kTile + kQ6Hi + 16 * li);
                sm[i][s] = *(const uint4 *)(b + s * kTile + kQ6Scales + 16 * r);
                dd[i][s] = *(const uint16_t *)(b + s * kTile + kQ6D + 2 * r);
            } else {
                sm[i][s] = *(const uint4 *)(b + s * kTile + kQ4Scales + 16 * r);
                dd[i][s] = *(const uint32_t *)(b + s * kTile + kQ4D + 4 * r);
            }
        }
    }
    // nothing moves across: the weight loads stay ahead of the first wait on x
    __builtin_amdgcn_sched_barrier(0);

    if (lane < 16) *(uint32_t *)(s_zero[wave] + 4 * lane) = 0;
    double S0[NSB], S1[NSB];
    float wgt[NSB], ss = 0.f;
    uint32_t plain = 0;
#pragma unroll
    for (int s = 0; s < NSB; s++) {
        float v[4] = {xv[s].x, xv[s].y, xv[s].z, xv[s].w};
        const float g[4] = {gv[s].x, gv[s].y, gv[s].z, gv[s].w};
        if constexpr (MODE == 1) {  // Ops.RmsNorm (Ops.cs:12-90); the factor comes at the end
            ss += (v[0] * v[0] + v[1] * v[1]) + (v[2] * v[2] + v[3] * v[3]);
#pragma unroll
            for (int e = 0; e < 4; e++) v[e] *= g[e];
        }
        if constexpr (MODE == 2) {  // Ops.SiLUMulRange (Ops.cs:1016-1052)
#pragma unroll
            for (int e = 0; e < 4; e++) v[e] = v[e] / (1.f + expf(-v[e])) * g[e];
        }
        if constexpr (!Q6 && !Q8) {  // sums over the sub-blocks (8 lanes) of this lane group: 2 grp, 2 grp + 1
            double a = ((double)v[0] + v[1]) + ((double)v[2] + v[3]);
            a += dpp<0xB1>(a);
            a += dpp<0x4E>(a);
            a += dpp<0x141>(a);
            const double b = dpp<0x128>(a);  // the other 8 lanes of the row
            S0[s] = (lane & 8) ? b : a;
            S1[s] = (lane & 8) ? a : b;
        }
        // largest |x'|, as bits (their order is the values', NaN above all)
        uint32_t mx = 0;
#pragma unroll
        for (int j = 0; j < 4; j++) mx = max(mx, __float_as_uint(v[j]) & 0x7FFFFFFFu);
        mx = max(mx, dpp<0xB1>(mx));
        mx = max(mx, dpp<0x4E>(mx));
        mx = max(mx, dpp<0x141>(mx));
        mx = max(mx, dpp<0x140>(mx));
        mx = __builtin_amdgcn_readfirstlane(rows_max(mx));
        // 2^k with mx 2^k in [2^29, 2^30), both it and its inverse normal
        const int e = min(max((int)(mx >> 23), 30), 254);
        const float sc = __uint_as_float((uint32_t)(283 - e) << 23);
        wgt[s] = __uint_as_float((uint32_t)(e - 29 + 8 * grp) << 23);  // of digit `grp`
        // x' 2^k = h + l 2^-30, each 30 bits and a sign; what is then left is
        // of values below 2^-36 of the largest, or an infinity or NaN
        int t[2][4];
        bool left = false;
#pragma unroll
        for (int j = 0; j < 4; j++) {
            const float u = v[j] * sc;
            t[0][j] = (int)u;
            const float r = (u - (float)t[0][j]) * 1073741824.f;
            t[1][j] = (int)r;
            left |= r != (float)t[1][j];
        }
        // no digits: plain_dot takes the super-block.  So it does where the
        // largest value is 2^74 or more, whose scale could take another to 0
        // unnoticed; below that only values under 2^-105 beside one over 2^30
        // are lost to it, which is 2^-135 of it
        if (__ballot(left) != 0 || e > 200) {
            plain |= 1u << s;
            wgt[s] = S0[s] = S1[s] = 0.f;
            *(float4 *)(s_x[wave][s][0] + 16 * lane) = make_float4(v[0], v[1], v[2], v[3]);
            continue;
        }
#pragma unroll
        for (int d = 0; d < 2; d++) {
            // four signed digits of each column: with 0x80 added to the lower
            // three bytes they are the bytes less 0x80
            uint32_t b[4];
#pragma unroll
            for (int j = 0; j < 4; j++) b[j] = ((uint32_t)t[d][j] + 0x00808080u) ^ 0x00808080u;
            // digit p of the 4 columns as one dword
            const uint32_t a0 = __builtin_amdgcn_perm(b[1], b[0], 0x05010400u), a1 = __builtin_amdgcn_perm(b[1], b[0], 0x07030602u);
            const uint32_t b0 = __builtin_amdgcn_perm(b[3], b[2], 0x05010400u), b1 = __builtin_amdgcn_perm(b[3], b[2], 0x07030602u);
            uint32_t *p = (uint32_t *)(s_x[wave][s][d] + grp * 256 + 4 * (lane & 15));
            p[0] = __builtin_amdgcn_perm(b0, a0, 0x05040100u);
            p[16] = __builtin_amdgcn_perm(b0, a0, 0x07060302u);
            p[32] = __builtin_amdgcn_perm(b1, a1, 0x05040100u);
            p[48] = __builtin_amdgcn_perm(b1, a1, 0x07060302u);
        }
    }
    wave_order();
    // Q4_K's products and minima cancel: fp64 until they have
    using Sum = std::conditional_t<Q6 || Q8, float, double>;
    Sum acc[RT] = {};
    // row c of the A operand: digit c / 4 in the columns of group c % 4
    const int zoff = (c & 3) == grp ? grp * 256 + (c >> 2) * 64 : -1;
#pragma unroll
    for (int s = 0; s < NSB; s++) {
        const i32x4 *xp[2];
#pragma unroll
        for (int d = 0; d < 2; d++) xp[d] = (const i32x4 *)(zoff < 0 ? s_zero[wave] : s_x[wave][s][d] + zoff);
        i32x4 xa[2][4];  // Q4_K: low codes' columns, high codes'
        if constexpr (!kLean) {
#pragma unroll
            for (int d = 0; d < 2; d++)
#pragma unroll
                for (int m = 0; m < 4; m++) xa[d][m] = xp[d][m];
        }
        // Two tiles (kLean): xa's pieces read again for each tile, none moved
        // ahead of the products before, instead of 32 registers held over both.
        // Where the grid is long (MANY) six waves then fit a SIMD: 120818 x 2048
        // of Q6_K 38.0 -> 35.9 us, of Q4_K 29.4 -> 28.3 (Q8_0 does not gain, 44.5 /
        // 45.3, nor a short grid, Q4_K 12288 x 2048 + SwiGLU 6.17 / 6.00); with more
        // than 8 super-blocks it saves spills.
        auto again = [&](int d, int m) {
            asm volatile("" ::: "memory");
            xa[d][m] = xp[d][m];
        };
#pragma unroll
        for (int i = 0; i < RT; i++) {
            const uint4 a = q0[i][s], b = q1[i][s];
            const uint32_t k[4] = {sm[i][s].x, sm[i][s].y, sm[i][s].z, sm[i][s].w};
            if constexpr (Q8) {
                const uint4 e = q2[i][s], f = q3[i][s];
                const i32x4 l0 = {(int)a.x, (int)a.y, (int)a.z, (int)a.w}, l1 = {(int)b.x, (int)b.y, (int)b.z, (int)b.w};
                const i32x4 h0 = {(int)e.x, (int)e.y, (int)e.z, (int)e.w}, h1 = {(int)f.x, (int)f.y, (int)f.z, (int)f.w};
                float t[2];
#pragma unroll
                for (int d = 0; d < 2; d++) {
                    i32x4 L = {0, 0, 0, 0}, H = {0, 0, 0, 0};
                    L = __builtin_amdgcn_mfma_i32_16x16x64_i8(xa[d][0], l0, L, 0, 0, 0);
                    H = __builtin_amdgcn_mfma_i32_16x16x64_i8(xa[d][2], h0, H, 0, 0, 0);
                    L = __builtin_amdgcn_mfma_i32_16x16x64_i8(xa[d][1], l1, L, 0, 0, 0);
                    H = __builtin_amdgcn_mfma_i32_16x16x64_i8(xa[d][3], h1, H, 0, 0, 0);
                    t[d] = 0.f;
#pragma unroll
                    for (int g = 0; g < 4; g++) {
                        t[d] = fmaf(h2f(k[g] & 0xFFFF), (float)L[g], t[d]);
                        t[d] = fmaf(h2f(k[g] >> 16), (float)H[g], t[d]);
                    }
                }
                acc[i] = fmaf(fmaf(t[1], 0x1p-30f, t[0]), wgt[s], acc[i]);
                continue;
            }
            if constexpr (Q6) {
                const uint32_t h[4] = {q2[i][s].x, q2[i][s].y, q2[i][s].z, q2[i][s].w};
                const uint32_t lo[2][4] = {{a.x, a.y, a.z, a.w}, {b.x, b.y, b.z, b.w}};
                int t[2] = {0, 0};
#pragma unroll
                for (int m = 0; m < 4; m++) {  // columns 64 g + 16 m + [0, 16): sub-block 4 g + m
                    if constexpr (kLean) {
                        if (m % 2 == 0) __builtin_amdgcn_sched_barrier(0);
                        again(0, m);
                        again(1, m);
                    }
                    i32x4 f;
#pragma unroll
                    for (int j = 0; j < 4; j++) {
                        const uint32_t l = m & 1 ? lo[m >> 1][j] >> 2 : lo[m >> 1][j] << 2;
                        f[j] = (int)(((h[j] << (2 * m)) & 0xC0C0C0C0u) | (l & 0x3C3C3C3Cu));
                    }
#pragma unroll
                    for (int d = 0; d < 2; d++) {
                        const i32x4 D = __builtin_amdgcn_mfma_i32_16x16x64_i8(xa[d][m], f, i32x4{0, 0, 0, 0}, 0, 0, 0);
#pragma unroll
                        for (int g = 0; g < 4; g++) t[d] += __mul24((int)(int8_t)(k[g] >> (8 * m)), D[g]);
                    }
                }
                acc[i] = fmaf(h2f(dd[i][s]), fmaf((float)t[1], 0x1p-30f, (float)t[0]) * 0.25f * wgt[s], acc[i]);
                continue;
            }
            constexpr uint32_t M = 0x0F0F0F0Fu;
            const i32x4 l0 = {(int)(a.x & M), (int)(a.y & M), (int)(a.z & M), (int)(a.w & M)};
            const i32x4 l1 = {(int)(b.x & M), (int)(b.y & M), (int)(b.z & M), (int)(b.w & M)};
            const i32x4 h0 = {(int)((a.x >> 4) & M), (int)((a.y >> 4) & M), (int)((a.z >> 4) & M), (int)((a.w >> 4) & M)};
            const i32x4 h1 = {(int)((b.x >> 4) & M), (int)((b.y >> 4) & M), (int)((b.z >> 4) & M), (int)((b.w >> 4) & M)};
            int t[2] = {0, 0};
#pragma unroll
            for (int d = 0; d < 2; d++) {
                if constexpr (kLean) {
                    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
                    for (int m = 0; m < 4; m++) again(d, m);
                }
                i32x4 L = {0, 0, 0, 0}, H = {0, 0, 0, 0};
                L = __builtin_amdgcn_mfma_i32_16x16x64_i8(xa[d][0], l0, L, 0, 0, 0);
                H = __builtin_amdgcn_mfma_i32_16x16x64_i8(xa[d][2], h0, H, 0, 0, 0);
                L = __builtin_amdgcn_mfma_i32_16x16x64_i8(xa[d][1], l1, L, 0, 0, 0);
                H = __builtin_amdgcn_mfma_i32_16x16x64_i8(xa[d][3], h1, H, 0, 0, 0);
#pragma unroll
                for (int g = 0; g < 4; g++)
                    t[d] += __mul24((int)(k[g] & 0xFFu), L[g]) + __mul24((int)((k[g] >> 8) & 0xFFu), H[g]);
            }
            const float d = h2f(dd[i][s] & 0xFFFF), dmin = h2f(dd[i][s] >> 16);
            const uint32_t kg = grp & 2 ? (grp & 1 ? k[3] : k[2]) : (grp & 1 ? k[1] : k[0]);
            const float m0 = (float)((kg >> 16) & 0xFFu), m1 = (float)(kg >> 24);
            acc[i] = fma((double)(-dmin * m0), S0[s], acc[i]);
            acc[i] = fma((double)(-dmin * m1), S1[s], acc[i]);
            acc[i] = fma((double)(d * wgt[s]), fma((double)t[1], 0x1p-30, (double)t[0]), acc[i]);
        }
    }
    if (plain) {
#pragma unroll 1
        for (uint32_t left = plain; left; left &= left - 1) {
            const int s = __builtin_ctz(left);
#pragma unroll
            for (int i = 0; i < RT; i++) {
                const int row = row_of(i);
                const uint8_t *b = (const uint8_t *)w.q + ((size_t)(row >> 4) * nsb + sb0 + s) * kTile;
                acc[i] += plain_dot<T>(b, row & 15, grp, (const float *)s_x[wave][s][0] + 64 * grp);
            }
        }
    }
#pragma unroll
    for (int i = 0; i < RT; i++) {
        const float r = (float)rows_sum(acc[i]);  // the digits' and the groups' shares of row c
        if (grp == 0) s_p[wave][i][c] = r;
    }
    if constexpr (MODE == 1) {
        ss = group_sum(ss, 64);
        if (lane == 0) s_ss[wave] = ss;
    }
    __syncthreads();
    const int outs = out_swiglu ? RT * 8 : RT * 16;
    if (tid >= outs) return;
    float rr = 1.f;
    if constexpr (MODE == 1) {
        float t = 0.f;
#pragma unroll
        for (int v = 0; v < NW; v++) t += s_ss[v];
        rr = 1.0f / sqrtf(t / (float)w.cols + eps);
    }
    auto sum = [&](int i, int r) {  // pairwise: half the roundings of a chain
        float t[NW];
#pragma unroll
        for (int v = 0; v < NW; v++) t[v] = s_p[v][i][r];
#pragma unroll
        for (int n = NW; n > 1; n = (n + 1) / 2)
#pragma unroll
            for (int v = 0; v < n / 2; v++) t[v] = t[v] + t[n - 1 - v];
        return MODE == 1 ? t[0] * rr : t[0];
    };
    const int i = tid >> 4, r = tid & 15;
    if (out_swiglu) {
        const int o = RT == 1 ? 8 * (int)blockIdx.x + r : 16 * ((int)(blockIdx.x * RT >> 1) + i) + r;
        if (o >= F) return;
        const float gt = RT == 1 ? sum(0, r) : sum(2 * i, r), up = RT == 1 ? sum(0, 8 + r) : sum(2 * i + 1, r);
        y[o] = gt / (1.f + expf(-gt)) * up;  // Ops.SiLUMul (Ops.cs:1016-1052)
        return;
    }
    const int row = 16 * (int)(blockIdx.x * RT + i) + r;
    if (row >= w.rows) return;
    const float t = sum(i, r);
    y[row] = (flags & kGemvAccumulate) ? y[row] + t : t;
}

// GGUF blocks (fp16 d and dmin, 12 bytes of 6-bit scales and mins, 128 code
// bytes; rows x cols / 256 of 144 bytes) into the tiles of weights.hpp: a wave
// per tile, its lane the tile's lane (group g, row c).
__global__ __launch_bounds__(256) void q4k_tiles_kernel(const uint8_t *__restrict__ blocks, int rows, int nsb, int tiles,
                                                        uint8_t *__restrict__ out) {
    const int tile = blockIdx.x * 4 + (threadIdx.x >> 6), lane = threadIdx.x & 63, g = lane >> 4, c = lane & 15;
    if (tile >= tiles) return;
    const int row = tile / nsb * 16 + c, sb = tile % nsb;
    uint4 hdr = make_uint4(0, 0, 0, 0), q0 = hdr, q1 = hdr;
    if (row < rows) {
        const uint8_t *b = blocks + ((size_t)row * nsb + sb) * 144;
        hdr = *(const uint4 *)b;
        q0 = *(const uint4 *)(b + 16 + 32 * g);
        q1 = *(const uint4 *)(b + 32 + 32 * g);
    }
    uint32_t sm = 0;  // GetScaleMin (Q4K.cs:8-19) of sub-blocks 2 g, 2 g + 1; scale bytes 0-3, 4-7, 8-11 in y, z, w
#pragma unroll
    for (int h = 0; h < 2; h++) {
        const int j = 2 * g + h, k = 8 * (j & 3);
        const uint32_t y = (hdr.y >> k) & 0xFFu, z = (hdr.z >> k) & 0xFFu, w = (hdr.w >> k) & 0xFFu;
        const uint32_t sc = j < 4 ? y & 63 : (w & 0xF) | ((y >> 6) << 4), m = j < 4 ? z & 63 : (w >> 4) | ((z >> 6) << 4);
        sm |= sc << (8 * h) | m << (16 + 8 * h);
    }
    uint8_t *t = out + (size_t)tile * kQ4Tile;
    *(uint4 *)(t + 16 * lane) = q0;
    *(uint4 *)(t + 1024 + 16 * lane) = q1;
    *(uint32_t *)(t + kQ4Scales + 16 * c + 4 * g) = sm;
    if (g == 0) *(uint32_t *)(t + kQ4D + 4 * c) = hdr.x;
}

// The same for Q6_K's GGUF blocks (ql 128, qh 64, int8 scales 16, fp16 d: 210
// bytes, so 2-byte aligned).
__global__ __launch_bounds__(256) void q6k_tiles_kernel(const uint8_t *__restrict__ blocks, int rows, int nsb, int tiles,
                                                        uint8_t *__restrict__ out) {
    const int tile = blockIdx.x * 4 + (threadIdx.x >> 6), lane = threadIdx.x & 63, g = lane >> 4, c = lane & 15;
    if (tile >= tiles) return;
    const int row = tile / nsb * 16 + c, sb = tile % nsb;
    uint32_t q[2][4] = {}, hi[4] = {}, sc = 0, d = 0;
    if (row < rows) {
        const uint8_t *b = blocks + ((size_t)row * nsb + sb) * 210;
        auto rd = [&](int at) {  // 4 bytes, 2-byte aligned
            return *(const uint16_t *)(b + at) | (uint32_t)*(const uint16_t *)(b + at + 2) << 16;
        };
        // columns 64 g + 32 h + [0, 32) are quarter j = 2 (g & 1) + h of half g / 2
        const int n = g >> 1, nib = 4 * (g & 1);
#pragma unroll
        for (int h = 0; h < 2; h++)
#pragma unroll
            for (int i = 0; i < 4; i++) {
                const int j2 = 4 * (g & 1) + 2 * h, at = 64 * n + 32 * h + 4 * i;  // 2 j
                q[h][i] = ((rd(at) >> nib) & 0x0F0F0F0Fu) | ((rd(at + 16) >> nib) & 0x0F0F0F0Fu) << 4;
                const uint32_t h0 = (rd(128 + 32 * n + 4 * i) >> j2) & 0x03030303u;
                const uint32_t h1 = (rd(128 + 32 * n + 16 + 4 * i) >> j2) & 0x03030303u;
                // bits 7:6 for m = 0 down to 1:0 for m = 3, the upper one (32) flipped
                hi[i] |= (h0 ^ 0x02020202u) << (6 - 4 * h) | (h1 ^ 0x02020202u) << (4 - 4 * h);
            }
        sc = rd(192 + 4 * g);
        d = *(const uint16_t *)(b + 208);
    }
    uint8_t *t = out + (size_t)tile * kQ6Tile;
    *(uint4 *)(t + 16 * lane) = make_uint4(q[0][0], q[0][1], q[0][2], q[0][3]);
    *(uint4 *)(t + 1024 + 16 * lane) = make_uint4(q[1][0], q[1][1], q[1][2], q[1][3]);
    *(uint4 *)(t + kQ6Hi + 16 * lane) = make_uint4(hi[0], hi[1], hi[2], hi[3]);
    *(uint32_t *)(t + kQ6Scales + 16 * c + 4 * g) = sc;
    if (g == 0) *(uint16_t *)(t + kQ6D + 2 * c) = (uint16_t)d;
}

// The same for Q8_0's GGUF blocks (fp16 d, 32 int8: 34 bytes, 2-byte aligned).
__global__ __launch_bounds__(256) void q80_tiles_kernel(const uint8_t *__restrict__ blocks, int rows, int nsb, int tiles,
                                                        uint8_t *__restrict__ out) {
    const int tile = blockIdx.x * 4 + (threadIdx.x >> 6), lane = threadIdx.x & 63, g = lane >> 4, c = lane & 15;
    if (tile >= tiles) return;
    const int row = tile / nsb * 16 + c, sb = tile % nsb;
    uint32_t q[4][4] = {}, d = 0;
    if (row < rows) {
        const uint8_t *b = blocks + (((size_t)row * nsb + sb) * 8 + 2 * g) * 34;
        auto rd = [&](int at) {  // 4 bytes, 2-byte aligned
            return *(const uint16_t *)(b + at) | (uint32_t)*(const uint16_t *)(b + at + 2) << 16;
        };
#pragma unroll
        for (int m = 0; m < 4; m++)
#pragma unroll
            for (int i = 0; i < 4; i++) q[m][i] = rd(34 * (m >> 1) + 2 + 16 * (m & 1) + 4 * i);
        d = *(const uint16_t *)b | (uint32_t)*(const uint16_t *)(b + 34) << 16;
    }
    uint8_t *t = out + (size_t)tile * kQ8Tile;
#pragma unroll
    for (int m = 0; m < 4; m++) *(uint4 *)(t + 1024 * m + 16 * lane) = make_uint4(q[m][0], q[m][1], q[m][2], q[m][3]);
    *(uint32_t *)(t + kQ8D + 16 * c + 4 * g) = d;
}

const char *gemv_span_name(int type) {
    switch (type) {
    case kW_F32: return "gemv_f32";
    case kW_F16: return "gemv_f16";
    case kW_Q8_0: return "gemv_q8_0";
    case kW_Q4_K: return "gemv_q4_k";
    case kW_Q6_K: return "gemv_q6_k";
    case kW_Q2_0C: return "gemv_q2_0c";
    default: return "gemv_stq1_0";
    }
}

template <typename Unit, bool STQ>
hipError_t launch_t(const WeightDev &w, const float *x, float *y, int flags, const float *nw, float eps,
                    hipStream_t s) {
    const int upr = w.cols / 32;
    // a row's units must fit a wave; a thread stages at most 4 x 8 values of x
    if (w.cols % 2048 != 0 || w.cols > 8192 || upr > Unit::kMax * 64) return hipErrorInvalidValue;
    // lanes per row: the fewest (most units in flight per lane, K <= kMax), but
    // more until the grid has 512 workgroups: the dequantising arithmetic is
    // then spread over more waves (gate|up GEMVs are a little slower at 1024).
    int lpr = 8;
    while (upr / lpr > Unit::kMax) lpr *= 2;
    auto blocks = [&](int l) { return (w.rows + 4 * (64 / l) - 1) / (4 * (64 / l)); };
    while (lpr < 64 && blocks(lpr) < 512) lpr *= 2;
    const size_t lds = ((size_t)w.cols + w.cols / 16) * 4 + (size_t)w.cols / 8 * 4;
    const dim3 grid(blocks(lpr));
    KernelSpan span(gemv_span_name(w.type), s, true);
    const int K = upr / lpr;  // 64 NJ / lpr with lpr 8..64: a power of two, or 3 or 6 for NJ = 3
    const int mode = (flags & kGemvInRmsNorm) ? 1 : (flags & kGemvInSwiGLU) ? 2 : 0;
    bool ok = false;
    auto go = [&](auto nj_tag, auto k_tag) {
        constexpr int NJ = decltype(nj_tag)::value, KK = decltype(k_tag)::value;
        if constexpr (KK <= Unit::kMax) {
            if (w.cols / 2048 == NJ && K == KK) {
                if (mode == 1)
                    launch(span, gemv_kernel<Unit, STQ, NJ, KK, 1>, grid, dim3(256), lds, s, w, x, y, lpr, flags, nw,
                           eps);
                else if (mode == 2)
                    launch(span, gemv_kernel<Unit, STQ, NJ, KK, 2>, grid, dim3(256), lds, s, w, x, y, lpr, flags, nw,
                           eps);
                else
                    launch(span, gemv_kernel<Unit, STQ, NJ, KK, 0>, grid, dim3(256), lds, s, w, x, y, lpr, flags, nw,
                           eps);
                ok = true;
            }
        }
    };
    using std::integral_constant;
    go(integral_constant<int, 1>{}, integral_constant<int, 1>{});
    go(integral_constant<int, 1>{}, integral_constant<int, 2>{});
    go(integral_constant<int, 1>{}, integral_constant<int, 4>{});
    go(integral_constant<int, 1>{}, integral_constant<int, 8>{});
    go(integral_constant<int, 2>{}, integral_constant<int, 2>{});
    go(integral_constant<int, 2>{}, integral_constant<int, 4>{});
    go(integral_constant<int, 2>{}, integral_constant<int, 8>{});
    go(integral_constant<int, 3>{}, integral_constant<int, 3>{});
    go(integral_constant<int, 3>{}, integral_constant<int, 6>{});
    go(integral_constant<int, 4>{}, integral_constant<int, 4>{});
    go(integral_constant<int, 4>{}, integral_constant<int, 8>{});
    if (!ok) return hipErrorInvalidValue;
    return hipGetLastError();
}

template <int T, int RT, int NW, int NSB, bool MANY>
void launch_kq_mode(const WeightDev &w, const float *x, float *y, int flags, const float *nw, float eps, int grid,
                    const KernelSpan &span, hipStream_t s) {
    const dim3 g(grid), b(64 * NW);
    if (flags & kGemvInRmsNorm) launch(span, gemv_kq_kernel<T, RT, NW, NSB, 1, MANY>, g, b, 0, s, w, x, y, flags, nw, eps);
    else if (flags & kGemvInSwiGLU) launch(span, gemv_kq_kernel<T, RT, NW, NSB, 2, MANY>, g, b, 0, s, w, x, y, flags, nw, eps);
    else launch(span, gemv_kq_kernel<T, RT, NW, NSB, 0, MANY>, g, b, 0, s, w, x, y, flags, nw, eps);
}

// One tile per workgroup (with SwiGLU a gate and an up tile) and k over as many
// waves as leave each one or two super-blocks, while that is at most 512
// workgroups; beyond, 8 waves and two tiles that share a preparation of x'
// (one at 8192 columns, where two would hold 200 registers).  us per call in a
// recorded chain, W from HBM, the VALU form / here: 3072 x 2048 + norm 3.7 /
// 3.3, 2048 x 2048 3.05 / 2.9, 12288 x 2048 + norm + SwiGLU 6.8 / 6.0, 2048 x
// 6144 4.7 / 4.75 in 12 waves of two super-blocks, 2048 x 8192 5.6 / 5.6 in 16;
// with the norm 16384 x 2048 8.6 / 6.4, 40000 x 2048 25.5 / 11.7, 120818 x 2048
// 72.5 / 28.3.
// Q6_K by the same rule, the VALU form / here: 3072 x 2048 + norm 4.0 / 3.5, 2048 x
// 2048 3.2 / 2.95, 12288 x 2048 + norm + SwiGLU 8.4 / 7.1, 2048 x 6144 5.9 / 5.3,
// 2048 x 8192 7.2 / 6.2, with the norm 16384 x 2048 10.3 / 7.6, 40000 x 2048
// 17.7 / 14.0, 120818 x 2048 42 / 36.1 (5.65 TB/s).
// Q8_0 likewise (its VALU form had a byte convert and an fma per weight and fp32
// scales): 3.95 / 3.6, 3.1 / 2.9, 7.3 / 7.15, 5.7 / 5.1, 6.9 / 6.1, 9.4 / 8.5, 18.0 /
// 16.7, 48.3 / 44.9 (5.85 TB/s).  With SwiGLU Q8_0 takes tiles of 8 gate and 8 up
// rows, twice the workgroups (768 rather than 384 for 12288 rows, three per CU):
// half a tile's codes are whole 128-byte lines, as its 4352 bytes are 34 lines.
// One token through eight layers 164.0 -> 160.0 us when that was measured; the
// other types' tiles start within a line, and halves cost them (Q6_K 161.6 ->
// 169.5, Q4_K 149.1 -> 151.3).
template <int T>
hipError_t launch_kq(const WeightDev &w, const float *x, float *y, int flags, const float *nw, float eps,
                     hipStream_t s) {
    if (w.cols % 2048 != 0 || w.cols > 8192) return hipErrorInvalidValue;
    const bool glu = flags & kGemvOutSwiGLU;
    const int tiles = glu ? 2 * ((w.rows / 2 + 15) / 16) : (w.rows + 15) / 16;
    const bool few = (glu ? tiles / 2 : tiles) <= 512, half = T == kW_Q8_0 && glu && few;
    KernelSpan span(gemv_span_name(w.type), s, true);
    auto go = [&](auto waves, auto sbs, int rt) {
        constexpr int NW = decltype(waves)::value, NSB = decltype(sbs)::value;
        if (rt == 2) {  // 8 waves of several super-blocks each: long grids only
            if (NW == 8 && (NSB > 1 || !few)) {
                if constexpr (NW == 8) launch_kq_mode<T, 2, NW, NSB, true>(w, x, y, flags, nw, eps, (tiles + 1) / 2, span, s);
            } else if constexpr (NW > 8 || NSB == 1) {
                launch_kq_mode<T, 2, NW, NSB, false>(w, x, y, flags, nw, eps, (tiles + 1) / 2, span, s);
            }
        } else if constexpr (NW > 8 || NSB == 1 || NSB == 4) {
            launch_kq_mode<T, 1, NW, NSB, false>(w, x, y, flags, nw, eps, half ? (w.rows / 2 + 7) / 8 : tiles, span, s);
        }
    };
    using I1 = std::integral_constant<int, 1>;
    using I2 = std::integral_constant<int, 2>;
    using I3 = std::integral_constant<int, 3>;
    using I4 = std::integral_constant<int, 4>;
    using I8 = std::integral_constant<int, 8>;
    using I12 = std::integral_constant<int, 12>;
    using I16 = std::integral_constant<int, 16>;
    const int rt = half || (!glu && few) ? 1 : 2;
    switch (w.cols / 2048) {
    case 1: go(I8{}, I1{}, rt); break;
    case 2: few ? go(I16{}, I1{}, rt) : go(I8{}, I2{}, rt); break;
    case 3: few ? go(I12{}, I2{}, rt) : go(I8{}, I3{}, rt); break;
    default: few ? go(I16{}, I2{}, rt) : go(I8{}, I4{}, glu ? 2 : 1); break;
    }
    return hipGetLastError();
}

// Rows of the matrix, dequantized to fp32: workgroup b writes row
// rows[b] (or row0 + b when rows is null) at out + b * cols.  Embedding of a
// prompt (HunyuanDenseModel.Embed's row loop, HunyuanDenseModel.cs:541-556)
// and the source of the dense copies the prefill GEMMs read.
template <typename Unit, bool STQ>
__global__ __launch_bounds__(256) void rows_kernel(WeightDev w, const int *__restrict__ rows, int row0,
                                                   float *__restrict__ out) {
    __shared__ uint8_t book[32];
    if (STQ && threadIdx.x < 32) book[threadIdx.x] = kStqBook[threadIdx.x];
    __syncthreads();
    const int row = rows ? rows[blockIdx.x] : row0 + (int)blockIdx.x;
    float *o = out + (size_t)blockIdx.x * w.cols;
    for (int u = threadIdx.x; u < w.cols / 32; u += 256) {
        Unit un;
        un.load(w, row, u);
        if constexpr (STQ) un.store(u, book, o);
        else un.store(u, 0.f, o);
    }
}

template <typename Unit, bool STQ>
hipError_t launch_rows_t(const WeightDev &w, const int *rows, int row0, int n, float *out, hipStream_t s) {
    KernelSpan span("weight_rows", s, true);
    launch(span, rows_kernel<Unit, STQ>, dim3(n), dim3(256), 0, s, w, rows, row0, out);
    return hipGetLastError();
}

template <typename Unit, bool STQ>
hipError_t launch_embed_t(const WeightDev &w, int row, float *out, hipStream_t s) {
    KernelSpan span("embed", s, true);
    launch(span, embed_kernel<Unit, STQ>, dim3(1), dim3(256), 0, s, w, row, out);
    return hipGetLastError();
}

}  // namespace

hipError_t launch_gemv(const WeightDev &w, const float *x, float *y, int flags, const float *nw, float eps,
                       hipStream_t s) {
    switch (w.type) {
    case kW_F32: return launch_t<UnitF32, false>(w, x, y, flags, nw, eps, s);
    case kW_F16: return launch_t<UnitF16, false>(w, x, y, flags, nw, eps, s);
    case kW_Q8_0: return launch_kq<kW_Q8_0>(w, x, y, flags, nw, eps, s);
    case kW_Q4_K: return launch_kq<kW_Q4_K>(w, x, y, flags, nw, eps, s);
    case kW_Q6_K: return launch_kq<kW_Q6_K>(w, x, y, flags, nw, eps, s);
    case kW_Q2_0C: return launch_t<UnitQ2_0C, false>(w, x, y, flags, nw, eps, s);
    case kW_STQ1_0: return launch_t<UnitSTQ1_0, true>(w, x, y, flags, nw, eps, s);
    default: return hipErrorInvalidValue;
    }
}

hipError_t launch_kq_tiles(int type, const void *blocks, int rows, int cols, void *tiles, hipStream_t s) {
    const int nsb = cols / 256, n = (rows + 15) / 16 * nsb;
    hipLaunchKernelGGL(type == kW_Q8_0 ? q80_tiles_kernel : type == kW_Q6_K ? q6k_tiles_kernel : q4k_tiles_kernel,
                       dim3((n + 3) / 4), dim3(256), 0, s, (const uint8_t *)blocks, rows, nsb, n, (uint8_t *)tiles);
    return hipGetLastError();
}

hipError_t launch_rows(const WeightDev &w, const int *rows, int row0, int n, float *out, hipStream_t s) {
    if (n <= 0) return hipSuccess;
    switch (w.type) {
    case kW_F32: return launch_rows_t<UnitF32, false>(w, rows, row0, n, out, s);
    case kW_F16: return launch_rows_t<UnitF16, false>(w, rows, row0, n, out, s);
    case kW_Q8_0: return launch_rows_t<UnitQ8_0, false>(w, rows, row0, n, out, s);
    case kW_Q4_K: return launch_rows_t<UnitQ4_K, false>(w, rows, row0, n, out, s);
    case kW_Q6_K: return launch_rows_t<UnitQ6_K, false>(w, rows, row0, n, out, s);
    case kW_Q2_0C: return launch_rows_t<UnitQ2_0C, false>(w, rows, row0, n, out, s);
    case kW_STQ1_0: return launch_rows_t<UnitSTQ1_0, true>(w, rows, row0, n, out, s);
    default: return hipErrorInvalidValue;
    }
}

hipError_t launch_embed(const WeightDev &w, int row, float *out, hipStream_t s) {
    switch (w.type) {
    case kW_F32: return launch_embed_t<UnitF32, false>(w, row, out, s);
    case kW_F16: return launch_embed_t<UnitF16, false>(w, row, out, s);
    case kW_Q8_0: return launch_embed_t<UnitQ8_0, false>(w, row, out, s);
    case kW_Q4_K: return launch_embed_t<UnitQ4_K, false>(w, row, out, s);
    case kW_Q6_K: return launch_embed_t<UnitQ6_K, false>(w, row, out, s);
    case kW_Q2_0C: return launch_embed_t<UnitQ2_0C, false>(w, row, out, s);
    case kW_STQ1_0: return launch_embed_t<UnitSTQ1_0, true>(w, row, out, s);
    default: return hipErrorInvalidValue;
    }
}

}  // namespace hymt
