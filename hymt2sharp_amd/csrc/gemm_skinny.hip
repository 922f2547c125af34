// gemm_skinny.hip -- the prefill GEMMs of short prompts (gfx950): y[m][n] (+)=
// x[m][k] . W[n][k]^T, bf16 operands, fp32 accumulation, for outputs so small
// that the tiles of gemm_mfma.hip leave most of the chip idle.
//
// What bounds it: reading W once (q/k/v and o 8-13 MB, down 25 MB, gate/up
// 50 MB per layer).  The 128 x 64 tiles gave 32 to 192 workgroups, each
// walking its whole k range (or half of it) through one ring behind a barrier
// per stage: for 2 to 187 tokens a layer's four GEMMs took 53-63 us whatever
// the token count, 1.1-1.3 TB/s.  Here a workgroup owns a small tile (16 A
// features x 16 B tokens) and its four waves split k: each wave streams its
// own quarter of the tile's W and x rows through an LDS ring of its own
// (global_load_lds_dwordx4, whole 128-byte lines), so there is no barrier
// before the end, four independent load streams run per workgroup, and a k
// step's serial chain is a quarter as long.  The four partial tiles meet in
// LDS and are added in wave order.
//
// k is always split in four equal parts whatever the tile, so that an output's
// sum -- four 32-k MFMA chains, added in order -- does not depend on the tile:
// all tiles give the same bits, and the fused gate/up + SwiGLU form (GLU)
// gives those of the GEMM followed by the row kernel.
//
// Tile choice (skinny_plan): the smallest tile that gives at most 256
// workgroups, one per CU; a second round costs more than a larger tile
// (2048 x 2048, 187 tokens: 32 x 32 in 384 workgroups 7.3 us, 32 x 64 in 192
// 6.3).  Where even 96 x 64 needs more than 256, the chip is full and the
// tiles of gemm_mfma.hip, which read fewer operand bytes per flop, take over.
// us per call with W from HBM, here / gemm_mfma.hip:
//   tokens      q/k/v 3072x2048  o 2048x2048  down 2048x6144  gate/up 12288x2048
//      2            3.8 /  9.3     3.2 /  9.2     5.5 / 17.9     10.3 / 13 (+ SwiGLU 3.9)
//     61            5.0 /  9.9     4.1 / 10.5     8.3 / 19.6     13.2 / 13.3
//    128            5.9 / 10.1     5.0 / 10.7    10.8 / 20.5     16.4 / 20.0 (both fused)
//    300            8.6 / 10.7     8.3 / 11.1    18.9 / 21.4     (gemm_mfma.hip)
//    700       (gemm_mfma.hip)    11.9 / 21.4    25.5 / 29.4     (gemm_mfma.hip)
#include <hip/hip_runtime.h>

#include <cstdint>

#include "device_common.hpp"
#include "ktimer.hpp"
#include "weights.hpp"

namespace hymt {
namespace {

typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef float f32x4 __attribute__((ext_vector_type(4)));

constexpr int kWaves = 4;    // waves of a workgroup: parts of k
constexpr int kBK = 64;      // k per stage
constexpr int kBlock = 2048; // bytes of one row block's 16 rows x 64 k

struct SkinnyArgs {
    const uint16_t *W;   // [n][k]; GLU: the gate rows [n / 2][k]
    const uint16_t *W2;  // GLU: the up rows [n / 2][k]
    const uint16_t *x;   // [m][k]
    void *y;             // [m][ldy], fp32 or bf16
    int k, m, ldy;
    int tiles, tiles_t;  // tiles in all, along the tokens
    int per_xcd;         // workgroups per XCD: ceil(tiles / 8)
    int stages;          // 64-k stages per wave: k / 256, >= S
};

enum Out { kF32, kAcc, kBf16, kGlu };

// s_waitcnt with vmcnt n (<= 63) alone, and lgkmcnt 0 alone (gfx9 encoding:
// vmcnt in bits 3:0 and 15:14, expcnt 6:4, lgkmcnt 11:8)
template <int N> __device__ __forceinline__ void wait_vm() {
    __builtin_amdgcn_s_waitcnt((N & 15) | ((N >> 4) << 14) | (7 << 4) | (15 << 8));
    asm volatile("" ::: "memory");
}
__device__ __forceinline__ void wait_lgkm() {
    __builtin_amdgcn_s_waitcnt(15 | (3 << 14) | (7 << 4));
    asm volatile("" ::: "memory");
}

// The last S stages of a wave, no copies left to issue: stage S - LEFT of them
// has landed once at most LEFT - 1 stages are outstanding.
template <int LEFT, int C, typename F> __device__ __forceinline__ void drain(F &&stage) {
    if constexpr (LEFT > 0) {
        wait_vm<(LEFT - 1) * C>();
        stage();
        drain<LEFT - 1, C>(stage);
    }
}

// Workgroup tile: 16 A features x 16 B tokens, wave w the k range
// [w, w + 1) k / 4 of it, S stages of 64 k in the wave's ring.  GLU: the first
// A / 2 row blocks are gate rows, the others the same rows of up, and the tile
// writes 8 A outputs silu(g) u of each token (g and u rounded to bf16 first, as
// the unfused calls do).
template <int A, int B, int S, int OUT>
__global__ __launch_bounds__(64 * kWaves) void skinny_kernel(SkinnyArgs a) {
    constexpr bool GLU = OUT == kGlu;
    constexpr int C = 2 * (A + B);  // copies (1 KiB each) of a stage
    constexpr int kStage = C * 1024, kRing = S * kStage, NT = 64 * kWaves;
    constexpr int AO = GLU ? A / 2 : A;                      // output row blocks
    constexpr int Q = AO * B * 64, NQ = (Q + NT - 1) / NT;   // 4-feature outputs, per thread
    static_assert(kWaves * kRing <= 160 * 1024 && C * (S - 1) <= 63, "ring");
    static_assert(A * B * 1024 <= kRing, "a wave's partial tile is handed over in its ring");
    static_assert(!GLU || A % 2 == 0, "gate and up row blocks");
    __shared__ __attribute__((aligned(1024))) uint8_t lds[kWaves * kRing];
    const int tid = threadIdx.x, lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int grp = lane >> 4, c = lane & 15;
    // Workgroup b runs on XCD b % 8: each XCD takes a contiguous run of tiles,
    // token tiles of one W slab next to each other, so that a slab is read
    // from HBM into one L2 and x (0.25 MB for 61 tokens) is read by all of them.
    const int L = (blockIdx.x & 7) * a.per_xcd + (blockIdx.x >> 3);
    if (L >= a.tiles) return;
    const int tf = L / a.tiles_t, tt = L - tf * a.tiles_t;
    const int f0 = tf * 16 * AO, t0 = tt * 16 * B;

    // output q (of Q): 4 features 4 grp.. of row block i, token c of token
    // block j, as the MFMA hands them over (q = 64 (i B + j) + lane)
    float4 old[NQ];
    if constexpr (OUT == kAcc) {  // the residual, loaded ahead of the stream
#pragma unroll
        for (int u = 0; u < NQ; u++) {
            const int q = tid + NT * u, fr = q >> 6, i = fr / B, j = fr - i * B;
            const int f = f0 + 16 * i + 4 * grp, t = t0 + 16 * j + c;
            old[u] = make_float4(0.f, 0.f, 0.f, 0.f);
            if (q < Q && t < a.m) old[u] = *(const float4 *)((const float *)a.y + (size_t)t * a.ldy + f);
        }
    }

    // Copy g of a stage brings half h = g & 1 of row block g >> 1 (W blocks,
    // then x): 8 whole 128-byte lines, placed as in gemm_mfma.hip so that
    // every operand read is free of bank conflicts: row r + 8 i of a block
    // keeps its 16-byte piece p in slot 16 r + 8 i + (p ^ r).  Token rows past
    // the end repeat the last one; their outputs are not written.
    uint32_t voff[C];
#pragma unroll
    for (int g = 0; g < C; g++) {
        const int gb = g >> 1, ga = 8 * (g & 1) + (lane >> 3);
        const int rl = (ga >> 1) + 8 * (ga & 1), piece = (lane & 7) ^ (ga >> 1);
        const int row = gb < A ? f0 + 16 * (GLU && gb >= AO ? gb - AO : gb) + rl : min(t0 + 16 * (gb - A) + rl, a.m - 1);
        voff[g] = (uint32_t)(((size_t)row * a.k + 8 * piece) * 2);
    }
    const size_t kbase = (size_t)wave * a.stages * kBK;
    const uint16_t *wb = a.W + kbase, *wb2 = GLU ? a.W2 + kbase : nullptr, *xb = a.x + kbase;
    const uint32_t ring = lds_addr(lds) + wave * kRing;
    auto copy = [&](int t, int slot) __attribute__((always_inline)) {
#pragma unroll
        for (int g = 0; g < C; g++) {
            const int gb = g >> 1;
            const uint16_t *base = gb >= A ? xb : GLU && gb >= AO ? wb2 : wb;
            lds_dma16_sv(base + t * kBK, voff[g], ring + slot * kStage + g * 1024);
        }
    };
    uint32_t off[2];
#pragma unroll
    for (int ks = 0; ks < 2; ks++) off[ks] = 16 * (16 * (c & 7) + 8 * (c >> 3) + ((4 * ks + grp) ^ (c & 7)));

    f32x4 acc[A][B];
#pragma unroll
    for (int i = 0; i < A; i++)
#pragma unroll
        for (int j = 0; j < B; j++) acc[i][j] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int t = 0; t < S; t++) copy(t, t);

    const uint8_t *my = lds + wave * kRing;
    bf16x8 w[2][A], x[2][B];
    int slot = 0;
    auto read = [&]() __attribute__((always_inline)) {
        const uint8_t *p = my + slot * kStage;
#pragma unroll
        for (int ks = 0; ks < 2; ks++) {
#pragma unroll
            for (int i = 0; i < A; i++) w[ks][i] = *(const bf16x8 *)(p + off[ks] + i * kBlock);
#pragma unroll
            for (int j = 0; j < B; j++) x[ks][j] = *(const bf16x8 *)(p + off[ks] + (A + j) * kBlock);
        }
    };
    auto mma = [&]() __attribute__((always_inline)) {
        slot = slot + 1 == S ? 0 : slot + 1;
#pragma unroll
        for (int ks = 0; ks < 2; ks++)
#pragma unroll
            for (int i = 0; i < A; i++)
#pragma unroll
                for (int j = 0; j < B; j++)
                    acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(w[ks][i], x[ks][j], acc[i][j], 0, 0, 0);
    };
    // A wave's copies retire in order: a stage has landed once at most S - 1
    // younger stages are outstanding.  Its slot is refilled as soon as this
    // wave has its operands in registers; no other wave touches the ring.
    for (int t = S; t < a.stages; t++) {
        wait_vm<(S - 1) * C>();
        read();
        wait_lgkm();
        copy(t, slot);
        mma();
    }
    drain<S, C>([&]() __attribute__((always_inline)) {
        read();
        mma();
    });
    wait_lgkm();

    // the partial tiles, each in its wave's ring (idle now), added in wave order
#pragma unroll
    for (int i = 0; i < A; i++)
#pragma unroll
        for (int j = 0; j < B; j++) *(f32x4 *)(lds + wave * kRing + (64 * (i * B + j) + lane) * 16) = acc[i][j];
    __syncthreads();
    auto sum = [&](int q) __attribute__((always_inline)) {
        f32x4 s = *(const f32x4 *)(lds + q * 16);
#pragma unroll
        for (int p = 1; p < kWaves; p++) s += *(const f32x4 *)(lds + p * kRing + q * 16);
        return s;
    };
    auto pack4 = [](float p, float q, float r, float s) {
        return make_uint2((uint32_t)f32_to_bf16(p) | ((uint32_t)f32_to_bf16(q) << 16),
                          (uint32_t)f32_to_bf16(r) | ((uint32_t)f32_to_bf16(s) << 16));
    };
#pragma unroll
    for (int u = 0; u < NQ; u++) {
        const int q = tid + NT * u, fr = q >> 6, i = fr / B, j = fr - i * B;
        const int f = f0 + 16 * i + 4 * grp, t = t0 + 16 * j + c;
        if (q >= Q || t >= a.m) continue;
        const f32x4 s = sum(q);
        if constexpr (GLU) {
            const f32x4 v = sum(q + Q);
            float o[4];
#pragma unroll
            for (int e = 0; e < 4; e++)  // swiglu8's arithmetic
                o[e] = silu_fast(bf16_to_f32(f32_to_bf16(s[e]))) * bf16_to_f32(f32_to_bf16(v[e]));
            *(uint2 *)((uint16_t *)a.y + (size_t)t * a.ldy + f) = pack4(o[0], o[1], o[2], o[3]);
        } else if constexpr (OUT == kBf16) {
            *(uint2 *)((uint16_t *)a.y + (size_t)t * a.ldy + f) = pack4(s[0], s[1], s[2], s[3]);
        } else {
            float4 o = make_float4(s[0], s[1], s[2], s[3]);
            if constexpr (OUT == kAcc) o = make_float4(old[u].x + o.x, old[u].y + o.y, old[u].z + o.z, old[u].w + o.w);
            *(float4 *)((float *)a.y + (size_t)t * a.ldy + f) = o;
        }
    }
}

// The tiles, smallest first: row blocks A, token blocks B, ring depth S.
// Depths: more stages in flight did not help once each wave has two or three
// (16 x 16: 4 stages 3.2 us, 8 stages 3.5 on the o projection), and a smaller
// ring lets two workgroups share a CU.
struct Tile {
    int A, B;
};
constexpr Tile kTiles[] = {{1, 1}, {1, 2}, {3, 1}, {2, 2}, {3, 2}, {2, 4}, {3, 4}, {4, 4}, {6, 4}, {4, 6}};
constexpr Tile kGluTiles[] = {{2, 1}, {4, 1}, {2, 2}, {4, 2}, {6, 2}, {4, 4}, {6, 4}, {4, 6}};
constexpr int kMaxStages = 4;  // the deepest ring
constexpr int kCus = 256;

template <int A, int B, int S> void launch_glu(const SkinnyArgs &a, const KernelSpan &span, hipStream_t s) {
    launch(span, skinny_kernel<A, B, S, kGlu>, dim3(8 * a.per_xcd), dim3(64 * kWaves), 0, s, a);
}
template <int A, int B, int S> void launch_out(int out, const SkinnyArgs &a, const KernelSpan &span, hipStream_t s) {
    const dim3 grid(8 * a.per_xcd), block(64 * kWaves);
    if (out == kBf16) launch(span, skinny_kernel<A, B, S, kBf16>, grid, block, 0, s, a);
    else if (out == kAcc) launch(span, skinny_kernel<A, B, S, kAcc>, grid, block, 0, s, a);
    else launch(span, skinny_kernel<A, B, S, kF32>, grid, block, 0, s, a);
}

long tiles_of(Tile t, int n, int m) { return (long)(n / (16 * t.A)) * ((m + 16 * t.B - 1) / (16 * t.B)); }

SkinnyArgs args_of(Tile t, const uint16_t *W, int n, int k, const uint16_t *x, int m, void *y, int ldy) {
    SkinnyArgs a{};
    a.W = W;
    a.x = x;
    a.y = y;
    a.k = k;
    a.m = m;
    a.ldy = ldy;
    a.tiles_t = (m + 16 * t.B - 1) / (16 * t.B);
    a.tiles = (int)tiles_of(t, n, m);
    a.per_xcd = (a.tiles + 7) / 8;
    a.stages = k / (kWaves * kBK);
    return a;
}

}  // namespace

int gemm_skinny_plan(int n, int k, int m) {
    if (n < 128 || n % 128 || m < 1 || k % (kWaves * kBK) || k / (kWaves * kBK) < kMaxStages) return -1;
    for (int i = 0; i < (int)(sizeof(kTiles) / sizeof(kTiles[0])); i++)
        if (n % (16 * kTiles[i].A) == 0 && tiles_of(kTiles[i], n, m) <= kCus) return i;
    return -1;
}

hipError_t gemm_skinny(const uint16_t *W, int n, int k, const uint16_t *x, int m, void *y, int ldy, bool y_bf16,
                       bool accumulate, hipStream_t s) {
    const int i = gemm_skinny_plan(n, k, m);
    if (i < 0 || !gemm_mfma_fits(W, n, k, x, m, y, ldy) || (accumulate && y_bf16)) return hipErrorInvalidValue;
    const SkinnyArgs a = args_of(kTiles[i], W, n, k, x, m, y, ldy);
    const int out = y_bf16 ? kBf16 : accumulate ? kAcc : kF32;
    KernelSpan span(y_bf16 ? "gemm_mfma_out_bf16" : "gemm_mfma_out_f32", s, true);
    switch (i) {
    case 0: launch_out<1, 1, 4>(out, a, span, s); break;
    case 1: launch_out<1, 2, 3>(out, a, span, s); break;
    case 2: launch_out<3, 1, 2>(out, a, span, s); break;
    case 3: launch_out<2, 2, 2>(out, a, span, s); break;
    case 4: launch_out<3, 2, 4>(out, a, span, s); break;
    case 5: launch_out<2, 4, 2>(out, a, span, s); break;
    case 6: launch_out<3, 4, 2>(out, a, span, s); break;
    case 7: launch_out<4, 4, 2>(out, a, span, s); break;
    case 8: launch_out<6, 4, 2>(out, a, span, s); break;
    default: launch_out<4, 6, 2>(out, a, span, s); break;
    }
    return hipGetLastError();
}

hipError_t gemm_skinny_swiglu(const uint16_t *Wg, const uint16_t *Wu, int f, int k, const uint16_t *x, int m,
                              uint16_t *act, int ld, hipStream_t s) {
    if (!gemm_swiglu_fits(Wg, Wu, f, k, x, m, act, ld) || k % (kWaves * kBK) || k / (kWaves * kBK) < kMaxStages)
        return hipErrorInvalidValue;
    // as skinny_plan over the 2 f rows; the largest tile that divides them
    // where all need more than one round
    int i = -1;
    for (int t = 0; t < (int)(sizeof(kGluTiles) / sizeof(kGluTiles[0])); t++) {
        if (2 * f % (16 * kGluTiles[t].A)) continue;
        i = t;
        if (tiles_of(kGluTiles[t], 2 * f, m) <= kCus) break;
    }
    SkinnyArgs a = args_of(kGluTiles[i], Wg, 2 * f, k, x, m, act, ld);
    a.W2 = Wu;
    KernelSpan span("gemm_mfma_swiglu", s, true);
    switch (i) {
    case 0: launch_glu<2, 1, 3>(a, span, s); break;
    case 1: launch_glu<4, 1, 2>(a, span, s); break;
    case 2: launch_glu<2, 2, 2>(a, span, s); break;
    case 3: launch_glu<4, 2, 3>(a, span, s); break;
    case 4: launch_glu<6, 2, 2>(a, span, s); break;
    case 5: launch_glu<4, 4, 2>(a, span, s); break;
    case 6: launch_glu<6, 4, 2>(a, span, s); break;
    default: launch_glu<4, 6, 2>(a, span, s); break;
    }
    return hipGetLastError();
}

}  // namespace hymt
