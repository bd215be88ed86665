// Learned initial guess for the Newton/PCG solves: a small 3D U-Net on a
// 64^3 voxel grid (inclusion indicator, damage, step residual, previous load
// increment -> displacement correction), trained and evaluated on the device
// with this file's own kernels.
//
//  * every convolution is an implicit GEMM on bf16 MFMA tiles
//    (v_mfma_f32_16x16x16bf16_1k, FP32 accumulation);
//  * activations are stored channels-last in bf16; gradients leave their FP32
//    sums behind the ReLU mask as bf16 MFMA operands, FP32 where a skip
//    connection adds them on; weights are FP32 masters with bf16 copies per
//    step in fragment order (forward matrix [Cout][T*Cin], data-gradient matrix
//    [Cin][T*Cout]);
//  * Adam in FP32.
//
// Layers (64^3 x 8 input):
//   a1 = relu(conv3(x))            16 @ 64^3
//   a2 = relu(down2(a1))           32 @ 32^3
//   a3 = relu(conv3(a2))           32 @ 32^3
//   a4 = relu(down2(a3))           64 @ 16^3
//   a5 = relu(conv3(a4))           64 @ 16^3
//   a6 = relu(up2(a5) + a3)        32 @ 32^3
//   a7 = relu(up2(a6) + a1)        16 @ 64^3
//   y  = conv3(a7)                 16 @ 64^3 (channels 0..2 used)
// conv3: 3x3x3, stride 1, zero padding 1; down2: 2x2x2 stride 2; up2: its
// transpose (each output voxel has exactly one tap).
#include <hip/hip_runtime.h>

#include <algorithm>
#include <cmath>
#include <cstdint>
#include <cstring>
#include <string>
#include <vector>

#include "pgf_copy.hpp"
#include "../../../include/pgfem_learn.h"

namespace pgfn {

typedef short v4s __attribute__((ext_vector_type(4)));
typedef float v4f __attribute__((ext_vector_type(4)));
typedef uint16_t bf16;

constexpr int GRID = 64;  // the interface's; the kernels' tiles are laid out for it
constexpr int NVOX = GRID * GRID * GRID;
constexpr int IN_CH = 8;
constexpr int OUT_CH = 3;
enum Mode { CONV3 = 0, DOWN = 1, UP = 2 };
constexpr int N_LAYERS = 8;

struct LayerSpec {
    int mode, cin, cout, din;  // din: input grid size
};
constexpr LayerSpec SPECS[N_LAYERS] = {
    {CONV3, 8, 16, GRID},      {DOWN, 16, 32, GRID},     {CONV3, 32, 32, GRID / 2}, {DOWN, 32, 64, GRID / 2},
    {CONV3, 64, 64, GRID / 4}, {UP, 64, 32, GRID / 4},   {UP, 32, 16, GRID / 2},    {CONV3, 16, 16, GRID},
};
__host__ __device__ constexpr int taps(int mode) { return mode == CONV3 ? 27 : 8; }
__host__ __device__ constexpr int dout_of(int mode, int din) { return mode == DOWN ? din / 2 : (mode == UP ? din * 2 : din); }

__device__ __host__ inline bf16 f2bf(float f) {
    uint32_t u;
    memcpy(&u, &f, 4);
    u += 0x7fffu + ((u >> 16) & 1u);  // round to nearest even (finite inputs)
    return (bf16)(u >> 16);
}
__device__ __host__ inline float bf2f(bf16 h) {
    uint32_t u = (uint32_t)h << 16;
    float f;
    memcpy(&f, &u, 4);
    return f;
}

// ---------------------------------------------------------------------------
// Implicit-GEMM convolution, forward form.
//   out[p][n] = sum_{t,c} in[src(p,t)][c] * B[n][t*C + c]
// CONV3: src = p + off(t) - 1 (zero outside); DOWN: src = 2p + off(t);
// UP: the output's parity is the tap, t = parity, and src = p / 2.  Epilogue of
// the forward pass: + bias, + skip (bf16, same shape as out), ReLU; of the data
// gradients (BACK): + the skip connection's gradient, the mask of the ReLU in
// front of it, and the sums per channel, which are that layer's bias gradient.
//
// MFMA tiles with M = 16 channels, N = 16 positions along x, so that a lane
// ends with four consecutive channels of one position: 8- and 16-byte stores.
// The weights lie in fragment order (k_weights_bf16), 512 contiguous bytes a
// step.  The layers are small (one to four waves per SIMD), so latency bounds
// them: sizes are template parameters, the steps of the sum (16 wide) are
// unrolled and loaded KB steps ahead of their products.  4.5 to 20 us a layer,
// 64 us for a forward pass; loaded step by step, 9 to 105 and 0.28 ms.
struct ConvArgs {
    const bf16* in;      // [DIN^3][C]
    const bf16* B;       // fragments of [N][T*C]
    bf16* out_bf;        // [dout^3][N] or null
    float* out_f;        // [dout^3][N] or null
    // forward
    const float* bias;   // [N]
    const bf16* skip;    // [dout^3][N] or null
    int relu;
    // data gradient
    const float* add;    // [dout^3][N] or null
    const bf16* act;     // [dout^3][N]
    float* bpart;        // [blocks][N] sums
};

__device__ inline v4s frag(uint32_t a, uint32_t b) {
    union { uint32_t u[2]; v4s v; } f;
    f.u[0] = a;
    f.u[1] = b;
    return f.v;
}
__device__ inline v4s frag_at(const bf16* p) {
    const uint2 v = *(const uint2*)p;
    return frag(v.x, v.y);
}

// channels n .. n + 3 of the output position whose first channel is element e
template <bool BACK>
__device__ inline void conv_out(const ConvArgs& a, size_t e, int n, v4f acc, float4& bs) {
    float4 v = {acc[0], acc[1], acc[2], acc[3]};
    if (!BACK) {
        const float4 b = *(const float4*)(a.bias + n);
        v = float4{v.x + b.x, v.y + b.y, v.z + b.z, v.w + b.w};
        if (a.skip) {
            const ushort4 k = *(const ushort4*)(a.skip + e);
            v = float4{v.x + bf2f(k.x), v.y + bf2f(k.y), v.z + bf2f(k.z), v.w + bf2f(k.w)};
        }
        if (a.relu) v = float4{v.x > 0.f ? v.x : 0.f, v.y > 0.f ? v.y : 0.f, v.z > 0.f ? v.z : 0.f, v.w > 0.f ? v.w : 0.f};
    } else {
        if (a.add) {
            const float4 d = *(const float4*)(a.add + e);
            v = float4{d.x + v.x, d.y + v.y, d.z + v.z, d.w + v.w};
        }
        const ushort4 m = *(const ushort4*)(a.act + e);
        v = float4{bf2f(m.x) > 0.f ? v.x : 0.f, bf2f(m.y) > 0.f ? v.y : 0.f, bf2f(m.z) > 0.f ? v.z : 0.f,
                   bf2f(m.w) > 0.f ? v.w : 0.f};
        bs = float4{bs.x + v.x, bs.y + v.y, bs.z + v.z, bs.w + v.w};
    }
    if (a.out_bf) *(ushort4*)(a.out_bf + e) = ushort4{f2bf(v.x), f2bf(v.y), f2bf(v.z), f2bf(v.w)};
    if (a.out_f) *(float4*)(a.out_f + e) = v;
}

// the block's sums of the channels n0 .. n0 + 16 NT of bs, to dst
template <int NT>
__device__ inline void conv_bias_sums(float4 (&bs)[NT], float* dst) {
    __shared__ float sb[4][16 * NT];
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
#pragma unroll
    for (int j = 0; j < NT; ++j) {
#pragma unroll
        for (int m = 1; m < 16; m *= 2) {
            bs[j].x += __shfl_xor(bs[j].x, m);
            bs[j].y += __shfl_xor(bs[j].y, m);
            bs[j].z += __shfl_xor(bs[j].z, m);
            bs[j].w += __shfl_xor(bs[j].w, m);
        }
        if ((lane & 15) == 0) *(float4*)&sb[wave][j * 16 + (lane >> 4) * 4] = bs[j];
    }
    __syncthreads();
    const int n = threadIdx.x;
    if (n < 16 * NT) dst[n] = sb[0][n] + sb[1][n] + sb[2][n] + sb[3][n];
}

// CONV3.  A block takes YB lines of a plane and 16 channels: the lines around
// them go to LDS once, with the zeros outside the grid, so a tap is an offset
// within the block's lines, while the weights travel to registers; the loads
// are one latency, and every input is read from memory 18 / YB times instead
// of 27.  Positions are padded by 8 bytes from 32 channels on (bank conflicts).
template <bool BACK, int C, int N, int D, int YB>
__global__ __launch_bounds__(256) void k_conv3(ConvArgs a) {
    constexpr int KS = (27 * C + 15) / 16, KB = 9, NB = (KS + KB - 1) / KB, NCT = N / 16;
    constexpr int LI = (YB + 2) * 3, PS = C + (C >= 32 ? 4 : 0), LINE = (D + 2) * PS;
    static_assert(D % 16 == 0 && 64 % D == 0 && D % YB == 0, "four wavefronts share whole lines of 16-position tiles");
    constexpr int XT = D / 16, WY = 4 / XT, PT = YB / WY, H8 = C / 8, LOADS = (LI * D * H8 + 255) / 256;
    __shared__ __align__(16) bf16 s_in[LI * LINE];
    const int lane = threadIdx.x & 63, row = lane & 15, kq = lane >> 4, wave = threadIdx.x >> 6;
    const int tch = blockIdx.x % NCT, y0 = blockIdx.x / NCT % (D / YB) * YB, z = blockIdx.x / NCT / (D / YB);
    v4s w[KS];
#pragma unroll
    for (int s = 0; s < KS; ++s) w[s] = frag_at(a.B + ((size_t)(tch * KS + s) * 64 + lane) * 4);
    uint4 v[LOADS];
#pragma unroll
    for (int k = 0; k < LOADS; ++k) {
        const int i = k * 256 + threadIdx.x, h = i % H8, x = i / H8 % D, l = i / (H8 * D);
        const int ly = y0 + l % (YB + 2) - 1, lz = z + l / (YB + 2) - 1;
        v[k] = uint4{0u, 0u, 0u, 0u};
        if (l < LI && (unsigned)ly < (unsigned)D && (unsigned)lz < (unsigned)D)
            v[k] = *(const uint4*)(a.in + ((size_t)(lz * D + ly) * D + x) * C + h * 8);
    }
    for (int i = threadIdx.x; i < LI * 2 * (C / 4); i += 256) {
        const int c4 = i % (C / 4), side = i / (C / 4) & 1, l = i / (C / 4 * 2);
        *(uint2*)&s_in[l * LINE + side * (D + 1) * PS + c4 * 4] = uint2{0u, 0u};
    }
#pragma unroll
    for (int k = 0; k < LOADS; ++k) {
        const int i = k * 256 + threadIdx.x, h = i % H8, x = i / H8 % D, l = i / (H8 * D);
        if (l < LI) {
            bf16* q = &s_in[l * LINE + (x + 1) * PS + h * 8];
            *(uint2*)q = uint2{v[k].x, v[k].y};
            *(uint2*)(q + 4) = uint2{v[k].z, v[k].w};
        }
    }
    __syncthreads();
    const int x = wave % XT * 16 + row, wy = wave / XT * PT;
    float4 bs[1] = {{0.f, 0.f, 0.f, 0.f}};
#pragma unroll 1
    for (int t = wy; t < wy + PT; ++t) {
        const bf16* base = &s_in[t * LINE + x * PS + (C >= 16 ? kq : kq & 1) * 4];
        auto off = [&](int tap) { return (tap / 9 * (YB + 2) + tap / 3 % 3) * LINE + tap % 3 * PS; };
        v4s av[2][KB];
        auto fetch = [&](int b) {
#pragma unroll
            for (int i = 0; i < KB; ++i) {
                const int s = b * KB + i;
                if (s >= KS) break;
                if (C >= 16) {
                    av[b & 1][i] = frag_at(base + off(s * 16 / C) + s * 16 % C);
                } else {  // 8 channels: two taps a step, the last alone
                    const int o0 = off(2 * s), o1 = 2 * s + 1 < 27 ? off(2 * s + 1) : o0;
                    const v4s f = frag_at(base + (kq < 2 ? o0 : o1));
                    av[b & 1][i] = 2 * s + 1 < 27 || kq < 2 ? f : v4s{0, 0, 0, 0};
                }
            }
        };
        v4f acc = {0.f, 0.f, 0.f, 0.f};
        fetch(0);
#pragma unroll
        for (int b = 0; b < NB; ++b) {
            if (b + 1 < NB) fetch(b + 1);
            __builtin_amdgcn_sched_barrier(0);  // else the loads sink to their products
#pragma unroll
            for (int i = 0; i < KB; ++i)
                if (b * KB + i < KS) acc = __builtin_amdgcn_mfma_f32_16x16x16bf16_1k(w[b * KB + i], av[b & 1][i], acc, 0, 0, 0);
        }
        const int n = tch * 16 + kq * 4;
        conv_out<BACK>(a, ((size_t)(z * D + y0 + t) * D + x) * N + n, n, acc, bs[0]);
    }
    if (BACK) conv_bias_sums<1>(bs, a.bpart + (size_t)(blockIdx.x / NCT) * N + tch * 16);
}

// DOWN and UP, no input read twice: fragments straight from memory.  A
// wavefront takes one tile of positions (UP: of the input's, both parities in
// x) and 16 NT channels.
template <bool BACK, int MODE, int C, int N, int DIN, int NT>
__global__ __launch_bounds__(256) void k_conv2(ConvArgs a) {
    constexpr int S = MODE == DOWN ? DIN / 2 : DIN, DOUT = dout_of(MODE, DIN), CS = C / 16, KST = 8 * CS;
    constexpr int KS = MODE == UP ? CS : KST, KB = KS < 8 ? KS : 8, NB = KS / KB;
    static_assert(S % 16 == 0 && S * S * S % 64 == 0, "whole tiles of 16 positions along x, four to a block");
    constexpr int XT = S / 16, NCT = N / (16 * NT), CLS = MODE == UP ? 2 : 1;
    const int lane = threadIdx.x & 63, row = lane & 15, kq = lane >> 4;
    // x tile fastest, then y, z, for UP the parity in y and z
    const int tch = blockIdx.x % NCT;
    int u = blockIdx.x / NCT * 4 + (threadIdx.x >> 6);
    const int x = u % XT * 16 + row;
    u /= XT;
    const int y = u % S, z = u / S % S, par = u / (S * S);  // par = oy + 2 oz
    const bf16* src = a.in + ((size_t)((MODE == DOWN ? 2 * z : z) * DIN + (MODE == DOWN ? 2 * y : y)) * DIN +
                              (MODE == DOWN ? 2 * x : x)) * C + kq * 4;
    const bf16* wts = a.B + ((size_t)(tch * NT * KST + 2 * par * CS) * 64 + lane) * 4;
    v4s av[2][KB], bv[2][KB][NT][CLS];
    auto fetch = [&](int b) {
#pragma unroll
        for (int i = 0; i < KB; ++i) {
            const int s = b * KB + i, t = s / CS;
            av[b & 1][i] = frag_at(src + (MODE == UP ? 0 : (((t >> 2) * DIN + (t >> 1 & 1)) * DIN + (t & 1)) * C) + s % CS * 16);
#pragma unroll
            for (int j = 0; j < NT; ++j)
#pragma unroll
                for (int c = 0; c < CLS; ++c) bv[b & 1][i][j][c] = frag_at(wts + (size_t)(j * KST + c * CS + s) * 256);
        }
    };
    v4f acc[NT][CLS];
#pragma unroll
    for (int j = 0; j < NT; ++j)
#pragma unroll
        for (int c = 0; c < CLS; ++c) acc[j][c] = v4f{0.f, 0.f, 0.f, 0.f};
    fetch(0);
#pragma unroll
    for (int b = 0; b < NB; ++b) {
        if (b + 1 < NB) fetch(b + 1);
        __builtin_amdgcn_sched_barrier(0);  // else the loads sink to their products
#pragma unroll
        for (int i = 0; i < KB; ++i)
#pragma unroll
            for (int j = 0; j < NT; ++j)
#pragma unroll
                for (int c = 0; c < CLS; ++c)
                    acc[j][c] = __builtin_amdgcn_mfma_f32_16x16x16bf16_1k(bv[b & 1][i][j][c], av[b & 1][i], acc[j][c], 0, 0, 0);
    }
    float4 bs[NT];
#pragma unroll
    for (int j = 0; j < NT; ++j) {
        bs[j] = float4{0.f, 0.f, 0.f, 0.f};
        const int n = (tch * NT + j) * 16 + kq * 4;
#pragma unroll
        for (int c = 0; c < CLS; ++c) {
            const size_t p = MODE == UP ? (size_t)((2 * z + (par >> 1)) * DOUT + 2 * y + (par & 1)) * DOUT + 2 * x + c
                                        : (size_t)(z * DOUT + y) * DOUT + x;
            conv_out<BACK>(a, p * N + n, n, acc[j][c], bs[j]);
        }
    }
    if (BACK) conv_bias_sums<NT>(bs, a.bpart + (size_t)(blockIdx.x / NCT) * N + tch * NT * 16);
}

// ---------------------------------------------------------------------------
// Weight gradients dW[t][c][n] = sum_p in[src(p,t)][c] * g[p][n] over the
// layer's output positions p, as MFMA tiles (M = 16 channels n, N = 16 channels
// c, K = p).
//
// Activations are channels-last, so both operands of a product over positions
// lie across memory; loading them element by element (2 bytes a lane) took 34
// to 280 us a layer.  A block instead stages 128 output positions at a time in
// LDS, transposed to [channel][x]: there a lane's four consecutive positions
// are one 8-byte read, and the lines staged once serve every tap.  A block owns
// one tile pair (16 c, 16 n), a wavefront the taps of one offset in z (3 x 3 x
// 3) or in y and z (2 x 2 x 2), whose sums stay in its registers over the
// block's stages; the partials of the blocks go to part[chunk][N][T*C] and are
// added by k_wgrad_reduce.  6 to 21 us a layer so, 0.09 ms for all eight
// (0.94 ms before), bound by the stages' latency: two blocks per CU.
struct WgArgs {
    int stages;      // stages per block
    const bf16* in;  // [din^3][C]
    const bf16* g;   // [dout^3][N]
    float* part;     // [chunks][N][T*C]
};
constexpr int WG_POS = 128;  // positions per stage

// 8 channels of one position into rows of a transposed tile
__device__ inline void put8(bf16* tile, int ld, int x, uint4 v) {
    const uint32_t w[4] = {v.x, v.y, v.z, v.w};
#pragma unroll
    for (int i = 0; i < 4; ++i) {
        tile[(2 * i) * ld + x] = (bf16)(w[i] & 0xffffu);
        tile[(2 * i + 1) * ld + x] = (bf16)(w[i] >> 16);
    }
}
template <int C, int N, int D>
__global__ __launch_bounds__(192) void k_wgrad3(WgArgs a) {
    static_assert(WG_POS % D == 0 && D % (WG_POS / D) == 0, "a stage is whole lines of one plane");
    constexpr int R = WG_POS / D, LI = (R + 2) * 3, LD = D + 4, LG = WG_POS + 4, TC = 27 * C;
    constexpr int CH = C < 16 ? C : 16, H8 = CH / 8;  // staged input channels, in groups of 8
    constexpr int CT = C < 16 ? 1 : C / 16, NT = N / 16;
    __shared__ __align__(16) bf16 s_in[LI][CH][LD], s_g[16][LG];
    const int lane = threadIdx.x & 63, oz = threadIdx.x >> 6, row = lane & 15, kq = lane >> 4;
    const int ct = blockIdx.x % CT, nt = blockIdx.x / CT % NT, chunk = blockIdx.x / (CT * NT);
    v4f acc[3][3];
#pragma unroll
    for (int i = 0; i < 3; ++i)
#pragma unroll
        for (int j = 0; j < 3; ++j) acc[i][j] = v4f{0.f, 0.f, 0.f, 0.f};
    // columns outside the grid (x + 1 of 0 and beyond D) stay zero
    for (int i = threadIdx.x; i < LI * CH * LD / 2; i += 192) ((uint32_t*)s_in)[i] = 0u;
    for (int st = chunk * a.stages; st < (chunk + 1) * a.stages; ++st) {
        const int z = st / (D / R), y0 = st % (D / R) * R;
        __syncthreads();
        for (int i = threadIdx.x; i < LI * D * H8; i += 192) {
            const int h = i % H8, x = i / H8 % D, l = i / (H8 * D), lz = z + l / (R + 2) - 1, ly = y0 + l % (R + 2) - 1;
            uint4 v = {0u, 0u, 0u, 0u};
            if ((unsigned)lz < (unsigned)D && (unsigned)ly < (unsigned)D)
                v = *(const uint4*)(a.in + ((size_t)(lz * D + ly) * D + x) * C + ct * CH + h * 8);
            put8(&s_in[l][h * 8][0], LD, x + 1, v);
        }
        for (int i = threadIdx.x; i < WG_POS * 2; i += 192) {
            const int h = i & 1, p = i >> 1;
            put8(&s_g[h * 8][0], LG, p, *(const uint4*)(a.g + ((size_t)(z * D + y0) * D + p) * N + nt * 16 + h * 8));
        }
        __syncthreads();
#pragma unroll 2
        for (int k = 0; k < WG_POS / 16; ++k) {
            const int p = k * 16 + kq * 4, r = p / D, x = p % D;
            const v4s av = frag_at(&s_g[row][p]);
#pragma unroll
            for (int oy = 0; oy < 3; ++oy) {
                // inputs x - 1 .. x + 6 of the tap's line: the three x offsets
                const bf16* q = &s_in[oz * (R + 2) + r + oy][row % CH][x];
                const uint2 lo = *(const uint2*)q, hi = *(const uint2*)(q + 4);
                const v4s b0 = frag(lo.x, lo.y);
                const v4s b1 = frag(__builtin_amdgcn_alignbit(lo.y, lo.x, 16), __builtin_amdgcn_alignbit(hi.x, lo.y, 16));
                const v4s b2 = frag(lo.y, hi.x);
                if (C >= 16) {
                    acc[oy][0] = __builtin_amdgcn_mfma_f32_16x16x16bf16_1k(av, b0, acc[oy][0], 0, 0, 0);
                    acc[oy][1] = __builtin_amdgcn_mfma_f32_16x16x16bf16_1k(av, b1, acc[oy][1], 0, 0, 0);
                    acc[oy][2] = __builtin_amdgcn_mfma_f32_16x16x16bf16_1k(av, b2, acc[oy][2], 0, 0, 0);
                } else {
                    // 8 channels: x offsets 0 and 1 side by side, then 2 alone
                    const v4s b01 = row < 8 ? b0 : b1;
                    acc[oy][0] = __builtin_amdgcn_mfma_f32_16x16x16bf16_1k(av, b01, acc[oy][0], 0, 0, 0);
                    acc[oy][1] = __builtin_amdgcn_mfma_f32_16x16x16bf16_1k(av, b2, acc[oy][1], 0, 0, 0);
                }
            }
        }
    }
    // lane holds channels n = nt*16 + kq*4 + i, column `row`
#pragma unroll
    for (int oy = 0; oy < 3; ++oy)
#pragma unroll
        for (int j = 0; j < (C >= 16 ? 3 : 2); ++j) {
            const int ox = C >= 16 ? j : (j == 0 ? row >> 3 : 2), c = C >= 16 ? ct * 16 + row : row & 7;
            if (C < 16 && j == 1 && row >= 8) continue;
            const int t = ox + 3 * oy + 9 * oz;
#pragma unroll
            for (int i = 0; i < 4; ++i)
                a.part[((size_t)chunk * N + nt * 16 + kq * 4 + i) * TC + t * C + c] = acc[oy][j][i];
        }
}

// 2 x 2 x 2 stride 2 between a fine grid (2H)^3 with CF channels and a coarse
// one H^3 with CQ: DOWN has in fine and g coarse, UP in coarse and g fine.
template <int CF, int CQ, int H, bool IS_UP>
__global__ __launch_bounds__(256) void k_wgrad2(WgArgs a) {
    static_assert(WG_POS % H == 0 && H % (WG_POS / H) == 0, "a stage is whole lines of one plane");
    constexpr int R = WG_POS / H, LD = H + 4, LG = WG_POS + 4, D = 2 * H;
    constexpr int C = IS_UP ? CQ : CF, N = IS_UP ? CF : CQ, TC = 8 * C;
    constexpr int FT = CF / 16, QT = CQ / 16;
    __shared__ __align__(16) bf16 s_f[R * 4][2][16][LD], s_q[16][LG];
    const bf16* fine = IS_UP ? a.g : a.in;
    const bf16* coarse = IS_UP ? a.in : a.g;
    const int lane = threadIdx.x & 63, oyz = threadIdx.x >> 6, row = lane & 15, kq = lane >> 4;
    const int ft = blockIdx.x % FT, qt = blockIdx.x / FT % QT, chunk = blockIdx.x / (FT * QT);
    v4f acc[2];
    acc[0] = acc[1] = v4f{0.f, 0.f, 0.f, 0.f};
    for (int st = chunk * a.stages; st < (chunk + 1) * a.stages; ++st) {
        const int z = st / (H / R), y0 = st % (H / R) * R;
        __syncthreads();
        for (int i = threadIdx.x; i < R * 4 * D * 2; i += 256) {
            const int h = i & 1, x = (i >> 1) % D, l = (i >> 1) / D, r = l >> 2, oy = l & 1, o2 = (l >> 1) & 1;
            const size_t p = ((size_t)(2 * z + o2) * D + 2 * (y0 + r) + oy) * D + x;
            put8(&s_f[l][x & 1][h * 8][0], LD, x >> 1, *(const uint4*)(fine + p * CF + ft * 16 + h * 8));
        }
        for (int i = threadIdx.x; i < WG_POS * 2; i += 256) {
            const int h = i & 1, p = i >> 1;
            put8(&s_q[h * 8][0], LG, p, *(const uint4*)(coarse + ((size_t)(z * H + y0) * H + p) * CQ + qt * 16 + h * 8));
        }
        __syncthreads();
#pragma unroll
        for (int k = 0; k < WG_POS / 16; ++k) {
            const int p = k * 16 + kq * 4, r = p / H, x = p % H;
            const v4s qv = frag_at(&s_q[row][p]);
#pragma unroll
            for (int ox = 0; ox < 2; ++ox) {
                const v4s fv = frag_at(&s_f[r * 4 + oyz][ox][row][x]);
                acc[ox] = IS_UP ? __builtin_amdgcn_mfma_f32_16x16x16bf16_1k(fv, qv, acc[ox], 0, 0, 0)
                                : __builtin_amdgcn_mfma_f32_16x16x16bf16_1k(qv, fv, acc[ox], 0, 0, 0);
            }
        }
    }
    const int nt = IS_UP ? ft : qt, c = (IS_UP ? qt : ft) * 16 + row;
#pragma unroll
    for (int ox = 0; ox < 2; ++ox)
#pragma unroll
        for (int i = 0; i < 4; ++i)
            a.part[((size_t)chunk * N + nt * 16 + kq * 4 + i) * TC + (ox + 2 * oyz) * C + c] = acc[ox][i];
}

// gW[t][c][n] = sum over chunks of part[chunk][n][t*C + c], every layer in one
// launch: 32 entries per block, 8 threads an entry.  Bound by memory: the
// partials, 62 MB in 14 us (eight launches of 10 us before).
struct WgLayers {
    int first[N_LAYERS + 1];  // blocks
    int chunks[N_LAYERS], N[N_LAYERS], TC[N_LAYERS];
    const float* part[N_LAYERS];
    float* gW[N_LAYERS];
};
__global__ __launch_bounds__(256) void k_wgrad_reduce(WgLayers w) {
    __shared__ float sh[8][32];
    int l = 0;
    while ((int)blockIdx.x >= w.first[l + 1]) ++l;
    const int nchunks = w.chunks[l], N = w.N[l], TC = w.TC[l];
    const float* part = w.part[l];
    const int idx = (blockIdx.x - w.first[l]) * 32 + (threadIdx.x & 31), q = threadIdx.x >> 5;
    float s = 0.f;
    if (idx < N * TC) {
#pragma unroll 8
        for (int k = q; k < nchunks; k += 8) s += part[(size_t)k * N * TC + idx];
    }
    sh[q][threadIdx.x & 31] = s;
    __syncthreads();
    if (q != 0 || idx >= N * TC) return;
    for (int k = 1; k < 8; ++k) s += sh[k][threadIdx.x];
    const int n = idx / TC, col = idx % TC;
    w.gW[l][(size_t)col * N + n] = s;  // col = t*C + c
}

// bf16(d) of the output layer's gradient and the block's sums of d per channel,
// its bias gradient's partials (the other layers' come from the convolutions).
// Bound by memory.  A thread's four elements have the same channels in every
// trip (1024 is a multiple of N).
constexpr int RB_BLOCKS = 512;
__global__ __launch_bounds__(256) void k_out_back(int64_t n4, int N, const float4* __restrict__ d,
                                                  ushort4* __restrict__ gbf, float* __restrict__ part) {
    __shared__ float sh[1024];
    float4 s = {0.f, 0.f, 0.f, 0.f};
    for (int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x; i < n4; i += (int64_t)gridDim.x * 256) {
        const float4 v = d[i];
        gbf[i] = ushort4{f2bf(v.x), f2bf(v.y), f2bf(v.z), f2bf(v.w)};
        s.x += v.x;
        s.y += v.y;
        s.z += v.z;
        s.w += v.w;
    }
    ((float4*)sh)[threadIdx.x] = s;
    __syncthreads();
    // entry e of the block's 1024 sums has channel e % N
    if ((int)threadIdx.x < N) {
        float t = 0.f;
        for (int e = threadIdx.x; e < 1024; e += N) t += sh[e];
        part[(size_t)blockIdx.x * N + threadIdx.x] = t;
    }
}

// gb[n] = sum over blocks of part[block][n], every layer in one launch (a block
// each)
struct BiasLayers {
    int blocks[N_LAYERS], N[N_LAYERS];
    float* gb[N_LAYERS];
};
constexpr int BIAS_PART = 512 * 64;  // floats per layer, the most any has (blocks x channels)
__global__ __launch_bounds__(1024) void k_bias_reduce(const float* __restrict__ part, BiasLayers b) {
    __shared__ float sh[1024];
    const int l = blockIdx.x, N = b.N[l];
    part += (size_t)l * BIAS_PART;
    float s = 0.f;
#pragma unroll 4
    for (int e = threadIdx.x; e < b.blocks[l] * N; e += 1024) s += part[e];
    sh[threadIdx.x] = s;
    __syncthreads();
    if ((int)threadIdx.x >= N) return;
    for (int e = threadIdx.x + N; e < 1024; e += N) s += sh[e];
    b.gb[l][threadIdx.x] = s;
}

// the three used channels of y [NVOX][16], and dy [NVOX][3] with the others zero
__global__ __launch_bounds__(256) void k_pick_out(const float* __restrict__ y, float* __restrict__ y3) {
    const int p = blockIdx.x * 256 + threadIdx.x;
    if (p >= NVOX) return;
    const float4 v = ((const float4*)y)[4 * (size_t)p];
    y3[3 * (size_t)p] = v.x;
    y3[3 * (size_t)p + 1] = v.y;
    y3[3 * (size_t)p + 2] = v.z;
}
__global__ __launch_bounds__(256) void k_widen_out(const float* __restrict__ d3, float* __restrict__ dy) {
    const int i = blockIdx.x * 256 + threadIdx.x, p = i / 4, q = i % 4;
    if (p >= NVOX) return;
    float4 v = {0.f, 0.f, 0.f, 0.f};
    if (q == 0) v = float4{d3[3 * (size_t)p], d3[3 * (size_t)p + 1], d3[3 * (size_t)p + 2], 0.f};
    ((float4*)dy)[i] = v;
}

__global__ void k_to_bf16(int64_t n, const float* x, bf16* y) {
    const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i < n) y[i] = f2bf(x[i]);
}

// bf16 weight copies from the FP32 master W[t][c][n]:
//   Bf[n][t*C + c] = W[t][c][n]             (forward)
//   Bd[c][t*N + n] = W[flip(t)][c][n]       (data gradient; flip = 26 - t for conv3)
// both as fragments: 16 rows by 16 columns, the columns padded to 16, a lane's
// four consecutive columns of a row side by side.
__host__ __device__ constexpr int frag_count(int rows, int cols) { return (rows + 15) / 16 * ((cols + 15) / 16) * 256; }
__device__ inline int frag_index(int r, int k, int cols) {
    return ((r >> 4) * ((cols + 15) >> 4) + (k >> 4)) * 256 + ((k & 15) >> 2) * 64 + (r & 15) * 4 + (k & 3);
}
__global__ void k_weights_bf16(int mode, int T, int C, int N, const float* W, bf16* Bf, bf16* Bd) {
    const int idx = blockIdx.x * blockDim.x + threadIdx.x;
    if (idx >= T * C * N) return;
    const int t = idx / (C * N), c = (idx / N) % C, n = idx % N;
    const bf16 h = f2bf(W[idx]);
    Bf[frag_index(n, t * C + c, T * C)] = h;
    const int tf = mode == CONV3 ? 26 - t : t;
    Bd[frag_index(c, tf * N + n, T * N)] = h;
}

// Adam (FP32): m = b1 m + (1-b1) g; v = b2 v + (1-b2) g^2; w -= lr mhat / (sqrt(vhat) + eps)
__global__ void k_adam(int64_t n, float* w, const float* g, float* m, float* v, float lr, float b1, float b2, float eps,
                       float c1, float c2) {
    const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= n) return;
    const float gi = g[i];
    const float mi = b1 * m[i] + (1.f - b1) * gi;
    const float vi = b2 * v[i] + (1.f - b2) * gi * gi;
    m[i] = mi;
    v[i] = vi;
    w[i] -= lr * (mi / c1) / (sqrtf(vi / c2) + eps);
}

// MSE over the 3 used output channels: dy = 2 (y - t) / (3 NVOX); per-block loss partials
__global__ void k_mse(const float* y, const float* tgt, float* dy, float* part) {
    __shared__ float sh[256];
    const int p = blockIdx.x * blockDim.x + threadIdx.x;
    float s = 0.f;
    if (p < NVOX)
        for (int c = 0; c < 16; ++c) {
            float d = 0.f;
            if (c < OUT_CH) {
                d = y[(size_t)p * 16 + c] - tgt[(size_t)p * OUT_CH + c];
                s += d * d;
            }
            dy[(size_t)p * 16 + c] = c < OUT_CH ? 2.f * d / (3.f * NVOX) : 0.f;
        }
    sh[threadIdx.x] = s;
    __syncthreads();
    for (int w = blockDim.x / 2; w > 0; w >>= 1) {
        if ((int)threadIdx.x < w) sh[threadIdx.x] += sh[threadIdx.x + w];
        __syncthreads();
    }
    if (threadIdx.x == 0) part[blockIdx.x] = sh[0];
}

}  // namespace pgfn

// ===========================================================================
// Host side
// ===========================================================================
using namespace pgfn;

#define NCHK(x)                                                                      \
    do {                                                                             \
        hipError_t e_ = (x);                                                         \
        if (e_ != hipSuccess) throw std::string("HIP error: ") + hipGetErrorString(e_); \
    } while (0)

struct pgf_net {
    std::string err;
    hipStream_t stream = nullptr;
    pgfd::HostCopy copy;
    int64_t n_params = 0;
    int64_t w_off[N_LAYERS], b_off[N_LAYERS];
    float *params = nullptr, *grads = nullptr, *adam_m = nullptr, *adam_v = nullptr;
    bf16 *Bf[N_LAYERS] = {}, *Bd[N_LAYERS] = {};
    // activations (bf16), layer outputs a1..a7, input x, final y (fp32)
    bf16* act[N_LAYERS] = {};  // act[l] = output of layer l (l < 7); act input separately
    bf16* x = nullptr;
    float* y = nullptr;
    float* gbuf[N_LAYERS] = {};  // gradient behind the ReLU, FP32 where a skip connection needs it
    bf16* gbf[N_LAYERS] = {};
    float* part = nullptr;       // weight-gradient partials, layer after layer
    size_t part_off[N_LAYERS];
    float* lossp = nullptr;
    float* bpart = nullptr;  // bias-gradient partials
    float* io = nullptr;     // [NVOX][8] staging of host inputs and outputs
    float* dy = nullptr;
    // dataset on the device
    std::vector<bf16*> ds_x;
    std::vector<float*> ds_t;
    int64_t step = 0;
    ~pgf_net();
};

static int64_t act_count(int l) {
    const int d = dout_of(SPECS[l].mode, SPECS[l].din);
    return (int64_t)d * d * d * SPECS[l].cout;
}

template <typename T>
static T* nalloc(size_t n) {
    void* p = nullptr;
    NCHK(hipMalloc(&p, sizeof(T) * (n ? n : 1)));
    return (T*)p;
}

pgf_net::~pgf_net() {
    void* ptrs[] = {params, grads, adam_m, adam_v, x, y, part, lossp, dy, bpart, io};
    for (void* p : ptrs)
        if (p) (void)hipFree(p);
    for (int l = 0; l < N_LAYERS; ++l) {
        void* q[] = {Bf[l], Bd[l], act[l], gbuf[l], gbf[l]};
        for (void* p : q)
            if (p) (void)hipFree(p);
    }
    for (auto p : ds_x) (void)hipFree(p);
    for (auto p : ds_t) (void)hipFree(p);
    if (stream) (void)hipStreamDestroy(stream);
}

static std::string g_net_err;

// One of the layer forms, both ways; returns the rows of bias partials that the
// data gradient leaves.  Four lines per block: 9.2, 20, 10.8 us for the first
// three below, against 10.9, 20, 12.9 with two and 9.6, 21, 10.4 with eight.
// Two channel tiles per wavefront for down_fine, 4.8 us against 5.3, one where
// two leave half the chip's wavefront slots empty.
template <int C, int N, int D, int YB>
static int conv3(pgf_net* net, const ConvArgs& a) {
    constexpr int rows = D / YB * D;
    static_assert(rows * N <= BIAS_PART, "the layer's bias partials fit their place");
    const dim3 grid(rows * (N / 16));
    if (!a.act) hipLaunchKernelGGL((k_conv3<false, C, N, D, YB>), grid, dim3(256), 0, net->stream, a);
    // (the network's input has no gradient)
    else if constexpr (C != IN_CH) hipLaunchKernelGGL((k_conv3<true, C, N, D, YB>), grid, dim3(256), 0, net->stream, a);
    NCHK(hipGetLastError());
    return rows;
}
template <int MODE, int C, int N, int DIN, int NT>
static int conv2(pgf_net* net, const ConvArgs& a) {
    constexpr int S = MODE == DOWN ? DIN / 2 : DIN;
    constexpr int rows = S * S * S / 64 * (MODE == UP ? 4 : 1);
    static_assert(rows * N <= BIAS_PART, "the layer's bias partials fit their place");
    const dim3 grid(rows * (N / (16 * NT)));
    if (a.act) hipLaunchKernelGGL((k_conv2<true, MODE, C, N, DIN, NT>), grid, dim3(256), 0, net->stream, a);
    else hipLaunchKernelGGL((k_conv2<false, MODE, C, N, DIN, NT>), grid, dim3(256), 0, net->stream, a);
    NCHK(hipGetLastError());
    return rows;
}
static int conv_first(pgf_net* net, const ConvArgs& a) { return conv3<IN_CH, 16, GRID, 4>(net, a); }
static int conv_fine(pgf_net* net, const ConvArgs& a) { return conv3<16, 16, GRID, 4>(net, a); }
static int conv_mid(pgf_net* net, const ConvArgs& a) { return conv3<32, 32, GRID / 2, 4>(net, a); }
static int conv_coarse(pgf_net* net, const ConvArgs& a) { return conv3<64, 64, GRID / 4, 4>(net, a); }
static int down_fine(pgf_net* net, const ConvArgs& a) { return conv2<DOWN, 16, 32, GRID, 2>(net, a); }
static int down_mid(pgf_net* net, const ConvArgs& a) { return conv2<DOWN, 32, 64, GRID / 2, 1>(net, a); }
static int up_coarse(pgf_net* net, const ConvArgs& a) { return conv2<UP, 64, 32, GRID / 4, 1>(net, a); }
static int up_mid(pgf_net* net, const ConvArgs& a) { return conv2<UP, 32, 16, GRID / 2, 1>(net, a); }

// blocks of a weight gradient: tile pairs times chunks of its stages (about 512,
// two per CU)
struct WgShape {
    int tiles, chunks, stages;
};
static WgShape wgrad_shape(int l) {
    const LayerSpec& s = SPECS[l];
    const int h = s.mode == UP ? s.din : dout_of(s.mode, s.din);  // positions of the sum: the coarser grid
    const int tiles = std::max(s.cin / 16, 1) * (s.cout / 16), stages = h * h * h / WG_POS;
    const int per = std::max(1, tiles * stages / 512);
    return {tiles, stages / per, per};
}

// layer l's partials, from its input; k_wgrad_reduce adds them up
static void launch_wgrad(pgf_net* net, int l, const bf16* in) {
    const WgShape w = wgrad_shape(l);
    const WgArgs a{w.stages, in, net->gbf[l], net->part + net->part_off[l]};
    const dim3 grid(w.tiles * w.chunks);
    hipStream_t st = net->stream;
    switch (l) {
        case 0: hipLaunchKernelGGL((k_wgrad3<8, 16, GRID>), grid, dim3(192), 0, st, a); break;
        case 1: hipLaunchKernelGGL((k_wgrad2<16, 32, GRID / 2, false>), grid, dim3(256), 0, st, a); break;
        case 2: hipLaunchKernelGGL((k_wgrad3<32, 32, GRID / 2>), grid, dim3(192), 0, st, a); break;
        case 3: hipLaunchKernelGGL((k_wgrad2<32, 64, GRID / 4, false>), grid, dim3(256), 0, st, a); break;
        case 4: hipLaunchKernelGGL((k_wgrad3<64, 64, GRID / 4>), grid, dim3(192), 0, st, a); break;
        case 5: hipLaunchKernelGGL((k_wgrad2<32, 64, GRID / 4, true>), grid, dim3(256), 0, st, a); break;
        case 6: hipLaunchKernelGGL((k_wgrad2<16, 32, GRID / 2, true>), grid, dim3(256), 0, st, a); break;
        default: hipLaunchKernelGGL((k_wgrad3<16, 16, GRID>), grid, dim3(192), 0, st, a); break;
    }
    NCHK(hipGetLastError());
}

static void refresh_bf16(pgf_net* net) {
    for (int l = 0; l < N_LAYERS; ++l) {
        const LayerSpec& s = SPECS[l];
        const int n = taps(s.mode) * s.cin * s.cout;
        hipLaunchKernelGGL(k_weights_bf16, dim3((n + 255) / 256), dim3(256), 0, net->stream, s.mode, taps(s.mode), s.cin,
                           s.cout, (const float*)(net->params + net->w_off[l]), net->Bf[l], net->Bd[l]);
    }
    NCHK(hipGetLastError());
}

static void forward(pgf_net* net, const bf16* x) {
    auto& act = net->act;
    // a1 .. a7
    auto args = [&](int l, const bf16* in, const bf16* skip) {
        return ConvArgs{in, net->Bf[l], l < 7 ? act[l] : nullptr, l < 7 ? nullptr : net->y, net->params + net->b_off[l],
                        skip, l < 7, nullptr, nullptr, nullptr};
    };
    conv_first(net, args(0, x, nullptr));
    down_fine(net, args(1, act[0], nullptr));
    conv_mid(net, args(2, act[1], nullptr));
    down_mid(net, args(3, act[2], nullptr));
    conv_coarse(net, args(4, act[3], nullptr));
    up_coarse(net, args(5, act[4], act[2]));
    up_mid(net, args(6, act[5], act[0]));
    conv_fine(net, args(7, act[6], nullptr));
}

// gradients of sum(dy . y) with respect to every parameter, dy [NVOX][16] FP32 on the device
static void backward(pgf_net* net, const bf16* x, const float* dy) {
    float* G = net->grads;
    auto& act = net->act;
    BiasLayers b;
    // g7 = dy (the output layer has no ReLU)
    b.blocks[7] = RB_BLOCKS;
    hipLaunchKernelGGL(k_out_back, dim3(RB_BLOCKS), dim3(256), 0, net->stream, act_count(7) / 4, SPECS[7].cout,
                       (const float4*)dy, (ushort4*)net->gbf[7], net->bpart + (size_t)7 * BIAS_PART);
    NCHK(hipGetLastError());
    // the gradient of layer l's output, from layer l + 1's: + that of a skip
    // connection (FP32, of the layer it leads to), behind layer l's ReLU
    auto args = [&](int l, const float* add) {
        return ConvArgs{net->gbf[l + 1], net->Bd[l + 1], net->gbf[l], net->gbuf[l], nullptr, nullptr, 0, add, act[l],
                        net->bpart + (size_t)l * BIAS_PART};
    };
    launch_wgrad(net, 7, act[6]);
    b.blocks[6] = conv_fine(net, args(6, nullptr));  // layer 6: up2 into a7, skip from a1
    launch_wgrad(net, 6, act[5]);
    b.blocks[5] = down_fine(net, args(5, nullptr));  // up2^T, down form
    launch_wgrad(net, 5, act[4]);
    b.blocks[4] = down_mid(net, args(4, nullptr));
    launch_wgrad(net, 4, act[3]);
    b.blocks[3] = conv_coarse(net, args(3, nullptr));
    launch_wgrad(net, 3, act[2]);
    b.blocks[2] = up_coarse(net, args(2, net->gbuf[5]));  // down2^T, up form; skip into a6
    launch_wgrad(net, 2, act[1]);
    b.blocks[1] = conv_mid(net, args(1, nullptr));
    launch_wgrad(net, 1, act[0]);
    b.blocks[0] = up_mid(net, args(0, net->gbuf[6]));  // skip into a7
    launch_wgrad(net, 0, x);
    WgLayers w;
    w.first[0] = 0;
    for (int l = 0; l < N_LAYERS; ++l) {
        const LayerSpec& s = SPECS[l];
        w.chunks[l] = wgrad_shape(l).chunks;
        w.N[l] = b.N[l] = s.cout;
        w.TC[l] = taps(s.mode) * s.cin;
        w.part[l] = net->part + net->part_off[l];
        w.gW[l] = G + net->w_off[l];
        w.first[l + 1] = w.first[l] + (s.cout * w.TC[l] + 31) / 32;
        b.gb[l] = G + net->b_off[l];
    }
    hipLaunchKernelGGL(k_wgrad_reduce, dim3(w.first[N_LAYERS]), dim3(256), 0, net->stream, w);
    NCHK(hipGetLastError());
    hipLaunchKernelGGL(k_bias_reduce, dim3(N_LAYERS), dim3(1024), 0, net->stream, (const float*)net->bpart, b);
    NCHK(hipGetLastError());
}

template <typename F>
static int nguard(pgf_net* net, F&& f) {
    try {
        f();
        return 0;
    } catch (const std::string& s) {
        if (net) net->err = s;
        else g_net_err = s;
        return PGF_EDEVICE;
    }
}

// host input to bf16 on the device (the upload is FP32, the rounding f2bf's)
static void upload_x(pgf_net* net, const float* xh, bf16* dst) {
    const int64_t n = (int64_t)NVOX * IN_CH;
    NCHK(hipMemcpyAsync(net->io, xh, sizeof(float) * n, hipMemcpyHostToDevice, net->stream));
    hipLaunchKernelGGL(k_to_bf16, dim3((unsigned)((n + 255) / 256)), dim3(256), 0, net->stream, n, (const float*)net->io, dst);
    NCHK(hipGetLastError());
}

extern "C" {

PGF_API int pgf_net_create(uint64_t seed, pgf_net** out) {
    if (!out) return PGF_EARG;
    pgf_net* net = new pgf_net();
    int rc = nguard(nullptr, [&]() {
        NCHK(hipStreamCreateWithFlags(&net->stream, hipStreamNonBlocking));
        int64_t off = 0;
        for (int l = 0; l < N_LAYERS; ++l) {
            const LayerSpec& s = SPECS[l];
            net->w_off[l] = off;
            off += (int64_t)taps(s.mode) * s.cin * s.cout;
            net->b_off[l] = off;
            off += s.cout;
        }
        net->n_params = off;
        // He-normal initialisation from a fixed 64-bit LCG + Box-Muller; biases 0
        std::vector<float> h(off, 0.f);
        uint64_t st = seed * 6364136223846793005ull + 1442695040888963407ull;
        auto uni = [&]() {
            st = st * 6364136223846793005ull + 1442695040888963407ull;
            return ((st >> 11) + 0.5) * (1.0 / 9007199254740992.0);
        };
        for (int l = 0; l < N_LAYERS; ++l) {
            const LayerSpec& s = SPECS[l];
            const int fan_in = (s.mode == UP ? 1 : taps(s.mode)) * s.cin;
            const double sd = std::sqrt(2.0 / fan_in) * (l == N_LAYERS - 1 ? 0.1 : 1.0);
            for (int64_t i = 0; i < (int64_t)taps(s.mode) * s.cin * s.cout; ++i) {
                const double u1 = uni(), u2 = uni();
                h[net->w_off[l] + i] = (float)(sd * std::sqrt(-2.0 * std::log(u1)) * std::cos(6.283185307179586 * u2));
            }
        }
        net->params = nalloc<float>(off);
        net->grads = nalloc<float>(off);
        net->adam_m = nalloc<float>(off);
        net->adam_v = nalloc<float>(off);
        NCHK(hipMemcpy(net->params, h.data(), sizeof(float) * off, hipMemcpyHostToDevice));
        NCHK(hipMemset(net->adam_m, 0, sizeof(float) * off));
        NCHK(hipMemset(net->adam_v, 0, sizeof(float) * off));
        NCHK(hipMemset(net->grads, 0, sizeof(float) * off));
        size_t part = 0;
        for (int l = 0; l < N_LAYERS; ++l) {
            const LayerSpec& s = SPECS[l];
            const int T = taps(s.mode);
            const int nf = frag_count(s.cout, T * s.cin), nd = frag_count(s.cin, T * s.cout);
            net->Bf[l] = nalloc<bf16>(nf);
            net->Bd[l] = nalloc<bf16>(nd);
            // the padding stays zero
            NCHK(hipMemsetAsync(net->Bf[l], 0, sizeof(bf16) * nf, net->stream));
            NCHK(hipMemsetAsync(net->Bd[l], 0, sizeof(bf16) * nd, net->stream));
            net->act[l] = nalloc<bf16>(act_count(l));
            if (l == 5 || l == 6) net->gbuf[l] = nalloc<float>(act_count(l));  // skip connections
            net->gbf[l] = nalloc<bf16>(act_count(l));
            net->part_off[l] = part;
            part += (size_t)wgrad_shape(l).chunks * s.cout * T * s.cin;
        }
        net->part = nalloc<float>(part);
        net->x = nalloc<bf16>((size_t)NVOX * IN_CH);
        net->y = nalloc<float>((size_t)NVOX * 16);
        net->dy = nalloc<float>((size_t)NVOX * 16);
        net->lossp = nalloc<float>(NVOX / 256);
        net->bpart = nalloc<float>((size_t)N_LAYERS * BIAS_PART);
        net->io = nalloc<float>((size_t)NVOX * IN_CH);
        refresh_bf16(net);
        NCHK(hipStreamSynchronize(net->stream));
    });
    if (rc) {
        delete net;
        return rc;
    }
    *out = net;
    return 0;
}

PGF_API void pgf_net_destroy(pgf_net* net) { delete net; }

PGF_API const char* pgf_net_last_error(const pgf_net* net) { return net ? net->err.c_str() : g_net_err.c_str(); }

PGF_API int pgf_net_num_params(pgf_net* net, int64_t* n) {
    if (!net || !n) return PGF_EARG;
    *n = net->n_params;
    return 0;
}

PGF_API int pgf_net_get_params(pgf_net* net, float* w) {
    if (!net || !w) return PGF_EARG;
    return nguard(net, [&]() { NCHK(net->copy.down(w, net->params, sizeof(float) * net->n_params, net->stream)); });
}

PGF_API int pgf_net_set_params(pgf_net* net, const float* w) {
    if (!net || !w) return PGF_EARG;
    return nguard(net, [&]() {
        NCHK(hipMemcpy(net->params, w, sizeof(float) * net->n_params, hipMemcpyHostToDevice));
        refresh_bf16(net);
        NCHK(hipStreamSynchronize(net->stream));
    });
}

PGF_API int pgf_net_forward(pgf_net* net, const float* x, float* y) {
    if (!net || !x || !y) return PGF_EARG;
    return nguard(net, [&]() {
        upload_x(net, x, net->x);
        forward(net, net->x);
        hipLaunchKernelGGL(k_pick_out, dim3(NVOX / 256), dim3(256), 0, net->stream, (const float*)net->y, net->io);
        NCHK(hipGetLastError());
        NCHK(net->copy.down(y, net->io, sizeof(float) * NVOX * OUT_CH, net->stream));
    });
}

PGF_API int pgf_net_backward(pgf_net* net, const float* x, const float* dy, float* grads) {
    if (!net || !x || !dy || !grads) return PGF_EARG;
    return nguard(net, [&]() {
        upload_x(net, x, net->x);
        forward(net, net->x);
        NCHK(hipMemcpyAsync(net->io, dy, sizeof(float) * NVOX * OUT_CH, hipMemcpyHostToDevice, net->stream));
        hipLaunchKernelGGL(k_widen_out, dim3(NVOX / 64), dim3(256), 0, net->stream, (const float*)net->io, net->dy);
        NCHK(hipGetLastError());
        backward(net, net->x, net->dy);
        NCHK(net->copy.down(grads, net->grads, sizeof(float) * net->n_params, net->stream));
    });
}

PGF_API int pgf_net_add_sample(pgf_net* net, const float* x, const float* t) {
    if (!net || !x || !t) return PGF_EARG;
    return nguard(net, [&]() {
        bf16* dx = nalloc<bf16>((size_t)NVOX * IN_CH);
        float* dt = nalloc<float>((size_t)NVOX * OUT_CH);
        net->ds_x.push_back(dx);
        net->ds_t.push_back(dt);
        upload_x(net, x, dx);
        NCHK(hipMemcpyAsync(dt, t, sizeof(float) * NVOX * OUT_CH, hipMemcpyHostToDevice, net->stream));
        NCHK(hipStreamSynchronize(net->stream));
    });
}

PGF_API int pgf_net_num_samples(pgf_net* net, int32_t* n) {
    if (!net || !n) return PGF_EARG;
    *n = (int32_t)net->ds_x.size();
    return 0;
}

// `epochs` passes over the device dataset in sample order, one Adam step per
// sample; loss[e] = mean MSE of epoch e (before each step's update)
PGF_API int pgf_net_train(pgf_net* net, int32_t epochs, float lr, float* loss) {
    if (!net || epochs < 0) return PGF_EARG;
    if (net->ds_x.empty()) return PGF_ESTATE;
    return nguard(net, [&]() {
        const int nb = NVOX / 256;
        std::vector<float> lp(nb);
        for (int e = 0; e < epochs; ++e) {
            double tot = 0.0;
            for (size_t s = 0; s < net->ds_x.size(); ++s) {
                forward(net, net->ds_x[s]);
                hipLaunchKernelGGL(k_mse, dim3(nb), dim3(256), 0, net->stream, (const float*)net->y,
                                   (const float*)net->ds_t[s], net->dy, net->lossp);
                backward(net, net->ds_x[s], net->dy);
                ++net->step;
                const float b1 = 0.9f, b2 = 0.999f;
                const float c1 = 1.f - std::pow(b1, (float)net->step), c2 = 1.f - std::pow(b2, (float)net->step);
                hipLaunchKernelGGL(k_adam, dim3((unsigned)((net->n_params + 255) / 256)), dim3(256), 0, net->stream,
                                   net->n_params, net->params, (const float*)net->grads, net->adam_m, net->adam_v, lr, b1, b2,
                                   1e-8f, c1, c2);
                refresh_bf16(net);
                NCHK(hipMemcpyAsync(lp.data(), net->lossp, sizeof(float) * nb, hipMemcpyDeviceToHost, net->stream));
                NCHK(hipStreamSynchronize(net->stream));
                double s2 = 0.0;
                for (float v : lp) s2 += v;
                tot += s2 / (3.0 * NVOX);
            }
            if (loss) loss[e] = (float)(tot / net->ds_x.size());
        }
    });
}

}  // extern "C"

// ===========================================================================
// Learned initial guess inside the Newton step
// ===========================================================================
#include "pgf_device.hpp"

namespace pgfn {

// voxel of a point of the box [lo, lo + ext)
__device__ inline int vox_of(const double* X, int64_t n_all, int64_t node, const double* lo, const double* ext) {
    int v[3];
    for (int d = 0; d < 3; ++d) {
        int i = (int)floor((X[d * n_all + node] - lo[d]) / ext[d] * GRID);
        v[d] = i < 0 ? 0 : (i >= GRID ? GRID - 1 : i);
    }
    return (v[2] * GRID + v[1]) * GRID + v[0];
}

struct Box {
    double lo[3], ext[3];
};

__global__ void k_node_vox(int64_t n_all, const double* X, Box b, int32_t* node_vox) {
    const int64_t n = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (n < n_all) node_vox[n] = vox_of(X, n_all, n, b.lo, b.ext);
}

// cohesive point -> voxel of its cut element's centroid (regular slots 0..3)
__global__ void k_cpt_vox(int64_t n_cut, int dim, int64_t n_all, const double* X, const int32_t* ce_nodes, const int64_t* cpt_ptr,
                          Box b, int32_t* cpt_vox) {
    const int64_t c = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (c >= n_cut) return;
    const int nv = dim == 2 ? 4 : 4;
    int v[3] = {0, 0, 0};
    for (int d = 0; d < dim; ++d) {
        double s = 0.0;
        for (int k = 0; k < nv; ++k) s += X[d * n_all + ce_nodes[c * 16 + k]];
        int i = (int)floor((s / nv - b.lo[d]) / b.ext[d] * GRID);
        v[d] = i < 0 ? 0 : (i >= GRID ? GRID - 1 : i);
    }
    const int vox = (v[2] * GRID + v[1]) * GRID + v[0];
    for (int64_t q = cpt_ptr[c]; q < cpt_ptr[c + 1]; ++q) cpt_vox[q] = vox;
}

__global__ void k_feat_init(const float* ind, float* feat, float* cnt) {
    const int v = blockIdx.x * blockDim.x + threadIdx.x;
    if (v >= NVOX) return;
    feat[(size_t)v * IN_CH + 0] = ind ? ind[v] : 0.f;
    for (int c = 1; c < IN_CH; ++c) feat[(size_t)v * IN_CH + c] = 0.f;
    cnt[v] = 0.f;
}

// damage channel: max over the voxel's cohesive points of delta_max / delta_c
__global__ void k_feat_damage(int64_t n_cpt, const int32_t* cpt_vox, const double* dmax, const int32_t* cpt_law,
                              const pgfk::CohParams* laws, float* feat) {
    const int64_t q = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (q >= n_cpt) return;
    const float val = (float)(dmax[q] / laws[cpt_law[q]].dc);
    // non-negative floats order like their bit patterns
    atomicMax(reinterpret_cast<int*>(&feat[(size_t)cpt_vox[q] * IN_CH + 1]), __float_as_int(val > 0.f ? val : 0.f));
}

// residual channels: sum of the free-dof residual of the nodes in each voxel
__global__ void k_feat_res(int64_t nf, int64_t n_all, const int64_t* free_slot, const double* r, const int32_t* node_vox,
                           float* feat) {
    const int64_t f = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (f >= nf) return;
    const int64_t s = free_slot[f];
    const int d = (int)(s / n_all);
    atomicAdd(&feat[(size_t)node_vox[s - d * n_all] * IN_CH + 2 + d], (float)r[f]);
}

// averaged nodal field a - b (or a alone when b is null) into channels ch..ch+dim-1
__global__ void k_feat_nodal(int64_t n_all, int dim, const double* a, const double* b, const int32_t* node_vox, float* out,
                             int ld, int ch, float* cnt) {
    const int64_t n = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (n >= n_all) return;
    const int v = node_vox[n];
    for (int d = 0; d < dim; ++d) {
        const double x = a[d * n_all + n] - (b ? b[d * n_all + n] : 0.0);
        atomicAdd(&out[(size_t)v * ld + ch + d], (float)x);
    }
    atomicAdd(&cnt[v], 1.f);
}

__global__ void k_feat_avg(float* out, int ld, int ch, int nc, const float* cnt) {
    const int v = blockIdx.x * blockDim.x + threadIdx.x;
    if (v >= NVOX) return;
    const float c = cnt[v];
    for (int k = 0; k < nc; ++k) out[(size_t)v * ld + ch + k] = c > 0.f ? out[(size_t)v * ld + ch + k] / c : 0.f;
}

// sum of squares of channels ch..ch+nc-1 (one double per block)
__global__ void k_sumsq(const float* x, int ld, int ch, int nc, double* part) {
    __shared__ double sh[256];
    double s = 0.0;
    for (int v = blockIdx.x * blockDim.x + threadIdx.x; v < NVOX; v += gridDim.x * blockDim.x)
        for (int k = 0; k < nc; ++k) {
            const double t = x[(size_t)v * ld + ch + k];
            s += t * t;
        }
    sh[threadIdx.x] = s;
    __syncthreads();
    for (int w = blockDim.x / 2; w > 0; w >>= 1) {
        if ((int)threadIdx.x < w) sh[threadIdx.x] += sh[threadIdx.x + w];
        __syncthreads();
    }
    if (threadIdx.x == 0) part[blockIdx.x] = sh[0];
}

__global__ void k_scale_ch(float* x, int ld, int ch, int nc, float s) {
    const int v = blockIdx.x * blockDim.x + threadIdx.x;
    if (v >= NVOX) return;
    for (int k = 0; k < nc; ++k) x[(size_t)v * ld + ch + k] *= s;
}

// Z columns on the free dofs: j < 3 the network output, channel j, trilinear
// at the node (cell-centred grid) on dofs of component j, zero elsewhere;
// column 3 the previous load increment.
__global__ void k_prolong(int64_t nf, int64_t n_all, const int64_t* free_slot, const double* X, Box b, const float* y,
                          int ldy, int use_net, const double* up, const double* upp, double* Z) {
    const int64_t f = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (f >= nf) return;
    const int64_t s = free_slot[f];
    const int d = (int)(s / n_all);
    const int64_t node = s - d * n_all;
    double val = 0.0;
    if (use_net && d < 3) {
        int i0[3];
        double w[3];
        for (int k = 0; k < 3; ++k) {
            double t = (X[k * n_all + node] - b.lo[k]) / b.ext[k] * GRID - 0.5;
            int i = (int)floor(t);
            if (i < 0) { i = 0; t = 0.0; }
            if (i > GRID - 2) { i = GRID - 2; t = GRID - 1; }
            i0[k] = i;
            w[k] = t - i;
        }
        for (int c = 0; c < 8; ++c) {
            const int dx = c & 1, dy = (c >> 1) & 1, dz = c >> 2;
            const double wc = (dx ? w[0] : 1.0 - w[0]) * (dy ? w[1] : 1.0 - w[1]) * (dz ? w[2] : 1.0 - w[2]);
            const int v = ((i0[2] + dz) * GRID + i0[1] + dy) * GRID + i0[0] + dx;
            val += wc * y[(size_t)v * ldy + d];
        }
    }
    for (int j = 0; j < 3; ++j) Z[j * nf + f] = (j == d) ? val : 0.0;
    Z[3 * nf + f] = up ? up[s] - upp[s] : 0.0;
}

// y = K_ff x for one of the four columns (K in FP64 or FP32, vectors FP64)
template <typename T>
__global__ void k_spmv_col(int64_t nf, const int32_t* rowptr, const int32_t* rowsplit, const int32_t* colidx, const T* K,
                           const double* x, double* y) {
    const int64_t r = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (r >= nf) return;
    double s = 0.0;
    for (int32_t j = rowptr[r]; j < rowptr[r] + rowsplit[r]; ++j) s += (double)K[j] * x[colidx[j]];
    y[r] = s;
}

// 14 dot products: G_ij = Z_i . KZ_j (i <= j, 10) and b_i = Z_i . r (4); per-block partials
constexpr int NDOT = 14;
__global__ void k_dots(int64_t nf, const double* Z, const double* KZ, const double* r, double* part) {
    __shared__ double sh[NDOT][256];
    double acc[NDOT];
    for (int k = 0; k < NDOT; ++k) acc[k] = 0.0;
    for (int64_t f = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; f < nf; f += (int64_t)gridDim.x * blockDim.x) {
        double z[4], kz[4];
        for (int j = 0; j < 4; ++j) { z[j] = Z[j * nf + f]; kz[j] = KZ[j * nf + f]; }
        int k = 0;
        for (int i = 0; i < 4; ++i)
            for (int j = i; j < 4; ++j) acc[k++] += z[i] * kz[j];
        for (int i = 0; i < 4; ++i) acc[10 + i] += z[i] * r[f];
    }
    for (int k = 0; k < NDOT; ++k) sh[k][threadIdx.x] = acc[k];
    __syncthreads();
    for (int w = blockDim.x / 2; w > 0; w >>= 1) {
        if ((int)threadIdx.x < w)
            for (int k = 0; k < NDOT; ++k) sh[k][threadIdx.x] += sh[k][threadIdx.x + w];
        __syncthreads();
    }
    if (threadIdx.x < NDOT) part[threadIdx.x * gridDim.x + blockIdx.x] = sh[threadIdx.x][0];
}

__global__ void k_combine(int64_t nf, const double* Z, double a0, double a1, double a2, double a3, double* x) {
    const int64_t f = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (f < nf) x[f] = a0 * Z[f] + a1 * Z[nf + f] + a2 * Z[2 * nf + f] + a3 * Z[3 * nf + f];
}

}  // namespace pgfn

namespace pgfd {

struct LearnState {
    pgf_net* net = nullptr;
    pgfn::Box box{};
    float* ind = nullptr;      // [NVOX] indicator
    float* feat = nullptr;     // [NVOX][8] step-start features
    float* cnt = nullptr;      // [NVOX]
    float* tgt = nullptr;      // [NVOX][3]
    int32_t* node_vox = nullptr;
    int32_t* cpt_vox = nullptr;
    double *U_prev = nullptr, *U_prevprev = nullptr, *U_start = nullptr, *U_iter = nullptr;
    int n_commits = 0;
    bool have_features = false;
    double* Z = nullptr;       // [4][n_free]
    double* KZ = nullptr;
    double* part = nullptr;    // [NDOT][DOT_BLOCKS]
    double* h_part = nullptr;
    double last_alpha[4] = {0, 0, 0, 0};
    int last_cols = 0;
    double last_ms = 0.0;
};
constexpr int DOT_BLOCKS = 512;

void learn_free(LearnState* s) {
    if (!s) return;
    void* p[] = {s->ind, s->feat, s->cnt, s->tgt, s->node_vox, s->cpt_vox, s->U_prev, s->U_prevprev, s->U_start, s->U_iter,
                 s->Z, s->KZ, s->part};
    for (void* q : p)
        if (q) (void)hipFree(q);
    if (s->h_part) (void)hipHostFree(s->h_part);
    delete s;
}

static unsigned gfor(int64_t n) { return (unsigned)((n + 255) / 256); }

// normalise channels ch..ch+nc-1 of x [NVOX][ld] to unit RMS (left as is when zero)
static void normalise(Ctx& c, LearnState& L, float* x, int ld, int ch, int nc) {
    hipLaunchKernelGGL(pgfn::k_sumsq, dim3(DOT_BLOCKS), dim3(256), 0, c.stream, (const float*)x, ld, ch, nc, L.part);
    NCHK(hipMemcpyAsync(L.h_part, L.part, sizeof(double) * DOT_BLOCKS, hipMemcpyDeviceToHost, c.stream));
    NCHK(hipStreamSynchronize(c.stream));
    double s = 0.0;
    for (int b = 0; b < DOT_BLOCKS; ++b) s += L.h_part[b];
    const double rms = std::sqrt(s / ((double)pgfn::NVOX * nc));
    if (rms > 0.0)
        hipLaunchKernelGGL(pgfn::k_scale_ch, dim3(gfor(pgfn::NVOX)), dim3(256), 0, c.stream, x, ld, ch, nc, (float)(1.0 / rms));
}

// features at the start of a load step (or of a later Newton iteration: the
// residual channels then hold that iteration's residual): indicator, damage,
// residual, previous increment
static void build_features(Ctx& c, LearnState& L, bool step_start) {
    using namespace pgfn;
    hipLaunchKernelGGL(k_feat_init, dim3(gfor(NVOX)), dim3(256), 0, c.stream, (const float*)L.ind, L.feat, L.cnt);
    if (c.n_cpt > 0)
        hipLaunchKernelGGL(k_feat_damage, dim3(gfor(c.n_cpt)), dim3(256), 0, c.stream, c.n_cpt, (const int32_t*)L.cpt_vox,
                           (const double*)c.dmax_conv, (const int32_t*)c.cpt_law, (const pgfk::CohParams*)c.laws, L.feat);
    hipLaunchKernelGGL(k_feat_res, dim3(gfor(c.n_free)), dim3(256), 0, c.stream, c.n_free, c.n_all,
                       (const int64_t*)c.free_slot, (const double*)c.r, (const int32_t*)L.node_vox, L.feat);
    if (L.n_commits >= 2) {
        hipLaunchKernelGGL(k_feat_nodal, dim3(gfor(c.n_all)), dim3(256), 0, c.stream, c.n_all, c.dim, (const double*)L.U_prev,
                           (const double*)L.U_prevprev, (const int32_t*)L.node_vox, L.feat, IN_CH, 5, L.cnt);
        hipLaunchKernelGGL(k_feat_avg, dim3(gfor(NVOX)), dim3(256), 0, c.stream, L.feat, IN_CH, 5, c.dim, (const float*)L.cnt);
    }
    NCHK(hipGetLastError());
    normalise(c, L, L.feat, IN_CH, 2, 3);
    normalise(c, L, L.feat, IN_CH, 5, 3);
    if (step_start) {
        NCHK(hipMemcpyAsync(L.U_start, c.U, sizeof(double) * c.dim * c.n_all, hipMemcpyDeviceToDevice, c.stream));
        L.have_features = true;
    }
}

bool learn_guess(Ctx& c, int use_guess, bool fp32, int it) {
    using namespace pgfn;
    LearnState& L = *c.learn;
    hipEvent_t e0, e1;
    NCHK(hipEventCreate(&e0));
    NCHK(hipEventCreate(&e1));
    NCHK(hipEventRecord(e0, c.stream));
    const bool guess = use_guess == 2 || use_guess == 3;
    if (it == 0 || (guess && use_guess == 2)) build_features(c, L, it == 0);
    // column 3: the previous load increment at iteration 0, the previous Newton
    // correction U - U_iter afterwards
    const double* c3a = nullptr;
    const double* c3b = nullptr;
    if (it == 0) {
        if (L.n_commits >= 2) { c3a = L.U_prev; c3b = L.U_prevprev; }
    } else {
        c3a = c.U;
        c3b = L.U_iter;
    }
    if (!guess) {
        NCHK(hipMemcpyAsync(L.U_iter, c.U, sizeof(double) * c.dim * c.n_all, hipMemcpyDeviceToDevice, c.stream));
        (void)hipEventDestroy(e0);
        (void)hipEventDestroy(e1);
        return false;
    }
    const bool use_net = use_guess == 2 && L.net != nullptr;
    if (use_net) {
        hipLaunchKernelGGL(k_to_bf16, dim3(gfor((int64_t)NVOX * IN_CH)), dim3(256), 0, c.stream, (int64_t)NVOX * IN_CH,
                           (const float*)L.feat, L.net->x);
        // the network runs on the solver's stream
        hipStream_t keep = L.net->stream;
        L.net->stream = c.stream;
        forward(L.net, L.net->x);
        L.net->stream = keep;
    }
    const bool have_prev = c3a != nullptr;
    const int64_t nf = c.n_free;
    hipLaunchKernelGGL(k_prolong, dim3(gfor(nf)), dim3(256), 0, c.stream, nf, c.n_all, (const int64_t*)c.free_slot,
                       (const double*)c.X, L.box, (const float*)(use_net ? L.net->y : nullptr), 16, use_net ? 1 : 0, c3a, c3b,
                       L.Z);
    NCHK(hipMemcpyAsync(L.U_iter, c.U, sizeof(double) * c.dim * c.n_all, hipMemcpyDeviceToDevice, c.stream));
    for (int j = 0; j < 4; ++j) {
        if (fp32)
            hipLaunchKernelGGL(k_spmv_col<float>, dim3(gfor(nf)), dim3(256), 0, c.stream, nf, (const int32_t*)c.rowptr,
                               (const int32_t*)c.rowsplit, (const int32_t*)c.colidx, (const float*)c.K32,
                               (const double*)(L.Z + j * nf), L.KZ + j * nf);
        else
            hipLaunchKernelGGL(k_spmv_col<double>, dim3(gfor(nf)), dim3(256), 0, c.stream, nf, (const int32_t*)c.rowptr,
                               (const int32_t*)c.rowsplit, (const int32_t*)c.colidx, (const double*)c.K,
                               (const double*)(L.Z + j * nf), L.KZ + j * nf);
    }
    hipLaunchKernelGGL(k_dots, dim3(DOT_BLOCKS), dim3(256), 0, c.stream, nf, (const double*)L.Z, (const double*)L.KZ,
                       (const double*)c.r, L.part);
    NCHK(hipGetLastError());
    NCHK(hipMemcpyAsync(L.h_part, L.part, sizeof(double) * NDOT * DOT_BLOCKS, hipMemcpyDeviceToHost, c.stream));
    NCHK(hipStreamSynchronize(c.stream));
    double d[NDOT];
    for (int k = 0; k < NDOT; ++k) {
        d[k] = 0.0;
        for (int b = 0; b < DOT_BLOCKS; ++b) d[k] += L.h_part[k * DOT_BLOCKS + b];
    }
    // Galerkin system G a = b over the usable columns (energy-optimal
    // combination: the guess never has a larger K-norm error than zero)
    double G[4][4], bb[4];
    {
        int k = 0;
        for (int i = 0; i < 4; ++i)
            for (int j = i; j < 4; ++j) G[i][j] = G[j][i] = d[k++];
        for (int i = 0; i < 4; ++i) bb[i] = d[10 + i];
    }
    bool act[4];
    double gmax = 0.0;
    for (int i = 0; i < 4; ++i) gmax = std::max(gmax, G[i][i]);
    for (int i = 0; i < 4; ++i) act[i] = gmax > 0.0 && G[i][i] > 1e-14 * gmax && (i < 3 ? use_net : have_prev);
    double alpha[4] = {0, 0, 0, 0};
    for (int attempt = 0; attempt < 4; ++attempt) {
        // Cholesky on the active set; a small pivot drops that column
        int idx[4], m = 0;
        for (int i = 0; i < 4; ++i)
            if (act[i]) idx[m++] = i;
        if (m == 0) break;
        double Lm[4][4] = {}, y[4];
        int drop = -1;
        for (int i = 0; i < m && drop < 0; ++i) {
            for (int j = 0; j <= i; ++j) {
                double s = G[idx[i]][idx[j]];
                for (int k = 0; k < j; ++k) s -= Lm[i][k] * Lm[j][k];
                if (i == j) {
                    if (s <= 1e-10 * G[idx[i]][idx[i]]) { drop = idx[i]; break; }
                    Lm[i][i] = std::sqrt(s);
                } else {
                    Lm[i][j] = s / Lm[j][j];
                }
            }
        }
        if (drop >= 0) { act[drop] = false; continue; }
        for (int i = 0; i < m; ++i) {
            double s = bb[idx[i]];
            for (int k = 0; k < i; ++k) s -= Lm[i][k] * y[k];
            y[i] = s / Lm[i][i];
        }
        for (int i = m - 1; i >= 0; --i) {
            double s = y[i];
            for (int k = i + 1; k < m; ++k) s -= Lm[k][i] * alpha[idx[k]];
            alpha[idx[i]] = s / Lm[i][i];
        }
        break;
    }
    int cols = 0;
    for (int i = 0; i < 4; ++i) cols += alpha[i] != 0.0;
    for (int i = 0; i < 4; ++i) L.last_alpha[i] = alpha[i];
    L.last_cols = cols;
    if (cols == 0) {
        (void)hipEventDestroy(e0);
        (void)hipEventDestroy(e1);
        return false;
    }
    hipLaunchKernelGGL(k_combine, dim3(gfor(nf)), dim3(256), 0, c.stream, nf, (const double*)L.Z, alpha[0], alpha[1], alpha[2],
                       alpha[3], c.guess);
    NCHK(hipEventRecord(e1, c.stream));
    NCHK(hipEventSynchronize(e1));
    float ms;
    NCHK(hipEventElapsedTime(&ms, e0, e1));
    L.last_ms = ms;
    (void)hipEventDestroy(e0);
    (void)hipEventDestroy(e1);
    return true;
}

}  // namespace pgfd

// dataset sample from device features / targets
static void net_add_device_sample(pgf_net* net, const float* feat, const float* tgt, hipStream_t st) {
    bf16* dx = nalloc<bf16>((size_t)NVOX * IN_CH);
    float* dt = nalloc<float>((size_t)NVOX * OUT_CH);
    net->ds_x.push_back(dx);
    net->ds_t.push_back(dt);
    hipLaunchKernelGGL(k_to_bf16, dim3((unsigned)(((int64_t)NVOX * IN_CH + 255) / 256)), dim3(256), 0, st,
                       (int64_t)NVOX * IN_CH, feat, dx);
    NCHK(hipMemcpyAsync(dt, tgt, sizeof(float) * NVOX * OUT_CH, hipMemcpyDeviceToDevice, st));
    NCHK(hipStreamSynchronize(st));
}

template <typename F>
static int cguard(pgfd::Ctx* c, F&& f) {
    try {
        return f();
    } catch (const std::string& s) {
        c->err = s;
        return PGF_EDEVICE;
    }
}

extern "C" {

PGF_API int pgf_learn_attach(pgf_ctx* h, pgf_net* net, const double* box, const float* indicator) {
    if (!h || !box) return PGF_EARG;
    pgfd::Ctx* c = pgfd::ctx_of(h);
    // the voxel features and the prolongation map one node per free dof;
    // periodic images share dofs at different positions
    if (c->image) {
        c->err = "the learned guess does not support periodic meshes";
        return PGF_EUNSUPPORTED;
    }
    return cguard(c, [&]() -> int {
        if (c->learn) pgfd::learn_free(c->learn);
        c->learn = nullptr;
        auto* L = new pgfd::LearnState();
        c->learn = L;
        L->net = net;
        for (int d = 0; d < 3; ++d) {
            L->box.lo[d] = box[d];
            L->box.ext[d] = box[3 + d] - box[d];
            if (!(L->box.ext[d] > 0.0)) {
                if (d < c->dim) throw std::string("learn box must have positive extent");
                L->box.ext[d] = 1.0;
            }
        }
        L->ind = nalloc<float>(NVOX);
        if (indicator) NCHK(hipMemcpy(L->ind, indicator, sizeof(float) * NVOX, hipMemcpyHostToDevice));
        else NCHK(hipMemset(L->ind, 0, sizeof(float) * NVOX));
        L->feat = nalloc<float>((size_t)NVOX * IN_CH);
        L->cnt = nalloc<float>(NVOX);
        L->tgt = nalloc<float>((size_t)NVOX * OUT_CH);
        L->node_vox = nalloc<int32_t>(c->n_all);
        L->cpt_vox = nalloc<int32_t>(std::max<int64_t>(c->n_cpt, 1));
        L->U_prev = nalloc<double>((size_t)c->dim * c->n_all);
        L->U_prevprev = nalloc<double>((size_t)c->dim * c->n_all);
        L->U_start = nalloc<double>((size_t)c->dim * c->n_all);
        L->U_iter = nalloc<double>((size_t)c->dim * c->n_all);
        L->Z = nalloc<double>((size_t)4 * c->n_free);
        L->KZ = nalloc<double>((size_t)4 * c->n_free);
        L->part = nalloc<double>((size_t)pgfn::NDOT * pgfd::DOT_BLOCKS);
        NCHK(hipHostMalloc((void**)&L->h_part, sizeof(double) * pgfn::NDOT * pgfd::DOT_BLOCKS, hipHostMallocDefault));
        hipLaunchKernelGGL(pgfn::k_node_vox, dim3(pgfd::gfor(c->n_all)), dim3(256), 0, c->stream, c->n_all, (const double*)c->X,
                           L->box, L->node_vox);
        if (c->n_cut > 0)
            hipLaunchKernelGGL(pgfn::k_cpt_vox, dim3(pgfd::gfor(c->n_cut)), dim3(256), 0, c->stream, c->n_cut, c->dim, c->n_all,
                               (const double*)c->X, (const int32_t*)c->ce_nodes, (const int64_t*)c->cpt_ptr, L->box,
                               L->cpt_vox);
        NCHK(hipGetLastError());
        // the state at attach time is the first "previous" converged field
        NCHK(hipMemcpyAsync(L->U_prev, c->U, sizeof(double) * c->dim * c->n_all, hipMemcpyDeviceToDevice, c->stream));
        L->n_commits = 1;
        NCHK(hipStreamSynchronize(c->stream));
        return 0;
    });
}

PGF_API int pgf_learn_detach(pgf_ctx* h) {
    if (!h) return PGF_EARG;
    pgfd::Ctx* c = pgfd::ctx_of(h);
    if (c->learn) pgfd::learn_free(c->learn);
    c->learn = nullptr;
    return 0;
}

// the converged U of an accepted load step (the previous increment channel)
PGF_API int pgf_learn_commit(pgf_ctx* h) {
    if (!h) return PGF_EARG;
    pgfd::Ctx* c = pgfd::ctx_of(h);
    if (!c->learn) return PGF_ESTATE;
    return cguard(c, [&]() -> int {
        pgfd::LearnState& L = *c->learn;
        const size_t n = sizeof(double) * c->dim * c->n_all;
        NCHK(hipMemcpyAsync(L.U_prevprev, L.U_prev, n, hipMemcpyDeviceToDevice, c->stream));
        NCHK(hipMemcpyAsync(L.U_prev, c->U, n, hipMemcpyDeviceToDevice, c->stream));
        NCHK(hipStreamSynchronize(c->stream));
        ++L.n_commits;
        return 0;
    });
}

// training sample from the last step: its start features and the normalised
// voxel average of the converged increment U - U_start
PGF_API int pgf_learn_record(pgf_ctx* h) {
    if (!h) return PGF_EARG;
    pgfd::Ctx* c = pgfd::ctx_of(h);
    if (!c->learn || !c->learn->net || !c->learn->have_features) return PGF_ESTATE;
    return cguard(c, [&]() -> int {
        pgfd::LearnState& L = *c->learn;
        NCHK(hipMemsetAsync(L.tgt, 0, sizeof(float) * NVOX * OUT_CH, c->stream));
        NCHK(hipMemsetAsync(L.cnt, 0, sizeof(float) * NVOX, c->stream));
        hipLaunchKernelGGL(pgfn::k_feat_nodal, dim3(pgfd::gfor(c->n_all)), dim3(256), 0, c->stream, c->n_all, c->dim,
                           (const double*)c->U, (const double*)L.U_start, (const int32_t*)L.node_vox, L.tgt, OUT_CH, 0, L.cnt);
        hipLaunchKernelGGL(pgfn::k_feat_avg, dim3(pgfd::gfor(NVOX)), dim3(256), 0, c->stream, L.tgt, OUT_CH, 0, c->dim,
                           (const float*)L.cnt);
        NCHK(hipGetLastError());
        pgfd::normalise(*c, L, L.tgt, OUT_CH, 0, 3);
        net_add_device_sample(L.net, L.feat, L.tgt, c->stream);
        return 0;
    });
}

// last guess: out[0..3] Galerkin coefficients (3 network channels, previous
// increment), out[4] number of columns used, out[5] device time of the guess (ms)
PGF_API int pgf_learn_last(pgf_ctx* h, double* out) {
    if (!h || !out) return PGF_EARG;
    pgfd::Ctx* c = pgfd::ctx_of(h);
    if (!c->learn) return PGF_ESTATE;
    for (int i = 0; i < 4; ++i) out[i] = c->learn->last_alpha[i];
    out[4] = c->learn->last_cols;
    out[5] = c->learn->last_ms;
    return 0;
}

// host copy of the last step-start features [64^3][8]
PGF_API int pgf_learn_features(pgf_ctx* h, float* out) {
    if (!h || !out) return PGF_EARG;
    pgfd::Ctx* c = pgfd::ctx_of(h);
    if (!c->learn) return PGF_ESTATE;
    return cguard(c, [&]() -> int {
        NCHK(hipMemcpy(out, c->learn->feat, sizeof(float) * NVOX * IN_CH, hipMemcpyDeviceToHost));
        return 0;
    });
}

}  // extern "C"
