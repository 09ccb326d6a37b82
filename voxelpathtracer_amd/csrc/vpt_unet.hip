// Learned denoiser: a 3-level U-Net over the tracer's 1-spp irradiance.
//
//   x (32 ch: log1p irradiance, albedo, normal, depth, zero padding)
//   e0a = relu(conv3x3(x))            32   full res
//   e0b = relu(conv3x3(e0a))          32          p0 = avgpool2(e0b)
//   e1a = relu(conv3x3(p0))           64   1/2
//   e1b = relu(conv3x3(e1a))          64          p1 = avgpool2(e1b)
//   b0  = relu(conv3x3(p1))          128   1/4
//   b1  = relu(conv3x3(b0))          128
//   d1a = relu(conv3x3(cat(up2(b1), e1b)))   64   1/2
//   d1b = relu(conv3x3(d1a))          64
//   d0a = relu(conv3x3(cat(up2(d1b), e0b)))  32   full
//   d0b = relu(conv3x3(d0a))          32
//   out = conv1x1(d0b) -> 3 (log1p irradiance; fp32)
//
// Activations are bf16 NHWC (channels a multiple of 32); weights are bf16
// [tap][cout][cin] copies of fp32 master weights; every product accumulates
// in fp32 on the MFMA units (v_mfma_f32_16x16x32_bf16).  A 3x3 convolution
// is an implicit GEMM: M = 16 output channels, N = 16 pixels of an output
// row, K = 32 input channels of one tap.  A pixel tile and its one-pixel
// halo are loaded into LDS per 32-channel slice together with the slice's
// weights for all nine taps; upsampling and concatenation are folded into
// that load, bias / ReLU / 2x2 average pooling / the output head into the
// epilogue.  vpt_unet_denoise's input has 16 stored channels (10 are used).
// The backward pass reuses the forward kernel with flipped, transposed
// weights (data gradient, ReLU mask in the epilogue) and an MFMA kernel for
// the weight gradient (K = pixels, transposing LDS reads, per-slice partials
// reduced in a fixed order, so gradients are deterministic).  Adam updates
// the fp32 master weights and refreshes the bf16 copies.
#include <hip/hip_runtime.h>
#include <math.h>
#include <string.h>

#include <algorithm>
#include <random>
#include <vector>

#include "vpt_device.h"
#include "vpt_gi.h"
#include "vpt_internal.h"

using vpt::set_error;

#define HIP_TRY(expr)                                                                          \
    do {                                                                                       \
        hipError_t e_ = (expr);                                                                \
        if (e_ != hipSuccess)                                                                  \
            return set_error(VPT_EDEVICE, "%s failed: %s", #expr, hipGetErrorString(e_));      \
    } while (0)

namespace {

typedef __attribute__((__vector_size__(8 * sizeof(__bf16)))) __bf16 bf16x8;
typedef __attribute__((__vector_size__(4 * sizeof(float)))) float f32x4;

// bf16 <-> fp32 (round to nearest even; NaN stays NaN), identical on host
// and device.
__host__ __device__ inline uint16_t f2bf(float f)
{
    uint32_t u;
    memcpy(&u, &f, 4);
    if ((u & 0x7fffffffu) > 0x7f800000u) return (uint16_t)((u >> 16) | 0x40u);
    u += 0x7fffu + ((u >> 16) & 1u);
    return (uint16_t)(u >> 16);
}

__host__ __device__ inline float bf2f(uint16_t h)
{
    uint32_t u = (uint32_t)h << 16;
    float f;
    memcpy(&f, &u, 4);
    return f;
}

// a bf16 value > 0 (the ReLU mask of a stored activation)
__device__ inline bool bf_pos(uint16_t h) { return h != 0 && !(h & 0x8000u); }

// Two bf16 values of v kept where the matching halves of m are > 0.
__device__ inline uint32_t mask_pair(uint32_t v, uint32_t m)
{
    const uint32_t lo = bf_pos((uint16_t)(m & 0xffffu)) ? (v & 0xffffu) : 0u;
    const uint32_t hi = bf_pos((uint16_t)(m >> 16)) ? (v & 0xffff0000u) : 0u;
    return lo | hi;
}

constexpr int kCi = 32;            // input channels per K slice

// What the last forward pass left in the activation buffers, written by its
// kernels, so that it also holds for replays of a captured pass.
struct LastPass {
    int x16;             // act[X] holds 16 channels per pixel (vpt_unet_denoise), not 32
    int n, h, w;         // the pass's sizes where its D0B was not stored (n = 0: it was)
    float bias[32];      // then also the last layer's parameters as the pass read them
    uint16_t w_[9 * 32 * 32];
};

struct ConvArgs {
    const uint16_t* a;   // input A, NHWC with ca channels (half resolution when a_up)
    const uint16_t* b;   // concatenated input B, NHWC with cb channels (full resolution)
    const uint16_t* w;   // [9][cout][cin] bf16
    const float* bias;   // [cout] or null
    const uint16_t* mask;// [n][h][w][cout]: y = acc where mask > 0, else 0 (no bias / ReLU)
    uint16_t* y;         // [n][h][w][cout]
    uint16_t* pool;      // [n][h/2][w/2][cout] 2x2 average of y, or null
    const uint16_t* zero;// 1 KiB of zeros (read for pixels outside the image)
    const float* head_w;  // [3][32], [3]: the 1x1 output head over y (32 channels), or null
    const float* head_b;
    float* head_out;     // [n][h][w][3]
    int head_exp;        // head_out = max(exp(.) - 1, 0)
    int ca, cb, a_up, relu;
    int a16;             // input A holds only its first 16 channels (the others are zero)
    LastPass* pass;      // the first layer notes a16 here, the last one the rest; or null
    int n, h, w_, cout;
    int near;            // 32-bit byte offsets reach over a tile's halo
};

typedef __attribute__((address_space(1))) const void GlobalPtr;
typedef __attribute__((address_space(3))) void LdsPtr;

// Two floats rounded to bf16 (nearest even, as f2bf), a in the low half.
__device__ inline uint32_t pack_bf(float a, float b)
{
    typedef __attribute__((__vector_size__(2 * sizeof(__bf16)))) __bf16 bf16x2;
    const bf16x2 v = {(__bf16)a, (__bf16)b};
    return __builtin_bit_cast(uint32_t, v);
}

// v of the other lane of each even-odd pair.
__device__ inline float next_lane(float v)
{
    return __int_as_float(__builtin_amdgcn_mov_dpp(__float_as_int(v), 0xB1, 0xF, 0xF, true));   // quad_perm [1,0,3,2]
}

// The sum of v over the lanes with the same lane % 16: v_permlane16_swap of
// v with itself leaves the even and the odd row of each pair of 16-lane rows
// in both rows, v_permlane32_swap likewise the halves.
__device__ inline float sum_rows(float v)
{
    const auto a = __builtin_amdgcn_permlane16_swap(__float_as_uint(v), __float_as_uint(v), false, false);
    v = __uint_as_float(a[0]) + __uint_as_float(a[1]);
    const auto b = __builtin_amdgcn_permlane32_swap(__float_as_uint(v), __float_as_uint(v), false, false);
    return __uint_as_float(b[0]) + __uint_as_float(b[1]);
}

// This wave's LDS reads and asynchronous loads have ended, and every wave's
// of the workgroup.  (The empty asm keeps the compiler from moving memory
// operations across.)
__device__ inline void wait_and_sync()
{
    asm volatile("" ::: "memory");
    __builtin_amdgcn_s_waitcnt(0x0070);   // vmcnt(0) lgkmcnt(0)
    __builtin_amdgcn_s_barrier();
    asm volatile("" ::: "memory");
}

// The 16-byte piece q (0..3) of the 64-byte row `row` (32 bf16 values of a
// pixel or of a weight row) lies at place (q + row / 2) % 4 of it: a 16-byte
// read of the same piece of any 16 consecutive rows is then free of bank
// conflicts (measured; q ^ (row / 2) % 4 is not for every first row).
__device__ inline int piece_place(int q, int row) { return (q + (row >> 1)) & 3; }
__device__ inline int place_piece(int place, int row) { return (place - (row >> 1)) & 3; }

// 3x3 convolution, stride 1, zero padding, as an implicit GEMM: M = 16
// output channels, N = 16 pixels of an output row, K = 32 input channels of
// one tap.  A workgroup of WR x WC waves owns a tile of WR * R rows and
// WC * 16 columns (wave (i, j): R rows, 16 columns) and is persistent: it
// walks (tile, 32-channel slice) steps, tile = blockIdx.x + k * gridDim.x.
// A step's halo slice (and, where the layer has more than one slice, its
// weight slice) is loaded straight into LDS (global_load_lds, no registers)
// while the step before is multiplied, two buffers, one barrier per step;
// pixels outside the image read p.zero.  A pixel fragment is read once per
// (halo row, dx) and multiplied into the up to three output rows that use
// it, so a step reads 3 * (R + 2) pixel fragments for 9 * R * NT products.
// The weight rows are ordered so that a lane ends with 8 consecutive
// channels of its pixel for each 32 channels: bias, ReLU, mask, 2x2 pooling
// and the 1x1 head run in registers, and a wave stores 1 KiB of consecutive
// pixels (COUT = 32), 16 bytes a lane.
// kOneSlice (32 input channels): the weights are loaded once per launch.
// kHead: the network's last convolution, with the 1x1 output head over its
// stored values in registers (p.y null: the values themselves are not
// stored).
// What bounds it at 1920x1080 (profiled): of the 32-channel layers at full
// resolution, memory where they store their activation (e0a 199 MB in 49 us,
// e0b 299 MB in 67 us, 4 to 4.5 TB/s), the epilogue in the last one, which
// with the head moves 158 MB in 76 us (2.1 TB/s); the 64-channel ones are
// held by the products' issue and what a step does between them (d1a 100 us,
// 1.15 PFLOP/s of the 2.0 that random data sustains; its two waves per SIMD
// leave the barrier together), those of two and three slices also by their
// weights, loaded again each step (d0a 136 us, 0.84 PFLOP/s).  Measured,
// whole denoise call: 1920x1080 894 -> 608
// us, 640x360 204 -> 135 us, against a kernel that staged through registers
// behind two barriers a step, read each pixel fragment for each of the three
// rows and stored through LDS, with the head and a 32-channel input apart.
// A second workgroup per CU on 16x16 tiles was slower for these layers.
template <int NT, int R, int WR, int WC, bool kOneSlice, bool kHead>
__global__ void __launch_bounds__(64 * WR * WC) conv3x3_kernel(ConvArgs p)
{
    constexpr int NW = WR * WC, COUT = NT * 16;
    // a halo row in LDS: TW + 2 pixels and 2 unused, so that a fragment's
    // address is one of two per dx plus a constant (see below)
    constexpr int TH = WR * R, TW = WC * 16, HW = TW + 4, HH = TH + 2;
    constexpr int A_LOADS = (HH * HW * 4 + 63) / 64;      // 1 KiB wave loads of the halo slice
    constexpr int B_LOADS = (9 * COUT * 4 + 63) / 64;     // of the weight slice
    constexpr int A_PER = (A_LOADS + NW - 1) / NW, B_PER = (B_LOADS + NW - 1) / NW;
    static_assert(9 * COUT * 4 % 64 == 0, "whole weight loads");
    __shared__ __attribute__((aligned(16))) uint8_t sA0[A_LOADS * 1024], sA1[A_LOADS * 1024];
    __shared__ __attribute__((aligned(16))) uint8_t sB0[B_LOADS * 1024], sB1[kOneSlice ? 16 : B_LOADS * 1024];

    const int tiles_x = (p.w_ + TW - 1) / TW, tiles_y = (p.h + TH - 1) / TH;
    const int per_img = tiles_x * tiles_y;
    const int ntiles = p.n * per_img;
    const int co0 = (int)blockIdx.y * COUT;
    const int cin = p.ca + p.cb;
    const int nch = kOneSlice ? 1 : cin / kCi;
    const int lane = (int)threadIdx.x & 63;
    const int wave = __builtin_amdgcn_readfirstlane((int)threadIdx.x >> 6);
    const int lm = lane & 15, g = lane >> 4;
    const int wr = (wave / WC) * R, wc = (wave % WC) * 16;
    if ((int)blockIdx.x >= ntiles) return;
    const int my_tiles = (ntiles - (int)blockIdx.x + (int)gridDim.x - 1) / (int)gridDim.x;
    const int nsteps = my_tiles * nch;

    // This lane's byte offsets of its halo pieces from the halo's first
    // pixel, in input A and in input B, and of its weight pieces from the
    // slice's first channel: tiles inside the image then load with a scalar
    // base and no address arithmetic.  LDS weight row tap * COUT + j * 16 +
    // m holds output channel (j / 2) * 32 + (m / 4) * 8 + (j % 2) * 4 + m % 4.
    uint32_t off_a[A_PER], off_b[kOneSlice ? 1 : A_PER], off_w[B_PER];
    uint32_t upper = 0;   // bit k: piece k lies in channels 16..31
    const int stride_a = kOneSlice && p.a16 ? 16 : p.ca;
#pragma unroll
    for (int k = 0; k < A_PER; k++) {
        const int piece = (wave + k * NW) * 64 + lane, pix = min(piece >> 2, HH * HW - 1);
        const int q = place_piece(piece & 3, piece >> 2);
        const int hy = pix / HW, hx = min(pix % HW, TW + 1);
        const int ya = p.a_up ? (hy + 1) >> 1 : hy, xa = p.a_up ? (hx + 1) >> 1 : hx;
        off_a[k] = (uint32_t)(((ya * (p.w_ >> p.a_up) + xa) * stride_a + q * 8) * 2);
        upper |= (uint32_t)(q >> 1) << k;
        if (!kOneSlice) off_b[k] = (uint32_t)(((hy * p.w_ + hx) * p.cb + q * 8) * 2);
    }
#pragma unroll
    for (int k = 0; k < B_PER; k++) {
        const int piece = (wave + k * NW) * 64 + lane, row = piece >> 2;
        const int q = place_piece(piece & 3, row);
        const int tap = row / COUT, j = row % COUT / 16, m = row % 16;
        const int co = co0 + (j >> 1) * 32 + (m >> 2) * 8 + (j & 1) * 4 + (m & 3);
        off_w[k] = (uint32_t)(((tap * p.cout + co) * cin + q * 8) * 2);
    }
    // The loads of a step, issued one by one between the products of the
    // step before (issued together they stall a wave for some 2,000
    // cycles): the addresses of this lane's halo pieces and weights.  A step
    // on the same input and tile as the one before moves on by 64 bytes
    // (p.zero has room for that); integer divisions and bounds are left to
    // the steps that begin a tile or the other input.
    const uint8_t* src_a[A_PER];
    const uint16_t* src_w = p.w;
    auto aim = [&](int t, int c) __attribute__((always_inline)) {
        src_w = p.w + c * kCi;
        if (c > 0 && c * kCi != p.ca) {
#pragma unroll
            for (int k = 0; k < A_PER; k++) src_a[k] += kCi * sizeof(uint16_t);
            return;
        }
        const int img = t / per_img, rem = t % per_img;
        const int y0 = (rem / tiles_x) * TH, x0 = (rem % tiles_x) * TW;
        const bool in_a = kOneSlice || c == 0;
        const uint16_t* src = in_a ? p.a : p.b;
        const int up = in_a ? p.a_up : 0;
        const int ch = in_a ? stride_a : p.cb, hh = p.h >> up, ww = p.w_ >> up;
        src += (size_t)img * hh * ww * ch;
        if (p.near && y0 > 0 && x0 > 0 && y0 + TH < p.h && x0 + TW < p.w_) {
            const uint8_t* base =
                reinterpret_cast<const uint8_t*>(src + ((ptrdiff_t)((y0 >> up) - 1) * ww + (x0 >> up) - 1) * ch);
#pragma unroll
            for (int k = 0; k < A_PER; k++) src_a[k] = base + (kOneSlice || in_a ? off_a[k] : off_b[kOneSlice ? 0 : k]);
        } else {
#pragma unroll
            for (int k = 0; k < A_PER; k++) {
                const int piece = (wave + k * NW) * 64 + lane, pix = piece >> 2;
                const int gy = y0 + pix / HW - 1, gx = x0 + pix % HW - 1;
                const int q = place_piece(piece & 3, pix);
                const bool in = (uint32_t)gy < (uint32_t)p.h && (uint32_t)gx < (uint32_t)p.w_ && pix < HH * HW &&
                                pix % HW < TW + 2;
                const uint16_t* at = src + ((ptrdiff_t)(gy >> up) * ww + (gx >> up)) * ch + q * 8;
                src_a[k] = reinterpret_cast<const uint8_t*>(in ? at : p.zero);
            }
        }
        if (kOneSlice && p.a16) {
            // channels 16..31 of the input are not stored: zeros
#pragma unroll
            for (int k = 0; k < A_PER; k++)
                if (upper >> k & 1) src_a[k] = reinterpret_cast<const uint8_t*>(p.zero);
        }
    };
    auto load = [&](int k, bool weights, uint8_t* la, uint8_t* lb) __attribute__((always_inline)) {
        if (k < A_PER) {
            const int i = wave + k * NW;
            if (i < A_LOADS)
                __builtin_amdgcn_global_load_lds((GlobalPtr*)src_a[k], (LdsPtr*)(la + i * 1024), 16, 0, 0);
        } else if (weights && k < A_PER + B_PER) {
            const int i = wave + (k - A_PER) * NW;
            if (i < B_LOADS)
                __builtin_amdgcn_global_load_lds(
                    (GlobalPtr*)(reinterpret_cast<const uint8_t*>(src_w) + off_w[k - A_PER]), (LdsPtr*)(lb + i * 1024),
                    16, 0, 0);
        }
    };
    auto frag = [&](const uint8_t* s, int row) __attribute__((always_inline)) {
        return *reinterpret_cast<const bf16x8*>(s + row * 64 + piece_place(g, row) * 16);
    };

    f32x4 acc[R][NT];
    constexpr bool kRegs = kOneSlice && NT == 2;   // 72 registers; 64 channels' weights stay in LDS
    bf16x8 wreg[kRegs ? 9 : 1][NT];
    // One step's products; hook(i) runs before item i's (an item: one halo
    // row and dx).  Fragments are read ahead of their use: pixel fragments
    // two items ahead, the weights of (dx, dy), which items dy .. dy + R - 1
    // of dx use, into the registers that the dx before has just left.  The
    // scheduling barriers keep the compiler from sinking the reads to the
    // products that wait for them.
    constexpr int kItems = 3 * (R + 2);
    // this lane's pixel of the wave's first halo row, for each dx and for
    // even and odd halo rows: HW / 2 = 2 (mod 4), so a piece's place moves by
    // two from row to row
    static_assert(HW % 8 == 4 && R * HW % 8 == 0, "places repeat every two halo rows");
    uint32_t pix_at[3][2];
#pragma unroll
    for (int dx = 0; dx < 3; dx++)
#pragma unroll
        for (int v = 0; v < 2; v++) {
            const int row = wr * HW + wc + lm + dx;
            pix_at[dx][v] = (uint32_t)(row * 64 + piece_place(g, row + v * HW) * 16);
        }
    auto multiply = [&](const uint8_t* sA, const uint8_t* sB, auto&& hook) __attribute__((always_inline)) {
        bf16x8 px[3], wf[kRegs ? 1 : 3][NT];
        auto pixels = [&](int i) __attribute__((always_inline)) {
            const int hy = i % (R + 2);
            return *reinterpret_cast<const bf16x8*>(sA + pix_at[i / (R + 2)][hy & 1] + hy * (HW * 64));
        };
        auto weights = [&](int dx, int dy) __attribute__((always_inline)) {
            if (kRegs || dx > 2) return;
#pragma unroll
            for (int j = 0; j < NT; j++)
                wf[kRegs ? 0 : dy][j] = frag(kOneSlice ? sB0 : sB, (dy * 3 + dx) * COUT + j * 16 + lm);
        };
        weights(0, 0);
        px[0] = pixels(0);
        px[1] = pixels(1);
        weights(0, 1);
#pragma unroll
        for (int i = 0; i < kItems; i++) {
            const int dx = i / (R + 2), hy = i % (R + 2);
            if (i + 2 < kItems) px[(i + 2) % 3] = pixels(i + 2);
            if (hy == 0) weights(dx, 2);
            if (hy == R) weights(dx + 1, 0);
            if (hy == R + 1) weights(dx + 1, 1);
            hook(i);
            __builtin_amdgcn_sched_barrier(0);
#pragma unroll
            for (int dy = 0; dy < 3; dy++) {
                const int r = hy - dy;
                if (r < 0 || r >= R) continue;
#pragma unroll
                for (int j = 0; j < NT; j++)
                    acc[r][j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(
                        kRegs ? wreg[kRegs ? dy * 3 + dx : 0][j] : wf[kRegs ? 0 : dy][j], px[i % 3], acc[r][j], 0, 0,
                        0);
            }
            __builtin_amdgcn_sched_barrier(0);
        }
    };

    // this lane's biases and head weights, read once (in each tile's finish
    // their latency was exposed)
    float bias[NT * 4], head[kHead ? 24 : 1], head_b = 0.0f;
#pragma unroll
    for (int i = 0; i < NT * 4; i++) bias[i] = p.bias ? p.bias[co0 + (i >> 3) * 32 + g * 8 + (i & 7)] : 0.0f;
    if (kHead) {
#pragma unroll
        for (int i = 0; i < (kHead ? 24 : 1); i++) head[i] = p.head_w[(i >> 3) * 32 + g * 8 + (i & 7)];
        head_b = p.head_b[min(g, 2)];
    }
    // The finished tile: its values in bf16; with 32 channels stored one by
    // one between the products of the next tile (64 channels' values would
    // not fit in the registers).
    constexpr bool kLater = NT == 2;
    constexpr int kStores = R * (NT / 2);
    uint4 out[kLater ? kStores : R];
    uint16_t* out_at = nullptr;   // this lane's first pixel and channel
    int out_rows = 0;             // its rows inside the image (0: its column is outside)
    auto store = [&](int k) __attribute__((always_inline)) {
        const int jp = k / R, r = k % R;
        if (r < out_rows && (!kHead || p.y))
            *reinterpret_cast<uint4*>(out_at + (size_t)r * p.w_ * p.cout + jp * 32) = out[kLater ? k : r];
    };
    auto finish = [&](int t) __attribute__((always_inline)) {
        const int img = t / per_img;
        const int ty0 = ((t % per_img) / tiles_x) * TH + wr, gx = ((t % per_img) % tiles_x) * TW + wc + lm;
        const size_t first = (((size_t)img * p.h + ty0) * p.w_ + gx) * p.cout + co0 + g * 8;
        out_at = p.y + first;
        out_rows = gx < p.w_ ? min(R, p.h - ty0) : 0;
#pragma unroll
        for (int jp = 0; jp < NT / 2; jp++) {
            uint4* o = out + (kLater ? jp * R : 0);
#pragma unroll
            for (int r = 0; r < R; r++) {
                float v[8];
#pragma unroll
                for (int i = 0; i < 8; i++) {
                    v[i] = acc[r][2 * jp + (i >> 2)][i & 3];
                    if (p.relu) v[i] = fmaxf(v[i] + bias[jp * 8 + i], 0.0f);
                }
                o[r] = make_uint4(pack_bf(v[0], v[1]), pack_bf(v[2], v[3]), pack_bf(v[4], v[5]), pack_bf(v[6], v[7]));
            }
            if (p.mask) {
                uint4 mk[R];
#pragma unroll
                for (int r = 0; r < R; r++)
                    mk[r] = r < out_rows ? *reinterpret_cast<const uint4*>(p.mask + first + (size_t)r * p.w_ * p.cout +
                                                                           jp * 32)
                                         : make_uint4(0u, 0u, 0u, 0u);
#pragma unroll
                for (int r = 0; r < R; r++)
                    o[r] = make_uint4(mask_pair(o[r].x, mk[r].x), mask_pair(o[r].y, mk[r].y),
                                      mask_pair(o[r].z, mk[r].z), mask_pair(o[r].w, mk[r].w));
            }
            if (kHead) {
                // the head over the stored values: 8 channels here, the
                // other 24 of the pixel in lanes +-16, +-32
#pragma unroll
                for (int r = 0; r < R; r++) {
                    const uint32_t u[4] = {o[r].x, o[r].y, o[r].z, o[r].w};
                    float s[3] = {0.0f, 0.0f, 0.0f};
#pragma unroll
                    for (int i = 0; i < 8; i++) {
                        const float v = __uint_as_float(i & 1 ? u[i >> 1] & 0xffff0000u : u[i >> 1] << 16);
#pragma unroll
                        for (int j = 0; j < 3; j++) s[j] += head[j * 8 + i] * v;
                    }
#pragma unroll
                    for (int j = 0; j < 3; j++) {
                        s[j] = sum_rows(s[j]);
                    }
                    // lane group g writes component g
                    float m = (g == 0 ? s[0] : (g == 1 ? s[1] : s[2])) + head_b;
                    if (p.head_exp) m = fmaxf(expm1f(m), 0.0f);
                    if (g < 3 && r < out_rows)
                        p.head_out[(((size_t)img * p.h + ty0 + r) * p.w_ + gx) * 3 + g] = m;
                }
            }
            if (!kLater) {
#pragma unroll
                for (int r = 0; r < R; r++) store(jp * R + r);
            }
            if (p.pool) {
                // 2x2 averages of the stored values: the right neighbour's
                // pixel is the next lane's
                const int ph = p.h >> 1, pw = p.w_ >> 1;
#pragma unroll
                for (int r = 0; r < R; r += 2) {
                    const uint32_t u[4] = {o[r].x, o[r].y, o[r].z, o[r].w};
                    const uint32_t d[4] = {o[r + 1].x, o[r + 1].y, o[r + 1].z, o[r + 1].w};
                    uint32_t q[4];
#pragma unroll
                    for (int i = 0; i < 4; i++) {
                        float s[2];
#pragma unroll
                        for (int h = 0; h < 2; h++) {
                            const float a = __uint_as_float(h ? u[i] & 0xffff0000u : u[i] << 16);
                            const float b = __uint_as_float(h ? d[i] & 0xffff0000u : d[i] << 16);
                            const float a1 = next_lane(a), b1 = next_lane(b);
                            s[h] = ((a + a1) + (b + b1)) * 0.25f;
                        }
                        q[i] = pack_bf(s[0], s[1]);
                    }
                    if ((lm & 1) == 0 && r < out_rows)
                        *reinterpret_cast<uint4*>(p.pool +
                                                  (((size_t)img * ph + ((ty0 + r) >> 1)) * pw + (gx >> 1)) * p.cout +
                                                  co0 + jp * 32 + g * 8) = make_uint4(q[0], q[1], q[2], q[3]);
                }
            }
        }
    };
    if (p.pass && blockIdx.x == 0) {
        if (!kHead) {
            if (threadIdx.x == 0) p.pass->x16 = p.a16;
        } else {
            if (threadIdx.x == 0) {
                p.pass->n = p.y ? 0 : p.n;
                p.pass->h = p.h;
                p.pass->w = p.w_;
            }
            if (!p.y) {
                if (threadIdx.x < COUT) p.pass->bias[threadIdx.x] = p.bias[threadIdx.x];
                const uint32_t* from = reinterpret_cast<const uint32_t*>(p.w);
                uint32_t* to = reinterpret_cast<uint32_t*>(p.pass->w_);
                for (int i = (int)threadIdx.x; i < 9 * COUT * kCi / 2; i += 64 * NW) to[i] = from[i];
            }
        }
    }
    {
        aim((int)blockIdx.x, 0);
#pragma unroll
        for (int k = 0; k < A_PER + B_PER; k++) load(k, true, sA0, sB0);
    }
    if (kRegs) {
        wait_and_sync();
#pragma unroll
        for (int tap = 0; tap < (kRegs ? 9 : 1); tap++)
#pragma unroll
            for (int j = 0; j < NT; j++) wreg[tap][j] = frag(sB0, tap * COUT + j * 16 + lm);
    }
    // step st: its loads have ended; between its products go the next
    // step's loads, into the other buffers, and the stores of the tile that
    // the step before finished
    int t = (int)blockIdx.x, c = 0;
    auto step = [&](int st, const uint8_t* a, const uint8_t* b, uint8_t* na, uint8_t* nb)
        __attribute__((always_inline)) {
            wait_and_sync();
            const bool more = st + 1 < nsteps, done = c == 0 && st > 0;
            const bool last = c + 1 == nch;
            if (more) aim(last ? t + (int)gridDim.x : t, last ? 0 : c + 1);
            if (done) finish(t - (int)gridDim.x);
            if (c == 0) {
#pragma unroll
                for (int r = 0; r < R; r++)
#pragma unroll
                    for (int j = 0; j < NT; j++) acc[r][j] = f32x4{0.0f, 0.0f, 0.0f, 0.0f};
            }
            multiply(a, b, [&](int i) __attribute__((always_inline)) {
                if (more) load(i, !kOneSlice, na, nb);
                if (kLater && done && i < kStores) store(i);
            });
            c = last ? 0 : c + 1;
            t = last ? t + (int)gridDim.x : t;
        };
    static_assert(A_PER + B_PER <= kItems && kStores <= kItems, "a step holds its loads and stores");
    for (int st = 0; st < nsteps; st += 2) {
        step(st, sA0, sB0, sA1, sB1);
        if (st + 1 < nsteps) step(st + 1, sA1, sB1, sA0, sB0);
    }
    finish(t - (int)gridDim.x);
    if (kLater) {
#pragma unroll
        for (int k = 0; k < kStores; k++) store(k);
    }
}

typedef short s16x4 __attribute__((ext_vector_type(4)));
typedef __attribute__((address_space(3))) s16x4 LdsS16x4;

// Weight gradient of a 3x3 convolution:
//   dW[tap][co][ci] = sum_px m[px][co] * X[px + off(tap)][ci],  db[co] = sum_px m[px][co]
// as MFMA products with K = 32 pixels of one output row.  A wave owns 32
// output x 32 input channels of all nine taps (144 accumulators); the four
// waves of a workgroup are CO x CI of them over the same pixels, times KS =
// 4 / (CO * CI) over different pixel tiles.  A tile is 4 rows x 32 columns of
// m with the 6 x 34 pixels of X around it, loaded into LDS as they lie in
// memory (a row of 64 bytes per pixel and 32 channels); ds_read_b64_tr_b16
// then gives a lane 4 pixels of its channel, so neither tile is transposed
// on the way and a dx shift is another first row.  A pixel fragment of X is
// used for the three output rows around it.  Grid: x = slices of the tiles,
// y, z = output and input channel blocks.  Each workgroup writes a partial
// [9][32 CO][32 CI] block (and the bias partial), its KS waves added in a
// fixed order, for the fixed-order reduction over slices.
// Measured at 16 x 128 x 128: all ten layers 530 -> 207 us against a kernel
// that wrote transposed, shifted copies to LDS two bytes at a time.  Bound by
// latency: a workgroup has about two tiles, one wave per SIMD (held to 256
// registers for a second workgroup per CU the 64 x 64 blocks spilled and took
// twice as long).
constexpr int kWgRows = 4, kWgPitch = 36, kWgXRows = (kWgRows + 2) * kWgPitch;
constexpr int kWgM = kWgRows * 32 * 64, kWgX = (kWgXRows * 64 + 1023) / 1024 * 1024;   // bytes per 32 channels

// Place of the 16-byte piece q of row `row`: the halves swap every 8 rows,
// so that the 8-row groups that a transposing read touches lie in different
// banks.
__device__ inline int wg_place(int q, int row) { return q ^ ((row >> 2) & 2); }

// 8 pixels (rows row0 + 8 (lane / 16) ...) of channel c0 + lane % 16 of LDS
// rows of 32 channels.
__device__ inline bf16x8 wg_frag(const uint8_t* s, int row0, int c0)
{
    const int lane = (int)threadIdx.x & 63, i = lane & 15, row = row0 + (lane >> 4) * 8 + (i >> 2);
    const int piece = (c0 >> 3) + ((i >> 1) & 1);
    union {
        s16x4 h[2];
        bf16x8 v;
    } u;
    u.h[0] = __builtin_amdgcn_ds_read_tr16_b64_v4i16(
        (LdsS16x4*)(s + row * 64 + wg_place(piece, row) * 16 + (i & 1) * 8));
    u.h[1] = __builtin_amdgcn_ds_read_tr16_b64_v4i16(
        (LdsS16x4*)(s + (row + 4) * 64 + wg_place(piece, row + 4) * 16 + (i & 1) * 8));
    return u.v;
}

template <int CO, int CI>
__global__ void __launch_bounds__(256) wgrad_kernel(ConvArgs p, const uint16_t* __restrict__ m, int cin,
                                                    float* __restrict__ part, float* __restrict__ part_b)
{
    constexpr int KS = 4 / (CO * CI);
    constexpr int STAGE = CO * kWgM + CI * kWgX;                   // one tile
    constexpr int ACC = 9 * 32 * 32 * 4;                           // one wave's sums
    constexpr int BYTES = KS * STAGE > 2 * ACC || KS == 1 ? KS * STAGE : 2 * ACC;
    constexpr int LOADS = STAGE / 1024, PER = (LOADS + CO * CI - 1) / (CO * CI);
    __shared__ __attribute__((aligned(16))) uint8_t smem[BYTES];
    const int lane = (int)threadIdx.x & 63, lm = lane & 15, g = lane >> 4;
    const int wave = __builtin_amdgcn_readfirstlane((int)threadIdx.x >> 6);
    const int ks = wave / (CO * CI), sub = wave % (CO * CI), wco = sub / CI, wci = sub % CI;
    const int co0 = ((int)blockIdx.y * CO) * 32, ci0 = ((int)blockIdx.z * CI) * 32;
    const int tiles_x = (p.w_ + 31) / 32, tiles_y = (p.h + kWgRows - 1) / kWgRows;
    const int total = p.n * tiles_x * tiles_y, groups = (total + KS - 1) / KS;
    uint8_t* stage = smem + ks * STAGE;

    f32x4 acc[9][2][2], accb[2];   // [tap][ci half][co half]
#pragma unroll
    for (int t = 0; t < 9; t++)
#pragma unroll
        for (int i = 0; i < 4; i++) acc[t][i >> 1][i & 1] = f32x4{0.0f, 0.0f, 0.0f, 0.0f};
    accb[0] = accb[1] = f32x4{0.0f, 0.0f, 0.0f, 0.0f};
    bf16x8 ones;
#pragma unroll
    for (int i = 0; i < 8; i++) ones[i] = (__bf16)1.0f;

    for (int gr = (int)blockIdx.x; gr < groups; gr += (int)gridDim.x) {
        const int tile = gr * KS + ks;
        const int img = tile / (tiles_x * tiles_y), rem = tile % (tiles_x * tiles_y);
        const int y0 = rem / tiles_x * kWgRows, x0 = rem % tiles_x * 32;
        __syncthreads();   // the tile before has been read
        if (tile < total) {
#pragma unroll
            for (int k = 0; k < PER; k++) {
                const int i = sub + k * CO * CI;   // 1 KiB of the stage
                if (i >= LOADS) continue;
                const uint16_t* at = nullptr;
                if (i < CO * (kWgM / 1024)) {
                    const int piece = i % (kWgM / 1024) * 64 + lane, row = piece >> 2;
                    const int c = co0 + i / (kWgM / 1024) * 32 + wg_place(piece & 3, row) * 8;
                    const int y = y0 + (row >> 5), x = x0 + (row & 31);
                    if (y < p.h && x < p.w_) at = m + (((size_t)img * p.h + y) * p.w_ + x) * p.cout + c;
                } else {
                    const int j = i - CO * (kWgM / 1024), piece = j % (kWgX / 1024) * 64 + lane, row = piece >> 2;
                    int c = ci0 + j / (kWgX / 1024) * 32 + wg_place(piece & 3, row) * 8;
                    const int y = y0 + row / kWgPitch - 1, x = x0 + row % kWgPitch - 1;
                    if ((uint32_t)y < (uint32_t)p.h && (uint32_t)x < (uint32_t)p.w_ && row < kWgXRows) {
                        const bool in_a = c < p.ca;
                        const int up = in_a ? p.a_up : 0, ch = in_a ? p.ca : p.cb;
                        if (!in_a) c -= p.ca;
                        at = (in_a ? p.a : p.b) +
                             (((size_t)img * (p.h >> up) + (y >> up)) * (p.w_ >> up) + (x >> up)) * ch + c;
                    }
                }
                __builtin_amdgcn_global_load_lds((GlobalPtr*)(at ? at : p.zero), (LdsPtr*)(stage + i * 1024), 16, 0,
                                                 0);
            }
        }
        wait_and_sync();
        if (tile >= total) continue;
        const uint8_t* sm = stage + wco * kWgM;
        const uint8_t* sx = stage + CO * kWgM + wci * kWgX;
        bf16x8 mf[kWgRows][2];
#pragma unroll
        for (int r = 0; r < kWgRows; r++)
#pragma unroll
            for (int h = 0; h < 2; h++) mf[r][h] = wg_frag(sm, r * 32, h * 16);
#pragma unroll
        for (int hy = 0; hy < kWgRows + 2; hy++) {
#pragma unroll
            for (int dx = 0; dx < 3; dx++) {
                bf16x8 xf[2];
#pragma unroll
                for (int h = 0; h < 2; h++) xf[h] = wg_frag(sx, hy * kWgPitch + dx, h * 16);
#pragma unroll
                for (int dy = 0; dy < 3; dy++) {
                    const int r = hy - dy;
                    if (r < 0 || r >= kWgRows) continue;
#pragma unroll
                    for (int i = 0; i < 4; i++)
                        acc[dy * 3 + dx][i >> 1][i & 1] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(
                            xf[i >> 1], mf[r][i & 1], acc[dy * 3 + dx][i >> 1][i & 1], 0, 0, 0);
                }
            }
            if (hy < kWgRows && wci == 0) {
#pragma unroll
                for (int h = 0; h < 2; h++)
                    accb[h] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(ones, mf[hy][h], accb[h], 0, 0, 0);
            }
        }
    }
    // the KS waves of a channel block: ks + KS / 2 into ks, then 1 into 0
    float4* const red = reinterpret_cast<float4*>(smem);
    float* const redb = reinterpret_cast<float*>(smem);
#pragma unroll
    for (int half = KS / 2; half >= 1; half >>= 1) {
        __syncthreads();
        const int at = ((ks % half) * CO * CI + sub) * 36 * 64 + lane;
        static_assert(KS == 1 || (KS / 2) * CO * CI * 36 * 64 * 16 <= BYTES, "the sums fit in the stage's LDS");
        if (ks >= half && ks < 2 * half) {
#pragma unroll
            for (int t = 0; t < 9; t++)
#pragma unroll
                for (int i = 0; i < 4; i++) red[at + (t * 4 + i) * 64] = *reinterpret_cast<float4*>(&acc[t][i >> 1][i & 1]);
        }
        __syncthreads();
        if (ks < half) {
#pragma unroll
            for (int t = 0; t < 9; t++)
#pragma unroll
                for (int i = 0; i < 4; i++) {
                    const float4 v = red[at + (t * 4 + i) * 64];
                    acc[t][i >> 1][i & 1] += f32x4{v.x, v.y, v.z, v.w};
                }
        }
        __syncthreads();
        if (ks >= half && ks < 2 * half && wci == 0)
#pragma unroll
            for (int h = 0; h < 2; h++) redb[(((ks % half) * CO + wco) * 2 + h) * 64 + lane] = accb[h][0];
        __syncthreads();
        if (ks < half && wci == 0)
#pragma unroll
            for (int h = 0; h < 2; h++) accb[h][0] += redb[(((ks % half) * CO + wco) * 2 + h) * 64 + lane];
    }
    if (ks != 0) return;
    // products give D[ci][co]: a lane holds 4 consecutive input channels
    float* dst = part + (size_t)blockIdx.x * 9 * p.cout * cin;
#pragma unroll
    for (int t = 0; t < 9; t++)
#pragma unroll
        for (int i = 0; i < 4; i++) {
            const int co = co0 + wco * 32 + (i & 1) * 16 + lm, ci = ci0 + wci * 32 + (i >> 1) * 16 + g * 4;
            *reinterpret_cast<float4*>(dst + ((size_t)t * p.cout + co) * cin + ci) =
                *reinterpret_cast<float4*>(&acc[t][i >> 1][i & 1]);
        }
    if (blockIdx.z == 0 && wci == 0 && g == 0)
#pragma unroll
        for (int h = 0; h < 2; h++)
            part_b[(size_t)blockIdx.x * p.cout + co0 + wco * 32 + h * 16 + lm] = accb[h][0];
}

// out[i] = sum over z of part[z][i], for n values (a multiple of 4), and the
// same for a second array in the same launch (its blocks come after the
// first's).  32 groups of a block take every 32nd slice and are added in
// order, so the sum does not depend on the launch.  Reads of one value's
// slices in turn (one thread each) had taken 60 us for the 9.4 MB of a 32 ->
// 32 layer and 235 us for the head's 1,024 partials; now 5 and 7 us.
__global__ void __launch_bounds__(1024) reduce_parts_kernel(const float* __restrict__ part, int slices, int n,
                                                            float* __restrict__ out, const float* __restrict__ part2,
                                                            int n2, float* __restrict__ out2)
{
    __shared__ float4 red[32][33];
    const int blocks1 = (n / 4 + 31) / 32;
    const bool second = (int)blockIdx.x >= blocks1;
    const float* src = second ? part2 : part;
    float* dst = second ? out2 : out;
    const int len = second ? n2 : n;
    const int x = (int)threadIdx.x & 31, y = (int)threadIdx.x >> 5;
    const int i = (((int)blockIdx.x - (second ? blocks1 : 0)) * 32 + x) * 4;
    float4 s = make_float4(0.0f, 0.0f, 0.0f, 0.0f);
    if (i < len) {
#pragma unroll 8
        for (int z = y; z < slices; z += 32) {
            const float4 v = *reinterpret_cast<const float4*>(src + (size_t)z * len + i);
            s.x += v.x;
            s.y += v.y;
            s.z += v.z;
            s.w += v.w;
        }
    }
    red[y][x] = s;
    __syncthreads();
    if (y == 0 && i < len) {
        for (int k = 1; k < 32; k++) {
            const float4 v = red[k][x];
            s.x += v.x;
            s.y += v.y;
            s.z += v.z;
            s.w += v.w;
        }
        // d_g's layers start at multiples of 4 bytes only
        dst[i] = s.x;
        dst[i + 1] = s.y;
        dst[i + 2] = s.z;
        dst[i + 3] = s.w;
    }
}

// wt[tap][ci][co] = w[8 - tap][co][ci] of every layer (at the layer's own
// offset): the data gradient of a convolution is the convolution of the
// output gradient with these weights.
struct FlipLayers {
    uint32_t off[10], cout[10], cin[10];
};
__global__ void flip_transpose_kernel(const uint16_t* __restrict__ w, const FlipLayers layers,
                                      uint16_t* __restrict__ wt)
{
    const uint32_t l = blockIdx.y, cout = layers.cout[l], cin = layers.cin[l];
    const uint32_t i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= 9u * cout * cin) return;
    const uint32_t tap = i / (cout * cin), rem = i % (cout * cin), ci = rem / cout, co = rem % cout;
    wt[layers.off[l] + i] = w[layers.off[l] + ((8u - tap) * cout + co) * cin + ci];
}

// Loss and head gradient, one thread per pixel; 256-thread blocks write
// partial sums [block][100]: 96 dW, 3 db, 1 loss.
//   L = mean |pred - target|,  g = sign(pred - target) / (3 npx)
//   m_d0b[px][c] = (sum_j W[j][c] g[px][j]) where d0b > 0
__global__ void __launch_bounds__(256) head_bwd_kernel(const uint16_t* __restrict__ x, size_t npx,
                                                       const float* __restrict__ wh, const float* __restrict__ pred,
                                                       const float* __restrict__ target, uint16_t* __restrict__ m,
                                                       float* __restrict__ part)
{
    __shared__ float sv[256][33], sg[4][256], red[2][96], red4[4][16];
    const size_t i = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
    float g[3] = {0.0f, 0.0f, 0.0f}, loss = 0.0f;
    float v[32];
    const float inv = 1.0f / (3.0f * (float)npx);
    if (i < npx) {
        const uint4* src = reinterpret_cast<const uint4*>(x + i * 32);
#pragma unroll
        for (int q = 0; q < 4; q++) {
            const uint4 u = src[q];
            const uint16_t* h = reinterpret_cast<const uint16_t*>(&u);
#pragma unroll
            for (int k = 0; k < 8; k++) v[q * 8 + k] = bf2f(h[k]);
        }
#pragma unroll
        for (int j = 0; j < 3; j++) {
            const float d = pred[i * 3 + j] - target[i * 3 + j];
            loss += fabsf(d);
            g[j] = (d > 0.0f ? inv : (d < 0.0f ? -inv : 0.0f));
        }
        uint16_t out[32];
#pragma unroll
        for (int c = 0; c < 32; c++) {
            const float s = (wh[c] * g[0] + wh[32 + c] * g[1]) + wh[64 + c] * g[2];
            out[c] = v[c] > 0.0f ? f2bf(s) : (uint16_t)0;
        }
        uint4* dstm = reinterpret_cast<uint4*>(m + i * 32);
#pragma unroll
        for (int q = 0; q < 4; q++) dstm[q] = *reinterpret_cast<const uint4*>(&out[q * 8]);
    } else {
#pragma unroll
        for (int c = 0; c < 32; c++) v[c] = 0.0f;
    }
    // the block's 96 weight sums, two threads each (128 pixels), from LDS;
    // the other 64 threads take the three bias sums and the loss (16 pixels
    // each, then in order).  Wave shuffles of all 100 sums took 41 us at 16 x
    // 128 x 128, this 15.
#pragma unroll
    for (int c = 0; c < 32; c++) sv[threadIdx.x][c] = v[c];
#pragma unroll
    for (int j = 0; j < 3; j++) sg[j][threadIdx.x] = g[j];
    sg[3][threadIdx.x] = loss;
    __syncthreads();
    const int k = (int)threadIdx.x;
    if (k < 192) {
        const int c = k & 31, j = (k >> 5) % 3, h = k / 96;
        float s = 0.0f;
#pragma unroll 8
        for (int q = 0; q < 128; q++) s += sg[j][h * 128 + q] * sv[h * 128 + q][c];
        red[h][j * 32 + c] = s;
    } else {
        const int j = (k - 192) >> 4, q0 = (k & 15) * 16;
        float s = 0.0f;
#pragma unroll
        for (int q = 0; q < 16; q++) s += sg[j][q0 + q];
        red4[j][k & 15] = s;
    }
    __syncthreads();
    if (k < 96) part[(size_t)blockIdx.x * 100 + k] = red[0][k] + red[1][k];
    if (k >= 96 && k < 100) {
        float s = 0.0f;
#pragma unroll
        for (int q = 0; q < 16; q++) s += red4[k - 96][q];
        part[(size_t)blockIdx.x * 100 + k] = s;
    }
}

// Eight bf16 values as floats, and back (rounded), kept where the matching
// value of y is > 0.
__device__ inline void unpack8(const uint4& q, float v[8])
{
    const uint32_t u[4] = {q.x, q.y, q.z, q.w};
#pragma unroll
    for (int i = 0; i < 8; i++) v[i] = __uint_as_float(i & 1 ? u[i >> 1] & 0xffff0000u : u[i >> 1] << 16);
}

__device__ inline uint4 pack8_where(const float v[8], const uint4& y)
{
    return make_uint4(mask_pair(pack_bf(v[0], v[1]), y.x), mask_pair(pack_bf(v[2], v[3]), y.y),
                      mask_pair(pack_bf(v[4], v[5]), y.z), mask_pair(pack_bf(v[6], v[7]), y.w));
}

// Upsample branch of a concatenated-input gradient, 8 channels a thread:
//   out[n][y][x][c] = (sum of g[n][2y+i][2x+j][c]) where y_low > 0
// for the first c of g's cg channels.
__global__ void sum2x2_mask_kernel(const uint16_t* __restrict__ g, int cg, int c, int n, int h, int w,
                                   const uint16_t* __restrict__ ylow, uint16_t* __restrict__ out)
{
    const size_t i = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
    const int hh = h >> 1, ww = w >> 1, c8 = c >> 3;
    if (i >= (size_t)n * hh * ww * c8) return;
    const size_t px = i / c8;
    const int ch = (int)(i % c8) * 8, x = (int)(px % ww);
    const size_t row = px / ww;   // img * hh + y; the full-resolution row is 2 * row
    const uint16_t* at = g + ((2 * row * w) + 2 * x) * cg + ch;
    float v[4][8], s[8];
#pragma unroll
    for (int k = 0; k < 4; k++)
        unpack8(*reinterpret_cast<const uint4*>(at + ((size_t)(k >> 1) * w + (k & 1)) * cg), v[k]);
#pragma unroll
    for (int k = 0; k < 8; k++) s[k] = (v[0][k] + v[1][k]) + (v[2][k] + v[3][k]);
    *reinterpret_cast<uint4*>(out + i * 8) = pack8_where(s, *reinterpret_cast<const uint4*>(ylow + i * 8));
}

// Skip branch, 8 channels a thread: out = g[..][c_off + c] + 0.25
// gpool[n][y/2][x/2][c], kept where y_skip > 0.
__global__ void skip_mask_kernel(const uint16_t* __restrict__ g, int cg, int c_off, int c, int n, int h, int w,
                                 const uint16_t* __restrict__ gpool, const uint16_t* __restrict__ yskip,
                                 uint16_t* __restrict__ out)
{
    const size_t i = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
    const int c8 = c >> 3;
    if (i >= (size_t)n * h * w * c8) return;
    const size_t px = i / c8;
    const int ch = (int)(i % c8) * 8, x = (int)(px % w);
    const size_t row = px / w;   // img * h + y; h is even, so its half is the pooled row
    float s[8], q[8];
    unpack8(*reinterpret_cast<const uint4*>(g + px * cg + c_off + ch), s);
    unpack8(*reinterpret_cast<const uint4*>(gpool + ((row >> 1) * (w >> 1) + (x >> 1)) * c + ch), q);
#pragma unroll
    for (int k = 0; k < 8; k++) s[k] += 0.25f * q[k];
    *reinterpret_cast<uint4*>(out + i * 8) = pack8_where(s, *reinterpret_cast<const uint4*>(yskip + i * 8));
}

// Adam on the fp32 master parameters; refreshes the bf16 copies.
__global__ void adam_kernel(float* __restrict__ w, uint16_t* __restrict__ wb, const float* __restrict__ g,
                            float* __restrict__ m1, float* __restrict__ m2, size_t n, float lr, float b1, float b2,
                            float eps, float c1, float c2)
{
    const size_t i = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= n) return;
    const float gi = g[i];
    const float a = b1 * m1[i] + (1.0f - b1) * gi;
    const float b = b2 * m2[i] + (1.0f - b2) * gi * gi;
    m1[i] = a;
    m2[i] = b;
    const float v = w[i] - lr * (a * c1) / (sqrtf(b * c2) + eps);
    w[i] = v;
    wb[i] = f2bf(v);
}

__global__ void to_bf16_kernel(const float* __restrict__ w, uint16_t* __restrict__ wb, size_t n)
{
    const size_t i = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i < n) wb[i] = f2bf(w[i]);
}

// ---- tracer outputs -> network input / reference -------------------------

struct Decoded {
    float r, g, b;
};

// SHToIrridiance (ColorPassFrag.glsl:356-368) of SH-Y (4) + CoCg with the
// face normal, as the SVGF chain's final decode.
__device__ inline Decoded sh_decode(const float sh[4], float co, float cg, int face)
{
    const vpt::Vec3 v = vpt::face_normal(face, 1.0f);
    const float x = (sh[0] * v.x + sh[1] * v.y) + sh[2] * v.z;
    float Y = 2.0f * (1.023326f * x + 0.886226f * sh[3]);
    Y = fmaxf(Y, 0.0f);
    const float k = (Y * 0.282095f) / (sh[3] + 1e-6f);
    const float c0 = co * k, c1 = cg * k;
    const float T = Y - c1 * 0.5f;
    const float G = c1 + T;
    const float B = T - c0 * 0.5f;
    const float R = B + c0;
    return Decoded{fmaxf(R, 0.0f), fmaxf(G, 0.0f), fmaxf(B, 0.0f)};
}

__device__ inline void texel_values(const vpt_svgf_texel& t, float v[6])
{
#pragma unroll
    for (int k = 0; k < 6; k++) v[k] = vpt::hw_h2f(t.h[k]);
}

// Network input: ch 0-2 log1p(1-spp irradiance), 3-5 albedo of the hit
// block, 6-8 face normal, 9 log1p(hit distance) / 8, 10-31 zero.  Sky
// pixels: irradiance of their texel, zero albedo / normal / depth.
template <int kPieces>   // 16-byte pieces stored per pixel: 4, or 2 (channels 0..15)
__global__ void assemble_kernel(int npx, const float* __restrict__ gb_t, const uint8_t* __restrict__ gb_face,
                                const uint8_t* __restrict__ gb_block, const vpt_svgf_texel* __restrict__ tex,
                                const vpt::AlbedoTable albedo, uint16_t* __restrict__ x)
{
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= npx) return;
    float v[6];
    texel_values(tex[i], v);
    const int face = gb_face[i];
    const Decoded d = sh_decode(v, v[4], v[5], face);
    uint16_t o[8 * kPieces];
#pragma unroll
    for (int k = 0; k < 8 * kPieces; k++) o[k] = 0;
    o[0] = f2bf(log1pf(d.r));
    o[1] = f2bf(log1pf(d.g));
    o[2] = f2bf(log1pf(d.b));
    const float t = gb_t[i];
    if (t >= 0.0f && face < 6) {
        const int blk = gb_block[i] & 127;
        o[3] = f2bf(albedo.v[blk * 3]);
        o[4] = f2bf(albedo.v[blk * 3 + 1]);
        o[5] = f2bf(albedo.v[blk * 3 + 2]);
        const vpt::Vec3 nrm = vpt::face_normal(face, 0.0f);
        o[6] = f2bf(nrm.x);
        o[7] = f2bf(nrm.y);
        o[8] = f2bf(nrm.z);
        o[9] = f2bf(log1pf(t) * 0.125f);
    }
    uint4* dst = reinterpret_cast<uint4*>(x + (size_t)i * 8 * kPieces);
#pragma unroll
    for (int q = 0; q < kPieces; q++) dst[q] = *reinterpret_cast<const uint4*>(&o[q * 8]);
}

// acc[i][0..5] (+)= SH-Y, Co, Cg of texel i.
__global__ void accumulate_kernel(int npx, const vpt_svgf_texel* __restrict__ tex, int reset, float* __restrict__ acc)
{
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= npx) return;
    float v[6];
    texel_values(tex[i], v);
#pragma unroll
    for (int k = 0; k < 6; k++) acc[(size_t)i * 6 + k] = (reset ? 0.0f : acc[(size_t)i * 6 + k]) + v[k];
}

// rgb = decode of the texel (tex) or of acc * scale.
__global__ void decode_irr_kernel(int npx, const uint8_t* __restrict__ gb_face, const vpt_svgf_texel* __restrict__ tex,
                                  const float* __restrict__ acc, float scale, float* __restrict__ rgb)
{
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= npx) return;
    float v[6];
    if (tex) {
        texel_values(tex[i], v);
    } else {
#pragma unroll
        for (int k = 0; k < 6; k++) v[k] = acc[(size_t)i * 6 + k] * scale;
    }
    const Decoded d = sh_decode(v, v[4], v[5], gb_face[i]);
    rgb[(size_t)i * 3] = d.r;
    rgb[(size_t)i * 3 + 1] = d.g;
    rgb[(size_t)i * 3 + 2] = d.b;
}

// ---- network description ---------------------------------------------------

enum Buf { X, E0A, E0B, P0, E1A, E1B, P1, B0, B1, D1A, D1B, D0A, D0B, NBUF };

struct Layer {
    int in_a, in_b;   // activation buffers (in_b = -1: none)
    int a_up;         // in_a is at half resolution
    int out, pool;    // output buffer, pooled output buffer (-1: none)
    int cin, cout;
    int level;        // resolution level of the output (0 full, 1 half, 2 quarter)
    size_t w_off, b_off;
};

const int kChannels[NBUF] = {32, 32, 32, 32, 64, 64, 64, 128, 128, 64, 64, 32, 32};
const int kLevel[NBUF] = {0, 0, 0, 1, 1, 1, 2, 2, 2, 1, 1, 0, 0};
constexpr int kLayers = 10;
const Layer kNet[kLayers] = {
    {X, -1, 0, E0A, -1, 32, 32, 0, 0, 0},       {E0A, -1, 0, E0B, P0, 32, 32, 0, 0, 0},
    {P0, -1, 0, E1A, -1, 32, 64, 1, 0, 0},      {E1A, -1, 0, E1B, P1, 64, 64, 1, 0, 0},
    {P1, -1, 0, B0, -1, 64, 128, 2, 0, 0},      {B0, -1, 0, B1, -1, 128, 128, 2, 0, 0},
    {B1, E1B, 1, D1A, -1, 192, 64, 1, 0, 0},    {D1A, -1, 0, D1B, -1, 64, 64, 1, 0, 0},
    {D1B, E0B, 1, D0A, -1, 96, 32, 0, 0, 0},    {D0A, -1, 0, D0B, -1, 32, 32, 0, 0, 0},
};

// Persistent workgroups: one per CU and output-channel block (the large
// tiles' LDS holds one workgroup per CU), never more than the tiles.
int g_cus = 0;

template <int NT, int R, int WR, int WC, bool kOneSlice, bool kHead = false>
void conv_go(const ConvArgs& a, int per_cu, hipStream_t s)
{
    const int th = WR * R, tw = WC * 16;
    const int tiles = a.n * ((a.h + th - 1) / th) * ((a.w_ + tw - 1) / tw);
    const int blocks_y = a.cout / (NT * 16);
    const int gx = std::min(tiles, std::max(1, per_cu * g_cus / blocks_y));
    ConvArgs b = a;
    b.near = (size_t)(th + 2) * a.w_ * std::max(a.ca, a.cb) * sizeof(uint16_t) < ((size_t)1 << 31);
    hipLaunchKernelGGL((conv3x3_kernel<NT, R, WR, WC, kOneSlice, kHead>), dim3((unsigned)gx, (unsigned)blocks_y),
                       dim3(64 * WR * WC), 0, s, b);
}

// 16 x 32 tiles, one workgroup per CU; where those would leave CUs idle (the
// lower levels of small images), 8 x 16 tiles, 32 channels a workgroup, two
// workgroups per CU.  The line is one large tile per CU: 120 large tiles
// (64 -> 64 channels at 320x180) take 15.0 us, in small ones 12.9 us; 460
// (96 -> 32 at 640x360) take 20.6 us, in small ones 24.5 us.
int launch_conv(const ConvArgs& a, hipStream_t s)
{
    const bool one = a.ca + a.cb == kCi, wide = a.cout % 64 == 0;
    const int tiles = a.n * ((a.h + 15) / 16) * ((a.w_ + 31) / 32);
    if (tiles * (wide ? a.cout / 64 : 1) < g_cus) {
        if (a.head_w) {
            conv_go<2, 2, 4, 1, true, true>(a, 2, s);
        } else {
            one ? conv_go<2, 2, 4, 1, true>(a, 2, s) : conv_go<2, 2, 4, 1, false>(a, 2, s);
        }
    } else if (a.head_w) {
        conv_go<2, 4, 4, 2, true, true>(a, 1, s);
    } else if (wide) {
        one ? conv_go<4, 4, 4, 2, true>(a, 1, s) : conv_go<4, 4, 4, 2, false>(a, 1, s);
    } else {
        one ? conv_go<2, 4, 4, 2, true>(a, 1, s) : conv_go<2, 4, 4, 2, false>(a, 1, s);
    }
    HIP_TRY(hipGetLastError());
    return VPT_OK;
}

unsigned blocks_for(size_t n, int t = 256) { return (unsigned)((n + t - 1) / t); }

}  // namespace

struct vpt_unet {
    vpt_ctx* ctx = nullptr;
    int device = 0;
    int max_n = 0, max_h = 0, max_w = 0;
    Layer net[kLayers];
    size_t n_params = 0, head_w = 0, head_b = 0;
    float* d_w = nullptr;        // fp32 master parameters
    uint16_t* d_wb = nullptr;    // bf16 copies (conv weights read these)
    float* d_g = nullptr;        // gradients
    float* d_m1 = nullptr;
    float* d_m2 = nullptr;
    uint16_t* d_wt = nullptr;    // flipped / transposed weights of every layer
    uint16_t* act[NBUF] = {};    // activations
    uint16_t* grad[NBUF] = {};   // masked gradients (pre-activation) of each buffer
    uint16_t* d_gcat[2] = {};    // data gradients of the concatenated inputs (of D0A, D1A)
    uint16_t* d_gpool[2] = {};   // gradients of P0, P1
    float* d_pred = nullptr;
    uint16_t* d_zero = nullptr;  // zeros, read for pixels outside the image
    float* d_part = nullptr;     // weight-gradient partials
    size_t part_floats = 0;
    float* d_head_part = nullptr;
    int slices = 0;
    int adam_t = 0;
    LastPass* d_pass = nullptr;
    float last_loss = 0.0f;
};

namespace {

size_t level_px(const vpt_unet* u, int n, int h, int w, int level) { return (size_t)n * (h >> level) * (w >> level); }

int check_dims(const vpt_unet* u, int n, int h, int w, const char* fn)
{
    if (n < 1 || h < 4 || w < 4 || (h & 3) || (w & 3))
        return set_error(VPT_EINVAL, "%s: %dx%dx%d: sizes must be positive multiples of 4", fn, n, h, w);
    if ((size_t)n * h * w > (size_t)u->max_n * u->max_h * u->max_w)
        return set_error(VPT_EINVAL, "%s: %dx%dx%d exceeds the capacity %dx%dx%d", fn, n, h, w, u->max_n, u->max_h,
                         u->max_w);
    return VPT_OK;
}

ConvArgs conv_args(vpt_unet* u, const Layer& L, int n, int h, int w)
{
    ConvArgs a;
    memset(&a, 0, sizeof(a));
    a.a = u->act[L.in_a];
    a.ca = kChannels[L.in_a];
    a.a_up = L.a_up;
    a.b = L.in_b >= 0 ? u->act[L.in_b] : nullptr;
    a.cb = L.in_b >= 0 ? kChannels[L.in_b] : 0;
    a.w = u->d_wb + L.w_off;
    a.bias = u->d_w + L.b_off;
    a.y = u->act[L.out];
    a.pool = L.pool >= 0 ? u->act[L.pool] : nullptr;
    a.relu = 1;
    a.zero = u->d_zero;
    a.n = n;
    a.h = h >> L.level;
    a.w_ = w >> L.level;
    a.cout = L.cout;
    return a;
}

// The network from act[X] to `out` (exp: irradiance, else log space).  The
// last layer's activation is stored only when keep_last is set (the backward
// pass reads it): vpt_unet_read_activation makes it from the layer before
// and the parameters in LastPass.
int forward(vpt_unet* u, int n, int h, int w, bool x16, bool keep_last, float* out, bool exp, hipStream_t s)
{
    for (int l = 0; l < kLayers; l++) {
        ConvArgs a = conv_args(u, u->net[l], n, h, w);
        if (l == 0) {
            a.a16 = x16;
            a.pass = u->d_pass;
        }
        if (l == kLayers - 1) {
            a.pass = u->d_pass;
            a.head_w = u->d_w + u->head_w;
            a.head_b = u->d_w + u->head_b;
            a.head_out = out;
            a.head_exp = exp;
            if (!keep_last) a.y = nullptr;
        }
        if (int rc = launch_conv(a, s)) return rc;
    }
    return VPT_OK;
}

// Weight gradient of a layer.  Channel blocks of 64 x 64, 64 x 32 or 32 x
// 32; one workgroup per CU in all (more slices would move more partial sums,
// fewer leave CUs idle), at most one per group of pixel tiles.
int wgrad(vpt_unet* u, const Layer& L, int n, int h, int w, const uint16_t* m, hipStream_t s)
{
    const ConvArgs a = conv_args(u, L, n, h, w);
    const int wsz = 9 * L.cout * L.cin;
    const int co = L.cout % 64 == 0 ? 2 : 1, ci = co == 2 && L.cin % 64 == 0 ? 2 : 1, ks = 4 / (co * ci);
    const int by = L.cout / (32 * co), bz = L.cin / (32 * ci);
    const long tiles = (long)a.n * ((a.h + kWgRows - 1) / kWgRows) * ((a.w_ + 31) / 32);
    const int slices = (int)std::min<long>((tiles + ks - 1) / ks, std::min(u->slices, std::max(1, g_cus / (by * bz))));
    float* part_b = u->d_part + (size_t)slices * wsz;
    auto go = [&](auto kern) {
        hipLaunchKernelGGL(kern, dim3((unsigned)slices, (unsigned)by, (unsigned)bz), dim3(256), 0, s, a, m, L.cin,
                           u->d_part, part_b);
    };
    ci == 2 ? go(wgrad_kernel<2, 2>) : (co == 2 ? go(wgrad_kernel<2, 1>) : go(wgrad_kernel<1, 1>));
    HIP_TRY(hipGetLastError());
    hipLaunchKernelGGL(reduce_parts_kernel, dim3((unsigned)((wsz / 4 + 31) / 32 + (L.cout / 4 + 31) / 32)), dim3(1024),
                       0, s, u->d_part, slices, wsz, u->d_g + L.w_off, part_b, L.cout, u->d_g + L.b_off);
    HIP_TRY(hipGetLastError());
    return VPT_OK;
}

// Data gradient of layer L's input: g_in = conv(m_out, flipped W^T), with
// the ReLU mask of the input buffer applied in the epilogue when the input
// is a single activation (mask_buf), else raw (concatenated inputs).
int dgrad(vpt_unet* u, const Layer& L, int n, int h, int w, const uint16_t* m, const uint16_t* mask, uint16_t* out,
          hipStream_t s)
{
    ConvArgs a;
    memset(&a, 0, sizeof(a));
    a.a = m;
    a.ca = L.cout;
    a.w = u->d_wt + L.w_off;
    a.mask = mask;
    a.y = out;
    a.zero = u->d_zero;
    a.n = n;
    a.h = h >> L.level;
    a.w_ = w >> L.level;
    a.cout = L.cin;
    return launch_conv(a, s);
}

int backward(vpt_unet* u, const float* d_target, int n, int h, int w, hipStream_t s)
{
    const size_t npx = level_px(u, n, h, w, 0);
    const Layer* N = u->net;
    {
        FlipLayers f;
        int most = 0;
        for (int l = 0; l < kLayers; l++) {
            f.off[l] = (uint32_t)N[l].w_off;
            f.cout[l] = (uint32_t)N[l].cout;
            f.cin[l] = (uint32_t)N[l].cin;
            most = std::max(most, 9 * N[l].cout * N[l].cin);
        }
        hipLaunchKernelGGL(flip_transpose_kernel, dim3(blocks_for((size_t)most), kLayers), dim3(256), 0, s, u->d_wb, f,
                           u->d_wt);
        HIP_TRY(hipGetLastError());
    }
    // head: loss, head gradients, masked gradient of D0B; the sums are 96 dW
    // and 3 db, which end the gradient vector, and the loss behind it
    const unsigned hb = blocks_for(npx);
    hipLaunchKernelGGL(head_bwd_kernel, dim3(hb), dim3(256), 0, s, u->act[D0B], npx, u->d_w + u->head_w, u->d_pred,
                       d_target, u->grad[D0B], u->d_head_part);
    HIP_TRY(hipGetLastError());
    hipLaunchKernelGGL(reduce_parts_kernel, dim3(1), dim3(1024), 0, s, u->d_head_part, (int)hb, 100,
                       u->d_g + u->head_w, (const float*)nullptr, 0, (float*)nullptr);
    HIP_TRY(hipGetLastError());

    auto sum2x2 = [&](const uint16_t* g, int cg, int c, int lh, int lw, const uint16_t* ylow, uint16_t* out) -> int {
        hipLaunchKernelGGL(sum2x2_mask_kernel, dim3(blocks_for((size_t)n * (lh >> 1) * (lw >> 1) * c / 8)), dim3(256),
                           0, s, g, cg, c, n, lh, lw, ylow, out);
        HIP_TRY(hipGetLastError());
        return VPT_OK;
    };
    auto skip = [&](const uint16_t* g, int cg, int off, int c, int lh, int lw, const uint16_t* gpool,
                    const uint16_t* y, uint16_t* out) -> int {
        hipLaunchKernelGGL(skip_mask_kernel, dim3(blocks_for((size_t)n * lh * lw * c / 8)), dim3(256), 0, s, g, cg, off,
                           c, n, lh, lw, gpool, y, out);
        HIP_TRY(hipGetLastError());
        return VPT_OK;
    };
    // layer 9: D0A -> D0B
    if (int rc = wgrad(u, N[9], n, h, w, u->grad[D0B], s)) return rc;
    if (int rc = dgrad(u, N[9], n, h, w, u->grad[D0B], u->act[D0A], u->grad[D0A], s)) return rc;
    // layer 8: cat(up(D1B), E0B) -> D0A; E0B's part waits in the
    // concatenated gradient until P0's is known
    if (int rc = wgrad(u, N[8], n, h, w, u->grad[D0A], s)) return rc;
    if (int rc = dgrad(u, N[8], n, h, w, u->grad[D0A], nullptr, u->d_gcat[0], s)) return rc;
    if (int rc = sum2x2(u->d_gcat[0], 96, 64, h, w, u->act[D1B], u->grad[D1B])) return rc;
    // layer 7: D1A -> D1B
    if (int rc = wgrad(u, N[7], n, h, w, u->grad[D1B], s)) return rc;
    if (int rc = dgrad(u, N[7], n, h, w, u->grad[D1B], u->act[D1A], u->grad[D1A], s)) return rc;
    // layer 6: cat(up(B1), E1B) -> D1A
    if (int rc = wgrad(u, N[6], n, h, w, u->grad[D1A], s)) return rc;
    if (int rc = dgrad(u, N[6], n, h, w, u->grad[D1A], nullptr, u->d_gcat[1], s)) return rc;
    if (int rc = sum2x2(u->d_gcat[1], 192, 128, h >> 1, w >> 1, u->act[B1], u->grad[B1])) return rc;
    // layer 5: B0 -> B1
    if (int rc = wgrad(u, N[5], n, h, w, u->grad[B1], s)) return rc;
    if (int rc = dgrad(u, N[5], n, h, w, u->grad[B1], u->act[B0], u->grad[B0], s)) return rc;
    // layer 4: P1 -> B0; gradient of P1 (no ReLU on a pooled buffer), then
    // E1B: skip gradient + pooled gradient, masked by E1B
    if (int rc = wgrad(u, N[4], n, h, w, u->grad[B0], s)) return rc;
    if (int rc = dgrad(u, N[4], n, h, w, u->grad[B0], nullptr, u->d_gpool[1], s)) return rc;
    if (int rc = skip(u->d_gcat[1], 192, 128, 64, h >> 1, w >> 1, u->d_gpool[1], u->act[E1B], u->grad[E1B])) return rc;
    // layer 3: E1A -> E1B
    if (int rc = wgrad(u, N[3], n, h, w, u->grad[E1B], s)) return rc;
    if (int rc = dgrad(u, N[3], n, h, w, u->grad[E1B], u->act[E1A], u->grad[E1A], s)) return rc;
    // layer 2: P0 -> E1A
    if (int rc = wgrad(u, N[2], n, h, w, u->grad[E1A], s)) return rc;
    if (int rc = dgrad(u, N[2], n, h, w, u->grad[E1A], nullptr, u->d_gpool[0], s)) return rc;
    if (int rc = skip(u->d_gcat[0], 96, 64, 32, h, w, u->d_gpool[0], u->act[E0B], u->grad[E0B])) return rc;
    // layer 1: E0A -> E0B
    if (int rc = wgrad(u, N[1], n, h, w, u->grad[E0B], s)) return rc;
    if (int rc = dgrad(u, N[1], n, h, w, u->grad[E0B], u->act[E0A], u->grad[E0A], s)) return rc;
    // layer 0: X -> E0A
    return wgrad(u, N[0], n, h, w, u->grad[E0A], s);
}

}  // namespace

// ---- C ABI -------------------------------------------------------------------

namespace {

struct DeviceGuard {
    int prev = -1;
    explicit DeviceGuard(int dev)
    {
        if (hipGetDevice(&prev) != hipSuccess) prev = -1;
        if (prev != dev) (void)hipSetDevice(dev);
    }
    ~DeviceGuard()
    {
        int cur = -1;
        if (prev >= 0 && hipGetDevice(&cur) == hipSuccess && cur != prev) (void)hipSetDevice(prev);
    }
};

int unet_upload(vpt_unet* u, const float* host)
{
    HIP_TRY(hipMemcpy(u->d_w, host, sizeof(float) * u->n_params, hipMemcpyHostToDevice));
    hipLaunchKernelGGL(to_bf16_kernel, dim3(blocks_for(u->n_params)), dim3(256), 0, nullptr, u->d_w, u->d_wb,
                       u->n_params);
    HIP_TRY(hipGetLastError());
    HIP_TRY(hipMemset(u->d_m1, 0, sizeof(float) * u->n_params));
    HIP_TRY(hipMemset(u->d_m2, 0, sizeof(float) * u->n_params));
    HIP_TRY(hipDeviceSynchronize());
    u->adam_t = 0;
    return VPT_OK;
}

}  // namespace

extern "C" VPT_API int vpt_unet_destroy(vpt_unet* u)
{
    if (!u) return VPT_OK;
    DeviceGuard g(u->device);
    (void)hipFree(u->d_w);
    (void)hipFree(u->d_wb);
    (void)hipFree(u->d_g);
    (void)hipFree(u->d_m1);
    (void)hipFree(u->d_m2);
    (void)hipFree(u->d_wt);
    for (int b = 0; b < NBUF; b++) {
        (void)hipFree(u->act[b]);
        (void)hipFree(u->grad[b]);
    }
    (void)hipFree(u->d_gcat[0]);
    (void)hipFree(u->d_gcat[1]);
    (void)hipFree(u->d_gpool[0]);
    (void)hipFree(u->d_gpool[1]);
    (void)hipFree(u->d_pred);
    (void)hipFree(u->d_zero);
    (void)hipFree(u->d_pass);
    (void)hipFree(u->d_part);
    (void)hipFree(u->d_head_part);
    delete u;
    return VPT_OK;
}

extern "C" VPT_API int vpt_unet_create(vpt_ctx* ctx, int max_n, int max_h, int max_w, vpt_unet** out)
{
    if (!ctx || !out) return set_error(VPT_EINVAL, "vpt_unet_create: null argument");
    if (max_n < 1 || max_h < 4 || max_w < 4 || (max_h & 3) || (max_w & 3) ||
        (size_t)max_n * max_h * max_w > ((size_t)1 << 26))
        return set_error(VPT_EINVAL, "vpt_unet_create: capacity %dx%dx%d (multiples of 4, at most 2^26 pixels)",
                         max_n, max_h, max_w);
    DeviceGuard g(ctx->device);
    vpt_unet* u = new vpt_unet();
    if (!g_cus) g_cus = vpt::device_cus(ctx->device);
    u->ctx = ctx;
    u->device = ctx->device;
    u->max_n = max_n;
    u->max_h = max_h;
    u->max_w = max_w;
    size_t off = 0, max_w_layer = 0;
    for (int l = 0; l < kLayers; l++) {
        u->net[l] = kNet[l];
        u->net[l].w_off = off;
        off += (size_t)9 * kNet[l].cout * kNet[l].cin;
        u->net[l].b_off = off;
        off += (size_t)kNet[l].cout;
        max_w_layer = std::max(max_w_layer, (size_t)9 * kNet[l].cout * kNet[l].cin);
    }
    u->head_w = off;
    u->head_b = off + 96;
    u->n_params = off + 99;
    const size_t full = (size_t)max_n * max_h * max_w;
    u->slices = 256;
    u->part_floats = (size_t)u->slices * (max_w_layer + 128);
    hipError_t e = hipSuccess;
    auto alloc = [&](void** p, size_t bytes) {
        if (e == hipSuccess) e = hipMalloc(p, std::max<size_t>(bytes, 256));
    };
    alloc((void**)&u->d_w, sizeof(float) * u->n_params);
    alloc((void**)&u->d_wb, sizeof(uint16_t) * u->n_params);
    alloc((void**)&u->d_g, sizeof(float) * (u->n_params + 1));
    alloc((void**)&u->d_m1, sizeof(float) * u->n_params);
    alloc((void**)&u->d_m2, sizeof(float) * u->n_params);
    alloc((void**)&u->d_wt, sizeof(uint16_t) * u->n_params);
    for (int b = 0; b < NBUF; b++) {
        const size_t px = full >> (2 * kLevel[b]);
        alloc((void**)&u->act[b], sizeof(uint16_t) * px * kChannels[b]);
        if (b != X && b != P0 && b != P1) alloc((void**)&u->grad[b], sizeof(uint16_t) * px * kChannels[b]);
    }
    alloc((void**)&u->d_gcat[0], sizeof(uint16_t) * full * 96);
    alloc((void**)&u->d_gcat[1], sizeof(uint16_t) * (full >> 2) * 192);
    alloc((void**)&u->d_gpool[0], sizeof(uint16_t) * (full >> 2) * 32);
    alloc((void**)&u->d_gpool[1], sizeof(uint16_t) * (full >> 4) * 64);
    alloc((void**)&u->d_pred, sizeof(float) * full * 3);
    alloc((void**)&u->d_zero, 1024);
    alloc((void**)&u->d_pass, sizeof(LastPass));
    alloc((void**)&u->d_part, sizeof(float) * u->part_floats);
    alloc((void**)&u->d_head_part, sizeof(float) * 100 * ((full + 255) / 256));
    if (e == hipSuccess) e = hipMemset(u->d_zero, 0, 1024);
    if (e == hipSuccess) e = hipMemset(u->d_pass, 0, sizeof(LastPass));
    if (e != hipSuccess) {
        vpt_unet_destroy(u);
        return set_error(VPT_ENOMEM, "vpt_unet_create: allocation failed (%s)", hipGetErrorString(e));
    }
    *out = u;
    return VPT_OK;
}

extern "C" VPT_API int vpt_unet_param_count(const vpt_unet* u, size_t* n)
{
    if (!u || !n) return set_error(VPT_EINVAL, "vpt_unet_param_count: null argument");
    *n = u->n_params;
    return VPT_OK;
}

extern "C" VPT_API int vpt_unet_init(vpt_unet* u, uint32_t seed)
{
    if (!u) return set_error(VPT_EINVAL, "vpt_unet_init: null network");
    std::vector<float> w(u->n_params, 0.0f);
    std::mt19937 rng(seed);
    for (int l = 0; l < kLayers; l++) {
        const Layer& L = u->net[l];
        std::normal_distribution<float> nd(0.0f, sqrtf(2.0f / (9.0f * (float)L.cin)));   // He initialisation
        for (size_t i = 0; i < (size_t)9 * L.cout * L.cin; i++) w[L.w_off + i] = nd(rng);
    }
    std::normal_distribution<float> nh(0.0f, sqrtf(1.0f / 32.0f));
    for (int i = 0; i < 96; i++) w[u->head_w + i] = nh(rng);
    DeviceGuard g(u->device);
    return unet_upload(u, w.data());
}

extern "C" VPT_API int vpt_unet_set_params(vpt_unet* u, const float* host, size_t n)
{
    if (!u || !host || n != u->n_params)
        return set_error(VPT_EINVAL, "vpt_unet_set_params: expected %zu floats", u ? u->n_params : (size_t)0);
    DeviceGuard g(u->device);
    return unet_upload(u, host);
}

extern "C" VPT_API int vpt_unet_get_params(vpt_unet* u, float* host, size_t n)
{
    if (!u || !host || n != u->n_params)
        return set_error(VPT_EINVAL, "vpt_unet_get_params: expected %zu floats", u ? u->n_params : (size_t)0);
    DeviceGuard g(u->device);
    HIP_TRY(hipDeviceSynchronize());
    HIP_TRY(hipMemcpy(host, u->d_w, sizeof(float) * n, hipMemcpyDeviceToHost));
    return VPT_OK;
}

extern "C" VPT_API int vpt_unet_get_grads(vpt_unet* u, float* host, size_t n)
{
    if (!u || !host || n != u->n_params)
        return set_error(VPT_EINVAL, "vpt_unet_get_grads: expected %zu floats", u ? u->n_params : (size_t)0);
    DeviceGuard g(u->device);
    HIP_TRY(hipDeviceSynchronize());
    HIP_TRY(hipMemcpy(host, u->d_g, sizeof(float) * n, hipMemcpyDeviceToHost));
    return VPT_OK;
}

extern "C" VPT_API int vpt_unet_forward(vpt_unet* u, const uint16_t* d_x, int n, int h, int w, int mode, float* d_out,
                                        void* stream)
{
    if (!u || !d_x || !d_out) return set_error(VPT_EINVAL, "vpt_unet_forward: null argument");
    if (int rc = check_dims(u, n, h, w, "vpt_unet_forward")) return rc;
    if (mode != 0 && mode != 1) return set_error(VPT_EINVAL, "vpt_unet_forward: mode 0 (log space) or 1 (irradiance)");
    DeviceGuard g(u->device);
    hipStream_t s = (hipStream_t)stream;
    const size_t npx = (size_t)n * h * w;
    HIP_TRY(hipMemcpyAsync(u->act[X], d_x, sizeof(uint16_t) * npx * 32, hipMemcpyDeviceToDevice, s));
    return forward(u, n, h, w, false, false, d_out, mode == 1, s);
}

extern "C" VPT_API int vpt_unet_backward(vpt_unet* u, const uint16_t* d_x, const float* d_target, int n, int h, int w,
                                         float* loss, void* stream)
{
    if (!u || !d_x || !d_target) return set_error(VPT_EINVAL, "vpt_unet_backward: null argument");
    if (int rc = check_dims(u, n, h, w, "vpt_unet_backward")) return rc;
    DeviceGuard g(u->device);
    hipStream_t s = (hipStream_t)stream;
    const size_t npx = (size_t)n * h * w;
    HIP_TRY(hipMemcpyAsync(u->act[X], d_x, sizeof(uint16_t) * npx * 32, hipMemcpyDeviceToDevice, s));
    if (int rc = forward(u, n, h, w, false, true, u->d_pred, false, s)) return rc;
    if (int rc = backward(u, d_target, n, h, w, s)) return rc;
    if (loss) {
        float sum = 0.0f;
        HIP_TRY(hipMemcpyAsync(&sum, u->d_g + u->n_params, sizeof(float), hipMemcpyDeviceToHost, s));
        HIP_TRY(hipStreamSynchronize(s));
        *loss = sum / (3.0f * (float)npx);
    }
    return VPT_OK;
}

extern "C" VPT_API int vpt_unet_adam_step(vpt_unet* u, float lr, void* stream)
{
    if (!u || !(lr > 0.0f)) return set_error(VPT_EINVAL, "vpt_unet_adam_step: bad arguments");
    DeviceGuard g(u->device);
    const float b1 = 0.9f, b2 = 0.999f;
    u->adam_t++;
    const float c1 = 1.0f / (1.0f - powf(b1, (float)u->adam_t));
    const float c2 = 1.0f / (1.0f - powf(b2, (float)u->adam_t));
    hipLaunchKernelGGL(adam_kernel, dim3(blocks_for(u->n_params)), dim3(256), 0, (hipStream_t)stream, u->d_w, u->d_wb,
                       u->d_g, u->d_m1, u->d_m2, u->n_params, lr, b1, b2, 1e-8f, c1, c2);
    HIP_TRY(hipGetLastError());
    return VPT_OK;
}

// The network's input; x16: only channels 0..15, 32 bytes a pixel.
static int assemble(const char* fn, vpt_unet* u, const vpt_gbuffer* gb, const vpt_svgf_texel* d_tex, uint16_t* d_x,
                    bool x16, void* stream)
{
    if (!u || !gb || !d_tex || !d_x || !gb->d_t || !gb->d_face || !gb->d_block)
        return set_error(VPT_EINVAL, "%s: null argument", fn);
    vpt::AlbedoTable albedo;
    {
        std::lock_guard<std::mutex> lk(u->ctx->mu);
        if (!u->ctx->albedo_valid) return set_error(VPT_ESTATE, "%s: no albedo table yet (trace GI first)", fn);
        memcpy(albedo.v, u->ctx->albedo_host, sizeof(albedo.v));
    }
    DeviceGuard g(u->device);
    const int npx = gb->width * gb->height;
    hipLaunchKernelGGL(x16 ? assemble_kernel<2> : assemble_kernel<4>, dim3(blocks_for((size_t)npx)), dim3(256), 0,
                       (hipStream_t)stream, npx, gb->d_t, gb->d_face, gb->d_block, d_tex, albedo, d_x);
    HIP_TRY(hipGetLastError());
    return VPT_OK;
}

extern "C" VPT_API int vpt_unet_assemble(vpt_unet* u, const vpt_gbuffer* gb, const vpt_svgf_texel* d_tex,
                                         uint16_t* d_x, void* stream)
{
    return assemble("vpt_unet_assemble", u, gb, d_tex, d_x, false, stream);
}

extern "C" VPT_API int vpt_unet_denoise(vpt_unet* u, const vpt_gbuffer* gb, const vpt_svgf_texel* d_tex, float* d_rgb,
                                        void* stream)
{
    if (!u || !gb || !d_rgb) return set_error(VPT_EINVAL, "vpt_unet_denoise: null argument");
    if (int rc = check_dims(u, 1, gb->height, gb->width, "vpt_unet_denoise")) return rc;
    if (int rc = assemble("vpt_unet_denoise", u, gb, d_tex, u->act[X], true, stream)) return rc;
    DeviceGuard g(u->device);
    return forward(u, 1, gb->height, gb->width, true, false, d_rgb, true, (hipStream_t)stream);
}

extern "C" VPT_API int vpt_texel_accumulate(const vpt_svgf_texel* d_tex, int npx, float* d_acc, int reset, void* stream)
{
    if (!d_tex || !d_acc || npx < 0) return set_error(VPT_EINVAL, "vpt_texel_accumulate: bad arguments");
    if (npx == 0) return VPT_OK;
    hipLaunchKernelGGL(accumulate_kernel, dim3(blocks_for((size_t)npx)), dim3(256), 0, (hipStream_t)stream, npx,
                       d_tex, reset, d_acc);
    HIP_TRY(hipGetLastError());
    return VPT_OK;
}

extern "C" VPT_API int vpt_irradiance_decode(const vpt_gbuffer* gb, const vpt_svgf_texel* d_tex, const float* d_acc,
                                             float acc_scale, float* d_rgb, void* stream)
{
    if (!gb || !gb->d_face || !d_rgb || (!d_tex && !d_acc))
        return set_error(VPT_EINVAL, "vpt_irradiance_decode: null argument");
    const int npx = gb->width * gb->height;
    hipLaunchKernelGGL(decode_irr_kernel, dim3(blocks_for((size_t)npx)), dim3(256), 0, (hipStream_t)stream, npx,
                       gb->d_face, d_tex, d_acc, acc_scale, d_rgb);
    HIP_TRY(hipGetLastError());
    return VPT_OK;
}

extern "C" VPT_API int vpt_unet_read_activation(vpt_unet* u, int index, int n, int h, int w, uint16_t* host)
{
    if (!u || !host || index < 0 || index >= NBUF) return set_error(VPT_EINVAL, "vpt_unet_read_activation: bad arguments");
    if (int rc = check_dims(u, n, h, w, "vpt_unet_read_activation")) return rc;
    DeviceGuard g(u->device);
    const size_t count = ((size_t)n * (h >> kLevel[index]) * (w >> kLevel[index])) * kChannels[index];
    HIP_TRY(hipDeviceSynchronize());
    int last[4] = {0, 0, 0, 0};   // x16, n, h, w
    if (index == X || index == D0B) HIP_TRY(hipMemcpy(last, u->d_pass, sizeof(last), hipMemcpyDeviceToHost));
    if (index == D0B && last[1]) {
        // made from the pass's own D0A, parameters and sizes, whatever part is read
        ConvArgs a = conv_args(u, u->net[kLayers - 1], last[1], last[2], last[3]);
        a.w = u->d_pass->w_;
        a.bias = u->d_pass->bias;
        if (int rc = launch_conv(a, nullptr)) return rc;
        HIP_TRY(hipDeviceSynchronize());
    }
    const bool half = index == X && last[0];   // 16 of the input's 32 channels are stored, the others are zero
    HIP_TRY(hipMemcpy(host, u->act[index], sizeof(uint16_t) * (half ? count / 2 : count), hipMemcpyDeviceToHost));
    if (half) {
        for (size_t i = count / 32; i-- > 0;) {
            memmove(host + i * 32, host + i * 16, 16 * sizeof(uint16_t));
            memset(host + i * 32 + 16, 0, 16 * sizeof(uint16_t));
        }
    }
    return VPT_OK;
}
