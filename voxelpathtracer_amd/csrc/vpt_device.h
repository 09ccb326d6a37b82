// Device-side building blocks shared by the gfx950 kernels: brick
// addressing, the DF traversal, ray generation.  Every floating-point
// expression here is the same IEEE operation sequence as the reference
// shader it cites (compiled with -ffp-contract=off), which is what makes hit
// cells, faces and distances reproducible bit for bit.
#pragma once

#include <hip/hip_runtime.h>
#include <stdint.h>

#include "vpt/vpt_numerics.h"
#include "vpt_tiles.h"

namespace vpt {

// A brick: 8 x 4 x 4 cells in one 128-byte line, x fastest, then y, then z.
constexpr int kBrickBytes = 128;

// Read-only view of a world's bricked planes, passed to kernels by value.
struct WorldView {
    const uint8_t* grid;
    const uint8_t* df;
    int nx, ny, nz;
    uint32_t row_stride;    // nbx * 128
    uint32_t slab_stride;   // nbx * nby * 128
    float xmax, ymax, zmax; // dims - 1 as float (IsInVolume bounds)
};

// Byte `off` of a world plane (grid or DF).  The planes are device
// allocations, so the read is a global one also where the view was loaded
// from memory (a served world) rather than passed as a kernel argument,
// which would otherwise make it a flat access.
__device__ inline uint8_t plane_byte(const uint8_t* p, uint32_t off)
{
    typedef const __attribute__((address_space(1))) uint8_t GlobalByte;
    return ((GlobalByte*)p)[off];   // address-space cast
}

// Byte offset of cell (x, y, z) in a bricked plane, bricks bx-fastest: the
// three axes contribute independent terms.  (x / 8) * 128 + x % 8 is x + (x /
// 8) * 120, and the others likewise; bricks and strides fit in 24-bit
// products.  Eight instructions in the traversal's turns, where the Morton
// order of 512-byte bricks that this layout replaced took fifteen; a line
// still covers 8 x 4 x 4 cells.
__host__ __device__ inline uint32_t brick_offset(uint32_t x, uint32_t y, uint32_t z, uint32_t row_stride,
                                                 uint32_t slab_stride)
{
    return (x + (x >> 3) * (kBrickBytes - 8u)) + ((y << 3) + (y >> 2) * (row_stride - 32u)) +
           ((z << 5) + (z >> 2) * (slab_stride - 128u));
}

// The same with 24-bit multiply-adds, for the traversal.
__device__ inline uint32_t brick_offset_fast(uint32_t x, uint32_t y, uint32_t z, uint32_t row_stride,
                                             uint32_t slab_stride)
{
    uint32_t off = __umul24(x >> 3, kBrickBytes - 8u) + x;
    off = __umul24(y >> 2, row_stride - 32u) + off;
    off = (y << 3) + off;
    off = __umul24(z >> 2, slab_stride - 128u) + off;
    return (z << 5) + off;
}

struct Vec3 {
    float x, y, z;
};

__device__ inline Vec3 mk3(float x, float y, float z)
{
    Vec3 r;
    r.x = x;
    r.y = y;
    r.z = z;
    return r;
}

__device__ inline float dot3(Vec3 a, Vec3 b) { return (a.x * b.x + a.y * b.y) + a.z * b.z; }

__device__ inline Vec3 normalize3(Vec3 v)
{
    float len = sqrtf((v.x * v.x + v.y * v.y) + v.z * v.z);
    return mk3(v.x / len, v.y / len, v.z / len);
}

__device__ inline Vec3 cross3(Vec3 a, Vec3 b)
{
    return mk3(a.y * b.z - b.y * a.z, a.z * b.x - b.z * a.x, a.x * b.y - b.x * a.y);
}

// mat4 * vec4 rows 0..n-1, GLSL column-major, summed in column order.
__device__ inline float mat_row(const float* m, int r, float v0, float v1, float v2, float v3)
{
    float acc = m[r] * v0;
    acc = acc + m[4 + r] * v1;
    acc = acc + m[8 + r] * v2;
    acc = acc + m[12 + r] * v3;
    return acc;
}

// GetRayStuff / GetRayDirectionAt (InitialRayTraceFrag.glsl:398-414,
// ShadowRayTraceFrag.glsl:292-297), normalised as in main() (:427).
__device__ inline Vec3 ray_dir_at(const float* inv_view, const float* inv_proj, float sx, float sy)
{
    float cx = sx * 2.0f - 1.0f;
    float cy = sy * 2.0f - 1.0f;
    float ex = mat_row(inv_proj, 0, cx, cy, -1.0f, 1.0f);
    float ey = mat_row(inv_proj, 1, cx, cy, -1.0f, 1.0f);
    Vec3 rd;
    rd.x = mat_row(inv_view, 0, ex, ey, -1.0f, 0.0f);
    rd.y = mat_row(inv_view, 1, ex, ey, -1.0f, 0.0f);
    rd.z = mat_row(inv_view, 2, ex, ey, -1.0f, 0.0f);
    return rd;
}

__device__ inline float texcoord(int p, int n) { return ((float)p + 0.5f) / (float)n; }

// GetNormalFromID for a face byte; `miss` is the value of the reference's
// out-of-range branch (1.0 in most passes, 0.5 in the diffuse pass).
__device__ inline Vec3 face_normal(int face, float miss)
{
    switch (face) {
    case 0: return mk3(0.0f, 0.0f, 1.0f);
    case 1: return mk3(0.0f, 0.0f, -1.0f);
    case 2: return mk3(0.0f, 1.0f, 0.0f);
    case 3: return mk3(0.0f, -1.0f, 0.0f);
    case 4: return mk3(-1.0f, 0.0f, 0.0f);
    case 5: return mk3(1.0f, 0.0f, 0.0f);
    default: return mk3(miss, miss, miss);
    }
}

// GetNormalID of the normal with component -s on `axis`
// (InitialRayTraceFrag.glsl:143-185).
__device__ inline int face_from_axis(int axis, int s)
{
    if (s == 0) return 0;
    int n = -s;
    if (axis == 2) return n > 0 ? 0 : 1;
    if (axis == 1) return n > 0 ? 2 : 3;
    return n < 0 ? 4 : 5;
}

// The DF step E of the reference for a DF byte: floor(M * 0.57735026918f),
// except M == 1 -> 1.  The unorm8 round trip (M/255)*255 is exact for every
// byte, so M is the byte itself (the host tests check this against
// vpt_df_step for all 256 values).  E is 0 only for M = 0 and 1 only for
// M = 1, 2, 3 (3 * 0.57735026918f = 1.73, 4 * 0.57735026918f = 2.31), which
// is how trav_advance branches on the byte; the jump length E - 1 is then
// df_jump.
__device__ inline int df_step(int m)
{
    return m == 1 ? 1 : (int)((float)m * 0.57735026918f);
}

// (float)(E - 1) for a byte M >= 4: truncf is floor for the positive
// product, and E - 1 < 2^24 subtracts exactly.
__device__ inline float df_jump(int m)
{
    return truncf((float)m * 0.57735026918f) - 1.0f;
}

struct Hit {
    float t;
    int face;
    int block;
    uint32_t voxel;
    int samples;
};

__device__ inline uint32_t pack_cell(int x, int y, int z)
{
    return (uint32_t)x | ((uint32_t)y << 10) | ((uint32_t)z << 20);
}

// VoxelTraversalDF (InitialRayTraceFrag.glsl:307-374; identical copies in
// ShadowRayTraceFrag.glsl:222-289 and DiffuseRayTraceFrag.glsl:1043-1110),
// split into resumable pieces so that a persistent kernel can interleave
// several rays per lane:
//   trav_init     the loop's set-up,
//   trav_prepare  the head of one iteration (iteration cap, IsInVolume, the
//                 DF address); false = the loop has ended,
//   trav_advance  the rest of the iteration once the DF byte has arrived;
//                 false = the loop has ended,
//   trav_finish   the code after the loop.
// The per-ray state is the reference's: origin, direction, the reciprocal
// direction, initial origin, MinIdx, Intersection.  `samples` counts the
// loop's turns (one DF sample each); the loop ends after max_iter of them.
struct Trav {
    float ox, oy, oz;
    float dx, dy, dz;
    float ix, iy, iz;
    float o0x, o0y, o0z;
    int max_iter;
    int min_idx;
    int inter;
    int samples;
};

// The cell of the position, found by trav_prepare and used by trav_advance
// in the same loop turn.
struct Cell {
    uint32_t x, y, z;
};

__device__ inline int sgn(float v) { return v > 0.0f ? 1 : (v < 0.0f ? -1 : 0); }

// c ? x : y with both values computed in every lane first (the empty asm
// only pins them to registers and emits nothing), so that the choice stays
// one v_cndmask_b32 instead of two exec-masked arms.
__device__ __attribute__((always_inline)) inline float pick(bool c, float x, float y)
{
    asm volatile("" : "+v"(x), "+v"(y));
    return c ? x : y;
}

__device__ __attribute__((always_inline)) inline void trav_init(Trav& r, Vec3 o, Vec3 d, int max_iter)
{
    // o + 0 turns a -0 component into +0 and leaves every other value as it
    // is.  The two behave alike in all the loop's arithmetic (both floor to a
    // zero inside the volume), and no later step can produce -0 (a sum is -0
    // only when both terms are), so trav_prepare's bounds test never sees it.
    r.ox = o.x + 0.0f;
    r.oy = o.y + 0.0f;
    r.oz = o.z + 0.0f;
    r.dx = d.x;
    r.dy = d.y;
    r.dz = d.z;
    r.ix = 1.0f / d.x;
    r.iy = 1.0f / d.y;
    r.iz = 1.0f / d.z;
    r.o0x = o.x;
    r.o0y = o.y;
    r.o0z = o.z;
    r.max_iter = max_iter;
    r.min_idx = 0;
    r.inter = 0;
    r.samples = 0;
}

// Bit pattern of (float)dim, dim = max + 1 (0 for the empty view, max = -1).
__device__ inline uint32_t trav_bound(float max) { return __float_as_uint(max + 1.0f); }

// IsInVolume(floor(o)), one unsigned compare per axis: floor(o) lies in
// [0, dim - 1] exactly when o lies in [+0, dim); non-negative floats order as
// their bit patterns, and negative values and NaN have patterns above every
// bound.
__device__ __attribute__((always_inline)) inline bool trav_inside(const WorldView& w, const Trav& r)
{
    return __float_as_uint(r.ox) < trav_bound(w.xmax) && __float_as_uint(r.oy) < trav_bound(w.ymax) &&
           __float_as_uint(r.oz) < trav_bound(w.zmax);
}

__device__ __attribute__((always_inline)) inline bool trav_prepare(const WorldView& w, Trav& r, uint32_t& off,
                                                                   Cell& c)
{
    if (r.samples >= r.max_iter) return false;
    if (!trav_inside(w, r)) {
        r.inter = 0;
        return false;
    }
    // truncation is floor for o >= 0
    c.x = (uint32_t)r.ox;
    c.y = (uint32_t)r.oy;
    c.z = (uint32_t)r.oz;
    off = brick_offset_fast(c.x, c.y, c.z, w.row_stride, w.slab_stride);
    return true;
}

// What the one-cell step needs of a ray's direction: the signs, h = (1 + s)
// / 2, e = s + 1 - h and s * 0.0001.
struct StepDir {
    int sx, sz;
    float hx, hy, hz, ex, ey, ez, tx, ty, tz;
};

__device__ __attribute__((always_inline)) inline StepDir step_dir(const Trav& r)
{
    const int sx = sgn(r.dx), sy = sgn(r.dy), sz = sgn(r.dz);
    const float hx = (float)((1 + sx) >> 1), hy = (float)((1 + sy) >> 1), hz = (float)((1 + sz) >> 1);
    return StepDir{sx,
                   sz,
                   hx,
                   hy,
                   hz,
                   (float)(sx + 1) - hx,
                   (float)(sy + 1) - hy,
                   (float)(sz + 1) - hz,
                   (float)sx * 0.0001f,
                   (float)sy * 0.0001f,
                   (float)sz * 0.0001f};
}

// E == 1: the one-cell step from cell c to (ax, ay, az) across axis mi, with
// selects on the step axis (no divergent branches: fewer exec-mask moves in
// the loop).  The reference forms float(int(o) + s) + w, then adds s * 0.0001
// on the step axis.  On that axis w is 1 - h, and the integers add exactly:
// (g + s) + (1 - h) = g + (s + 1 - h), also for the s = 0 that the y axis can
// be picked with.  On the others s is 0 and w moves by d * fm.
__device__ __attribute__((always_inline)) inline void one_cell(const Trav& r, const StepDir& s, const Cell& c,
                                                               float& ax, float& ay, float& az, int& mi)
{
    // float(int(o)) of the reference is the cell's corner
    const float gx = (float)c.x, gy = (float)c.y, gz = (float)c.z;
    const float wx = r.ox - gx, wy = r.oy - gy, wz = r.oz - gz;
    const float fxx = (s.hx - wx) * r.ix, fyy = (s.hy - wy) * r.iy, fzz = (s.hz - wz) * r.iz;
    const bool x_first = fxx < fyy && s.sx != 0;
    const float fxy = x_first ? fxx : fyy;
    const bool not_z = fxy < fzz || s.sz == 0;
    const float fm = not_z ? fxy : fzz;
    ax = pick(x_first && not_z, (gx + s.ex) + s.tx, gx + (wx + r.dx * fm));
    ay = pick(!x_first && not_z, (gy + s.ey) + s.ty, gy + (wy + r.dy * fm));
    az = pick(not_z, gz + (wz + r.dz * fm), (gz + s.ez) + s.tz);
    mi = not_z ? (x_first ? 0 : 1) : 2;
}

__device__ __attribute__((always_inline)) inline bool trav_advance(Trav& r, int m, const Cell& c)
{
    r.samples++;
    if (m == 0) return false;   // E == 0
    if (m < 4) {
        float ax, ay, az;
        int mi;
        one_cell(r, step_dir(r), c, ax, ay, az, mi);
        r.ox = ax;
        r.oy = ay;
        r.oz = az;
        r.min_idx = mi;
        r.inter = 1;
    } else {
        const float k = df_jump(m);
        r.ox = r.ox + k * r.dx;
        r.oy = r.oy + k * r.dy;
        r.oz = r.oz + k * r.dz;
    }
    return r.samples < r.max_iter;
}

__device__ __attribute__((always_inline)) inline Hit trav_finish(const WorldView& w, const Trav& r)
{
    Hit h;
    h.t = -1.0f;
    h.face = 255;
    h.block = 0;
    h.voxel = 0xffffffffu;
    h.samples = r.samples;
    if (r.inter) {
        float fx = floorf(r.ox), fy = floorf(r.oy), fz = floorf(r.oz);
        if (fx >= 0.0f && fy >= 0.0f && fz >= 0.0f && fx <= w.xmax && fy <= w.ymax && fz <= w.zmax) {
            int cx = (int)fx, cy = (int)fy, cz = (int)fz;
            int b = plane_byte(w.grid, brick_offset_fast(cx, cy, cz, w.row_stride, w.slab_stride));
            if (b > 0) {
                float dx = r.ox - r.o0x, dy = r.oy - r.o0y, dz = r.oz - r.o0z;
                h.t = sqrtf((dx * dx + dy * dy) + dz * dz);
                // the three signs first, then a select: an indexed pick of the
                // direction components can end up as a scratch-memory load
                const int sx = sgn(r.dx), sy = sgn(r.dy), sz = sgn(r.dz);
                int s = sx;
                s = r.min_idx == 1 ? sy : s;
                s = r.min_idx == 2 ? sz : s;
                h.face = face_from_axis(r.min_idx, s);
                h.block = b;
                h.voxel = pack_cell(cx, cy, cz);
            }
        }
    }
    return h;
}

// The loop's turns of a ray to its end or to r.max_iter, as trav_prepare and
// trav_advance make them, in a form with one exit and selects in place of
// most branches.  The position must be inside the volume and samples below
// the cap on entry; returns the last DF byte (0: stopped in a solid cell).
// Leaving the volume needs no flag: trav_finish finds the position outside.
// kEager: the one-cell step, which does not need the DF byte, is computed
// while that byte is on its way.  That shortens the chain from one position
// to the next, which is what the few long rays that end a launch wait for
// with most of the chip idle; it costs every turn both kinds of step, which
// the short rays of a full chip would pay for.
template <bool kEager>
__device__ __attribute__((always_inline)) inline int trav_run(const WorldView& w, Trav& r)
{
    const StepDir s = step_dir(r);
    const uint32_t bx = trav_bound(w.xmax), by = trav_bound(w.ymax), bz = trav_bound(w.zmax);
    int m;
    bool alive;
    do {
        const Cell c{(uint32_t)r.ox, (uint32_t)r.oy, (uint32_t)r.oz};
        m = plane_byte(w.df, brick_offset_fast(c.x, c.y, c.z, w.row_stride, w.slab_stride));
        float ax, ay, az;
        int mi;
        if (kEager) {
            one_cell(r, s, c, ax, ay, az, mi);
            // all of that before the byte is waited for
            asm volatile("" : "+v"(ax), "+v"(ay), "+v"(az), "+v"(mi));
            const bool solid = m == 0, one = m < 4;
            const float k = df_jump(m);
            const float nx = one ? ax : r.ox + k * r.dx, ny = one ? ay : r.oy + k * r.dy,
                        nz = one ? az : r.oz + k * r.dz;
            r.min_idx = one && !solid ? mi : r.min_idx;
            r.inter = one && !solid ? 1 : r.inter;
            r.ox = solid ? r.ox : nx;
            r.oy = solid ? r.oy : ny;
            r.oz = solid ? r.oz : nz;
        } else if (m < 4) {
            one_cell(r, s, c, ax, ay, az, mi);
            const bool solid = m == 0;
            r.ox = pick(solid, r.ox, ax);
            r.oy = pick(solid, r.oy, ay);
            r.oz = pick(solid, r.oz, az);
            r.min_idx = solid ? r.min_idx : mi;
            r.inter = solid ? r.inter : 1;
        } else {
            const float k = df_jump(m);
            r.ox = r.ox + k * r.dx;
            r.oy = r.oy + k * r.dy;
            r.oz = r.oz + k * r.dz;
        }
        r.samples++;
        alive = m != 0 && r.samples < r.max_iter && __float_as_uint(r.ox) < bx && __float_as_uint(r.oy) < by &&
                __float_as_uint(r.oz) < bz;
    } while (alive);
    return m;
}

// Steps of a ray after which traverse goes over to the eager turns: at once
// in a launch that leaves the chip idle lanes anyway.
constexpr int kLongRay = 24;
constexpr uint32_t kSmallLaunch = 1024;   // workgroups
__device__ inline int long_ray_after() { return gridDim.x <= kSmallLaunch ? 0 : kLongRay; }

__device__ inline Hit traverse(const WorldView& w, Vec3 o, Vec3 d, int max_iter)
{
    Trav r;
    const int after = long_ray_after();
    trav_init(r, o, d, min(max_iter, after));
    if (max_iter > 0 && trav_inside(w, r)) {
        int m = 1;
        if (after > 0) m = trav_run<false>(w, r);
        if (m != 0 && max_iter > after && trav_inside(w, r)) {
            r.max_iter = max_iter;
            trav_run<true>(w, r);
        }
    }
    return trav_finish(w, r);
}

// GetVoxel(ivec3(floor(p))) (InitialRayTraceFrag.glsl:79-87).
__device__ inline int voxel_at(const WorldView& w, Vec3 p)
{
    float fx = floorf(p.x), fy = floorf(p.y), fz = floorf(p.z);
    if (!(fx >= 0.0f && fy >= 0.0f && fz >= 0.0f && fx <= w.xmax && fy <= w.ymax && fz <= w.zmax)) return 0;
    return plane_byte(w.grid, brick_offset_fast((uint32_t)(int)fx, (uint32_t)(int)fy, (uint32_t)(int)fz,
                                                w.row_stride, w.slab_stride));
}

// Hardware binary16 conversions (v_cvt_f32_f16 is exact; v_cvt_f16_f32
// rounds to nearest even with fp16 denormals preserved), i.e. the same
// results as vpt_f16_to_f32 / vpt_f32_to_f16 of the shared numerics.
__device__ inline float hw_h2f(uint32_t h) { return (float)__builtin_bit_cast(_Float16, (uint16_t)h); }
__device__ inline uint32_t hw_f2h(float x) { return (uint32_t)__builtin_bit_cast(uint16_t, (_Float16)x); }

// Blocks are dealt to the 8 XCDs round-robin by hardware; remap the block
// index so that XCD k receives a contiguous 1/8 of the tiles, keeping
// neighbouring tiles in one L2.
__device__ inline uint32_t xcd_remap(uint32_t bid, uint32_t nblocks)
{
    uint32_t per = nblocks / 8u;
    if (per == 0u || bid >= per * 8u) return bid;
    return (bid & 7u) * per + (bid >> 3);
}

// The tile of a block in a launch of one block per tile: XCD k takes the
// k-th eighth of the tiles in strip order.
__device__ inline TileXY screen_tile(uint32_t tx, uint32_t ty)
{
    return strip_tile(xcd_remap(blockIdx.x, tx * ty), tx, ty);
}

// The same for the denoisers' passes over 32x8 tiles, in their order.
__device__ inline TileXY pass_tile(int W, int H)
{
    const uint32_t tx = (uint32_t)(W + 31) / 32u, ty = (uint32_t)(H + 7) / 8u;
    return pass_tile_at(xcd_remap(blockIdx.x, tx * ty), tx, ty, (uint32_t)(W - 1) % 32u < 7u);
}

}  // namespace vpt
