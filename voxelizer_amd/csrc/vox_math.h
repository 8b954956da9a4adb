// vox_math.h -- device-side arithmetic of the voxelizer, in the operation
// order of the reference's expressions (FP64 solid stage, FP32 surface stage).
// Compiled with -ffp-contract=off: no FMA contraction anywhere.
#pragma once

#include <hip/hip_runtime.h>
#include <stdint.h>

#define VOX_DBL_MIN 2.2250738585072014e-308

namespace vk {

struct D2 { double x, y; };
struct D3 { double x, y, z; };
struct F2 { float x, y; };
struct F3 { float x, y, z; };
struct I3 { int32_t x, y, z; };

__device__ __forceinline__ D3 dsub(D3 a, D3 b) { return {a.x - b.x, a.y - b.y, a.z - b.z}; }
__device__ __forceinline__ F3 fsub(F3 a, F3 b) { return {a.x - b.x, a.y - b.y, a.z - b.z}; }
// cross(a, b) = (a.y*b.z - a.z*b.y, a.z*b.x - a.x*b.z, a.x*b.y - a.y*b.x)
__device__ __forceinline__ D3 dcross(D3 a, D3 b) {
    return {a.y * b.z - a.z * b.y, a.z * b.x - a.x * b.z, a.x * b.y - a.y * b.x};
}
__device__ __forceinline__ F3 fcross(F3 a, F3 b) {
    return {a.y * b.z - a.z * b.y, a.z * b.x - a.x * b.z, a.x * b.y - a.y * b.x};
}
// dot evaluated left to right
__device__ __forceinline__ float fdot3(F3 a, F3 b) { return a.x * b.x + a.y * b.y + a.z * b.z; }

// Saturating conversions (truncate toward zero, clamp, NaN -> 0), the
// semantics of the hardware float->int conversions on both vendors.
__device__ __forceinline__ int32_t sat_i32(double v) {
    if (v != v) return 0;
    if (v >= 2147483648.0) return INT32_MAX;
    if (v <= -2147483649.0) return INT32_MIN;
    return (int32_t)v;
}
__device__ __forceinline__ uint32_t sat_u32(double v) {
    if (v != v) return 0u;
    if (v >= 4294967296.0) return UINT32_MAX;
    if (v <= -1.0) return 0u;
    return (uint32_t)v;
}
// sat_i32((double)v) without the double: v_cvt_i32_f32 truncates, saturates
// and returns 0 for NaN (a C++ conversion leaves those cases undefined).
__device__ __forceinline__ int32_t f2i(float v) {
    int32_t r;
    asm("v_cvt_i32_f32 %0, %1" : "=v"(r) : "v"(v));
    return r;
}

__device__ __forceinline__ F3 fetch_f(const float *__restrict__ V, const uint32_t *__restrict__ I,
                                      uint32_t t, int k) {
    uint32_t i = I[3u * t + (uint32_t)k];
    return {V[3u * i], V[3u * i + 1u], V[3u * i + 2u]};
}

// ---------------------------------------------------------------------------
// Solid stage (FP64)
// ---------------------------------------------------------------------------

// Work-queue filter of one triangle for a y/z subspace [smin, smax):
// ext voxel range of its yz bounding box intersected with the subspace
// ("commonSpace"), its 4x4 tile range, and edge functions oriented by the
// reference's tN expression (src/voxelizer.cu:861-945).
struct TileSetup {
    D2 ne[3];
    double de[3];
    uint32_t cmin[2], cmax[2];
    uint32_t tmin[2], tmax[2];
};

// x component of the normal in the reference's own expression
// (src/voxelizer.cu:882-884) and the edge functions it orients.
__device__ __forceinline__ double tri_tN(const D3 v[3]) {
    return (v[0].y * v[1].z + v[2].y * v[0].z + v[2].z * v[1].y) -
           (v[2].y * v[1].z + v[0].z * v[1].y + v[2].z * v[0].y);
}
__device__ __forceinline__ void edges_by_sign(const D3 v[3], bool pos, TileSetup &ts) {
#pragma unroll
    for (int i = 0; i < 3; i++) {
        const D3 a = v[i], b = v[(i + 1) % 3];
        if (pos)
            ts.ne[i] = {a.z - b.z, b.y - a.y};
        else
            ts.ne[i] = {b.z - a.z, a.y - b.y};
        ts.de[i] = -(ts.ne[i].x * a.y + ts.ne[i].y * a.z);
    }
}
// Edge functions only (the commonSpace box comes from the setup pass).
__device__ __forceinline__ void tile_edges(const D3 v[3], TileSetup &ts) {
    edges_by_sign(v, tri_tN(v) > 0.0, ts);
}

__device__ __forceinline__ bool tile_setup(const D3 v[3], double emy, double emz, double d,
                                           uint32_t sminy, uint32_t sminz, uint32_t smaxy,
                                           uint32_t smaxz, TileSetup &ts) {
    D2 bmin = {v[0].y, v[0].z}, bmax = bmin;
#pragma unroll
    for (int i = 1; i < 3; i++) {
        bmin.x = v[i].y < bmin.x ? v[i].y : bmin.x;
        bmin.y = v[i].z < bmin.y ? v[i].z : bmin.y;
        bmax.x = v[i].y > bmax.x ? v[i].y : bmax.x;
        bmax.y = v[i].z > bmax.y ? v[i].z : bmax.y;
    }
    double vb0 = (bmin.x - emy) / d, vb1 = (bmin.y - emz) / d;
    double vb2 = (bmax.x - emy) / d, vb3 = (bmax.y - emz) / d;
    int32_t vmin0 = sat_i32(ceil(vb0)), vmin1 = sat_i32(ceil(vb1));
    int32_t vmax0 = sat_i32(floor(vb2) + 1.0), vmax1 = sat_i32(floor(vb3) + 1.0);
    const double tN = tri_tN(v);
    if (tN == 0.0) return false;
    if (vmin0 >= vmax0 || vmin1 >= vmax1) return false;
    if (vmax0 <= (int32_t)sminy || vmax1 <= (int32_t)sminz) return false;
    if (vmin0 >= (int32_t)smaxy || vmin1 >= (int32_t)smaxz) return false;
    ts.cmin[0] = (uint32_t)max((int32_t)sminy, vmin0);
    ts.cmin[1] = (uint32_t)max((int32_t)sminz, vmin1);
    ts.cmax[0] = min(smaxy, (uint32_t)vmax0);
    ts.cmax[1] = min(smaxz, (uint32_t)vmax1);
    edges_by_sign(v, tN > 0.0, ts);
    ts.tmin[0] = ts.cmin[0] / 4u;
    ts.tmin[1] = ts.cmin[1] / 4u;
    ts.tmax[0] = (ts.cmax[0] - 1u) / 4u;
    ts.tmax[1] = (ts.cmax[1] - 1u) / 4u;
    return true;
}

// Tile (ty, tz) is queued if a voxel centre of it inside commonSpace passes
// all three (>= 0) edge tests (src/voxelizer.cu:998-1031).
__device__ __forceinline__ bool tile_hit(const TileSetup &ts, uint32_t ty, uint32_t tz,
                                         double emy, double emz, double d) {
    bool hit = false;
    for (uint32_t i = ty * 4u; i < ty * 4u + 4u && i < ts.cmax[0] && !hit; i++) {
        for (uint32_t j = tz * 4u; j < tz * 4u + 4u && j < ts.cmax[1] && !hit; j++) {
            if (i >= ts.cmin[0] && j >= ts.cmin[1]) {
                double px = double(i) * d + emy;
                double py = double(j) * d + emz;
                bool r = true;
#pragma unroll
                for (int k = 0; k < 3; k++)
                    r &= (ts.ne[k].x * px + ts.ne[k].y * py + ts.de[k] >= 0.0);
                hit = r;
            }
        }
    }
    return hit;
}

// Per-triangle data of the centre test (src/voxelizer.cu:1334-1372).  th: the
// DBL_MIN top-left tie break; r + DBL_MIN > 0 exactly where r > -DBL_MIN (the
// sign of a rounded sum is that of the exact one).
struct FillSetup {
    D3 n;
    D2 ne[3];
    double de[3], th[3];
};
__device__ __forceinline__ void fill_setup(const D3 v[3], FillSetup &fs) {
    fs.n = dcross(dsub(v[0], v[2]), dsub(v[1], v[0]));
#pragma unroll
    for (int i = 0; i < 3; i++) {
        const D3 a = v[i], b = v[(i + 1) % 3];
        if (fs.n.x > 0.0)
            fs.ne[i] = {a.z - b.z, b.y - a.y};
        else
            fs.ne[i] = {b.z - a.z, a.y - b.y};
        fs.de[i] = -(fs.ne[i].x * a.y + fs.ne[i].y * a.z);
        fs.th[i] = fs.ne[i].x > 0.0 || (fs.ne[i].x == 0.0 && fs.ne[i].y < 0.0) ? -VOX_DBL_MIN : 0.0;
    }
}
// Centre test (src/voxelizer.cu:1418-1436) at the centre (px, py).
__device__ __forceinline__ bool fill_inside(const FillSetup &fs, double px, double py) {
    bool in = true;
#pragma unroll
    for (int i = 0; i < 3; i++) in &= fs.ne[i].x * px + fs.ne[i].y * py + fs.de[i] > fs.th[i];
    return in;
}
// x crossing (src/voxelizer.cu:1437-1453) there, +1 for the x padding; ax: the
// first vertex's x from the grid's origin, times n.x; y0, z0: its y and z.
__device__ __forceinline__ uint32_t fill_crossing(const D3 &n, double ax, double y0, double z0,
                                                  double px, double py, double d) {
    const double ay = y0 - px, az = z0 - py;
    const double B = ax + ay * n.y + az * n.z;
    double x = B / n.x;
    x = x < 0.0 ? 0.0 : x;
    return sat_u32(ceil(x / d)) + 1u;
}

// ---------------------------------------------------------------------------
// Surface stage (FP32)
// ---------------------------------------------------------------------------
enum { BB_DEGEN = 0, BB_1D = 1, BB_2D = 2, BB_3D = 3 };
enum { AX_X = 0, AX_Y = 1, AX_Z = 2 };

struct VoxBB { I3 min, max; };

__device__ __forceinline__ void tri_bounds(const F3 t[3], F3 &mn, F3 &mx) {
    mn = t[0];
    mx = t[0];
#pragma unroll
    for (int i = 1; i < 3; i++) {
        if (t[i].x < mn.x) mn.x = t[i].x;
        if (t[i].y < mn.y) mn.y = t[i].y;
        if (t[i].z < mn.z) mn.z = t[i].z;
        if (t[i].x > mx.x) mx.x = t[i].x;
        if (t[i].y > mx.y) mx.y = t[i].y;
        if (t[i].z > mx.z) mx.z = t[i].z;
    }
}
// x / b, correctly rounded, from y = 1 / b correctly rounded: after the first
// correction the quotient is within one unit in the last place, and from there
// Markstein's theorem makes the second correction's result the rounded quotient
// (P. Markstein, IBM J. Res. Dev. 34, 1990), provided nothing overflows; a
// numerator so small that the residuals lose bits keeps its quotient tiny.  5
// instructions in place of the 11 (one of them quarter rate) of a division.
__device__ __forceinline__ float div_by(float x, float b, float y) {
    float q = x * y;
    q = __builtin_fmaf(__builtin_fmaf(-b, q, x), y, q);
    return __builtin_fmaf(__builtin_fmaf(-b, q, x), y, q);
}

// getVoxelBoundsHalf (src/voxelizer.cu:2471-2492).
__device__ __forceinline__ VoxBB voxel_bounds_half(F3 mn, F3 mx, F3 m, float d) {
    VoxBB b;
    b.min = {f2i(ceilf((mn.x - m.x) / d - 0.5f)), f2i(ceilf((mn.y - m.y) / d - 0.5f)),
             f2i(ceilf((mn.z - m.z) / d - 0.5f))};
    b.max = {f2i(floorf((mx.x - m.x) / d + 0.5f)), f2i(floorf((mx.y - m.y) / d + 0.5f)),
             f2i(floorf((mx.z - m.z) / d + 0.5f))};
    return b;
}
// The same with div_by (rd = 1 / d).
__device__ __forceinline__ VoxBB voxel_bounds_half_by(F3 mn, F3 mx, F3 m, float d, float rd) {
    VoxBB b;
    b.min = {f2i(ceilf(div_by(mn.x - m.x, d, rd) - 0.5f)),
             f2i(ceilf(div_by(mn.y - m.y, d, rd) - 0.5f)),
             f2i(ceilf(div_by(mn.z - m.z, d, rd) - 0.5f))};
    b.max = {f2i(floorf(div_by(mx.x - m.x, d, rd) + 0.5f)),
             f2i(floorf(div_by(mx.y - m.y, d, rd) + 0.5f)),
             f2i(floorf(div_by(mx.z - m.z, d, rd) + 0.5f))};
    return b;
}
__device__ __forceinline__ float vox_corner(int32_t c, float m, float d) {
    return m + (float(c) - 0.5f) * d;
}

// classifyTriangles + analyzeBoundingBox: class (0..3) and dominant axis,
// from the triangle's unclipped voxel range vb (voxel_bounds_half of its
// bounds).
__device__ __forceinline__ void classify_vb(const F3 t[3], const VoxBB &vb, int &bb, int &axis) {
    F3 n = fcross(fsub(t[0], t[2]), fsub(t[1], t[0]));
    if (!(n.x != 0.0f || n.y != 0.0f || n.z != 0.0f)) {
        bb = BB_DEGEN;
        axis = AX_X;
        return;
    }
    int32_t dx = vb.max.x - vb.min.x, dy = vb.max.y - vb.min.y, dz = vb.max.z - vb.min.z;
    if (dx == 0) {
        if (dy == 0) {
            bb = BB_1D;
            axis = dz == 0 ? AX_X : AX_Z;
        } else if (dz == 0) {
            bb = BB_1D;
            axis = AX_Y;
        } else {
            bb = BB_2D;
            axis = AX_X;
        }
    } else if (dy == 0) {
        if (dz == 0) {
            bb = BB_1D;
            axis = AX_X;
        } else {
            bb = BB_2D;
            axis = AX_Y;
        }
    } else if (dz == 0) {
        bb = BB_2D;
        axis = AX_Z;
    } else {
        bb = BB_3D;
        float ax = fabsf(n.x), ay = fabsf(n.y), az = fabsf(n.z);
        if (ax > ay && ax > az)
            axis = AX_X;
        else if (ay > ax && ay > az)
            axis = AX_Y;
        else
            axis = AX_Z;
    }
}

// setup{YZ,ZX,XY}OverlapTest (src/voxelizer.cu:2677-2757) for one edge a -> b
// of a triangle projected to the plane's (first, second) coordinates, pos =
// (normal component along the plane's axis >= 0).
__device__ __forceinline__ void overlap_edge(float a0, float a1, float b0, float b1, bool pos,
                                             float d, float &ne0, float &ne1, float &de) {
    const float s0 = a1 - b1, s1 = b0 - a0;  // exact negations below
    ne0 = pos ? s0 : -s0;
    ne1 = pos ? s1 : -s1;
    de = -(ne0 * a0 + ne1 * a1) + fmaxf(0.0f, d * ne0) + fmaxf(0.0f, d * ne1);
}
// The t for which x + de >= 0 and x >= t agree for every x: the sign of a
// rounded sum is that of the exact one, so t = -de; an infinite de takes its
// sum's value with the other infinity (NaN: false), and a NaN de is never met.
__device__ __forceinline__ float overlap_bound(float de) {
    return de == __builtin_inff()    ? -3.402823466e38f
           : de == -__builtin_inff() ? __builtin_nanf("")
                                     : -de;
}

// ---------------------------------------------------------------------------
// PartialNode volume ratio: processVoxel<PartialNode> (src/voxelizer.cu:
// 2997-3033) with calculateVoxelPlaneIntersectionVolume (4220-4307),
// boxParallelCutVolume (4313-4326), constructPolyhedronFaces (4333-4537),
// volumeOfPolyhedron (4548-4706), rotX / rotY (4719-4757) and
// volumeOfPyramid (4764-4785), FP32 in the reference's operation order.
// length(float2) is sqrt(x*x + y*y) and normalize(v) is v * rsqrt(dot(v, v))
// with rsqrt = 1 / sqrt: correctly rounded divide and square root.
// ---------------------------------------------------------------------------
__device__ __forceinline__ F3 fadd3(F3 a, F3 b) { return {a.x + b.x, a.y + b.y, a.z + b.z}; }
__device__ __forceinline__ F3 fscale3(float s, F3 a) { return {s * a.x, s * a.y, s * a.z}; }
__device__ __forceinline__ F3 rot_x(F3 v, float s, float c) {
    return {v.x, v.y * c - v.z * s, v.y * s + v.z * c};
}
__device__ __forceinline__ F3 rot_y(F3 v, float s, float c) {
    return {v.x * c + v.z * s, v.y, v.z * c - v.x * s};
}
__device__ __forceinline__ float len2f(float a, float b) { return sqrtf(a * a + b * b); }

// Turns the polygon and the apex so that rotN points along z, then returns
// the pyramid's volume (surveyor's formula times a third of the height).  The
// polygon is the points of pt with their `on` flag set, in order: with every
// index a constant the points stay in registers, where a list with a running
// count would live in scratch memory.
__device__ __forceinline__ float turned_pyramid(const F3 (&pt)[6], const bool (&on)[6], F3 rotN,
                                                F3 apex) {
    F3 h = apex;
    float sx = 0.0f, cx = 0.0f, sy = 0.0f, cy = 0.0f;
    const bool turn_x = rotN.y != 0.0f;
    if (turn_x) {
        const float pl = len2f(rotN.y, rotN.z);
        sx = rotN.y / pl;
        cx = rotN.z / pl;
        h = rot_x(h, sx, cx);
        rotN = rot_x(rotN, sx, cx);
    }
    const bool turn_y = rotN.x != 0.0f;
    if (turn_y) {
        const float pl = len2f(rotN.z, rotN.x);
        sy = -rotN.x / pl;
        cy = rotN.z / pl;
        h = rot_y(h, sy, cy);
    }
    float area = 0.0f, z0 = 0.0f;  // an empty polygon keeps area 0 and height h.z
    F3 first = {0.0f, 0.0f, 0.0f}, prev = first;
    bool any = false;
#pragma unroll
    for (int i = 0; i < 6; i++) {
        if (!on[i]) continue;
        F3 q = pt[i];
        if (turn_x) q = rot_x(q, sx, cx);
        if (turn_y) q = rot_y(q, sy, cy);
        if (any)
            area += 0.5f * (prev.x * q.y - q.x * prev.y);
        else {
            first = q;
            z0 = q.z;
        }
        prev = q;
        any = true;
    }
    if (any) area += 0.5f * (prev.x * first.y - first.x * prev.y);
    return fabsf((1.0f / 3.0f) * area * (h.z - z0));
}

// Volume of the pyramid over one face of the cut box (nothing for fewer than
// three points); the normal comes from its first three points.
__device__ __forceinline__ void face_pyramid(const F3 (&pt)[6], const bool (&on)[6], F3 apex,
                                             float &vol) {
    F3 p[3] = {{0.0f, 0.0f, 0.0f}, {0.0f, 0.0f, 0.0f}, {0.0f, 0.0f, 0.0f}};
    int n = 0;
#pragma unroll
    for (int i = 0; i < 6; i++)
        if (on[i]) {
#pragma unroll
            for (int k = 0; k < 3; k++)
                if (n == k) p[k] = pt[i];
            n++;
        }
    if (n > 2) {
        const F3 e = fcross(fsub(p[0], p[2]), fsub(p[1], p[0]));
        const float inv = 1.0f / sqrtf(fdot3(e, e));
        vol += turned_pyramid(pt, on, F3{e.x * inv, e.y * inv, e.z * inv}, apex);
    }
}

// Volume the reference computes for the box centred at m + d * node, cut by
// the plane through t0 with normal n (the part the normal points into for
// a plane through the box).
__device__ __forceinline__ float cut_volume(F3 t0, const int32_t node[3], F3 n, F3 m, float d) {
    const F3 vc = fadd3(m, fscale3(d, F3{float(node[0]), float(node[1]), float(node[2])}));
    if (fabsf(n.x) == 1.0f) return (d * d) * ((d / 2.0f) + t0.x - vc.x);
    if (fabsf(n.y) == 1.0f) return (d * d) * ((d / 2.0f) + t0.y - vc.y);
    if (fabsf(n.z) == 1.0f) return (d * d) * ((d / 2.0f) + t0.z - vc.z);
    const bool bx = n.x > 0.0f, by = n.y > 0.0f, bz = n.z > 0.0f;
    const float sx = float(!bx) * d + float(bx) * -d, sy = float(!by) * d + float(by) * -d,
                sz = float(!bz) * d + float(bz) * -d;
    const bool even = (int(bx) + int(by) + int(bz)) % 2 == 0;
    const F3 dx = {sx, 0.0f, 0.0f};
    const F3 dy = even ? F3{0.0f, sy, 0.0f} : F3{0.0f, 0.0f, sz};
    const F3 dz = even ? F3{0.0f, 0.0f, sz} : F3{0.0f, sy, 0.0f};
    const float dh = d / 2.0f;
    F3 v[8];
    v[0] = fadd3(vc, F3{dh * float(bx) - dh * float(!bx), dh * float(by) - dh * float(!by),
                        dh * float(bz) - dh * float(!bz)});
    v[1] = fadd3(v[0], dx);
    v[2] = fadd3(v[0], dy);
    v[3] = fadd3(v[0], dz);
    v[4] = fadd3(v[1], dz);
    v[5] = fadd3(v[2], dx);
    v[6] = fadd3(v[3], dy);
    v[7] = fadd3(v[4], dy);
    // Three paths from v0 (edges (0,a), (a,b), (b,7) and (a,c)).  Path k's
    // first crossed edge among the first three is `hit` (0, 1, 2; 3 if none),
    // crossed at ip; qp is the crossing of (a,c), if `cut`.
    constexpr int pa[3] = {1, 2, 3}, pb[3] = {4, 5, 6}, pc[3] = {5, 6, 4};
    F3 ip[3], qp[3];
    int hit[3];
    bool cut[3];
#pragma unroll
    for (int k = 0; k < 3; k++) {
        const F3 va = v[pa[k]], vb = v[pb[k]], vc2 = v[pc[k]];
        ip[k] = F3{0.0f, 0.0f, 0.0f};
        qp[k] = ip[k];
        float t = fdot3(n, fsub(t0, v[0])) / fdot3(n, fsub(va, v[0]));
        if (t < 0.0f || t > 1.0f) {
            t = fdot3(n, fsub(t0, va)) / fdot3(n, fsub(vb, va));
            if (t < 0.0f || t > 1.0f) {
                t = fdot3(n, fsub(t0, vb)) / fdot3(n, fsub(v[7], vb));
                hit[k] = 3;
                if (t >= 0.0f && t <= 1.0f) {
                    hit[k] = 2;
                    ip[k] = fadd3(vb, fscale3(t, fsub(v[7], vb)));
                }
            } else {
                hit[k] = 1;
                ip[k] = fadd3(va, fscale3(t, fsub(vb, va)));
            }
        } else {
            hit[k] = 0;
            ip[k] = fadd3(v[0], fscale3(t, fsub(va, v[0])));
        }
        t = fdot3(n, fsub(t0, va)) / fdot3(n, fsub(vc2, va));
        cut[k] = t >= 0.0f && t <= 1.0f;
        if (cut[k]) qp[k] = fadd3(va, fscale3(t, fsub(vc2, va)));
    }
    // The cut polygon: each path's crossings in path order.
    float vol = 0.0f;
    {
        const F3 pt[6] = {ip[0], qp[0], ip[1], qp[1], ip[2], qp[2]};
        const bool on[6] = {hit[0] < 3, cut[0], hit[1] < 3, cut[1], hit[2] < 3, cut[2]};
        vol += turned_pyramid(pt, on, n, v[0]);
    }
    // Face f: its own path's corners up to the crossing, the crossing and the
    // one of (a,c); and from the path whose third edge it shares (path 1 for
    // face 0, 2 for 1, and 0, walked before its own, for 2) that edge's
    // crossing and corner.
#pragma unroll
    for (int f = 0; f < 3; f++) {
        const int o = f == 2 ? 0 : f + 1;
        const F3 own[4] = {v[pa[f]], v[pb[f]], ip[f], qp[f]};
        const bool own_on[4] = {hit[f] >= 1, hit[f] >= 2, hit[f] == 1 || hit[f] == 2, cut[f]};
        const F3 sh[2] = {ip[o], v[pb[o]]};
        const bool sh_on[2] = {hit[o] == 2, hit[o] >= 2};
        F3 pt[6];
        bool on[6];
#pragma unroll
        for (int i = 0; i < 6; i++) {
            const bool mine = f == 2 ? i >= 2 : i < 4;
            const int q = f == 2 ? (mine ? i - 2 : i) : (mine ? i : i - 4);
            pt[i] = mine ? own[q & 3] : sh[q & 1];
            on[i] = mine ? own_on[q & 3] : sh_on[q & 1];
        }
        face_pyramid(pt, on, v[0], vol);
    }
    return vol;
}

// The ratio stored for the winner triangle t (class bb, 1 = 1D) at node
// coordinates `node` (the padded coordinates processVoxel receives): 1D
// triangles pass a zero normal; NaN is stored as 0x7FC00000.
__device__ __forceinline__ float partial_ratio(const float *__restrict__ V,
                                               const uint32_t *__restrict__ I, uint32_t t,
                                               uint32_t bb, const int32_t node[3], F3 m, float d) {
    const F3 t0 = fetch_f(V, I, t, 0), t1 = fetch_f(V, I, t, 1), t2 = fetch_f(V, I, t, 2);
    const F3 n = bb == 1u ? F3{0.0f, 0.0f, 0.0f} : fcross(fsub(t0, t2), fsub(t1, t0));
    const float vol = cut_volume(t0, node, n, m, d);
    const float r = fabsf(1.0f - vol / (d * d * d));
    return r != r ? __uint_as_float(0x7FC00000u) : r;
}

}  // namespace vk
