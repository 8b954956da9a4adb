// vox_kernels.hip -- HIP kernels of the voxelizer hot path for gfx950.
// The arithmetic of every test follows the reference expressions cited in
// vox_math.h; the data flow (binning, LDS staging, bitwise node stencils) is
// this library's own.
#include "vox_kernels.h"

#include <type_traits>

namespace vk {

// ---------------------------------------------------------------------------
// Scan
// ---------------------------------------------------------------------------
// Every scan writes out[0, n] (exclusive prefix, out[n] = total mod 2^32) and
// out[n + 1] = 1 if the true total reached 2^32 (the 32-bit offsets wrapped),
// else 0; partial sums are kept in 64 bits for that.

// Sum of one value per thread over a 256-thread block, in 64 bits.
__device__ __forceinline__ uint64_t block_sum_u64(uint64_t s) {
    __shared__ uint64_t wsum64[kScanThreads / kWave];
#pragma unroll
    for (int d = kWave / 2; d >= 1; d >>= 1) {
        const uint32_t lo = (uint32_t)__shfl_xor((int)(uint32_t)s, d);
        const uint32_t hi = (uint32_t)__shfl_xor((int)(uint32_t)(s >> 32), d);
        s += ((uint64_t)hi << 32) | lo;
    }
    if ((threadIdx.x & (kWave - 1u)) == 0u) wsum64[threadIdx.x / kWave] = s;
    __syncthreads();
    uint64_t t = 0;
#pragma unroll
    for (uint32_t w = 0; w < kScanThreads / kWave; w++) t += wsum64[w];
    __syncthreads();  // wsum64 may be reused by the caller's next call
    return t;
}

// Block-wide sum and exclusive prefix of one value per thread: a wave scan
// in registers, the four wave totals through LDS (one barrier).
__device__ __forceinline__ uint32_t block_excl_scan(uint32_t s, uint32_t &total) {
    __shared__ uint32_t wsum[kScanThreads / kWave];
    const uint32_t lane = threadIdx.x & (kWave - 1u), wave = threadIdx.x / kWave;
    const uint32_t incl = wave_incl_scan(s);
    if (lane == kWave - 1u) wsum[wave] = incl;
    __syncthreads();
    uint32_t before = 0u;
    total = 0u;
#pragma unroll
    for (uint32_t w = 0; w < kScanThreads / kWave; w++) {
        before += w < wave ? wsum[w] : 0u;
        total += wsum[w];
    }
    return before + incl - s;
}

// Sum over a 256-thread block of up to 2^32 / 256 per thread.
__device__ __forceinline__ uint32_t block_sum_u32(uint32_t s) {
    uint32_t total;
    block_excl_scan(s, total);
    __syncthreads();  // its LDS may be reused
    return total;
}

// A thread's 16 consecutive values of a tile (0 past n), in 16-byte loads.
__device__ __forceinline__ void scan_load(const uint32_t *in, uint32_t n, uint64_t base,
                                          uint32_t v[kScanItems]) {
    if (base + kScanItems <= n) {
#pragma unroll
        for (int q = 0; q < kScanItems / 4; q++) {
            const uint4 x = reinterpret_cast<const uint4 *>(in + base)[q];
            v[4 * q] = x.x;
            v[4 * q + 1] = x.y;
            v[4 * q + 2] = x.z;
            v[4 * q + 3] = x.w;
        }
    } else {
#pragma unroll
        for (int k = 0; k < kScanItems; k++) v[k] = base + k < n ? in[base + k] : 0u;
    }
}

// Tile sums of each segment's in[0, n) (blockIdx.y: the segment):
// low words in part[0, npart), high words in part[npart, 2 * npart) and, with a
// list, the nonzero entries in part[2 * npart, 3 * npart).
__global__ __launch_bounds__(kScanThreads) void k_scan_reduce(ScanSegs segs) {
    const ScanSeg &S = segs.s[blockIdx.y];
    if (blockIdx.x >= S.npart) return;  // uniform
    const uint64_t base = (uint64_t)blockIdx.x * kScanTile + (uint64_t)threadIdx.x * kScanItems;
    uint32_t v[kScanItems];
    scan_load(S.in, S.n, base, v);
    uint64_t s = 0u;
    uint32_t nz = 0u;
#pragma unroll
    for (int k = 0; k < kScanItems; k++) {
        s += v[k];
        nz += v[k] != 0u ? 1u : 0u;
    }
    const uint64_t total = block_sum_u64(s);
    if (S.list) nz = block_sum_u32(nz);
    if (threadIdx.x == 0) {
        S.part[blockIdx.x] = (uint32_t)total;
        S.part[S.npart + blockIdx.x] = (uint32_t)(total >> 32);
        if (S.list) S.part[2u * S.npart + blockIdx.x] = nz;
    }
}

// Exclusive scan of each segment's in[0, n) into out[0, n] (out[n] = total):
// a tile first adds the sums before it: those in part, each of
// 1 / per_tile of a tile, or with per_tile = 0 (at most kScanSmallTiles tiles)
// the values themselves.  The last tile also adds them in 64 bits and writes
// the wrap flag, and both to `host` if given.  in may be out.  With a list, the
// indices of the nonzero entries go there in order, their number to *n_list.
__global__ __launch_bounds__(kScanThreads) void k_scan_down(ScanSegs segs) {
    const ScanSeg &S = segs.s[blockIdx.y];
    const uint32_t n = S.n, tiles = n / kScanTile + 1u;
    if (blockIdx.x >= tiles) return;  // uniform
    const bool last = blockIdx.x == tiles - 1u, listed = S.list != nullptr;
    uint32_t p = 0u, pz = 0u;
    uint64_t p64 = 0u;
    if (S.per_tile) {
        const uint32_t before = min(blockIdx.x * S.per_tile, S.npart);
#pragma unroll 4
        for (uint32_t i = threadIdx.x; i < before; i += kScanThreads) {
            const uint32_t v = S.part[i];
            p += v;
            if (last) p64 += ((uint64_t)S.part[S.npart + i] << 32) | v;
            if (listed) pz += S.part[2u * S.npart + i];
        }
    } else {
        for (uint32_t b = 0; b < blockIdx.x; b++) {
            uint32_t v[kScanItems];
            scan_load(S.in, n, (uint64_t)b * kScanTile + threadIdx.x * kScanItems, v);
#pragma unroll
            for (int k = 0; k < kScanItems; k++) {
                p += v[k];
                if (last) p64 += v[k];
                pz += v[k] != 0u ? 1u : 0u;
            }
        }
    }
    const uint32_t off = block_sum_u32(p);
    const uint32_t zoff = listed ? block_sum_u32(pz) : 0u;
    const uint64_t base = (uint64_t)blockIdx.x * kScanTile + (uint64_t)threadIdx.x * kScanItems;
    uint32_t v[kScanItems];
    scan_load(S.in, n, base, v);
    uint32_t s = 0u, nz = 0u;
#pragma unroll
    for (int k = 0; k < kScanItems; k++) {
        s += v[k];
        nz += v[k] != 0u ? 1u : 0u;
        if (last) p64 += v[k];
    }
    uint32_t total;
    uint32_t excl = off + block_excl_scan(s, total);
    uint32_t e[kScanItems];
#pragma unroll
    for (int k = 0; k < kScanItems; k++) {
        e[k] = excl;
        excl += v[k];
    }
    if (base + kScanItems <= n) {
#pragma unroll
        for (int q = 0; q < kScanItems / 4; q++)
            reinterpret_cast<uint4 *>(S.out + base)[q] =
                make_uint4(e[4 * q], e[4 * q + 1], e[4 * q + 2], e[4 * q + 3]);
    } else {
#pragma unroll
        for (int k = 0; k < kScanItems; k++)
            if (base + k <= n) S.out[base + k] = e[k];
    }
    if (listed) {
        __syncthreads();  // block_excl_scan's LDS
        uint32_t ztotal;
        uint32_t at = zoff + block_excl_scan(nz, ztotal);
#pragma unroll
        for (int k = 0; k < kScanItems; k++)
            if (v[k] != 0u) S.list[at++] = (uint32_t)base + (uint32_t)k;
        if (last && threadIdx.x == 0) *S.n_list = zoff + ztotal;
    }
    if (last) {  // uniform
        const uint64_t all = block_sum_u64(p64);
        if (threadIdx.x == 0) {
            const uint32_t wrap = (all >> 32) != 0u ? 1u : 0u;
            S.out[(uint64_t)n + 1u] = wrap;
            if (S.host) {
                S.host[0] = (uint32_t)all;
                S.host[1] = wrap;
            }
        }
    }
}

// ---------------------------------------------------------------------------
// Bounding box: order-preserving uint keys of the float coordinates, six per
// block, left to the host to join (in its own memory: no clear, no atomics, no
// copy back).
// ---------------------------------------------------------------------------
__device__ __forceinline__ uint32_t fkey(float f) {
    uint32_t u = __float_as_uint(f);
    return (u & 0x80000000u) ? ~u : (u | 0x80000000u);
}

__global__ __launch_bounds__(256) void k_bbox(const float *__restrict__ V, uint32_t nv,
                                              uint32_t *__restrict__ out) {
    uint32_t mn[3] = {UINT32_MAX, UINT32_MAX, UINT32_MAX}, mx[3] = {0u, 0u, 0u};
    for (uint32_t i = blockIdx.x * blockDim.x + threadIdx.x; i < nv; i += gridDim.x * blockDim.x) {
#pragma unroll
        for (int c = 0; c < 3; c++) {
            uint32_t k = fkey(V[3u * i + c]);
            mn[c] = min(mn[c], k);
            mx[c] = max(mx[c], k);
        }
    }
#pragma unroll
    for (int c = 0; c < 3; c++) {
        for (int off = 32; off > 0; off >>= 1) {
            mn[c] = min(mn[c], (uint32_t)__shfl_xor((int)mn[c], off));
            mx[c] = max(mx[c], (uint32_t)__shfl_xor((int)mx[c], off));
        }
    }
    // Block reduction through LDS.
    __shared__ uint32_t red[6][256 / kWave];
    const uint32_t wv = threadIdx.x / kWave;
    if (lane_id() == 0) {
#pragma unroll
        for (int c = 0; c < 3; c++) {
            red[c][wv] = mn[c];
            red[3 + c][wv] = mx[c];
        }
    }
    __syncthreads();
    if (threadIdx.x < 6) {
        const int c = threadIdx.x;
        uint32_t r = red[c][0];
        for (uint32_t k = 1; k < blockDim.x / kWave; k++)
            r = c < 3 ? min(r, red[c][k]) : max(r, red[c][k]);
        out[6u * blockIdx.x + c] = r;
    }
}

// ---------------------------------------------------------------------------
// Solid stage
// ---------------------------------------------------------------------------
// The triangle's vertices widened to FP64 (fetchTriangleVertices,
// src/voxelizer.cu:2242-2253), from its 48-byte record.
__device__ __forceinline__ void load_tri_d(const SolidParams &p, uint32_t t, D3 v[3]) {
    const float4 r0 = p.rec[3 * (size_t)t], r1 = p.rec[3 * (size_t)t + 1],
                 r2 = p.rec[3 * (size_t)t + 2];
    v[0] = {(double)r0.x, (double)r0.y, (double)r0.z};
    v[1] = {(double)r0.w, (double)r1.x, (double)r1.y};
    v[2] = {(double)r1.z, (double)r1.w, (double)r2.x};
}

// Block starts of the candidate passes: first[b] = the triangle that holds
// candidate 256*b (the passes' blocks take 256 consecutive candidates), so a
// block bounds its triangles with two loads instead of a binary search over
// the whole offset array (about 21 dependent loads on the large hall).
// Candidates at or past `cap` are not processed.  blockIdx.y: the pass.
__global__ __launch_bounds__(256) void k_block_starts(BlockStarts a, BlockStarts b,
                                                      uint32_t nslots) {
    const BlockStarts &S = blockIdx.y ? b : a;
    const uint32_t total = S.off[nslots + 1u] ? 0u : min(S.off[nslots], S.cap);
    for (uint32_t t = blockIdx.x * 256u + threadIdx.x; t < nslots; t += gridDim.x * 256u) {
        const uint32_t lo = min(S.off[t], total), hi = min(S.off[t + 1u], total);
        for (uint32_t k = cand_blocks(lo); k < cand_blocks(hi); k++) S.first[k] = t;
    }
}

// The triangle of candidate 256 k + threadIdx.x, for a 256-thread block, among
// the n from that of its first candidate to that of the next block's first.
// Triangles without candidates count in n: where most of the mesh has none (a
// slice, a thin partition), a block beside such a run has most of the mesh there.
//
// Up to 256, a triangle per thread: those that start among the block's candidates
// leave their number where they start, and a running maximum over the block
// spreads them: one coalesced load and one scan, where a search takes eight
// dependent loads.  Triangles without candidates start where the next one does
// and lose to its larger number.  Above 256 every thread searches for the last
// triangle that starts at or before its candidate: 256 samples through LDS, then
// log2(n / 256) dependent loads.
//
// The hall (1.4 M triangles), calls with a walk of the n in steps of 256 instead,
// with one up to 1024 and with this: z slice at 800 voxels 3281, 301, 302 us (up
// to 5390 steps), x slice at 400 1664, 577, 573 us, solid bits at 400 246, 213,
// 212 us, at 1100 243, 234, 232 us, ShortNodes at 1533 1428, 1432, 1431 us.
__device__ __forceinline__ uint32_t block_owner(const uint32_t *__restrict__ off,
                                                const uint32_t *__restrict__ first,
                                                uint32_t nslots, uint32_t k, uint32_t total,
                                                CandLds &L) {
    const uint32_t base = k * 256u, nb = cand_blocks(total);
    const uint32_t t0 = first[k], t1 = k + 1u < nb ? first[k + 1u] : nslots - 1u;
    const uint32_t n = t1 - t0 + 1u;
    if (n > 256u) {  // uniform
        const uint32_t c = min(base + threadIdx.x, total - 1u);
        const uint32_t step = (n + 255u) / 256u, s = t0 + threadIdx.x * step;
        L.own[threadIdx.x] = s <= t1 ? off[s] : UINT32_MAX;
        __syncthreads();
        uint32_t i = 0u;
#pragma unroll
        for (uint32_t d = 128u; d; d >>= 1)
            if (L.own[i + d] <= c) i += d;
        uint32_t lo = t0 + i * step, hi = min(lo + step, t1 + 1u);
        while (lo + 1u < hi) {
            const uint32_t mid = (lo + hi) >> 1;
            if (off[mid] <= c)
                lo = mid;
            else
                hi = mid;
        }
        return lo;
    }
    L.own[threadIdx.x] = threadIdx.x == 0u ? t0 : 0u;
    __syncthreads();
    if (threadIdx.x < n) {
        const uint32_t o = off[t0 + threadIdx.x] - base;
        if (o < 256u) atomicMax(&L.own[o], t0 + threadIdx.x);
    }
    __syncthreads();
    const uint32_t incl = wave_incl_max(L.own[threadIdx.x]);
    const uint32_t wave = threadIdx.x / kWave;
    if (lane_id() == kWave - 1u) L.wmax[wave] = incl;
    __syncthreads();
    uint32_t t = incl;
#pragma unroll
    for (uint32_t w = 0; w + 1u < 256u / kWave; w++) t = max(t, w < wave ? L.wmax[w] : 0u);
    return t;
}

// Rows of tile (ty, tz) whose voxSplitRes subspace queues the triangle (bit
// r = centre (4 ty + (r & 3), 4 tz + (r >> 2))).  The reference builds its
// queue per y/z subspace (src/host_side.cpp:275-397): a tile is queued for a
// subspace when one of its centres inside that subspace passes the (>= 0)
// filter (src/voxelizer.cu:880-925, 998-1031), and the fill then tests only
// that subspace's centres.  So a centre's crossing counts only when some
// centre of the same subspace part of the tile passes.  sy/sz: the subspace
// start flags of the ext rows (Job::sstart).
__device__ __forceinline__ uint32_t tile_split_mask(const TileSetup &ts, uint32_t ty, uint32_t tz,
                                                    double emy, double emz, double d,
                                                    const uint8_t *__restrict__ sy, uint32_t ry,
                                                    const uint8_t *__restrict__ sz, uint32_t rz) {
    uint32_t pass = 0u;
#pragma unroll
    for (uint32_t r = 0; r < 16u; r++) {
        const uint32_t i = ty * 4u + (r & 3u), j = tz * 4u + (r >> 2);
        if (i >= ts.cmin[0] && i < ts.cmax[0] && j >= ts.cmin[1] && j < ts.cmax[1]) {
            const double px = double(i) * d + emy;
            const double py = double(j) * d + emz;
            bool ok = true;
#pragma unroll
            for (int k = 0; k < 3; k++)
                ok &= (ts.ne[k].x * px + ts.ne[k].y * py + ts.de[k] >= 0.0);
            pass |= (ok ? 1u : 0u) << r;
        }
    }
    if (!pass) return 0u;
    // Subspace parts of the tile's 4 y rows and 4 z rows: part ids grow by
    // one where a subspace starts.
    uint32_t gy[4], gz[4];
    gy[0] = gz[0] = 0u;
#pragma unroll
    for (uint32_t k = 1; k < 4u; k++) {
        const uint32_t y = ty * 4u + k, z = tz * 4u + k;
        gy[k] = gy[k - 1] + (y < ry && sy[y] ? 1u : 0u);
        gz[k] = gz[k - 1] + (z < rz && sz[z] ? 1u : 0u);
    }
    uint32_t ysame[4], zsame[4];  // rows in the same part as row k (4-bit sets)
#pragma unroll
    for (uint32_t k = 0; k < 4u; k++) {
        ysame[k] = zsame[k] = 0u;
#pragma unroll
        for (uint32_t q = 0; q < 4u; q++) {
            ysame[k] |= (gy[q] == gy[k] ? 1u : 0u) << q;
            zsame[k] |= (gz[q] == gz[k] ? 1u : 0u) << q;
        }
    }
    uint32_t mask = 0u;
#pragma unroll
    for (uint32_t r = 0; r < 16u; r++) {
        if (!((pass >> r) & 1u)) continue;
        const uint32_t ys = ysame[r & 3u], zs = zsame[r >> 2];
        const uint32_t yrows = ys | (ys << 4) | (ys << 8) | (ys << 12);
        const uint32_t zrows = ((zs & 1u) ? 0x000Fu : 0u) | ((zs & 2u) ? 0x00F0u : 0u) |
                               ((zs & 4u) ? 0x0F00u : 0u) | ((zs & 8u) ? 0xF000u : 0u);
        mask |= yrows & zrows;
    }
    return mask;
}

// Counts the block's candidates per bin and returns this one's place in its
// bin: its rank among the block's (LDS table), after those counted before (one
// global atomic per distinct bin).
__device__ __forceinline__ uint32_t bin_place(CandLds &L, bool live, uint32_t bin,
                                              uint32_t *__restrict__ hist) {
    uint32_t slot = 0u, rank = 0u;
    if (live) slot = agg_insert(L.agg, bin, rank);
    __syncthreads();
    for (uint32_t i = threadIdx.x; i < kAggSlots; i += 256u)
        if (L.agg.key[i] != kAggEmpty) L.agg.base[i] = atomicAdd(&hist[L.agg.key[i]], L.agg.cnt[i]);
    __syncthreads();
    return L.agg.base[slot] + rank;
}

// The solid pass's candidates: the reference's per-tile queue test, a thread
// per (triangle, tile) instead of one walking all tiles of a triangle.
template <bool kMulti>
__device__ __forceinline__ void count_solid(const Job *__restrict__ jobs,
                                            const uint32_t *__restrict__ tri_job, uint32_t nslots,
                                            const SolidPairs &a, uint32_t block, uint32_t blocks,
                                            CandLds &L) {
    // off[nslots + 1]: the candidate count reached 2^32 (the offsets wrapped).
    const uint32_t full = a.off[nslots], wrap = a.off[nslots + 1u];
    const uint32_t total = wrap ? 0u : min(full, a.cap);
    if (a.ovf && (full > a.cap || wrap) && block == 0u && threadIdx.x == 0) *a.ovf = 1u;
    for (CandRange r(block, blocks, total); r.more(); r.next()) {
        __syncthreads();
        agg_clear(L.agg);
        const uint32_t c = r.k * 256u + threadIdx.x;
        const uint32_t t = block_owner(a.off, a.first, nslots, r.k, total, L);
        bool hit = false;
        uint32_t tile = 0;
        if (c < total) {
            const Job &J = jobs[kMulti ? tri_job[t] : 0u];
            const SolidParams p = solid_params(J, a.rec);
            D3 v[3];
            load_tri_d(p, t, v);
            TileSetup ts;
            const uint4 cb = a.cbox[t];
            ts.cmin[0] = cb.x;
            ts.cmin[1] = cb.y;
            ts.cmax[0] = cb.z;
            ts.cmax[1] = cb.w;
            tile_edges(v, ts);
            const uint32_t tmin0 = cb.x / 4u, tmin1 = cb.y / 4u, tmax0 = (cb.z - 1u) / 4u;
            const uint32_t w = tmax0 - tmin0 + 1u;
            const uint32_t local = c - a.off[t];
            const uint32_t ty = tmin0 + local % w, tz = tmin1 + local / w;
            if (J.sstart) {  // several y/z subspaces
                const uint32_t m = tile_split_mask(ts, ty, tz, p.emy, p.emz, p.d, J.sstart,
                                                   (uint32_t)J.res[1], J.sstart + J.res[1],
                                                   (uint32_t)J.res[2]);
                hit = m != 0u;
                a.pmask[c] = (uint16_t)m;
            } else {
                hit = tile_hit(ts, ty, tz, p.emy, p.emz, p.d);
            }
            tile = J.tile_base + tz * p.tilesY + ty;
        }
        const uint32_t place = bin_place(L, hit, tile, a.hist);
        // One slot per candidate (no global counter); misses are skipped by
        // the placing pass.
        if (c < total) a.pairs[c] = make_uint2(hit ? tile : UINT32_MAX, place);
    }
}

// Brick of candidate c (of triangle t) of the surface pass.
template <bool kMulti>
__device__ __forceinline__ uint32_t cand_brick(const Job *__restrict__ jobs,
                                               const uint32_t *__restrict__ tri_job,
                                               const SurfPairs &a, uint32_t t, uint32_t c) {
    const Job &J = jobs[kMulti ? tri_job[t] : 0u];
    const uint4 ti = a.tri_info[t];
    const uint32_t bx0 = ti.y & 0xFFFFu, by0 = ti.y >> 16, bz0 = ti.z & 0xFFFFu;
    const uint32_t w0 = ti.z >> 16, w1 = ti.w & 0xFFFFu;
    const uint32_t local = c - a.off[t];
    const uint32_t bx = bx0 + local % w0;
    const uint32_t by = by0 + (local / w0) % w1;
    const uint32_t bz = bz0 + local / (w0 * w1);
    return J.brick_base + (bz * J.nb[1] + by) * J.nb[0] + bx;
}

template <bool kMulti>
__device__ __forceinline__ void count_surf(const Job *__restrict__ jobs,
                                           const uint32_t *__restrict__ tri_job, uint32_t nslots,
                                           const SurfPairs &a, uint32_t block, uint32_t blocks,
                                           CandLds &L) {
    const uint32_t full = a.off[nslots], wrap = a.off[nslots + 1u];
    const uint32_t total = wrap ? 0u : min(full, a.cap);
    if (a.ovf && (full > a.cap || wrap) && block == 0u && threadIdx.x == 0) *a.ovf = 1u;
    for (CandRange r(block, blocks, total); r.more(); r.next()) {
        __syncthreads();
        agg_clear(L.agg);
        const uint32_t c = r.k * 256u + threadIdx.x;
        const uint32_t t = block_owner(a.off, a.first, nslots, r.k, total, L);
        const bool live = c < total;
        const uint32_t b = live ? cand_brick<kMulti>(jobs, tri_job, a, t, c) : 0u;
        const uint32_t place = bin_place(L, live, b, a.hist);
        if (live && a.place) a.place[c] = place;
    }
}

// The counting sorts of (triangle, tile) and (triangle, brick) pairs by tile and
// by brick: this pass counts the pairs of each bin and keeps every pair's place
// in its bin, so the placing pass needs no counters of its own (unless there was
// no room for the bricks' places: then it counts again).  Both sorts
// share a launch: blocks [0, solid_blocks) take the first, the rest the second.
// Bound by the latency of its chain (starts, triangle, table, atomics): eight
// waves a SIMD, which the registers allow, against six, hall 86 -> 77 us.
template <bool kMulti>
__global__ __launch_bounds__(256, 8) void k_pairs_count(const Job *__restrict__ jobs,
                                                     const uint32_t *__restrict__ tri_job,
                                                     uint32_t nslots, SolidPairs a, SurfPairs b,
                                                     uint32_t solid_blocks) {
    __shared__ CandLds L;
    if (blockIdx.x < solid_blocks)
        count_solid<kMulti>(jobs, tri_job, nslots, a, blockIdx.x, solid_blocks, L);
    else
        count_surf<kMulti>(jobs, tri_job, nslots, b, blockIdx.x - solid_blocks,
                           gridDim.x - solid_blocks, L);
}

template <bool kMulti>
__global__ __launch_bounds__(256) void k_pairs_place(const Job *__restrict__ jobs,
                                                     const uint32_t *__restrict__ tri_job,
                                                     uint32_t nslots, SolidPairs a, SurfPairs b,
                                                     uint32_t solid_blocks) {
    __shared__ CandLds L;
    const bool solid = blockIdx.x < solid_blocks;
    const uint32_t block = solid ? blockIdx.x : blockIdx.x - solid_blocks;
    const uint32_t blocks = solid ? solid_blocks : gridDim.x - solid_blocks;
    const uint32_t *off = solid ? a.off : b.off, *first = solid ? a.first : b.first;
    const uint32_t total = off[nslots + 1u] ? 0u : min(off[nslots], solid ? a.cap : b.cap);
    const bool again = !solid && !b.place;
    for (CandRange r(block, blocks, total); r.more(); r.next()) {
        __syncthreads();
        if (again) agg_clear(L.agg);
        const uint32_t c = r.k * 256u + threadIdx.x;
        const uint32_t t = block_owner(off, first, nslots, r.k, total, L);
        if (again) {  // uniform
            const uint32_t brick = c < total ? cand_brick<kMulti>(jobs, tri_job, b, t, c) : 0u;
            const uint32_t place = bin_place(L, c < total, brick, b.cursor);
            if (c < total) b.list[b.bin_off[brick] + place] = t;
            continue;
        }
        if (c >= total) continue;  // the last trip
        if (solid) {
            const uint2 pr = a.pairs[c];
            if (pr.x == UINT32_MAX) continue;
            const uint32_t pos = a.bin_off[pr.x] + pr.y;
            a.list[pos] = t;
            if (a.list_mask) a.list_mask[pos] = a.pmask[c];
        } else {
            b.list[b.bin_off[cand_brick<kMulti>(jobs, tri_job, b, t, c)] + b.place[c]] = t;
        }
    }
}
template __global__ void k_pairs_count<false>(const Job *, const uint32_t *, uint32_t, SolidPairs,
                                              SurfPairs, uint32_t);
template __global__ void k_pairs_count<true>(const Job *, const uint32_t *, uint32_t, SolidPairs,
                                             SurfPairs, uint32_t);
template __global__ void k_pairs_place<false>(const Job *, const uint32_t *, uint32_t, SolidPairs,
                                              SurfPairs, uint32_t);
template __global__ void k_pairs_place<true>(const Job *, const uint32_t *, uint32_t, SolidPairs,
                                             SurfPairs, uint32_t);

// Bit i: parity of the bits above and at i (MSB first: x%32 == 0 is bit 31).
__device__ __forceinline__ uint32_t prefix_xor(uint32_t c) {
    c ^= c >> 1;
    c ^= c >> 2;
    c ^= c >> 4;
    c ^= c >> 8;
    return c ^ (c >> 16);
}

// Zeroes kPadBlock words of the pad rows (y or z at the alloc border).
__device__ __forceinline__ void zero_pad_rows(const Job *__restrict__ jobs,
                                              const uint32_t *__restrict__ pad_bases,
                                              uint32_t njobs, uint32_t block) {
    const Job &J = jobs[job_of(pad_bases, njobs, block)];
    const uint32_t W = J.gd.W, rowsY = J.gd.Y, rowsZ = J.gd.Z;
    const uint32_t i0 = (block - J.pad_base) * kPadBlock, n = pad_words(W, rowsY, rowsZ);
    for (uint32_t i = i0 + threadIdx.x; i < min(i0 + kPadBlock, n); i += kWave) {
        const uint32_t r = i / W, w = i % W;
        uint32_t y, z, bit;
        if (r < 2u * rowsZ) {
            z = r >> 1;
            y = (r & 1u) ? rowsY - 1u : 0u;
            bit = (r & 1u) ? 2u : 1u;
        } else {
            const uint32_t q = r - 2u * rowsZ;
            y = q >> 1;
            z = (q & 1u) ? rowsZ - 1u : 0u;
            bit = (q & 1u) ? 8u : 4u;
        }
        // Rows and planes that are a neighbouring partition's overlap hold
        // voxelized data (written by the fill) instead of padding.
        if (J.padmask & bit) gptr(J.bits)[((size_t)z * rowsY + y) * W + w] = 0u;
    }
}

// One wave per 4x4 tile of voxel-centre rows.  Every queued triangle's
// crossings toggle one bit each in an LDS copy of the tile's 16 rows
// (ds_xor); a per-row prefix XOR then turns crossings into solid runs
// (the suffix flips of src/voxelizer.cu:1487-1616) and each bit word is
// written to HBM once, coalesced, with no global atomics.  The workgroups past
// the tiles clear the pad rows.
//
// Bound by FP64 and integer instructions.  A triangle's lanes test centres, and
// the few that pass (their two divisions cost as much as the tests of four
// centres) are queued in LDS and worked off by full waves; the rows' words are
// taken 64 at a time whatever the row width.  With the divisions in line and a
// step per row: hall (1536x1024x768) 145 -> 111 us, hall at 1100 98 -> 73 us,
// 64-mesh batch 400 -> 210 us (225 with divisions in line), room 512x403x303
// 33 -> 21 us, LongFCC room 640x255x384 55 -> 33 us, 132 large triangles over
// 672x515x387 26 -> 19 us.
__global__ __launch_bounds__(kWave) void k_solid_fill(const Job *__restrict__ jobs,
                                                      const uint32_t *__restrict__ tile_bases,
                                                      const uint32_t *__restrict__ pad_bases,
                                                      uint32_t njobs,
                                                      const float4 *__restrict__ rec,
                                                      const uint32_t *__restrict__ tile_off,
                                                      const uint32_t *__restrict__ tile_hist,
                                                      const uint32_t *__restrict__ list,
                                                      const uint16_t *__restrict__ list_mask) {
    extern __shared__ __align__(16) uint32_t cross[];  // [16][SW]
    __shared__ double tri[6][kWave];     // per lane: its triangle for fill_crossing
    __shared__ uint16_t queue[2 * kWave];  // centres that await their crossing: lane, row
    const uint32_t n_tiles = tile_bases[njobs];
    if (blockIdx.x >= n_tiles) {
        zero_pad_rows(jobs, pad_bases, njobs, blockIdx.x - n_tiles);
        return;
    }
    const Job &J = jobs[job_of(tile_bases, njobs, blockIdx.x)];
    const SolidParams p = solid_params(J, rec);
    VK_G uint32_t *__restrict__ bits = gptr(J.bits);
    const uint32_t W = p.X >> 5;
    // Rows wider than kFillSegWords words are filled a segment at a time:
    // the tile's triangles are walked once per segment, and each row's
    // crossing parity carries from one segment into the next.
    const uint32_t SW = min(W, kFillSegWords);
    const uint32_t tid = threadIdx.x;
    const uint32_t local = blockIdx.x - J.tile_base;
    const uint32_t ty = local % p.tilesY;
    const uint32_t tz = local / p.tilesY;
    const uint32_t tile = blockIdx.x;
    const uint32_t cnt = tile_hist[tile];
    const uint32_t off = tile_off[tile];
    // The tile's 16 rows are split over 2^lg lanes per triangle (the largest
    // lg <= 4 with cnt << lg <= 64), so a tile with few triangles (the
    // median one on large meshes has 8) still keeps the wave's lanes busy;
    // crossings are XORed, so the split does not change the result.
    uint32_t lg = 0;
    while (lg < 4u && cnt <= (kWave >> (lg + 1u))) lg++;
    const uint32_t items = cnt << lg, rows = 16u >> lg;
    const uint32_t lane = tid;
    // Rows that hold voxel centres (bit r; the last tiles reach past the grid).
    const uint32_t ny = min(p.smax[0] - ty * 4u, 4u), nz = min(p.smax[1] - tz * 4u, 4u);
    const uint32_t inside = ((1u << ny) - 1u) * (0x1111u & ((1u << (4u * nz)) - 1u));
    const float rW = 1.0f / (float)W;
    uint32_t carries = 0u;  // bit r: crossing parity of row r before the segment
    for (uint32_t s0 = 0; s0 < W; s0 += SW) {
        const uint32_t sw = min(SW, W - s0);
        uint4 *cross4 = reinterpret_cast<uint4 *>(cross);  // 16 * SW words: 4 * SW uint4
        for (uint32_t i = tid; i < 4u * SW; i += kWave) cross4[i] = make_uint4(0u, 0u, 0u, 0u);
        __syncthreads();
        auto cross_at = [&](uint32_t e) {  // a queued centre's crossing
            const uint32_t k = e >> 4, r = e & 15u;
            const uint32_t cy = ty * 4u + (r & 3u), cz = tz * 4u + (r >> 2);
            const uint32_t vx = fill_crossing({tri[0][k], tri[1][k], tri[2][k]}, tri[3][k],
                                              tri[4][k], tri[5][k], double(cy) * p.d + p.emy,
                                              double(cz) * p.d + p.emz, p.d);
            const uint32_t wx = (vx >> 5) - s0;  // wraps for words before s0
            if (vx < p.X && wx < sw) atomicXor(&cross[r * SW + wx], 1u << (31u - (vx & 31u)));
        };
        for (uint32_t i0 = 0; i0 < items; i0 += kWave) {  // uniform
            const uint32_t i = i0 + lane, at = off + (i >> lg);
            const uint32_t r0 = (i & ((1u << lg) - 1u)) * rows;
            uint32_t rmask = 0u;  // rows to test
            FillSetup fs;
            if (i < items) {
                // Rows whose subspace queued the triangle (all with one subspace).
                rmask = inside & (list_mask ? (uint32_t)list_mask[at] : ~0u);
                D3 v[3];
                load_tri_d(p, list[at], v);
                fill_setup(v, fs);
                tri[0][lane] = fs.n.x;
                tri[1][lane] = fs.n.y;
                tri[2][lane] = fs.n.z;
                tri[3][lane] = (v[0].x - p.emx) * fs.n.x;
                tri[4][lane] = v[0].y;
                tri[5][lane] = v[0].z;
            }
            uint32_t nq = 0u;  // queued centres (uniform)
            for (uint32_t r = r0; r < r0 + rows; r++) {  // `rows` is uniform
                const uint32_t cy = ty * 4u + (r & 3u), cz = tz * 4u + (r >> 2);
                const bool in = ((rmask >> r) & 1u) &&
                                fill_inside(fs, double(cy) * p.d + p.emy, double(cz) * p.d + p.emz);
                const unsigned long long m = __ballot(in);
                if (in)
                    queue[nq + __builtin_amdgcn_mbcnt_hi(
                                   (uint32_t)(m >> 32),
                                   __builtin_amdgcn_mbcnt_lo((uint32_t)m, 0u))] =
                        (uint16_t)(lane << 4 | r);
                nq += (uint32_t)__popcll(m);
                wave_lds_sync();
                if (nq >= (uint32_t)kWave) {
                    nq -= (uint32_t)kWave;
                    cross_at(queue[nq + lane]);
                    wave_lds_sync();
                }
            }
            if (lane < nq) cross_at(queue[lane]);
            wave_lds_sync();
        }
        __syncthreads();
        // Crossing parity -> solid bits (MSB-first bits: x%32 == 0 is bit
        // 31): a prefix XOR inside each word, and across words the parity of
        // the crossings before it (one ballot per 64 words), written
        // straight out.
        if (SW == W) {
            // The 16 rows lie one after another in LDS, so 64 consecutive
            // words are taken at a time whatever the rows' width (a step per
            // row left most lanes idle on narrow grids): below counts the odd
            // words before the lane in its own row, and a row that began
            // before the step carries the parity of its words there.
            uint32_t carry = 0u;
            for (uint32_t i0 = 0; i0 < 16u * W; i0 += kWave) {
                const uint32_t i = i0 + lane;
                uint32_t r = (uint32_t)((float)i * rW);  // i / W: within one
                int32_t w = (int32_t)(i - r * W);
                if (w < 0) { r--; w += (int32_t)W; }
                if (w >= (int32_t)W) { r++; w -= (int32_t)W; }
                const bool valid = r < 16u && ((inside >> r) & 1u);
                const uint32_t c = i < 16u * W ? cross[i] : 0u;
                const uint32_t sx = prefix_xor(c);
                const unsigned long long odd = __ballot((__popc(c) & 1) != 0);
                // Odd words of the lane's row in this step, before it.
                const uint32_t from = (uint32_t)w < lane ? lane - (uint32_t)w : 0u;
                const unsigned long long mine = odd & ((1ull << lane) - 1ull) & (~0ull << from);
                const uint32_t before =
                    ((uint32_t)__popcll(mine) ^ ((uint32_t)w > lane ? carry : 0u)) & 1u;
                if (valid) {
                    const uint32_t cy = ty * 4u + (r & 3u), cz = tz * 4u + (r >> 2);
                    const size_t row = (size_t)(cz + p.oz) * p.rowsY + (cy + p.oy);
                    bits[row * W + (uint32_t)w] = sx ^ (before ? 0xFFFFFFFFu : 0u);
                }
                // The last lane's row goes on in the next step (or ends here).
                const uint32_t end = before ^ ((uint32_t)__popc(c) & 1u);
                carry = (uint32_t)__builtin_amdgcn_readlane((int)end, kWave - 1);
            }
            return;
        }
        for (uint32_t r = 0; r < 16u; r++) {
            if (!((inside >> r) & 1u)) continue;
            const uint32_t cy = ty * 4u + (r & 3u), cz = tz * 4u + (r >> 2);
            const size_t rowIdx = (size_t)(cz + p.oz) * p.rowsY + (cy + p.oy);
            uint32_t carry = (carries >> r) & 1u;
            for (uint32_t w0 = 0; w0 < sw; w0 += kWave) {
                const uint32_t w = w0 + lane;
                const uint32_t c = w < sw ? cross[r * SW + w] : 0u;
                const uint32_t sx = prefix_xor(c);
                const unsigned long long odd = __ballot((__popc(c) & 1) != 0);
                // Odd-crossing words below this lane, counted by mbcnt.
                const uint32_t below = __builtin_amdgcn_mbcnt_hi(
                    (uint32_t)(odd >> 32), __builtin_amdgcn_mbcnt_lo((uint32_t)odd, 0u));
                const uint32_t before = carry ^ (below & 1u);
                if (w < sw) bits[rowIdx * W + s0 + w] = sx ^ (before ? 0xFFFFFFFFu : 0u);
                carry ^= (uint32_t)__popcll(odd) & 1u;
            }
            carries = (carries & ~(1u << r)) | (carry << r);
        }
        __syncthreads();  // the next segment clears cross[]
    }
}

// ---------------------------------------------------------------------------
// Surface stage
// ---------------------------------------------------------------------------

// Voxel range vb of a triangle clipped to the whole ext space (the union of
// all matSplitRes subspaces); false if it lies outside (adjustVoxelRange,
// src/voxelizer.cu:3963-3993).
__device__ __forceinline__ bool surf_clip(const SurfParams &p, VoxBB &vb) {
    if (0 > vb.max.x || 0 > vb.max.y || 0 > vb.max.z) return false;
    if (vb.min.x > p.res[0] - 1 || vb.min.y > p.res[1] - 1 || vb.min.z > p.res[2] - 1) return false;
    vb.min = {max(vb.min.x, 0), max(vb.min.y, 0), max(vb.min.z, 0)};
    vb.max = {min(vb.max.x, p.res[0] - 1), min(vb.max.y, p.res[1] - 1), min(vb.max.z, p.res[2] - 1)};
    return true;
}
// Axis helpers: for dominant axis a, u and v are the other two axes in
// increasing order.
__device__ __forceinline__ int axis_u(int a) { return a == AX_X ? AX_Y : AX_X; }
__device__ __forceinline__ int axis_v(int a) { return a == AX_Z ? AX_Y : AX_Z; }
__device__ __forceinline__ int32_t pick3i(const I3 &p, int a) {
    return a == AX_X ? p.x : a == AX_Y ? p.y : p.z;
}

// Bricks are laid over alloc coordinates (ext + off).
__device__ __forceinline__ void brick_range(const SurfParams &p, const VoxBB &vb, uint32_t lo[3],
                                            uint32_t hi[3]) {
    lo[0] = (uint32_t)(vb.min.x + p.off[0]) / (uint32_t)p.bdim[0];
    lo[1] = (uint32_t)(vb.min.y + p.off[1]) / (uint32_t)p.bdim[1];
    lo[2] = (uint32_t)(vb.min.z + p.off[2]) / (uint32_t)p.bdim[2];
    hi[0] = (uint32_t)(vb.max.x + p.off[0]) / (uint32_t)p.bdim[0];
    hi[1] = (uint32_t)(vb.max.y + p.off[1]) / (uint32_t)p.bdim[1];
    hi[2] = (uint32_t)(vb.max.z + p.off[2]) / (uint32_t)p.bdim[2];
}

// Per triangle, from one read of its vertices: the 48-byte record, the solid
// pass's candidate tiles (its commonSpace tile rectangle; the box itself is kept
// so the candidate pass needs no divisions) and, for jobs with a surface stage,
// its class and dominant axis (classifyTriangles) and the box of bricks its
// clipped voxel range touches, packed as
// {info, lo.x | lo.y<<16, lo.z | w.x<<16, w.y | w.z<<16}.  With tri_ext, also
// its clipped voxel extents along (u, v, a) and its work items (voxels for 1D,
// dominant-plane columns otherwise), the cost model's inputs.  A block leaves
// the sums of its candidate counts for the scans.  The blocks past the
// triangles clear what the call counts into.
__global__ __launch_bounds__(256) void k_tri_setup(const Job *__restrict__ jobs,
                                                   const uint32_t *__restrict__ tri_bases,
                                                   uint32_t njobs, uint32_t tri_blocks,
                                                   TriSetup o, FillSegs clear) {
    if (blockIdx.x >= tri_blocks) {
        fill_segs(clear, blockIdx.x - tri_blocks, gridDim.x - tri_blocks);
        return;
    }
    const uint32_t t0 = blockIdx.x * 256u, j = job_of(tri_bases, njobs, t0);
    const Job &J = jobs[j];
    const uint32_t t = t0 + threadIdx.x, lt = t - J.tri_base;
    if (o.tri_job) o.tri_job[t] = j;
    uint32_t cs = 0u, cf = 0u;
    if (lt < J.nt) {  // not a padding slot
        const VK_G float *V = gptr(J.V);
        const VK_G uint32_t *I = gptr(J.I);
        const uint32_t ia = I[3u * lt], ib = I[3u * lt + 1u], ic = I[3u * lt + 2u];
        const F3 tri[3] = {{V[3u * ia], V[3u * ia + 1u], V[3u * ia + 2u]},
                           {V[3u * ib], V[3u * ib + 1u], V[3u * ib + 2u]},
                           {V[3u * ic], V[3u * ic + 1u], V[3u * ic + 2u]}};
        const uint32_t mat = J.mats ? (uint32_t)gptr(J.mats)[lt] : 0u;
        {
            const SolidParams p = solid_params(J, nullptr);
            D3 v[3];
#pragma unroll
            for (int k = 0; k < 3; k++)
                v[k] = {(double)tri[k].x, (double)tri[k].y, (double)tri[k].z};
            TileSetup ts;
            if (tile_setup(v, p.emy, p.emz, p.d, p.smin[0], p.smin[1], p.smax[0], p.smax[1],
                           ts)) {
                cs = (ts.tmax[0] - ts.tmin[0] + 1u) * (ts.tmax[1] - ts.tmin[1] + 1u);
                o.cbox[t] = make_uint4(ts.cmin[0], ts.cmin[1], ts.cmax[0], ts.cmax[1]);
            }
        }
        uint32_t info = 0u;
        if (o.off_f && J.use_mats) {
            const SurfParams p = surf_params(J);
            // One voxel range for the class and for the brick box.
            F3 mn, mx;
            tri_bounds(tri, mn, mx);
            VoxBB vb = voxel_bounds_half(mn, mx, p.m, p.d);
            int bb, axis;
            classify_vb(tri, vb, bb, axis);
            uint32_t lo[3] = {0, 0, 0}, w[3] = {0, 0, 0};
            uint4 ext = make_uint4(0u, 0u, 0u, 0u);
            if (bb != BB_DEGEN && surf_clip(p, vb)) {
                uint32_t hi[3];
                brick_range(p, vb, lo, hi);
                for (int a = 0; a < 3; a++) w[a] = hi[a] - lo[a] + 1u;
                cf = w[0] * w[1] * w[2];
                const uint32_t eu = (uint32_t)(pick3i(vb.max, axis_u(axis)) - pick3i(vb.min, axis_u(axis)) + 1);
                const uint32_t ev = (uint32_t)(pick3i(vb.max, axis_v(axis)) - pick3i(vb.min, axis_v(axis)) + 1);
                const uint32_t ea = (uint32_t)(pick3i(vb.max, axis) - pick3i(vb.min, axis) + 1);
                ext = make_uint4(eu, ev, ea, bb == BB_1D ? ea : eu * ev);
            }
            info = ((uint32_t)bb << 30) | ((uint32_t)axis << 28);
            o.tri_info[t] = make_uint4(info, lo[0] | (lo[1] << 16), lo[2] | (w[0] << 16),
                                       w[1] | (w[2] << 16));
            if (o.tri_ext) o.tri_ext[t] = ext;
        }
        // The class word goes into the record for the brick pass.
        o.rec[3 * (size_t)t] = make_float4(tri[0].x, tri[0].y, tri[0].z, tri[1].x);
        o.rec[3 * (size_t)t + 1] = make_float4(tri[1].y, tri[1].z, tri[2].x, tri[2].y);
        o.rec[3 * (size_t)t + 2] = make_float4(tri[2].z, __uint_as_float(info),
                                               __uint_as_float(mat), 0.0f);
    }
    o.off_s[t] = cs;
    const uint64_t ss = block_sum_u64(cs);
    if (threadIdx.x == 0) {
        o.part_s[blockIdx.x] = (uint32_t)ss;
        o.part_s[tri_blocks + blockIdx.x] = (uint32_t)(ss >> 32);
    }
    if (!o.off_f) return;
    o.off_f[t] = cf;
    const uint64_t sf = block_sum_u64(cf);
    if (threadIdx.x == 0) {
        o.part_f[blockIdx.x] = (uint32_t)sf;
        o.part_f[tri_blocks + blockIdx.x] = (uint32_t)(sf >> 32);
    }
}

// Winner key of a (triangle, voxel) hit; the largest key of a voxel wins
// (bbType first, then the mesh-local triangle index, as the oracle's rule).
// With `embed` (meshes of fewer than 2^22 triangles) the key carries the
// triangle's material in its low byte (the index is unique, so the byte
// never decides), and the brick pass reads no materials from memory; larger
// meshes keep the plain index and look the material up.
__device__ __forceinline__ uint32_t winner_key(uint32_t bb, uint32_t lt, uint32_t mat,
                                               bool embed) {
    return (bb << 30) | (embed ? (lt << 8) | (mat & 0xFFu) : lt);
}

// Per-triangle data of one brick's chunk, set up once in LDS.  Coordinates
// are named (u, v, a): a is the triangle's dominant axis, u and v the other
// two in increasing axis order (u = x unless a = x; v = z unless a = z).
// Every 2-term edge function of the reference, (ne.x*c0 + ne.y*c1) + de >= 0,
// is kept as c_first*p_first + c_second*p_second >= t with the two products
// in either order (IEEE addition is commutative) and t = overlap_bound(de).
// 44 words: a lane's 16-byte reads of neighbouring slots fall into different
// LDS banks.
struct __align__(16) SurfTri {
    float dom[3][3];    // dominant-plane edges: (coef of u, coef of v, t)
    float lu, lv;       // brick-clipped lowest u and v, less 1/2
    float rwu;          // ~ 1 / columns along u
    uint32_t ext;       // columns along u | voxels along a << 16
    uint32_t pk;        // LDS key index of the box's low corner (12 bits), log2 key strides of
                        // u, v, a (4 bits each), class, axis, kSlowDiv, kManySplits
    uint32_t key;       // LDS winner key (winner_key)
    // 3D triangles
    float nu, nv, na, rna;  // normal, 1 / na
    float t0u, t0v, ta;     // first vertex along u and v; its (vertex * normal) along a
    int32_t la;             // brick-clipped lowest a
    int32_t va, vb;         // range along a of the triangle's box in the brick's matSplitRes
                            // interval (kManySplits: of the box alone)
    float pl[2][3][3];      // the two other planes: (coef of a, coef of other, t)
};
static_assert(sizeof(SurfTri) == 176, "an odd number of 16-byte slots");
constexpr int kSurfChunk = 64;
constexpr uint32_t kPkU = 12, kPkV = 16, kPkA = 20, kPkClass = 24, kPkAxis = 26;
constexpr uint32_t kSlowDiv = 1u << 28;     // coordinates too large or small for div_by
constexpr uint32_t kManySplits = 1u << 29;  // the range along a crosses matSplitRes intervals

__device__ __forceinline__ F3 rotate_axes(const F3 &p, int a) {  // (u, v, a) up to a swap of u, v
    return a == AX_X ? F3{p.y, p.z, p.x} : a == AX_Y ? F3{p.z, p.x, p.y} : p;
}

// Sets up a triangle (its record r0..r2, mesh-local index lt) for the brick whose alloc-coordinate box starts at
// (ext coordinates) (blx, bly, blz), restricted to its z layers [z0, z1)
// (a sub-brick); returns its work items there: voxels along the axis for 1D,
// dominant-plane columns for 2D/3D.
__device__ __forceinline__ uint32_t surf_tri_setup(const SurfParams &p, bool fdiv,
                                                   const SplitTable &spl, const float4 &r0,
                                                   const float4 &r1, const float4 &r2,
                                                   uint32_t lt, bool embed, int32_t blx,
                                                   int32_t bly, int32_t blz, int32_t z0,
                                                   int32_t z1, SurfTri &st) {
    const F3 tri[3] = {{r0.x, r0.y, r0.z}, {r0.w, r1.x, r1.y}, {r1.z, r1.w, r2.x}};
    const uint32_t info = __float_as_uint(r2.y);
    F3 mn, mx;
    tri_bounds(tri, mn, mx);
    const bool near0 = fdiv && mn.x >= -0x1p24f && mn.y >= -0x1p24f && mn.z >= -0x1p24f &&
                       mx.x <= 0x1p24f && mx.y <= 0x1p24f && mx.z <= 0x1p24f;
    VoxBB vb = near0 ? voxel_bounds_half_by(mn, mx, p.m, p.d, p.rd)
                     : voxel_bounds_half(mn, mx, p.m, p.d);
    if (!surf_clip(p, vb)) return 0u;
    const int bb = (int)(info >> 30), a = (int)((info >> 28) & 3u);
    const int ua = axis_u(a), va = axis_v(a);
    const uint32_t lgx = 31u - (uint32_t)__clz(p.bdim[0]),
                   lgz = lgx + 31u - (uint32_t)__clz(p.bdim[1]);
    const int ax3[3] = {ua, va, a};
    int32_t lo[3], hi[3];
    uint32_t base = 0u, pk = (uint32_t)bb << kPkClass | (uint32_t)a << kPkAxis;
#pragma unroll
    for (int k = 0; k < 3; k++) {
        const int ax = ax3[k];
        const int32_t b0 = ax == AX_X ? blx : ax == AX_Y ? bly : blz;
        const int32_t bl = ax == AX_Z ? blz + z0 : b0;
        const int32_t bs = ax == AX_X ? p.bdim[0] : ax == AX_Y ? p.bdim[1] : z1 - z0;
        const uint32_t lg = ax == AX_X ? 0u : ax == AX_Y ? lgx : lgz;
        lo[k] = max(pick3i(vb.min, ax), bl);
        hi[k] = min(pick3i(vb.max, ax), bl + bs - 1);
        if (lo[k] > hi[k]) return 0u;
        base += (uint32_t)(lo[k] - b0) << lg;
        pk |= lg << (kPkU + 4u * (uint32_t)k);
    }
    const uint32_t wu = (uint32_t)(hi[0] - lo[0] + 1), wa = (uint32_t)(hi[2] - lo[2] + 1);
    st.ext = wu | wa << 16;
    st.key = winner_key((uint32_t)bb, lt, __float_as_uint(r2.z), embed);
    st.pk = pk |= base;
    if (bb == BB_1D) return wa;
    st.lu = (float)lo[0] - 0.5f;
    st.lv = (float)lo[1] - 0.5f;
    st.rwu = __builtin_amdgcn_rcpf((float)wu);
    const F3 n = fcross(fsub(tri[0], tri[2]), fsub(tri[1], tri[0]));
    // With the axes rotated so that a comes last, (x, y) is the dominant
    // plane in the reference's coordinate order, (y, z) the plane of x and
    // (z, x) the plane of y.  u and v are x and y, or y and x for a = y.
    const F3 rn = rotate_axes(n, a);
    const F3 rt[3] = {rotate_axes(tri[0], a), rotate_axes(tri[1], a), rotate_axes(tri[2], a)};
    const bool swap = a == AX_Y;
#pragma unroll
    for (int e = 0; e < 3; e++) {
        const F3 A = rt[e], B = rt[(e + 1) % 3];
        float n0, n1, de;
        overlap_edge(A.x, A.y, B.x, B.y, rn.z >= 0.0f, p.d, n0, n1, de);
        st.dom[e][0] = swap ? n1 : n0;
        st.dom[e][1] = swap ? n0 : n1;
        st.dom[e][2] = overlap_bound(de);
        if (bb == BB_3D) {
            overlap_edge(A.y, A.z, B.y, B.z, rn.x >= 0.0f, p.d, n0, n1, de);
            st.pl[0][e][0] = n1;
            st.pl[0][e][1] = n0;
            st.pl[0][e][2] = overlap_bound(de);
            overlap_edge(A.z, A.x, B.z, B.x, rn.y >= 0.0f, p.d, n0, n1, de);
            st.pl[1][e][0] = n0;
            st.pl[1][e][1] = n1;
            st.pl[1][e][2] = overlap_bound(de);
        }
    }
    if (bb == BB_3D) {
        st.nu = swap ? rn.y : rn.x;
        st.nv = swap ? rn.x : rn.y;
        st.na = rn.z;
        st.rna = 1.0f / rn.z;
        st.t0u = swap ? rt[0].y : rt[0].x;
        st.t0v = swap ? rt[0].x : rt[0].y;
        st.ta = rt[0].z * rn.z;
        st.la = lo[2];
        int32_t sa = pick3i(vb.min, a), sb = pick3i(vb.max, a);
        const uint32_t ns = spl.n[a];
        uint32_t si = 0;
        while (si + 1u < ns && (uint32_t)lo[2] >= spl.hi[a][si]) si++;
        if (si + 1u < ns && (uint32_t)hi[2] >= spl.hi[a][si]) {
            pk |= kManySplits;
        } else {
            sa = max(sa, (int32_t)spl.lo[a][si]);
            sb = min(sb, (int32_t)spl.hi[a][si] - 1);
        }
        st.va = sa;
        st.vb = sb;
        const bool safe = near0 && fabsf(n.x) <= 0x1p40f && fabsf(n.y) <= 0x1p40f &&
                          fabsf(n.z) <= 0x1p40f && fabsf(rn.z) >= 0x1p-40f;
        st.pk = pk | (safe ? 0u : kSlowDiv);
    }
    return wu * (uint32_t)(hi[1] - lo[1] + 1);
}

__device__ __forceinline__ void key_write(uint32_t *keys, uint8_t *touched, uint32_t idx,
                                          uint32_t nvox, uint32_t key) {
    if (idx >= nvox) return;  // unreachable: items lie in the brick
    atomicMax(&keys[idx], key);
    touched[idx >> 8] = 1;
}

// The dominant-plane half of work item k (a 1D triangle's voxel, or a column
// of the others' box), following the 1D/2D/3D kernels of the reference
// (src/voxelizer.cu:3307-3955).  1D and 2D hits are written; true for a 3D
// triangle's column that passes, whose depth part follows (surf_depth).
__device__ __forceinline__ bool surf_column(const SurfParams &p, const SurfTri &st, uint32_t k,
                                            uint32_t *keys, uint8_t *touched, uint32_t nvox,
                                            uint32_t &cu, uint32_t &cv) {
    const uint32_t pk = st.pk, base = pk & 0xFFFu;
    const uint32_t bb = (pk >> kPkClass) & 3u, a = (pk >> kPkAxis) & 3u;
    if (bb == BB_1D) {
        key_write(keys, touched, base + (k << ((pk >> kPkA) & 15u)), nvox, st.key);
        return false;
    }
    // k = cv * wu + cu
    const int32_t wu = (int32_t)(st.ext & 0xFFFFu);
    int32_t q = (int32_t)((float)k * st.rwu);
    int32_t r = (int32_t)k - (int32_t)__umul24(q, wu);
    if (r < 0) { q--; r += wu; }
    if (r >= wu) { q++; r -= wu; }
    cu = (uint32_t)r;
    cv = (uint32_t)q;
    const float mu = a == AX_X ? p.m.y : p.m.x, mv = a == AX_Z ? p.m.y : p.m.z;
    const float pu = mu + (st.lu + (float)r) * p.d;  // vox_corner
    const float pv = mv + (st.lv + (float)q) * p.d;
    bool in = true;
#pragma unroll
    for (int e = 0; e < 3; e++) in &= st.dom[e][0] * pu + st.dom[e][1] * pv >= st.dom[e][2];
    if (in && bb != BB_3D)
        key_write(keys, touched,
                  base + (cu << ((pk >> kPkU) & 15u)) + (cv << ((pk >> kPkV) & 15u)), nvox,
                  st.key);
    return in && bb == BB_3D;
}

// The depth part of a 3D triangle's column (determineDepthRange{X,Y,Z},
// src/voxelizer.cu:4004-4119, and the side-plane tests along the column).
// It costs about four times the dominant-plane test and only half of a box's
// columns reach it, so a wave queues those in LDS and works them off 64 at a
// time; its four divisions go by reciprocals.  k_surf_brick: room at 1 cm
// (512x403x303) 237 -> 198 us (89.4 -> 64.9 M wave instructions), hall
// (1536x1024x768) 930 -> 849 us (354 -> 295 M), LongFCC room 640x255x384
// 451 -> 417 us, 64-mesh batch 2002 -> 1835 us.
// Only the single-voxel shortcut depends on the matSplitRes subspace, through
// the interval along a that the voxel falls in.
__device__ __forceinline__ void surf_depth(const SurfParams &p, const SplitTable &spl,
                                           const SurfTri &st, uint32_t cu, uint32_t cv,
                                           uint32_t *keys, uint8_t *touched, uint32_t nvox) {
    const uint32_t pk = st.pk, a = (pk >> kPkAxis) & 3u, sa = (pk >> kPkA) & 15u;
    const float mu = a == AX_X ? p.m.y : p.m.x, mv = a == AX_Z ? p.m.y : p.m.z;
    const float ma = a == AX_X ? p.m.x : a == AX_Y ? p.m.y : p.m.z;
    const float pu = mu + (st.lu + (float)cu) * p.d, pv = mv + (st.lv + (float)cv) * p.d;
    // Depths of the plane over the column's two extreme corners: the dot
    // product's terms in x, y, z order, (u + v) + a for a = z, (u + a) + v
    // otherwise (IEEE addition is commutative).
    const float pu1 = pu + p.d, pv1 = pv + p.d;
    const bool fu = st.nu > 0.0f, fv = st.nv > 0.0f;
    const float u0 = (st.t0u - (fu ? pu1 : pu)) * st.nu, u1 = (st.t0u - (fu ? pu : pu1)) * st.nu;
    const float v0 = (st.t0v - (fv ? pv1 : pv)) * st.nv, v1 = (st.t0v - (fv ? pv : pv1)) * st.nv;
    const bool az = a == AX_Z;
    const float x0 = az ? v0 : st.ta, y0 = az ? st.ta : v0;
    const float x1 = az ? v1 : st.ta, y1 = az ? st.ta : v1;
    const float num0 = (u0 + x0) + y0, num1 = (u1 + x1) + y1;
    int32_t lo, hi;
    if (pk & kSlowDiv) {
        float d0 = num0 / st.na, d1 = num1 / st.na;
        if (d0 > d1) {
            const float tmp = d0;
            d0 = d1;
            d1 = tmp;
        }
        lo = f2i(ceilf((d0 - ma) / p.d - 0.5f));
        hi = f2i(floorf((d1 - ma) / p.d + 0.5f));
    } else {  // finite throughout
        const float d0 = div_by(num0, st.na, st.rna), d1 = div_by(num1, st.na, st.rna);
        lo = f2i(ceilf(div_by(fminf(d0, d1) - ma, p.d, p.rd) - 0.5f));
        hi = f2i(floorf(div_by(fmaxf(d0, d1) - ma, p.d, p.rd) + 0.5f));
    }
    const int32_t la = st.la;
    const int32_t ilo = max(lo, la), ihi = min(hi, la + (int32_t)(st.ext >> 16) - 1);
    if (ilo > ihi) return;
    // The two side planes' edge functions along the column, c * pa + k >= t.
    float sc[6], sk[6], se[6];
#pragma unroll
    for (int q = 0; q < 2; q++) {
        const float po = (q == 0) == (a == AX_Y) ? pu : pv;  // plane of v, then of u, for a = y
#pragma unroll
        for (int e = 0; e < 3; e++) {
            sc[3 * q + e] = st.pl[q][e][0];
            sk[3 * q + e] = st.pl[q][e][1] * po;
            se[3 * q + e] = st.pl[q][e][2];
        }
    }
    uint32_t idx = (pk & 0xFFFu) + (cu << ((pk >> kPkU) & 15u)) + (cv << ((pk >> kPkV) & 15u)) +
                   ((uint32_t)(ilo - la) << sa);
    const uint32_t key = st.key;
    float fa = (float)ilo - 0.5f;
    auto inside = [&]() {
        const float pa = ma + fa * p.d;  // vox_corner
        bool in = true;
#pragma unroll
        for (int e = 0; e < 6; e++) in &= sc[e] * pa + sk[e] >= se[e];
        return in;
    };
    if (!(pk & kManySplits)) {
        const bool single = max(lo, st.va) == min(hi, st.vb);
        for (int32_t i = ilo; i <= ihi; i++) {
            if (single || inside()) key_write(keys, touched, idx, nvox, key);
            fa += 1.0f;
            idx += 1u << sa;
        }
        return;
    }
    const uint32_t ns = spl.n[a];
    uint32_t si = 0;
    for (int32_t i = ilo; i <= ihi; i++) {
        while (si + 1u < ns && (uint32_t)i >= spl.hi[a][si]) si++;
        const int32_t rl = max(lo, max(st.va, (int32_t)spl.lo[a][si]));
        const int32_t rh = min(hi, min(st.vb, (int32_t)spl.hi[a][si] - 1));
        if (rl == rh || inside()) key_write(keys, touched, idx, nvox, key);
        fa += 1.0f;
        idx += 1u << sa;
    }
}

// Persistent workgroups over a list of non-empty bricks (`order`: brick ids
// in index order), before it the heavy bricks of the learned schedule
// (`hlist`).  A workgroup is kBrickWaves waves that voxelize and one that
// prepares: while the others work on a chunk of up to 64 triangles of a brick,
// it takes the next list entry, loads the next chunk's triangle ids and
// records, and, while the others write the finished brick, sets the chunk's
// triangles up in LDS (a lane per triangle).  So neither the chain entry ->
// brick -> ids -> records -> setup nor a global load stands in the voxelizing
// waves' way: they work from LDS and only store.
//
// All (triangle, column) items of the chunk are spread over the voxelizing
// threads; winners accumulate in LDS (ds_max of winner_key).  The 256-voxel steps
// that received a key are visited when the brick's last chunk is done: each lane
// takes four voxels, a word's eight lanes OR their bits into the solid grid,
// and the words that hold a surface voxel have their winners' materials
// stored in the brick's block of the material grid.  With `stats`, surface
// voxels are counted; with `cycles`, each brick's duration from its first
// item to its last store (s_memtime) is recorded.  The kKeys variant also
// stores surface words and winner keys for jobs with a keygrid (PartialNode).
//
// Before the split every brick paid that chain and its setup in series, and one
// counter handed out the list.  Together (fifteen voxelizing waves a CU and
// five preparing; with four and one a workgroup's registers allow four
// workgroups a CU, and the hall took 2050 instead of 1800 us as a whole):
// hall (1536x1024x768, 1.4 M triangles) 849 -> 650 us, room 512x403x303
// 198 -> 168 us, LongFCC room 640x255x384 417 -> 316 us, 64-mesh batch
// 1835 -> 1400 us, 132 large triangles over 672x515x387 278 -> 147 us,
// sphere 128^3 24.4 -> 19.0 us.
constexpr int kDppQuadSwap1 = 0xB1, kDppQuadSwap2 = 0x4E, kDppHalfMirror = 0x141;

// What the voxelizing waves need to know of a chunk.
struct BrickStep {
    uint32_t valid;         // 0: the list is done
    uint32_t ends;          // bit 0: the brick's first chunk, bit 1: its last
    uint32_t job, brick;    // brick within the job
    uint32_t bx, by, bz;    // its coordinates
    uint32_t layers;        // z0 | z1 << 16
    uint32_t total, ntri;   // work items, triangles with items
};

template <bool kKeys>
__global__ __launch_bounds__(kBrickThreads, 5) void k_surf_brick(
    const Job *__restrict__ jobs, const uint32_t *__restrict__ brick_bases, uint32_t njobs,
    const float4 *__restrict__ tri_rec, const uint32_t *__restrict__ brick_off,
    const uint32_t *__restrict__ brick_hist, const uint32_t *__restrict__ blist,
    uint32_t *__restrict__ stats, const uint32_t *__restrict__ order,
    const uint32_t *__restrict__ n_order, const uint32_t *__restrict__ hlist,
    const uint32_t *__restrict__ hsub, const uint32_t *__restrict__ n_heavy,
    const uint8_t *__restrict__ skip, uint32_t *__restrict__ next,
    uint64_t *__restrict__ cycles) {
    __shared__ __align__(16) uint32_t keys[kMaxBrickVox];
    __shared__ SurfTri tris[kSurfChunk];
    __shared__ uint32_t cstart[kSurfChunk], smask[kBrickWaves][2];
    __shared__ uint8_t cslot[kSurfChunk];
    __shared__ uint32_t wqueue[kBrickWaves][2 * kWave];  // columns that await their depth part
    // 256-voxel steps with a key, of this brick and (cleared) the next
    __shared__ uint8_t touched[2][kMaxBrickVox / 256];
    __shared__ BrickStep step;
    __shared__ SplitTable spl;
    const uint32_t tid = threadIdx.x, lane = lane_id();
    const uint32_t wave = __builtin_amdgcn_readfirstlane(tid / kWave);
    for (uint32_t i = tid; i < (uint32_t)kMaxBrickVox; i += kBrickThreads) keys[i] = 0u;
    if (tid < sizeof(touched)) (&touched[0][0])[tid] = 0;
    if (tid < 2u * kBrickWaves) (&smask[0][0])[tid] = 0u;

    if (wave == kBrickWaves) {
        // ---- the preparing wave ----
        const uint32_t nh = hlist ? *n_heavy : 0u;
        const uint32_t n_list = *n_order + nh;  // heavy entries first, then the plain list
        // Every workgroup starts with the entry of its own number; the rest
        // lies in kBrickLists parts, each with a counter that a workgroup
        // draws its next entry or two from: its own part's first (part and
        // XCD have the same number), then the others' when that is used up.
        // One counter bound the pass at 14-18 ns a draw (room 195 us against
        // 166 with eight), which longer runs only trade for imbalance: runs
        // of up to 16, 8, 4, 2 and 1 took 866, 658, 644, 640 and 660 us on
        // the hall, 16 and 32 counters no less than eight.
        const uint32_t dealt = min(gridDim.x, n_list);
        const uint32_t part = (n_list - dealt + kBrickLists - 1u) / kBrickLists;
        uint32_t list = blockIdx.x % kBrickLists, tried = 0u;
        // The run in hand, an entry per lane: brick, pairs, first pair, layers.
        uint32_t gb = 0u, cnt = 0u, off = 0u, sub = 0u;
        uint32_t rn = 0u, ri = 0u;
        // The next run on its way: its first entry (pending 1: being drawn),
        // its bricks (2: being read).
        uint32_t q0 = blockIdx.x, qk = 1u, qend = n_list, pending = 1u;
        uint32_t ngb = 0u, nsub = 0u;
        bool nskip = false;
        auto draw = [&](uint32_t seen) {  // seen: entries of the list before this were drawn
            const uint32_t lo = min(dealt + list * part, n_list);
            qend = min(dealt + (list + 1u) * part, n_list);
            const uint32_t left = qend - min(max(seen, lo), qend);
            qk = left * kBrickLists / (32u * gridDim.x) > 1u ? 2u : 1u;
            if (lane == 0u) q0 = lo + atomicAdd(next + list * kBrickListPitch, qk);
            pending = 1u;
        };
        auto bricks_of_run = [&]() {  // pending 1 -> 2
            q0 = __builtin_amdgcn_readfirstlane(q0);
            while (q0 >= qend && tried < kBrickLists) {
                list = list + 1u < kBrickLists ? list + 1u : 0u;
                tried++;
                draw(0u);
                q0 = __builtin_amdgcn_readfirstlane(q0);
            }
            qk = q0 < qend ? min(qk, qend - q0) : 0u;
            const uint32_t q = q0 + lane;
            ngb = 0u;
            nsub = 0xFFFF0000u;
            nskip = lane >= qk;
            if (!nskip) {
                if (q < nh) {
                    ngb = hlist[q];
                    nsub = hsub[q];
                } else {
                    ngb = order[q - nh];
                    // A plain entry already taken from the heavy list is passed over.
                    if (hlist) nskip = skip[q - nh] != 0;
                }
            }
            pending = 2u;
        };
        // The chunk in preparation.
        uint32_t cb = 0u, ccnt = 0u, coff = 0u, csub = 0u, c0 = 0u;
        bool more = true, first = false;
        uint32_t cjob = 0u, spl_job = UINT32_MAX;
        float4 r0, r1, r2;
        uint32_t t = 0u;
        auto fetch = [&]() {  // the next chunk's triangles
            first = false;
            if (c0 + kSurfChunk < ccnt) {
                c0 += kSurfChunk;
            } else {
                ccnt = 0u;
                while (ccnt == 0u) {
                    if (ri == rn) {
                        if (pending == 1u) bricks_of_run();
                        rn = qk;
                        ri = 0u;
                        if (rn == 0u) {
                            more = false;
                            return;
                        }
                        gb = ngb;
                        sub = nsub;
                        cnt = nskip ? 0u : brick_hist[gb];
                        off = nskip ? 0u : brick_off[gb];
                        pending = 0u;
                    }
                    cb = (uint32_t)__builtin_amdgcn_readlane((int)gb, (int)ri);
                    ccnt = (uint32_t)__builtin_amdgcn_readlane((int)cnt, (int)ri);
                    coff = (uint32_t)__builtin_amdgcn_readlane((int)off, (int)ri);
                    csub = (uint32_t)__builtin_amdgcn_readlane((int)sub, (int)ri);
                    ri++;
                    if (ri == rn) draw(q0 + rn);  // the next run, early
                }
                c0 = 0u;
                first = true;
            }
            if (c0 + lane < ccnt) {
                t = blist[coff + c0 + lane];
                r0 = tri_rec[3 * (size_t)t];
                r1 = tri_rec[3 * (size_t)t + 1];
                r2 = tri_rec[3 * (size_t)t + 2];
            }
        };
        auto publish = [&]() {
            if (!more) {
                if (lane == 0u) step.valid = 0u;
                return;
            }
            // Consecutive entries mostly share a job: its range is tested
            // before a search.
            if (njobs > 1u && !(spl_job != UINT32_MAX && cb >= brick_bases[cjob] &&
                                cb < brick_bases[cjob + 1u]))
                cjob = job_of(brick_bases, njobs, cb);
            const Job &J = jobs[cjob];
            if (cjob != spl_job) {  // the job's matSplitRes table into LDS
                const VK_G uint32_t *src = (const VK_G uint32_t *)gptr(J.splits);
                uint32_t *dst = (uint32_t *)&spl;
                for (uint32_t i = lane; i < sizeof(SplitTable) / 4; i += kWave) dst[i] = src[i];
                spl_job = cjob;
                wave_lds_sync();
            }
            const SurfParams p = surf_params(J);
            const uint32_t b = cb - J.brick_base;
            const uint32_t bx = b % p.nb[0], by = (b / p.nb[0]) % p.nb[1],
                           bz = b / (p.nb[0] * p.nb[1]);
            const uint32_t z0 = csub & 0xFFFFu, z1 = min(csub >> 16, (uint32_t)p.bdim[2]);
            // Bricks are laid over alloc coordinates; ext = alloc - off.
            uint32_t items = 0u;
            if (c0 + lane < ccnt)
                items = surf_tri_setup(p, J.fdiv != 0, spl, r0, r1, r2, t - J.tri_base,
                                       J.embed != 0, (int32_t)(bx * p.bdim[0]) - p.off[0],
                                       (int32_t)(by * p.bdim[1]) - p.off[1],
                                       (int32_t)(bz * p.bdim[2]) - p.off[2], (int32_t)z0,
                                       (int32_t)z1, tris[lane]);
            static_assert(kSurfChunk == kWave, "one wave sets up a chunk");
            const uint32_t incl = wave_incl_scan(items);
            // The triangles with items, in order: first item and LDS slot.
            const unsigned long long nz = __ballot(items != 0u);
            if (items) {
                const uint32_t r = __builtin_amdgcn_mbcnt_hi(
                    (uint32_t)(nz >> 32), __builtin_amdgcn_mbcnt_lo((uint32_t)nz, 0u));
                cstart[r] = incl - items;
                cslot[r] = (uint8_t)lane;
            }
            if (lane == kWave - 1u)
                step = BrickStep{1u, (first ? 1u : 0u) | (c0 + kSurfChunk >= ccnt ? 2u : 0u),
                                 cjob, b, bx, by, bz, z0 | z1 << 16, incl,
                                 (uint32_t)__popcll(nz)};
        };
        fetch();
        publish();
        while (true) {
            __syncthreads();  // the step is set up
            if (!more) return;
            fetch();
            __syncthreads();  // its items are done
            publish();
            if (pending == 1u) bricks_of_run();
        }
    }

    // ---- the voxelizing waves ----
    uint32_t nsurf = 0u;  // surface voxels found by this lane
    uint32_t par = 1u;
    uint64_t t_start = 0;
    while (true) {
        __syncthreads();  // the step is set up
        if (__builtin_amdgcn_readfirstlane(step.valid) == 0u) break;
        const uint32_t ends = __builtin_amdgcn_readfirstlane(step.ends);
        const uint32_t b = __builtin_amdgcn_readfirstlane(step.brick);
        const uint32_t total = __builtin_amdgcn_readfirstlane(step.total),
                       ntri = __builtin_amdgcn_readfirstlane(step.ntri);
        const uint32_t bx = __builtin_amdgcn_readfirstlane(step.bx),
                       by = __builtin_amdgcn_readfirstlane(step.by),
                       bz = __builtin_amdgcn_readfirstlane(step.bz),
                       layers = __builtin_amdgcn_readfirstlane(step.layers);
        const Job &J = jobs[__builtin_amdgcn_readfirstlane(step.job)];
        const SurfParams p = surf_params(J);
        const uint32_t nvox = (uint32_t)(p.bdim[0] * p.bdim[1] * p.bdim[2]);
        const uint32_t row_shift = 31u - (uint32_t)__clz(p.bdim[0]);
        if (ends & 1u) {
            par ^= 1u;
            if (tid < sizeof(touched[0])) touched[par ^ 1u][tid] = 0;  // the previous brick's
            if (cycles && tid == 0u) t_start = __builtin_amdgcn_s_memtime();
        }
        // Lane j holds the first item of the j-th triangle with items
        // (strictly increasing in j) and its slot.  A wave takes 64
        // consecutive items at a time: the triangle of its first item
        // is a ballot over the held starts, and each lane adds the
        // triangles starting between the first item and its own, read
        // from a 64-bit mask of start offsets that the starting lanes
        // OR together in LDS.
        const uint32_t cs = lane < ntri ? cstart[lane] : UINT32_MAX;
        const uint32_t sl = lane < ntri ? (uint32_t)cslot[lane] : 0u;
        uint32_t *sm = &smask[wave][0], *wq = wqueue[wave];
        uint8_t *steps = touched[par];
        uint32_t nq = 0u;  // columns in the wave's queue (uniform)
        auto depth = [&](uint32_t e) {
            surf_depth(p, spl, tris[e >> 24], e & 0xFFFu, (e >> 12) & 0xFFFu, keys, steps,
                       nvox);
        };
        for (uint32_t w0 = wave * kWave; w0 < total; w0 += kBrickWaves * kWave) {  // uniform
            const uint32_t t0 = (uint32_t)__popcll(__ballot(cs <= w0)) - 1u;
            const uint32_t ps = cs - w0 - 1u;  // start offset - 1, in 0..62
            if (cs > w0 && ps < kWave - 1u) atomicOr(&sm[ps >> 5], 1u << (ps & 31u));
            const uint32_t m_lo = sm[0], m_hi = sm[1];
            if (lane == 0u) {
                sm[0] = 0u;
                sm[1] = 0u;
            }
            const uint32_t ti =
                t0 + __builtin_amdgcn_mbcnt_hi(m_hi, __builtin_amdgcn_mbcnt_lo(m_lo, 0u));
            const uint32_t slot = (uint32_t)__shfl((int)sl, (int)ti);
            const uint32_t start = (uint32_t)__shfl((int)cs, (int)ti);
            const uint32_t c = w0 + lane;
            uint32_t cu = 0u, cv = 0u;
            const bool deep = c < total && surf_column(p, tris[slot], c - start, keys, steps,
                                                       nvox, cu, cv);
            const unsigned long long dm = __ballot(deep);
            if (deep)
                wq[nq + __builtin_amdgcn_mbcnt_hi(
                            (uint32_t)(dm >> 32),
                            __builtin_amdgcn_mbcnt_lo((uint32_t)dm, 0u))] =
                    slot << 24 | cv << 12 | cu;
            nq += (uint32_t)__popcll(dm);
            wave_lds_sync();
            if (nq >= (uint32_t)kWave) {
                nq -= (uint32_t)kWave;
                depth(wq[nq + lane]);
                wave_lds_sync();
            }
        }
        if (lane < nq) depth(wq[lane]);
        __syncthreads();  // the step's items are done
        if (!(ends & 2u)) continue;
        // The brick's rows, 256 voxels per wave step: each lane takes 4
        // consecutive voxels (one 16-byte LDS read of their keys), the 8
        // lanes of a 32-voxel word OR their nibbles together, and each lane
        // of a word holding a surface voxel writes its 4 material bytes as
        // one dword of the brick's block in the material grid (the winner's
        // material, 0 for the word's other voxels).  Steps that received no
        // key are passed over.  Keys are cleared for the next
        // brick.  With materials in the keys the loop issues no global loads,
        // so its stores never wait (a wait for a load also waits for earlier
        // stores here).
        VK_G uint32_t *__restrict__ bits = gptr(J.bits);
        VK_G uint32_t *__restrict__ mg =
            (VK_G uint32_t *)(gptr(J.matgrid) + (size_t)b * nvox);
        VK_G u32x4 *__restrict__ kg =
            kKeys && J.keygrid ? (VK_G u32x4 *)(gptr(J.keygrid) + (size_t)b * nvox) : nullptr;
        VK_G uint32_t *__restrict__ surf = kKeys ? gptr(J.surf) : nullptr;
        const VK_G uint8_t *__restrict__ materials = gptr(J.mats);
        const bool embed = J.embed != 0;
        const uint32_t z0 = layers & 0xFFFFu, z1 = layers >> 16;
        const uint32_t lwx = row_shift - 5u, lby = 31u - (uint32_t)__clz(p.bdim[1]);
        const uint32_t aw0 = bx << lwx, ay0 = by << lby, az0 = bz * (uint32_t)p.bdim[2];
        const uint32_t W = p.alloc[0] / 32u;
        const bool whole = z0 == 0u && z1 == (uint32_t)p.bdim[2];
        VK_G uint8_t *wm = (VK_G uint8_t *)gptr(J.wmask) + (size_t)b * 16u;
        constexpr uint32_t kSteps = kMaxBrickVox / 256;
        const uint32_t tmask =
            (uint32_t)__ballot(lane < kSteps && steps[lane & (kSteps - 1u)] != 0);
        for (uint32_t v0 = wave * 256u; v0 < nvox; v0 += kBrickWaves * 256u) {
            // This lane's word and its place in the grid.
            const uint32_t wi = (v0 >> 5) + (lane >> 3);
            const uint32_t aw = aw0 + (wi & ((1u << lwx) - 1u)),
                           ay = ay0 + ((wi >> lwx) & ((1u << lby) - 1u)),
                           lz = wi >> (lwx + lby), az = az0 + lz;
            const size_t gi = ((size_t)az * p.alloc[1] + ay) * W + aw;
            uint32_t w = 0u;
            if ((tmask >> (v0 >> 8)) & 1u) {  // uniform
                uint4 *kp = (uint4 *)&keys[v0 + 4u * lane];
                const uint4 kv = *kp;
                const uint32_t nib = (kv.x ? 8u : 0u) | (kv.y ? 4u : 0u) | (kv.z ? 2u : 0u) |
                                     (kv.w ? 1u : 0u);
                // OR over the word's 8 lanes in registers (DPP): the
                // quad swaps [1,0,3,2] and [2,3,0,1], then the half-row
                // mirror (lane i <-> 7 - i) joins the two quads.
                w = nib << (28u - 4u * (lane & 7u));
                w |= (uint32_t)__builtin_amdgcn_update_dpp(0, (int)w, kDppQuadSwap1, 0xF, 0xF, false);
                w |= (uint32_t)__builtin_amdgcn_update_dpp(0, (int)w, kDppQuadSwap2, 0xF, 0xF, false);
                w |= (uint32_t)__builtin_amdgcn_update_dpp(0, (int)w, kDppHalfMirror, 0xF, 0xF, false);
                // The words with a surface voxel: bit 8 i of the ballot is
                // word i of the step, gathered into its byte of the brick's
                // word mask (cleared each call; a part of a cut brick shares it).
                const unsigned long long wb = __ballot(w != 0u) & 0x0101010101010101ull;
                const uint32_t byte = (uint32_t)((wb * 0x0102040810204080ull) >> 56);
                if (lane == 0u && byte) {
                    if (whole)
                        wm[v0 >> 8] = (uint8_t)byte;
                    else
                        atomicOr((uint32_t *)(J.wmask + (size_t)b * 4u + (v0 >> 10)),
                                 byte << ((v0 >> 5) & 24u));
                }
                if (w) {
                    if ((lane & 7u) == 0u)
                        __hip_atomic_fetch_or(bits + gi, w, __ATOMIC_RELAXED,
                                              __HIP_MEMORY_SCOPE_AGENT);
                    nsurf += (uint32_t)__popc(nib);
                    uint32_t m;
                    if (embed) {
                        m = (kv.x & 0xFFu) | (kv.y & 0xFFu) << 8 | (kv.z & 0xFFu) << 16 |
                            (kv.w & 0xFFu) << 24;
                    } else {
                        auto mat = [&](uint32_t key) -> uint32_t {
                            return key && materials ? (uint32_t)materials[key & 0x3FFFFFFFu] : 0u;
                        };
                        m = mat(kv.x) | mat(kv.y) << 8 | mat(kv.z) << 16 | mat(kv.w) << 24;
                    }
                    if (nib) *kp = make_uint4(0u, 0u, 0u, 0u);
                    mg[(v0 >> 2) + lane] = m;
                    if (kKeys && kg) kg[(v0 >> 2) + lane] = u32x4{kv.x, kv.y, kv.z, kv.w};
                }
            }
            if (kKeys && surf && (lane & 7u) == 0u && lz >= z0 && lz < z1 && aw < W &&
                ay < p.alloc[1] && az < p.alloc[2])
                surf[gi] = w;
        }
        if (cycles && tid == 0u)
            cycles[J.brick_base + b] = __builtin_amdgcn_s_memtime() - t_start;
    }
    // One atomic per wave at exit: a shared counter bumped per brick would
    // serialise every workgroup on one address.
    if (stats) {
        for (int d = kWave / 2; d >= 1; d >>= 1) nsurf += (uint32_t)__shfl_xor((int)nsurf, d);
        if (lane == 0 && nsurf) atomicAdd(stats, nsurf);
    }
}
template __global__ void k_surf_brick<false>(const Job *, const uint32_t *, uint32_t,
                                             const float4 *, const uint32_t *, const uint32_t *,
                                             const uint32_t *, uint32_t *, const uint32_t *,
                                             const uint32_t *, const uint32_t *, const uint32_t *,
                                             const uint32_t *, const uint8_t *, uint32_t *,
                                             uint64_t *);
template __global__ void k_surf_brick<true>(const Job *, const uint32_t *, uint32_t,
                                            const float4 *, const uint32_t *, const uint32_t *,
                                            const uint32_t *, uint32_t *, const uint32_t *,
                                            const uint32_t *, const uint32_t *, const uint32_t *,
                                            const uint32_t *, const uint8_t *, uint32_t *,
                                            uint64_t *);

// ---------------------------------------------------------------------------
// Erosion: removal of solid voxels that lack a solid neighbour on some axis
// (the invalid-permutation removal of src/voxelizer.cu:1791-1913), repeated
// until a pass removes nothing (src/host_side.cpp:1183-1206).  The rule is
// monotone and only removes, so passes may run in place and in any order:
// every such (chaotic) iteration reaches the same greatest fixed point as
// the reference's.  The first pass of a subspace reads the whole grid; a
// later pass only visits blocks that changed, or that hold neighbours of
// words in blocks that changed, in the previous pass (stamp = 1 + last pass with a
// change), and a word is written only when it changes.  Voxels outside
// [y0,y1) x [z0,z1) are left alone.  Plane-linear launch: a block takes
// kChunk consecutive words of a plane over kErodeZ planes.
// ---------------------------------------------------------------------------
// Whether logical block GL of job J lies in the subspace and, after the
// subspace's first pass, is near a change of the previous pass: a word
// depends on words at most W positions away in its plane and on the same
// word in the planes next to it, so the block is visited when any chunk
// within W words, or this chunk in the plane groups next to it, changed.
// DPP controls: every lane takes the value of the lane one below (wave_shr:1)
// or one above (wave_shl:1); the wave's end lanes get 0.
constexpr int kDppWaveShl1 = 0x130, kDppWaveShr1 = 0x138;

__device__ __forceinline__ bool erode_visit(const Job &J, uint32_t GL, uint32_t y0, uint32_t y1,
                                            uint32_t z0, uint32_t z1,
                                            const uint32_t *__restrict__ stamp, uint32_t gpass,
                                            int full) {
    const GridDims g = J.gd;
    const uint32_t P = g.W * g.Y;  // words per plane
    const uint32_t nch = (P + kChunk - 1u) / kChunk;
    const uint32_t nzc = (g.Z + kErodeZ - 1) / kErodeZ;
    const uint32_t L = GL - J.erode_base;  // block within the job
    stamp += J.erode_base;
    const uint32_t c = L % nch, zg = L / nch;
    const uint32_t zb = zg * kErodeZ;
    const uint32_t i0 = c * kChunk;
    const uint32_t ylo = i0 / g.W, yhi = min(i0 + kChunk - 1u, P - 1u) / g.W;
    if (zb >= z1 || zb + kErodeZ <= z0 || yhi < y0 || ylo >= y1) return false;
    if (full) return true;
    const uint32_t r = g.W / kChunk + 1u;
    const uint32_t clo = c >= r ? c - r : 0u, chi = min(c + r, nch - 1u);
    bool visit = false;
    for (uint32_t cc = clo; cc <= chi; cc++) visit |= stamp[zg * nch + cc] >= gpass;
    if (zg > 0) visit |= stamp[L - nch] >= gpass;
    if (zg + 1 < nzc) visit |= stamp[L + nch] >= gpass;
    return visit;
}

// The voxels of word G that keep a solid neighbour on every axis: gm and gp are
// the words beside it in x, the others the words beside it in y and z.
__device__ __forceinline__ uint32_t erode_word(uint32_t G, uint32_t gm, uint32_t gp, uint32_t ym,
                                               uint32_t yp, uint32_t zm, uint32_t zp) {
    return G & ((G >> 1) | (gm << 31) | (G << 1) | (gp >> 31)) & (ym | yp) & (zm | zp);
}

// Sweeps a block makes over its own words before it leaves the rest to the
// next pass.  With one sweep a pass, a room's open sheets took 13 passes (each
// a launch, a read-back every four); swept to rest within the block, 3 and one
// that finds nothing: k_erode and the call, room 512x403x303 89 -> 39 us and
// 530 -> 493 us, 64-mesh batch 333 -> 205 us and 3340 -> 3113 us, room at
// 256x203x153 474 -> 442 us.  The hall (1536x1024x768), which converged in
// four passes as it was, pays for the barrier: 105 -> 108 us.
constexpr uint32_t kErodeIters = 64;

// A workgroup's LDS in the erosion pass: the block's words, and the planes with
// removals (see erode_block).
struct ErodeLds {
    uint32_t (*words)[kChunk];
    uint32_t (*act)[3];
    uint32_t set;
};

// One logical block GL (of job j) of an erosion pass.
__device__ __forceinline__ void erode_block(const Job &J, uint32_t j, uint32_t GL, uint32_t njobs,
                                            uint32_t y0, uint32_t y1, uint32_t z0, uint32_t z1,
                                            uint32_t *__restrict__ stamp,
                                            uint32_t *__restrict__ changes,
                                            uint32_t *__restrict__ totals,
                                            uint32_t *__restrict__ notconv, uint32_t pass,
                                            uint32_t gpass, ErodeLds &L) {
    const GridDims g = J.gd;
    VK_G uint32_t *__restrict__ bits = gptr(J.bits);
    const uint32_t P = g.W * g.Y;  // words per plane
    const uint32_t nch = (P + kChunk - 1u) / kChunk;
    const uint32_t blk = GL - J.erode_base;  // block within the job
    stamp += J.erode_base;
    const uint32_t c = blk % nch, zg = blk / nch;
    const uint32_t zb = zg * kErodeZ;
    const uint32_t i0 = c * kChunk;
    const uint32_t tid = threadIdx.x, lane = tid & (kWave - 1u);
    const uint32_t i = i0 + tid;
    const bool valid = i < P;
    const uint32_t y = valid ? i / g.W : 0u;
    const uint32_t w = valid ? i - y * g.W : 0u;
    const size_t rowW = g.W, planeW = P;
    const size_t col0 = valid ? i : 0;  // index of (w, y) in plane 0
    const bool hyn = valid && y > 0, hyp = valid && y + 1 < g.Y;
    // Column z = zb-1 .. zb+kErodeZ of this word, the rows above and below it
    // for the thread's planes, and the words across the wave's edges: all
    // loads are independent and in flight together (clamped addresses).
    uint32_t col[kErodeZ + 2], yn[kErodeZ], yp[kErodeZ], em[kErodeZ], ep[kErodeZ];
#pragma unroll
    for (uint32_t k = 0; k < kErodeZ + 2; k++) {
        const uint32_t z = zb + k - 1u;  // wraps to UINT32_MAX for zb == 0, k == 0
        const bool ok = valid && z < g.Z;
        col[k] = bits[ok ? (size_t)z * planeW + col0 : 0];
        if (!ok) col[k] = 0u;
    }
#pragma unroll
    for (uint32_t k = 0; k < kErodeZ; k++) {
        const uint32_t z = zb + k;
        const bool ok = valid && z < g.Z;
        const size_t wi = ok ? (size_t)z * planeW + col0 : 0;
        yn[k] = bits[ok && hyn ? wi - rowW : 0];
        yp[k] = bits[ok && hyp ? wi + rowW : 0];
        if (!(ok && hyn)) yn[k] = 0u;
        if (!(ok && hyp)) yp[k] = 0u;
        const bool lm = ok && lane == 0 && w > 0;
        const bool rp = ok && lane == kWave - 1 && w + 1 < g.W;
        em[k] = lm ? bits[wi - 1] : 0u;
        ep[k] = rp ? bits[wi + 1] : 0u;
    }
    uint32_t dirty = 0u;  // planes with a removal
#pragma unroll
    for (uint32_t k = 0; k < kErodeZ; k++) {
        const uint32_t z = zb + k;
        const uint32_t G = col[k + 1];
        // x neighbours: adjacent lanes hold the adjacent words of the plane
        // (whole-wave DPP shifts, no LDS round trip); across a row's ends
        // there is nothing.
        uint32_t gm = (uint32_t)__builtin_amdgcn_update_dpp(0, (int)G, kDppWaveShr1, 0xF, 0xF, false);
        uint32_t gp = (uint32_t)__builtin_amdgcn_update_dpp(0, (int)G, kDppWaveShl1, 0xF, 0xF, false);
        if (lane == 0) gm = em[k];
        if (lane == kWave - 1) gp = ep[k];
        if (w == 0) gm = 0u;
        if (w + 1 >= g.W) gp = 0u;
        if (!valid || !G || z >= g.Z || z < z0 || z >= z1 || y < y0 || y >= y1) continue;
        const uint32_t out = erode_word(G, gm, gp, yn[k], yp[k], col[k], col[k + 2]);
        if (out != G) {
            col[k + 1] = out;  // later planes of this column see the update
            dirty |= 1u << k;
        }
    }
    // A removal takes its neighbours along one voxel at a time (a sheet with a
    // free edge goes row by row), so a block that removed something repeats on
    // its own words, shared through LDS, until it is stable against what it
    // read of its surroundings; a sweep looks at the planes next to the last
    // one's removals.  Sweep n reads act[n % 3], gathers into the next and
    // clears the one after that; two blocks in a row use different sets, so a
    // wave that is ahead writes nothing that another still reads.
    uint32_t *act = L.act[L.set & 1u];
    L.set++;
    auto gather = [&](uint32_t planes, uint32_t *to) {
        if (!__ballot(planes != 0u)) return;
        uint32_t m = 0u;
#pragma unroll
        for (uint32_t k = 0; k < kErodeZ; k++)
            m |= __ballot((planes >> k) & 1u) ? 1u << k : 0u;
        if (lane == 0) atomicOr(to, m);
    };
    gather(dirty, &act[0]);
    __syncthreads();
    uint32_t m = __builtin_amdgcn_readfirstlane(act[0]);
    if (m) {  // uniform over the block
#pragma unroll
        for (uint32_t k = 0; k < kErodeZ; k++) L.words[k][tid] = col[k + 1];
        __syncthreads();
        const bool hm = tid >= g.W, hp = tid + g.W < kChunk;  // rows held by the block
        const bool xm = tid > 0u, xp = tid + 1u < kChunk;
        for (uint32_t it = 0; m && it < kErodeIters; it++) {
            const uint32_t near = m | m << 1 | m >> 1;
            uint32_t removed = 0u;
#pragma unroll
            for (uint32_t k = 0; k < kErodeZ; k++) {
                if (!((near >> k) & 1u)) continue;  // uniform
                const uint32_t z = zb + k;
                const uint32_t G = col[k + 1];
                if (!valid || !G || z >= g.Z || z < z0 || z >= z1 || y < y0 || y >= y1) continue;
                const uint32_t gm = w == 0u ? 0u : xm ? L.words[k][tid - 1u] : em[k];
                const uint32_t gp = w + 1u >= g.W ? 0u : xp ? L.words[k][tid + 1u] : ep[k];
                const uint32_t ym = hm ? L.words[k][tid - g.W] : yn[k];
                const uint32_t yq = hp ? L.words[k][tid + g.W] : yp[k];
                const uint32_t out = erode_word(G, gm, gp, ym, yq, col[k], col[k + 2]);
                if (out != G) {
                    col[k + 1] = out;
                    L.words[k][tid] = out;
                    removed |= 1u << k;
                }
            }
            dirty |= removed;
            gather(removed, &act[(it + 1u) % 3u]);
            if (tid == 0) act[(it + 2u) % 3u] = 0u;
            __syncthreads();
            m = __builtin_amdgcn_readfirstlane(act[(it + 1u) % 3u]);
        }
        __syncthreads();
        if (tid < 3u) act[tid] = 0u;
    }
#pragma unroll
    for (uint32_t k = 0; k < kErodeZ; k++)
        if ((dirty >> k) & 1u) bits[(size_t)(zb + k) * planeW + col0] = col[k + 1];
    const bool changed = dirty != 0u;
    // Flags, not counts: plain stores of 1 (atomics from every changing
    // wave to one address would serialise).
    const unsigned long long any = __ballot(changed);  // every lane takes part
    if (lane == 0 && any) {
        changes[pass * njobs + j] = 1u;
        totals[pass] = 1u;
        if (notconv) *notconv = 1u;
        stamp[blk] = gpass + 1u;
    }
}

// Persistent pass: the grid is at most the resident workgroups; each XCD
// walks a contiguous run of logical blocks (its L2 then holds the neighbour
// planes).  After the first pass only the jobs the previous pass changed are
// visited (a batch may have one slow job among many finished ones).
__global__ __launch_bounds__(256, 8) void k_erode(const Job *__restrict__ jobs,
                                               const uint32_t *__restrict__ erode_bases,
                                               uint32_t njobs, uint32_t y0, uint32_t y1,
                                               uint32_t z0, uint32_t z1,
                                               uint32_t *__restrict__ stamp,
                                               uint32_t *__restrict__ changes,
                                               uint32_t *__restrict__ totals,
                                               uint32_t *__restrict__ notconv, uint32_t pass,
                                               uint32_t gpass, int full) {
    const uint32_t total = erode_bases[njobs];  // bases[njobs] = all blocks
    const uint32_t nx = gridDim.x / kXcds;      // workgroups per XCD (grid: a multiple of 8)
    const uint32_t x = blockIdx.x % kXcds, slot = blockIdx.x / kXcds;
    const uint32_t per = (total + kXcds - 1u) / kXcds;
    const uint32_t lo = x * per, hi = min(lo + per, total);
    const uint32_t start = lo + slot;  // this workgroup takes start, start + nx, ...
    __shared__ uint32_t words[kErodeZ][kChunk], act[2][3];
    if (threadIdx.x < 6u) act[threadIdx.x / 3u][threadIdx.x % 3u] = 0u;
    __syncthreads();
    ErodeLds L{words, act, 0u};
    if (pass == 0) {
        for (uint32_t GL = start; GL < hi; GL += nx) {
            const uint32_t j = job_of(erode_bases, njobs, GL);
            if (erode_visit(jobs[j], GL, y0, y1, z0, z1, stamp, gpass, full))
                erode_block(jobs[j], j, GL, njobs, y0, y1, z0, z1, stamp, changes, totals,
                            notconv, pass, gpass, L);
        }
        return;
    }
    // Later passes: the workgroup's blocks are checked 256 at a time, one
    // per thread (its job changed in the previous pass, and the stamps near
    // it), and only the blocks that pass are visited, from a list in LDS.
    // (Checked one after another, each block would cost the workgroup a
    // round trip to memory, most of them to skip it.)
    __shared__ uint32_t s_list[256];
    __shared__ uint32_t s_n;
    const uint32_t tid = threadIdx.x;
    const uint32_t *prev = changes + (pass - 1u) * njobs;
    for (uint32_t k0 = 0; start + k0 * nx < hi; k0 += blockDim.x) {  // uniform
        if (tid == 0) s_n = 0u;
        __syncthreads();
        const uint32_t GLt = start + (k0 + tid) * nx;
        if (GLt < hi) {
            const uint32_t jt = job_of(erode_bases, njobs, GLt);
            if (prev[jt] != 0u && erode_visit(jobs[jt], GLt, y0, y1, z0, z1, stamp, gpass, full))
                s_list[atomicAdd(&s_n, 1u)] = GLt;
        }
        __syncthreads();
        const uint32_t n = s_n;
        for (uint32_t i = 0; i < n; i++) {
            const uint32_t GL = s_list[i];
            const uint32_t j = job_of(erode_bases, njobs, GL);
            erode_block(jobs[j], j, GL, njobs, y0, y1, z0, z1, stamp, changes, totals, notconv,
                        pass, gpass, L);
        }
        __syncthreads();
    }
}

// ---------------------------------------------------------------------------
// Node writing
// ---------------------------------------------------------------------------
// 16-byte slots between the pieces of a word in a wave's staging run: 64 lanes
// plus a shift of 16 LDS banks.
constexpr uint32_t kStagePitch = kWave + 4u;
// Buffer offset past every range used below: loads there return 0 and
// stores there are dropped (raw buffer range check, offset >= size).
constexpr uint32_t kOob = 0x80000000u;

typedef __amdgpu_buffer_rsrc_t Rsrc;
__device__ __forceinline__ Rsrc rsrc(const VK_G void *base, uint32_t bytes) {
    return __builtin_amdgcn_make_buffer_rsrc((void *)base, (short)0, (int)bytes, 0x00020000);
}
__device__ __forceinline__ uint32_t ld32(Rsrc r, uint32_t off) {
    return __builtin_amdgcn_raw_buffer_load_b32(r, (int)off, 0, 0);
}
__device__ __forceinline__ u32x4 ld128(Rsrc r, uint32_t off) {
    return __builtin_amdgcn_raw_buffer_load_b128(r, (int)off, 0, 0);
}
__device__ __forceinline__ void st128(Rsrc r, uint32_t off, u32x4 v) {
    __builtin_amdgcn_raw_buffer_store_b128(v, r, (int)off, 0, 0);
}

// (m & a) | (~m & b): one v_bfi_b32.
__device__ __forceinline__ uint32_t bfi(uint32_t m, uint32_t a, uint32_t b) {
    return (m & a) | (~m & b);
}
// Exchanges the bits of a above each group of kS bits with the bits of b
// below them: one step of a bit-matrix transpose (kM: the low kS bits of
// every 2 kS).
template <uint32_t kS, uint32_t kM>
__device__ __forceinline__ void swap_bits(uint32_t &a, uint32_t &b) {
    const uint32_t t = bfi(kM, a, b << kS);
    b = bfi(kM, a >> kS, b);
    a = t;
}
// Id bytes of a word's 32 voxels (four per dword, voxel order; voxel i at bit
// 31 - i of the planes): the five bit planes, padded to eight, are transposed
// as four 8x8 bit matrices side by side (bytes of the words), then the bytes
// are put in voxel order.  61 operations for any number of boundary voxels.
__device__ __forceinline__ void id_bytes(const IdPlanes &o, uint32_t idw[8]) {
    uint32_t r[8] = {o.b[0], o.b[1], o.b[2], o.b[3], o.b[4], 0u, 0u, 0u};
#pragma unroll
    for (int i = 0; i < 4; i++) swap_bits<4, 0x0F0F0F0Fu>(r[i], r[i + 4]);
#pragma unroll
    for (int i = 0; i < 2; i++) {
        swap_bits<2, 0x33333333u>(r[i], r[i + 2]);
        swap_bits<2, 0x33333333u>(r[i + 4], r[i + 6]);
    }
#pragma unroll
    for (int i = 0; i < 8; i += 2) swap_bits<1, 0x55555555u>(r[i], r[i + 1]);
    // r[j] byte k: the id of bit position 8 k + j.
#pragma unroll
    for (int h = 0; h < 2; h++) {
        const uint32_t a = r[7 - 4 * h], b = r[6 - 4 * h], c = r[5 - 4 * h], d = r[4 - 4 * h];
        const uint32_t ab0 = __builtin_amdgcn_perm(b, a, 0x05010400u);
        const uint32_t ab1 = __builtin_amdgcn_perm(b, a, 0x07030602u);
        const uint32_t cd0 = __builtin_amdgcn_perm(d, c, 0x05010400u);
        const uint32_t cd1 = __builtin_amdgcn_perm(d, c, 0x07030602u);
        idw[6 + h] = __builtin_amdgcn_perm(cd0, ab0, 0x05040100u);
        idw[4 + h] = __builtin_amdgcn_perm(cd0, ab0, 0x07060302u);
        idw[2 + h] = __builtin_amdgcn_perm(cd1, ab1, 0x05040100u);
        idw[0 + h] = __builtin_amdgcn_perm(cd1, ab1, 0x07060302u);
    }
}

// Cartesian node write: a block takes kChunk consecutive words of a plane
// (plane-linear, so no lane idles on narrow rows), each thread a column of
// kNodeZ planes.  All loads go through buffer resources, one per plane, so
// every address is a 32-bit lane offset and a neighbour outside the grid
// (z -1 / Z, rows -1 / Y, lanes past the plane) falls outside its range and
// reads 0 without a branch.  Every load of the column is issued before the
// first use, so a wave waits for memory once; the 32 material bytes of each
// surface word come in a second round trip.  x neighbours come from
// adjacent lanes.
//
// A word whose 32 voxels are all empty or all fully surrounded (the bulk of
// a grid) is stored as a constant.  Otherwise the bit planes of the ids come
// from the bit-sliced table (orient_planes; all six neighbours give id 27)
// and are transposed into bytes in registers (id_bytes), and surface voxels
// OR in their material (bytes of the word's other voxels are 0 in the
// material grid).  The transpose replaced a loop over the boundary voxels
// that patched their bytes in LDS: room at 1 cm (512x403x303 LongNodes) 38.9
// -> 31.2 us, hall (1536x1024x768 ShortNodes) 385 -> 362 us, both with 128x4x8
// bricks: 4.8 TB/s of the hall's 1.7 GB, where a large copy runs at 5.0.  With
// 32x8x16 bricks, whose material words of neighbouring lanes lie 4 KB apart, the
// hall takes 428 us (1.6 GB at 3.75 TB/s); the brick pass gains more.
//
// With several erosion subspaces (voxSplitRes y/z smaller than the grid) the
// reference computes a subspace's ids before later subspaces erode
// (src/host_side.cpp:1183-1206), so neighbours across a +y/+z seam are read
// from the pre-erosion snapshot `pre` (seam rows flagged in ystart/zstart);
// that path is a kernel of its own (k_nodes_cart_pre), so the common one
// holds no registers for it.
template <bool kPre>
__device__ __forceinline__ void nodes_cart(const Job *__restrict__ jobs,
                                           const uint32_t *__restrict__ node_bases,
                                           uint32_t njobs, const uint32_t *__restrict__ pre,
                                           const uint8_t *__restrict__ ystart,
                                           const uint8_t *__restrict__ zstart) {
    // A wave's node run of one plane on its way out: the 16-byte pieces of a
    // word kStagePitch apart, so that lanes write consecutive slots and the
    // pieces of neighbouring words read back from other banks.
    __shared__ uint4 stage[256 / kWave][4 * kStagePitch];
    const uint32_t GL = xcd_logical_block(node_bases[njobs]);  // bases[njobs] = all blocks
    if (GL == UINT32_MAX) return;  // uniform over the block
    const Job &J = jobs[job_of(node_bases, njobs, GL)];
    const GridDims g = J.gd;
    const int use_mats = J.use_mats, kind = J.kind;
    const bool zbrd = J.zero_border != 0, rot = J.rot_ids != 0;
    const BrickDims bd = J.bdn;
    const uint32_t P = g.W * g.Y;  // words per plane
    const uint32_t nch = (P + kChunk - 1u) / kChunk;
    const uint32_t lb = GL - J.node_base;  // block within the job
    const uint32_t tid = threadIdx.x, tx = tid & (kWave - 1u);
    const uint32_t zb = (lb / nch) * kNodeZ;
    const uint32_t i0 = (lb % nch) * kChunk, i = i0 + tid;
    const bool valid = i < P;
    const uint32_t y = valid ? i / g.W : 0u;
    const uint32_t w = valid ? i - y * g.W : 0u;
    const uint32_t P4 = P * 4u, W4 = g.W * 4u;
    // Byte offsets within a plane: the word, its y neighbours (row -1 wraps
    // past the range, row Y lands past it) and, for the wave's first and
    // last lane, the x neighbour held by the adjacent wave.
    const uint32_t o = valid ? i * 4u : kOob;
    const uint32_t oyn = valid ? o - W4 : kOob;
    const uint32_t oyp = o + W4;
    const uint32_t oex = valid && tx == 0u && w > 0u                 ? o - 4u
                         : valid && tx == kWave - 1u && w + 1u < g.W ? o + 4u
                                                                      : kOob;
    const VK_G uint32_t *bits = gptr(J.bits);
    auto plane = [&](const VK_G uint32_t *base, uint32_t z) {  // z -1 wraps to UINT32_MAX
        return z < g.Z ? rsrc(base + (size_t)z * P, P4) : rsrc(base, 0u);
    };
    // Round trip 1.
    uint32_t col[kNodeZ + 2], yn[kNodeZ], yp[kNodeZ], ex[kNodeZ];
#pragma unroll
    for (uint32_t k = 0; k < kNodeZ + 2; k++) col[k] = ld32(plane(bits, zb + k - 1u), o);
#pragma unroll
    for (uint32_t k = 0; k < kNodeZ; k++) {
        const Rsrc r = plane(bits, zb + k);
        yn[k] = ld32(r, oyn);
        yp[k] = ld32(r, oyp);
        ex[k] = ld32(r, oex);  // the x neighbour across the wave's edge (edge lanes)
    }
    uint32_t ypp[kNodeZ], zpp[kNodeZ];
    bool ys = false, zs[kNodeZ];
#pragma unroll
    for (uint32_t k = 0; k < kNodeZ; k++) {
        ypp[k] = 0u;
        zpp[k] = 0u;
        zs[k] = false;
    }
    if (kPre) {
        const VK_G uint32_t *pg = gptr(pre);
        ys = valid && y + 1u < g.Y && ystart[y + 1u] != 0;
#pragma unroll
        for (uint32_t k = 0; k < kNodeZ; k++) {
            const uint32_t z = zb + k;
            ypp[k] = ld32(plane(pg, z), oyp);
            zpp[k] = ld32(plane(pg, z + 1u), o);
            zs[k] = z + 1u < g.Z && zstart[z + 1u] != 0;
        }
    }
    // Surface words (a word holding a surface voxel) from the brick's word
    // mask, and the offsets of their material bytes.
    bool S[kNodeZ];
    uint32_t moff[kNodeZ];
#pragma unroll
    for (uint32_t k = 0; k < kNodeZ; k++) {
        S[k] = false;
        moff[k] = kOob;
    }
    Rsrc mr = rsrc(gptr(J.bits), 0u);
    if (use_mats) {  // uniform; the kNodeZ planes lie in one brick (kNodeZ divides its depth)
        // Material blocks relative to the first brick row the block touches.
        const uint32_t lbytes = bd.lwx + bd.lby + bd.lbz + 5u;  // log2 bytes per brick
        const uint32_t yb0 = (i0 / g.W) >> bd.lby;
        const uint32_t yb1 = ((min(i0 + kChunk, P) - 1u) / g.W) >> bd.lby;
        const uint32_t brow0 = ((zb >> bd.lbz) * bd.nby + yb0) * bd.nbx;
        const uint32_t nbrow = (yb1 - yb0 + 1u) * bd.nbx;  // bricks the block touches
        mr = rsrc(gptr(J.matgrid) + ((size_t)brow0 << lbytes), nbrow << lbytes);
        const uint32_t b = ((y >> bd.lby) - yb0) * bd.nbx + (w >> bd.lwx);
        const u32x4 hm = ld128(rsrc(gptr(J.wmask) + (size_t)brow0 * 4u, nbrow * 16u),
                               valid ? b * 16u : kOob);
        const uint32_t wib = word_in_brick(bd, w, y, zb);
        const uint32_t lane_off = (b << lbytes) + (wib << 5);
#pragma unroll
        for (uint32_t k = 0; k < kNodeZ; k++) {
            const uint32_t bit = wib + (k << (bd.lby + bd.lwx));
            const uint32_t q = bit >> 5;
            const uint32_t mw = q == 0u ? hm.x : q == 1u ? hm.y : q == 2u ? hm.z : hm.w;
            S[k] = ((mw >> (bit & 31u)) & 1u) != 0u;
            moff[k] = lane_off + ((k << (bd.lby + bd.lwx)) << 5);
        }
    }
    // Round trip 2: the 32 material bytes of each surface word.
    u32x4 ma[kNodeZ], mb[kNodeZ];
#pragma unroll
    for (uint32_t k = 0; k < kNodeZ; k++) {
        ma[k] = u32x4{0u, 0u, 0u, 0u};
        mb[k] = ma[k];
        if (S[k]) {
            ma[k] = ld128(mr, moff[k]);
            mb[k] = ld128(mr, moff[k] + 16u);
        }
    }
    const uint32_t nbw = kind == 0 ? 32u : 64u;  // node bytes per word
    VK_G uint8_t *nodes = (VK_G uint8_t *)gptr(J.nodes);
    const uint32_t lane = tx;
    uint4 *wst = stage[tid / kWave];  // this wave's staging run
    // The wave's 64 words are consecutive, so its nodes of a plane are one
    // run (2 KB ShortNode, 4 KB LongNode) starting at byte wrun: staged in
    // LDS in node order and stored lane by lane, each store writes 1 KB of
    // whole lines instead of every other 16 bytes.
    const uint32_t wrun = (i0 + (tid - lane)) * nbw;
#pragma unroll
    for (uint32_t k = 0; k < kNodeZ; k++) {
        const uint32_t z = zb + k;
        if (z >= g.Z) break;  // uniform
        const uint32_t G = col[k + 1];
        uint32_t gm = (uint32_t)__shfl_up((int)G, 1);
        uint32_t gp = (uint32_t)__shfl_down((int)G, 1);
        if (tx == 0) gm = ex[k];
        if (tx == kWave - 1) gp = ex[k];
        if (w == 0) gm = 0u;
        if (w + 1 >= g.W) gp = 0u;
        const uint32_t L = (G >> 1) | (gm << 31);
        const uint32_t R = (G << 1) | (gp >> 31);
        // Seam selects as masks: a select between two array elements
        // becomes a select between the arrays, which then live in scratch.
        const uint32_t ysm = ys ? ~0u : 0u, zsm = zs[k] ? ~0u : 0u;
        const uint32_t Yn = yn[k];
        const uint32_t Yp = (yp[k] & ~ysm) | (ypp[k] & ysm);
        const uint32_t Zn = col[k];
        const uint32_t Zp = (col[k + 2] & ~zsm) | (zpp[k] & zsm);
        const uint32_t interior = G & L & R & Yn & Yp & Zn & Zp;
        const uint32_t bnd = G & ~interior;  // solid, some neighbour missing
        uint32_t idw[8];
        if (bnd == 0u && !S[k]) {
            // All 32 voxels empty, or all fully surrounded (id 27).
            const uint32_t v = interior ? 0x1B1B1B1Bu : 0u;
#pragma unroll
            for (int j = 0; j < 8; j++) idw[j] = v;
        } else {
            // A model rotated about z (x slices) takes its ids in the
            // un-rotated frame: its -x/+x are the rotated -y/+y, its -y/+y
            // the rotated +x/-x.
            IdPlanes op = rot ? orient_planes(Yn, Yp, R, L, Zn, Zp)
                              : orient_planes(L, R, Yn, Yp, Zn, Zp);
#pragma unroll
            for (int j = 0; j < 5; j++) op.b[j] &= G;
            id_bytes(op, idw);
        }
        const uint32_t md[8] = {ma[k].x, ma[k].y, ma[k].z, ma[k].w,
                                mb[k].x, mb[k].y, mb[k].z, mb[k].w};
        const Rsrc nr = rsrc(nodes + (size_t)z * P * nbw, P * nbw);
        // A partition with neighbours clears its border (zeroPadding,
        // src/voxelizer.cu:4811-4844): whole rows and planes, and the first
        // and last node of each row.
        const uint32_t all =
            zbrd && (y == 0u || y + 1u == g.Y || z == 0u || z + 1u == g.Z) ? 0u : ~0u;
        const bool x0 = zbrd && w == 0u, x1 = zbrd && w + 1u == g.W;
        if (kind == 0) {  // ShortNode byte: id | material << 5
            uint32_t out[8];
#pragma unroll
            for (int j = 0; j < 8; j++) out[j] = (idw[j] | ((md[j] << 5) & 0xE0E0E0E0u)) & all;
            if (x0) out[0] &= 0xFFFFFF00u;
            if (x1) out[7] &= 0x00FFFFFFu;
            wst[lane] = make_uint4(out[0], out[1], out[2], out[3]);
            wst[kStagePitch + lane] = make_uint4(out[4], out[5], out[6], out[7]);
            wave_lds_sync();
#pragma unroll
            for (uint32_t q = 0; q < 2u; q++) {
                const uint32_t piece = q * kWave + lane;
                const uint4 v = wst[(piece & 1u) * kStagePitch + (piece >> 1)];
                st128(nr, wrun + piece * 16u, u32x4{v.x, v.y, v.z, v.w});
            }
        } else {  // LongNode halfword: id | material << 8
            uint32_t out[16];
#pragma unroll
            for (int j = 0; j < 8; j++) {
                out[2 * j] = __builtin_amdgcn_perm(md[j], idw[j], 0x05010400u) & all;
                out[2 * j + 1] = __builtin_amdgcn_perm(md[j], idw[j], 0x07030602u) & all;
            }
            if (x0) out[0] &= 0xFFFF0000u;
            if (x1) out[15] &= 0x0000FFFFu;
#pragma unroll
            for (uint32_t q = 0; q < 4u; q++)
                wst[q * kStagePitch + lane] =
                    make_uint4(out[4 * q], out[4 * q + 1], out[4 * q + 2], out[4 * q + 3]);
            wave_lds_sync();
#pragma unroll
            for (uint32_t q = 0; q < 4u; q++) {
                const uint32_t piece = q * kWave + lane;
                const uint4 v = wst[(piece & 3u) * kStagePitch + (piece >> 2)];
                st128(nr, wrun + piece * 16u, u32x4{v.x, v.y, v.z, v.w});
            }
        }
        wave_lds_sync();  // the run is read out before the next plane's writes
    }
}
__global__ __launch_bounds__(256) void k_nodes_cart(const Job *__restrict__ jobs,
                                                    const uint32_t *__restrict__ node_bases,
                                                    uint32_t njobs) {
    nodes_cart<false>(jobs, node_bases, njobs, nullptr, nullptr, nullptr);
}
// The seam path holds 8 more registers per thread; it runs at one wave per
// SIMD less rather than spill.
__global__ __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(1, 5))) void k_nodes_cart_pre(
    const Job *__restrict__ jobs, const uint32_t *__restrict__ node_bases, uint32_t njobs,
    const uint32_t *__restrict__ pre, const uint8_t *__restrict__ ystart,
    const uint8_t *__restrict__ zstart) {
    nodes_cart<true>(jobs, node_bases, njobs, pre, ystart, zstart);
}

// PartialNode expansion (processVoxel<PartialNode>, src/voxelizer.cu:
// 2997-3033; r = float(solid) from constructNodeList2, 1675, which erosion
// leaves alone, so the bits are read from the pre-erosion copy).  A surface
// node's winner key comes from the keygrid at the node's position in its
// brick (as its material in matgrid); the ratio is computed for the winner at
// the node's alloc coordinates.  A cleared partition border keeps r = 0
// (zeroPadding stores Node()).
//
// A block takes kPartialWords words.  The cut volume is over a thousand
// instructions and few nodes need it (about one in eight of a furnished
// room's, mostly one or two per 32-voxel word of a wall), so the block first
// lists its surface nodes in LDS and then computes their ratios with full
// waves, where a thread per node ran the whole path for a few lanes; the
// nodes are written once, two per lane.  Room at 2 cm (256x203x153 nodes,
// 64 MB): 579 us with a thread per node, 265 us with the list, 82 us with
// the cut polygons in registers too (vox_math.h), bound by the VALU work of
// about a million cut volumes.
__global__ __launch_bounds__(256) void k_nodes_partial(const Job *__restrict__ jobs, uint32_t j) {
    __shared__ uint32_t s_bits[kPartialWords], s_surf[kPartialWords], s_key[kPartialWords];
    __shared__ uint32_t s_pos[kPartialWords];
    __shared__ uint32_t s_y[kPartialWords], s_z[kPartialWords];
    __shared__ uint16_t s_queue[kPartialWords * 32];
    __shared__ float s_ratio[kPartialWords * 32];
    __shared__ uint32_t s_n;
    const Job &J = jobs[j];
    const GridDims g = J.gd;
    const BrickDims bd = J.bdn;
    const uint32_t tid = threadIdx.x, lane = lane_id();
    const bool mats = J.use_mats != 0, embed = J.embed != 0;
    const uint32_t nwords = g.W * g.Y * g.Z;  // < 2^27: at most 2^32 nodes
    const uint32_t wi0 = blockIdx.x * kPartialWords;
    const uint32_t lvox = bd.lwx + bd.lby + bd.lbz + 5u;  // log2 voxels per brick
    if (tid == 0) s_n = 0u;
    static_assert(kPartialWords == kWave, "one wave loads the block's words");
    if (tid < kPartialWords) {
        const uint32_t wi = wi0 + tid;
        uint32_t bits = 0u, surf = 0u, key = 0u, w = 0u, y = 0u, z = 0u;
        if (wi < nwords) {
            const uint32_t row = wi / g.W;
            w = wi - row * g.W;
            z = row / g.Y;
            y = row - z * g.Y;
            bits = gptr(J.pbits)[wi];  // before erosion
            if (mats) {
                const uint32_t b = brick_of_word(bd, w, y, z);
                if (gptr(J.bhist)[b]) surf = gptr(J.surf)[wi] & bits;
                // Word index in the keygrid: grids hold fewer than 2^32 voxels,
                // brick padding at most doubles each axis.
                key = (b << (lvox - 5u)) + word_in_brick(bd, w, y, z);
            }
            if (J.zero_border) {
                uint32_t keep = y == 0u || y + 1u == g.Y || z == 0u || z + 1u == g.Z ? 0u : ~0u;
                if (w == 0u) keep &= 0x7FFFFFFFu;
                if (w + 1u == g.W) keep &= ~1u;
                bits &= keep;
                surf &= keep;
            }
        }
        s_bits[tid] = bits;
        s_surf[tid] = surf;
        s_key[tid] = key;
        s_pos[tid] = w;
        s_y[tid] = y;
        s_z[tid] = z;
    }
    __syncthreads();
    // The block's surface nodes, in no particular order.
    for (uint32_t p = tid; p < kPartialWords * 32u; p += 256u) {
        const bool on = ((s_surf[p >> 5] >> (31u - (p & 31u))) & 1u) != 0u;
        const unsigned long long m = __ballot(on);
        if (!m) continue;
        uint32_t base = 0u;
        if (lane == 0u) base = atomicAdd(&s_n, (uint32_t)__popcll(m));
        base = (uint32_t)__builtin_amdgcn_readfirstlane((int)base);
        const uint32_t below = __builtin_amdgcn_mbcnt_hi(
            (uint32_t)(m >> 32), __builtin_amdgcn_mbcnt_lo((uint32_t)m, 0u));
        if (on) s_queue[base + below] = (uint16_t)p;
    }
    __syncthreads();
    const uint32_t n = s_n;
    for (uint32_t q = tid; q < n; q += 256u) {
        const uint32_t p = s_queue[q], k = p >> 5, x = p & 31u;
        const uint32_t key = gptr(J.keygrid)[((size_t)s_key[k] << 5) + x];
        const uint32_t t = embed ? (key >> 8) & 0x3FFFFFu : key & 0x3FFFFFFFu;
        const int32_t node[3] = {(int32_t)(s_pos[k] * 32u + x), (int32_t)s_y[k], (int32_t)s_z[k]};
        s_ratio[p] = partial_ratio(J.V, J.I, t, key >> 30, node, J.m, J.fd);
    }
    __syncthreads();
    const VK_G uint32_t *ln = (const VK_G uint32_t *)gptr(J.nodes);
    VK_G u32x4 *out = (VK_G u32x4 *)J.pnodes;
    const size_t h0 = (size_t)wi0 * 16u;  // first pair of nodes
    const uint32_t halves = min(kPartialWords, nwords - wi0) * 16u;
    for (uint32_t h = tid; h < halves; h += 256u) {
        const uint32_t p = 2u * h, k = p >> 5, s = 31u - (p & 31u);
        const uint32_t bits = s_bits[k], surf = s_surf[k];
        const uint32_t two = ln[h0 + h];
        const float r0 = (surf >> s) & 1u ? s_ratio[p] : (bits >> s) & 1u ? 1.0f : 0.0f;
        const float r1 = (surf >> (s - 1u)) & 1u ? s_ratio[p + 1u]
                         : (bits >> (s - 1u)) & 1u ? 1.0f : 0.0f;
        out[h0 + h] = u32x4{two & 0xFFFFu, __float_as_uint(r0), two >> 16, __float_as_uint(r1)};
    }
}

// ---------------------------------------------------------------------------
// FCC nodes
// ---------------------------------------------------------------------------
// 32 FCC nodes of one row: even x from the sub-grid with x shift 0 (word e),
// odd x from the one with x shift d/2 (word o), 16 voxels of each
// (convertToFCCGrid, src/voxelizer.cu:1756-1772).  half picks the 16: the
// bytes are laid out e o e o by one v_perm_b32, then the bits inside each
// 16-bit half are interleaved (a perfect shuffle).
__device__ __forceinline__ uint32_t fcc_word(uint32_t e, uint32_t o, uint32_t half) {
    uint32_t x = __builtin_amdgcn_perm(e, o, half);  // e1 o1 e0 o0
    x = (x & 0xF00FF00Fu) | ((x & 0x00F000F0u) << 4) | ((x >> 4) & 0x00F000F0u);
    x = (x & 0xC3C3C3C3u) | ((x & 0x0C0C0C0Cu) << 2) | ((x >> 2) & 0x0C0C0C0Cu);
    return (x & 0x99999999u) | ((x & 0x22222222u) << 1) | ((x >> 1) & 0x22222222u);
}

// FCC node write: the 12-bit neighbour mask of calculateFCCBoundaries
// (src/voxelizer.cu:1930-2048) as bitwise selects by the (x+z) parity mask,
// materials from the four sub-grids' material grids.
//
// Plane-linear like the Cartesian pass: the FCC words of a plane are numbered
// i = y * FW + fw, a wave takes kFccRun consecutive ones over kFccZ planes,
// its first and last lane hold the words before and after the run (so every
// x neighbour comes from an adjacent lane) and write nothing.  The words of a
// plane's three rows are interleaved from the sub-grids once and serve as the
// plane itself and as its neighbours' neighbour.  The twelve neighbour words
// of 32 nodes are turned into node masks by a bit-matrix transpose in
// registers (144 operations whatever the number of boundary nodes), and the
// wave's nodes go through LDS so that each store writes 1 KB of whole lines.
// Room at 1.6 cm (640x255x384 LongFCCNodes, 251 MB): 58 us, 4.3 TB/s of node
// writes; a wave per 64 words of one row (20 of them there), nine interleaved
// words per plane and a loop over the boundary nodes took 163 us.
__global__ __launch_bounds__(256) void k_nodes_fcc(const Job *__restrict__ jobs,
                                                   const uint32_t *__restrict__ fcc_first,
                                                   const uint32_t *__restrict__ fcc_bases,
                                                   uint32_t nfcc) {
    __shared__ uint4 stage[256 / kWave][8 * kFccPitch];
    const uint32_t GL = xcd_logical_block(fcc_bases[nfcc]);  // bases[nfcc] = all blocks
    if (GL == UINT32_MAX) return;
    const uint32_t f = job_of(fcc_bases, nfcc, GL);
    const Job *__restrict__ Js = jobs + fcc_first[f];
    const GridDims g = Js[0].gd;
    const int use_mats = Js[0].use_mats, kind = Js[0].kind;
    const BrickDims bd = Js[0].bdn;
    const uint32_t FW = 2u * g.W, P = FW * g.Y, FZ = 2u * g.Z;
    const uint32_t nch = fcc_chunks(g);
    const uint32_t L = GL - fcc_bases[f];  // block within the lattice
    const uint32_t lane = lane_id();
    const uint32_t wave = (uint32_t)__builtin_amdgcn_readfirstlane((int)(threadIdx.x / kWave));
    const uint32_t base = (L % nch) * (kFccRun * 4u) + wave * kFccRun;  // first word of the run
    const uint32_t z0 = (L / nch) * kFccZ;                              // first FCC plane
    const uint32_t i = base + lane - 1u;  // UINT32_MAX before the first word
    const bool valid = i < P;
    const uint32_t y = valid ? i / FW : 0u, fw = valid ? i - y * FW : 0u;
    const uint32_t gw = fw >> 1;
    // Byte offsets of the word's sub-grid word and its y neighbours within a
    // plane (row -1 wraps past the range, row Y lands past it: both read 0).
    const uint32_t SP = g.W * g.Y, W4 = g.W * 4u;  // words per sub-grid plane
    const uint32_t o0 = valid ? (y * g.W + gw) * 4u : kOob;
    const uint32_t om = valid ? o0 - W4 : kOob, op = valid ? o0 + W4 : kOob;
    const uint32_t half = (fw & 1u) ? 0x05010400u : 0x07030602u;  // odd words: the low half
    const VK_G uint32_t *sub[4] = {gptr(Js[0].bits), gptr(Js[1].bits), gptr(Js[2].bits),
                                   gptr(Js[3].bits)};
    // Raw words of planes z0 - 1 .. z0 + kFccZ: sub-grids 0 and 1 hold the
    // even planes, 2 and 3 the odd ones (z0 is even).
    uint32_t re[kFccZ + 2][3], ro[kFccZ + 2][3];
#pragma unroll
    for (uint32_t k = 0; k < kFccZ + 2u; k++) {
        const uint32_t fz = z0 + k - 1u;  // wraps for z0 == 0
        const uint32_t s = (k & 1u) ? 0u : 2u;
        const uint32_t bytes = fz < FZ ? SP * 4u : 0u;
        const size_t at = fz < FZ ? (size_t)(fz >> 1) * SP : 0u;
        const Rsrc e = rsrc(sub[s] + at, bytes), o = rsrc(sub[s + 1u] + at, bytes);
        re[k][0] = ld32(e, om); re[k][1] = ld32(e, o0); re[k][2] = ld32(e, op);
        ro[k][0] = ld32(o, om); ro[k][1] = ld32(o, o0); ro[k][2] = ld32(o, op);
    }
    // Surface words and then their material bytes: node k is voxel k / 2 of
    // the sub-grid with x parity k & 1, whose word's half holds 16 voxels.  A
    // word that holds a surface voxel has all 32 material bytes written in
    // the call (0 for its other voxels), so its half is read as 16 bytes.
    u32x4 ma[kFccZ][2];
#pragma unroll
    for (uint32_t k = 0; k < kFccZ; k++) ma[k][0] = ma[k][1] = u32x4{0u, 0u, 0u, 0u};
    if (use_mats) {
        uint32_t wm[kFccZ][2];
#pragma unroll
        for (uint32_t k = 0; k < kFccZ; k++) {
            const uint32_t gz = (z0 + k) >> 1, wib = word_in_brick(bd, gw, y, gz);
            const size_t b = brick_of_word(bd, gw, y, gz);
            const bool in = valid && z0 + k < FZ;
#pragma unroll
            for (uint32_t par = 0; par < 2u; par++) {
                const Job &S = Js[2u * (k & 1u) + par];
                wm[k][par] = in ? gptr(S.wmask)[b * 4u + (wib >> 5)] >> (wib & 31u) : 0u;
            }
        }
#pragma unroll
        for (uint32_t k = 0; k < kFccZ; k++) {
            const uint32_t gz = (z0 + k) >> 1, wib = word_in_brick(bd, gw, y, gz);
            const size_t b = brick_of_word(bd, gw, y, gz);
            const size_t at = (b << (bd.lwx + bd.lby + bd.lbz + 5u)) + (size_t)wib * 32u +
                              ((fw & 1u) ? 16u : 0u);
#pragma unroll
            for (uint32_t par = 0; par < 2u; par++)
                if (wm[k][par] & 1u)
                    ma[k][par] = *(const VK_G u32x4 *)(gptr(Js[2u * (k & 1u) + par].matgrid) + at);
        }
    }
    uint32_t word[kFccZ + 2][3];
#pragma unroll
    for (uint32_t k = 0; k < kFccZ + 2u; k++)
#pragma unroll
        for (uint32_t r = 0; r < 3u; r++) word[k][r] = fcc_word(re[k][r], ro[k][r], half);
    // The word shifted by one node: its -x (left) and +x (right) neighbours.
    const bool first = fw == 0u, last = fw + 1u == FW;
    auto left = [&](uint32_t w) {
        uint32_t p = (uint32_t)__builtin_amdgcn_update_dpp(0, (int)w, kDppWaveShr1, 0xF, 0xF, false);
        if (first) p = 0u;
        return (w >> 1) | (p << 31);
    };
    auto right = [&](uint32_t w) {
        uint32_t n = (uint32_t)__builtin_amdgcn_update_dpp(0, (int)w, kDppWaveShl1, 0xF, 0xF, false);
        if (last) n = 0u;
        return (w << 1) | (n >> 31);
    };
    const uint32_t nbw = kind == 3 ? 64u : 128u;  // node bytes per word
    const uint32_t ppw = nbw / 16u;               // 16-byte pieces per word
    const uint32_t run = base < P ? min(kFccRun, P - base) : 0u;
    VK_G uint8_t *nodes = (VK_G uint8_t *)gptr(Js[0].nodes);
    uint4 *wst = stage[wave];
#pragma unroll
    for (uint32_t k = 0; k < kFccZ; k++) {
        const uint32_t fz = z0 + k;
        if (fz >= FZ) break;  // uniform
        const uint32_t Dm = word[k][0], D0 = word[k][1], Dp = word[k][2];
        const uint32_t Mm = word[k + 1][0], M0 = word[k + 1][1], Mp = word[k + 1][2];
        const uint32_t Um = word[k + 2][0], U0 = word[k + 2][1], Up = word[k + 2][2];
        const uint32_t E = (k & 1u) ? 0x55555555u : 0xAAAAAAAAu;  // (x+z) even
        const uint32_t LM0 = left(M0), RM0 = right(M0);
        uint32_t n[16];
        n[0] = bfi(E, Dm, D0);
        n[1] = left(D0);
        n[2] = right(D0);
        n[3] = bfi(E, D0, Dp);
        n[4] = bfi(E, left(Mm), LM0);
        n[5] = bfi(E, right(Mm), RM0);
        n[6] = bfi(E, LM0, left(Mp));
        n[7] = bfi(E, RM0, right(Mp));
        n[8] = bfi(E, Um, U0);
        n[9] = left(U0);
        n[10] = right(U0);
        n[11] = bfi(E, U0, Up);
        uint32_t interior = M0;
#pragma unroll
        for (int j = 0; j < 12; j++) interior &= n[j];
        // Node masks, two per dword (node 2d in the low half).
        uint32_t mk[16];
        if (M0 == interior && (M0 == 0u || M0 == ~0u)) {  // all empty, or all surrounded
#pragma unroll
            for (int d = 0; d < 16; d++) mk[d] = M0 & 0x0FFF0FFFu;
        } else {
#pragma unroll
            for (int j = 0; j < 12; j++) n[j] &= M0;
#pragma unroll
            for (int j = 12; j < 16; j++) n[j] = 0u;
            // Two 16x16 bit matrices side by side (the halves of the words).
#pragma unroll
            for (int j = 0; j < 8; j++) {
                const uint32_t t = __builtin_amdgcn_perm(n[j + 8], n[j], 0x06020400u);
                n[j + 8] = __builtin_amdgcn_perm(n[j + 8], n[j], 0x07030501u);
                n[j] = t;
            }
#pragma unroll
            for (int j = 0; j < 16; j++)
                if (!(j & 4)) swap_bits<4, 0x0F0F0F0Fu>(n[j], n[j + 4]);
#pragma unroll
            for (int j = 0; j < 16; j++)
                if (!(j & 2)) swap_bits<2, 0x33333333u>(n[j], n[j + 2]);
#pragma unroll
            for (int j = 0; j < 16; j += 2) swap_bits<1, 0x55555555u>(n[j], n[j + 1]);
            // n[j] half h: the mask of bit position 16 h + j; node 31 - that.
#pragma unroll
            for (int d = 0; d < 16; d++)
                mk[d] = __builtin_amdgcn_perm(n[14 - 2 * (d & 7)], n[15 - 2 * (d & 7)],
                                              d < 8 ? 0x07060302u : 0x05040100u);
        }
        const uint32_t a4[4] = {ma[k][0].x, ma[k][0].y, ma[k][0].z, ma[k][0].w};
        const uint32_t c4[4] = {ma[k][1].x, ma[k][1].y, ma[k][1].z, ma[k][1].w};
        const Rsrc nr = rsrc(nodes + ((size_t)fz * P + base) * nbw, run * nbw);
        if (kind == 3) {  // ShortFCCNode: mat<<12 | bid&4095
#pragma unroll
            for (int q = 0; q < 4; q++) {
                uint32_t o[4];
#pragma unroll
                for (int e = 0; e < 4; e++) {
                    const uint32_t a = (a4[q] >> (8 * e)) & 0xFu, c = (c4[q] >> (8 * e)) & 0xFu;
                    o[e] = mk[4 * q + e] | (a << 12) | (c << 28);
                }
                wst[q * kFccPitch + lane] = make_uint4(o[0], o[1], o[2], o[3]);
            }
        } else {  // LongFCCNode: {u16 bid, u8 mat, u8 0}
#pragma unroll
            for (int q = 0; q < 8; q++) {
                uint32_t o[4];
#pragma unroll
                for (int e = 0; e < 2; e++) {
                    const int d = 2 * q + e;
                    const uint32_t a = (a4[d >> 2] >> (8 * (d & 3))) & 0xFFu;
                    const uint32_t c = (c4[d >> 2] >> (8 * (d & 3))) & 0xFFu;
                    o[2 * e] = (mk[d] & 0xFFFFu) | (a << 16);
                    o[2 * e + 1] = (mk[d] >> 16) | (c << 16);
                }
                wst[q * kFccPitch + lane] = make_uint4(o[0], o[1], o[2], o[3]);
            }
        }
        wave_lds_sync();
        // Pieces past the run's end lie outside the range and are dropped.
        const uint32_t lp = kind == 3 ? 2u : 3u;
#pragma unroll
        for (uint32_t s = 0; s < 8u; s++) {
            if (s >= ppw) break;  // uniform
            const uint32_t piece = s * kWave + lane;
            const uint32_t w = min((piece >> lp) + 1u, kWave - 1u);
            const uint4 v = wst[(piece & (ppw - 1u)) * kFccPitch + w];
            st128(nr, piece * 16u, u32x4{v.x, v.y, v.z, v.w});
        }
        wave_lds_sync();  // the run is read out before the next plane's writes
    }
}

}  // namespace vk
