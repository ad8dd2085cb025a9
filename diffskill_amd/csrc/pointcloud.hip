// Point-cloud losses on gfx950: the nearest-neighbour searches under the
// Chamfer losses of the reference (plb/engine/losses/loss.py:183-204, and the
// chamferdist.ChamferDistance loss of plb/engine/taichi_env.py:28-32), those
// losses and their gradients, and the Sinkhorn divergence of its EMD loss.
//
// Nearest neighbours, every pair: brute force over all (query, target) pairs,
// exact in fp32: a workgroup takes 256 queries (one per lane) and one chunk of
// targets staged in LDS; every lane scans the chunk (LDS broadcast reads)
// keeping its smallest squared distance and the first index reaching it.
// Chunks meet through one 64-bit atomicMin per query on (distance bits << 32 |
// index): distances are non-negative, so their bit patterns order like the
// values, and equal distances keep the smaller index.
#include <hip/hip_runtime.h>
#include <algorithm>
#include <cmath>
#include <cstdint>
#include <mutex>
#include <string>

#include "../../include/diffskill_pointcloud.h"

#define DEV_PC __device__ __forceinline__

namespace {

constexpr int PC_WG = 256;     // queries per workgroup
constexpr int PC_CHUNK = 2048; // targets per workgroup (24 KB of LDS)
constexpr unsigned long long PC_EMPTY = 0xffffffffffffffffull;

thread_local std::string g_pc_err;
int pc_fail(const std::string& m) {
    g_pc_err = m;
    return -1;
}

// device address of `scratch` on each GPU, looked up once per device (with
// that device current) on the first pc_nearest_noalloc call there
constexpr int PC_MAX_DEVICES = 64;
std::mutex g_scratch_mu;
unsigned long long* g_scratch_dev[PC_MAX_DEVICES] = {};
int noalloc_scratch(unsigned long long** out);

__global__ void __launch_bounds__(PC_WG) k_pc_clear(unsigned long long* __restrict__ best, int n) {
    int i = blockIdx.x * PC_WG + threadIdx.x;
    if (i < n) best[i] = PC_EMPTY;
}

__global__ void __launch_bounds__(PC_WG) k_pc_nearest(const float* __restrict__ q, int nq, const float* __restrict__ t, int nt,
                                                     unsigned long long* __restrict__ best) {
    __shared__ float sx[PC_CHUNK], sy[PC_CHUNK], sz[PC_CHUNK];
    int t0 = blockIdx.y * PC_CHUNK;
    int nc = min(PC_CHUNK, nt - t0);
    for (int k = threadIdx.x; k < nc; k += PC_WG) {
        const float* p = t + (size_t)(t0 + k) * 3;
        sx[k] = p[0];
        sy[k] = p[1];
        sz[k] = p[2];
    }
    __syncthreads();
    int i = blockIdx.x * PC_WG + threadIdx.x;
    if (i >= nq) return;
    float qx = q[(size_t)i * 3], qy = q[(size_t)i * 3 + 1], qz = q[(size_t)i * 3 + 2];
    float bd = __int_as_float(0x7f800000);
    int bk = -1;
    int k = 0;
    // four independent distances per step, compared in index order
    for (; k + 4 <= nc; k += 4) {
        float d[4];
#pragma unroll
        for (int u = 0; u < 4; u++) {
            float ex = qx - sx[k + u], ey = qy - sy[k + u], ez = qz - sz[k + u];
            d[u] = fmaf(ez, ez, fmaf(ey, ey, ex * ex));
        }
#pragma unroll
        for (int u = 0; u < 4; u++)
            if (d[u] < bd) { bd = d[u]; bk = k + u; }
    }
    for (; k < nc; k++) {
        float ex = qx - sx[k], ey = qy - sy[k], ez = qz - sz[k];
        float d = fmaf(ez, ez, fmaf(ey, ey, ex * ex));
        if (d < bd) { bd = d; bk = k; }
    }
    if (bk >= 0)
        atomicMin(&best[i], ((unsigned long long)__float_as_uint(bd) << 32) | (unsigned)(t0 + bk));
}

// ------------------------------------------------- nearest, spatially sorted
// The same results with most pairs left out.  Both clouds are sorted along a
// Morton curve of 16^3 cells over their own extent (counting sort; a few points far
// outside the others do not count for the extent and share its border cells, those
// with a NaN or infinite coordinate count nowhere), cut into blocks of 32 points
// with their bounding boxes, and a workgroup finds the
// targets of a block of queries: the target block nearest to it and its
// neighbours give every query an upper bound, blocks whose box is further from
// the queries' box than the largest bound are dropped, then those that no
// query's own bound reaches, and the rest is scanned.  The distances are those
// of k_pc_nearest, bit for bit, and equal ones keep the smaller index, so the
// order that the sort's atomics give points of one cell does not show.  Bounds
// are compared with a margin of 1e-6 (a distance's rounding is below 4e-7);
// a comparison that NaN or infinities spoil scans.
// What bounds it: five dependent launches (about 4 us each) and, in the search, the
// latency of the block loads.  Both ways, every pair -> sorted: 30000 x 25001
// points 309 -> 67 us, 10000 x 10000 166 -> 36, 3000 x 3000 164 -> 24 (the search
// over every pair gives a workgroup 2048 targets at least).
constexpr int NN_BITS = 4, NN_CELLS = 1 << (3 * NN_BITS);
constexpr int NN_BLOCK = 32;
constexpr int NN_RUNS = 1 << 16;    // points from which k_nn_box reads runs
constexpr int NN_BOXES = 61;       // workgroups, and partial boxes, of k_nn_box: a wave's lanes at most, and prime
constexpr int NN_LIST = 1024;      // target blocks tested at a time
constexpr float NN_MARGIN = 0.999999f;
typedef float nn4 __attribute__((ext_vector_type(4)));

// one cloud's part of the workspace
struct NnCloud {
    const float* p;
    int n, blocks;
    float* part;        // [NN_BOXES][6] partial boxes: min, -max
    int* count;         // [NN_CELLS]
    unsigned* at;       // [n] cell and rank
    nn4* sorted;        // [blocks * NN_BLOCK] x, y, z, index; padding at infinity
    nn4* box;           // [blocks][2] min, max
};
struct NnPair { NnCloud c[2]; };

// (no target is at a finite distance from it, and no query has it as its nearest)
DEV_PC bool nn_special(float x, float y, float z) { return !(fabsf(x) < INFINITY && fabsf(y) < INFINITY && fabsf(z) < INFINITY); }
DEV_PC int nn_spread(int v) { return (v & 1) | (v & 2) << 2 | (v & 4) << 4 | (v & 8) << 6; }

__global__ void __launch_bounds__(PC_WG) k_nn_box(NnPair a) {
    __shared__ float s[6][PC_WG / 64];
    NnCloud c = a.c[blockIdx.y];
    for (int k = blockIdx.x * PC_WG + threadIdx.x; k < NN_CELLS; k += NN_BOXES * PC_WG) c.count[k] = 0;
    float v[6] = {INFINITY, INFINITY, INFINITY, INFINITY, INFINITY, INFINITY};
    // every NN_BOXES'th point, or run of 8 in large clouds: each partial box is a sample
    // of the whole cloud (a prime number of them, so that the rows of a lattice, 16, 32
    // or 64 points long, do not give each sample a stretch of its own of the axis they
    // run along; points by themselves while there are few runs to a sample)
    int run = c.n > NN_RUNS ? 3 : 0, per = PC_WG >> run;
    for (long long r = blockIdx.x + (long long)(threadIdx.x >> run) * NN_BOXES; r << run < c.n; r += (long long)per * NN_BOXES) {
        long long i = (r << run) + (threadIdx.x & ((1 << run) - 1));
        if (i >= c.n) continue;
        float u[3] = {c.p[i * 3], c.p[i * 3 + 1], c.p[i * 3 + 2]};
        if (nn_special(u[0], u[1], u[2])) continue;
#pragma unroll
        for (int d = 0; d < 3; d++) {
            v[d] = fminf(v[d], u[d]);
            v[3 + d] = fminf(v[3 + d], -u[d]);
        }
    }
#pragma unroll
    for (int d = 0; d < 6; d++) {
        for (int o = 32; o > 0; o >>= 1) v[d] = fminf(v[d], __shfl_xor(v[d], o));
        if ((threadIdx.x & 63) == 0) s[d][threadIdx.x >> 6] = v[d];
    }
    __syncthreads();
    if (threadIdx.x < 6) {
        float m = s[threadIdx.x][0];
        for (int w = 1; w < PC_WG / 64; w++) m = fminf(m, s[threadIdx.x][w]);
        c.part[blockIdx.x * 6 + threadIdx.x] = m;
    }
}

// Each point's cell, and its rank in it.  The extent of an axis: of 16 samples (4
// partial boxes each) the innermost ends, so that points which some sample does not
// hold do not stretch it (with one outlier at 500 times the extent every other point
// fell into one cell: 30000 x 25001 points one way 192 us, every pair 160).  The
// others, by a few percent at the ends, go to the border cells; the blocks' boxes are
// the points' own.
__global__ void __launch_bounds__(PC_WG) k_nn_count(NnPair a) {
    NnCloud c = a.c[blockIdx.y];
    if ((int)blockIdx.x * PC_WG >= c.n) return;
    int lane = threadIdx.x & 63;
    float lo[3], scale[3];
#pragma unroll
    for (int d = 0; d < 3; d++) {
        float mn = lane < NN_BOXES ? c.part[lane * 6 + d] : INFINITY, mx = lane < NN_BOXES ? c.part[lane * 6 + 3 + d] : INFINITY;
        for (int o = 1; o < 4; o <<= 1) {
            mn = fminf(mn, __shfl_xor(mn, o));
            mx = fminf(mx, __shfl_xor(mx, o));
        }
        mn = mn < INFINITY ? mn : -INFINITY;   // (an empty sample)
        mx = mx < INFINITY ? mx : -INFINITY;
        for (int o = 4; o < 64; o <<= 1) {
            mn = fmaxf(mn, __shfl_xor(mn, o));
            mx = fmaxf(mx, __shfl_xor(mx, o));
        }
        lo[d] = mn;
        float w = -mx - mn;
        scale[d] = w > 0.f ? (1 << NN_BITS) / w : 0.f;
    }
    int i = blockIdx.x * PC_WG + threadIdx.x;
    if (i >= c.n) return;
    int cell = 0;
#pragma unroll
    for (int d = 0; d < 3; d++) {
        // (points outside the extent, at infinity or NaN end in a border cell)
        float u = (c.p[(size_t)i * 3 + d] - lo[d]) * scale[d];
        int k = (int)fminf(fmaxf(u, 0.f), (float)((1 << NN_BITS) - 1));
        cell |= nn_spread(k) << d;
    }
    unsigned rank = atomicAdd(&c.count[cell], 1);
    c.at[2 * (size_t)i] = cell;
    c.at[2 * (size_t)i + 1] = rank;
}

// prefix sums of the cells' counts (by every workgroup for itself) and the sort
__global__ void __launch_bounds__(1024) k_nn_sort(NnPair a) {
    __shared__ int start[NN_CELLS], wsum[16];
    NnCloud c = a.c[blockIdx.y];
    int total = c.blocks * NN_BLOCK;
    if ((int)blockIdx.x * 1024 >= total) return;
    constexpr int PER = NN_CELLS / 1024;
    int v[PER], sum = 0, t = threadIdx.x, lane = t & 63;
#pragma unroll
    for (int k = 0; k < PER; k++) {
        v[k] = sum;
        sum += c.count[t * PER + k];
    }
    int inc = sum;
    for (int o = 1; o < 64; o <<= 1) {
        int u = __shfl_up(inc, o);
        if (lane >= o) inc += u;
    }
    if (lane == 63) wsum[t >> 6] = inc;
    __syncthreads();
    int base = inc - sum;
    for (int w = 0; w < (t >> 6); w++) base += wsum[w];
#pragma unroll
    for (int k = 0; k < PER; k++) start[t * PER + k] = base + v[k];
    __syncthreads();
    int i = blockIdx.x * 1024 + t;
    if (i < c.n) {
        const float* p = c.p + (size_t)i * 3;
        c.sorted[start[c.at[2 * (size_t)i]] + c.at[2 * (size_t)i + 1]] = nn4{p[0], p[1], p[2], __int_as_float(i)};
    } else if (i < total) {
        c.sorted[i] = nn4{INFINITY, INFINITY, INFINITY, __int_as_float(0x7fffffff)};
    }
}

// the blocks' boxes, half a wave each; padding and special points do not count
__global__ void __launch_bounds__(PC_WG) k_nn_blocks(NnPair a) {
    NnCloud c = a.c[blockIdx.y];
    int i = blockIdx.x * PC_WG + threadIdx.x;
    if ((int)blockIdx.x * PC_WG >= c.blocks * NN_BLOCK) return;
    bool in = i < c.blocks * NN_BLOCK;
    nn4 p = c.sorted[in ? i : 0];
    bool real = in && __float_as_int(p.w) != 0x7fffffff && !nn_special(p.x, p.y, p.z);
    float v[6] = {real ? p.x : INFINITY, real ? p.y : INFINITY, real ? p.z : INFINITY,
                  real ? -p.x : INFINITY, real ? -p.y : INFINITY, real ? -p.z : INFINITY};
#pragma unroll
    for (int d = 0; d < 6; d++)
        for (int o = 16; o > 0; o >>= 1) v[d] = fminf(v[d], __shfl_xor(v[d], o));
    if (in && i % NN_BLOCK < 2)
        c.box[i / NN_BLOCK * 2 + i % NN_BLOCK] = i % NN_BLOCK ? nn4{-v[3], -v[4], -v[5], 0.f} : nn4{v[0], v[1], v[2], 0.f};
}

// One block of queries to a workgroup, its half-waves (lane h * 32 + q: query q)
// taking a block of targets each.  16 of them: queries far from the targets have
// long lists, whose groups the launch would wait for (both ways of 30000 x 25001
// points, 8, 16, 32: 73.7, 64.1, 78.6 us; 10000 x 10000: 41.9, 35.3, 40.1).
constexpr int NN_HALVES = 16;
DEV_PC unsigned long long nn_key(float d, int k) { return (unsigned long long)__float_as_uint(d) << 32 | (unsigned)k; }

// squared distance from a point to a box, scaled down by the margin
DEV_PC float nn_reach(float x, float y, float z, nn4 lo, nn4 hi) {
    float gx = fmaxf(0.f, fmaxf(lo.x - x, x - hi.x)), gy = fmaxf(0.f, fmaxf(lo.y - y, y - hi.y)), gz = fmaxf(0.f, fmaxf(lo.z - z, z - hi.z));
    return (gx * gx + gy * gy + gz * gz) * NN_MARGIN;
}
// the half-wave's queries against a block of targets, one per lane in t; `tile`
// is the half-wave's own.  (distance, index) pairs compare as 64-bit words; a
// NaN's bits are above infinity's.
DEV_PC void nn_scan(nn4 t, nn4* tile, float qx, float qy, float qz, unsigned long long* best) {
    unsigned long long old = *best, key = old;
    tile[threadIdx.x & 31] = t;
    __builtin_amdgcn_wave_barrier();
#pragma unroll 8
    for (int u = 0; u < NN_BLOCK; u++) {
        nn4 v = tile[u];
        float ex = qx - v.x, ey = qy - v.y, ez = qz - v.z;
        float d = fmaf(ez, ez, fmaf(ey, ey, ex * ex));
        unsigned long long k = nn_key(d, __float_as_int(v.w));
        key = k < key ? k : key;
    }
    __builtin_amdgcn_wave_barrier();
    if (key < old) atomicMin(best, key);
}

__global__ void __launch_bounds__(NN_HALVES * NN_BLOCK) k_nn_search(NnPair a, int first, int* __restrict__ idx0, float* __restrict__ d0,
                                                    int* __restrict__ idx1, float* __restrict__ d1) {
    __shared__ unsigned long long best[NN_BLOCK];
    __shared__ nn4 query[NN_BLOCK], tile[NN_HALVES][NN_BLOCK];
    __shared__ int list[2][NN_LIST], listed[2], started[NN_HALVES];
    int dir = first + blockIdx.y;
    NnCloud q = a.c[dir], t = a.c[dir ^ 1];
    if ((int)blockIdx.x >= q.blocks) return;
    int tid = threadIdx.x, half = tid >> 5, ql = tid & 31;
    nn4 me = q.sorted[(size_t)blockIdx.x * NN_BLOCK + ql];
    bool real = __float_as_int(me.w) != 0x7fffffff, live = real && !nn_special(me.x, me.y, me.z);
    if (!live) me.x = me.y = me.z = INFINITY;
    nn4 lo = q.box[2 * (size_t)blockIdx.x], hi = q.box[2 * (size_t)blockIdx.x + 1];
    if (half == 0) {
        query[ql] = me;
        // (a lane without a query, or with one at no finite distance from any target,
        // neither asks for anything nor takes anything)
        best[ql] = live ? nn_key(INFINITY, 0x7fffffff) : 0ull;
    }
    if (tid < 2) listed[tid] = 0;
    // half-wave h starts with the block, of h, h + NN_HALVES, ..., whose centre is nearest
    // to the queries': they come from one neighbourhood
    unsigned long long near = ~0ull;
    for (int b = ql * NN_HALVES + half; b < t.blocks; b += NN_HALVES * NN_BLOCK) {
        nn4 tl = t.box[2 * (size_t)b], th = t.box[2 * (size_t)b + 1];
        float cx = lo.x + hi.x - tl.x - th.x, cy = lo.y + hi.y - tl.y - th.y, cz = lo.z + hi.z - tl.z - th.z;
        float c = cx * cx + cy * cy + cz * cz;
        unsigned long long k = nn_key(c == c ? c : INFINITY, b);
        near = k < near ? k : near;
    }
    for (int o = 16; o > 0; o >>= 1) {
        unsigned long long k = __shfl_xor(near, o);
        near = k < near ? k : near;
    }
    int b0 = (int)(unsigned)near;   // (-1: none)
    if (ql == 0) started[half] = b0;
    __syncthreads();
    const nn4 none = {INFINITY, INFINITY, INFINITY, __int_as_float(0x7fffffff)};
    nn_scan(b0 >= 0 ? t.sorted[(size_t)b0 * NN_BLOCK + ql] : none, tile[half], me.x, me.y, me.z, &best[ql]);
    for (int c0 = 0; c0 < t.blocks; c0 += NN_LIST) {
        __syncthreads();
        // blocks that the queries' box may reach with the largest bound, ...
        float ub = __uint_as_float((unsigned)(best[ql] >> 32));
        for (int o = 16; o > 0; o >>= 1) ub = fmaxf(ub, __shfl_xor(ub, o));
        for (int b = c0 + tid; b < min(t.blocks, c0 + NN_LIST); b += NN_HALVES * NN_BLOCK) {
            nn4 tl = t.box[2 * (size_t)b], th = t.box[2 * (size_t)b + 1];
            float gx = fmaxf(0.f, fmaxf(tl.x - hi.x, lo.x - th.x)), gy = fmaxf(0.f, fmaxf(tl.y - hi.y, lo.y - th.y));
            float gz = fmaxf(0.f, fmaxf(tl.z - hi.z, lo.z - th.z));
            if (!((gx * gx + gy * gy + gz * gz) * NN_MARGIN > ub) && started[b % NN_HALVES] != b) list[0][atomicAdd(&listed[0], 1)] = b;
        }
        __syncthreads();
        // ... of these the ones that some query may reach with its own, ...
        int n0 = listed[0];
        for (int j = tid; j < n0; j += NN_HALVES * NN_BLOCK) {
            int b = list[0][j];
            nn4 tl = t.box[2 * (size_t)b], th = t.box[2 * (size_t)b + 1];
            bool reach = false;
#pragma unroll 8
            for (int k = 0; k < NN_BLOCK; k++) {
                nn4 p = query[k];
                float bd = __uint_as_float((unsigned)(best[k] >> 32));
                reach |= !(nn_reach(p.x, p.y, p.z, tl, th) > bd);
            }
            if (reach) list[1][atomicAdd(&listed[1], 1)] = b;
        }
        __syncthreads();
        // ... are scanned, unless the bounds have come down meanwhile
        int n = listed[1];
        nn4 v, bl, bh;
        auto fetch = [&](int j) {
            int b = j < n ? list[1][j] : 0;
            bl = t.box[2 * (size_t)b];
            bh = t.box[2 * (size_t)b + 1];
            v = j < n ? t.sorted[(size_t)b * NN_BLOCK + ql] : none;
        };
        fetch(half);
        for (int j = half & ~1; j < n; j += NN_HALVES) {
            nn4 tv = v, tl = bl, th = bh;
            fetch(j + (half & 1) + NN_HALVES);
            float bd = __uint_as_float((unsigned)(best[ql] >> 32));
            if (__any(!(nn_reach(me.x, me.y, me.z, tl, th) > bd))) nn_scan(tv, tile[half], me.x, me.y, me.z, &best[ql]);
        }
        __syncthreads();
        if (tid < 2) listed[tid] = 0;
    }
    __syncthreads();
    if (half != 0 || !real) return;
    unsigned long long k = best[ql];
    float bd = __uint_as_float((unsigned)(k >> 32));
    int at = __float_as_int(me.w);
    bool nothing = !live || !(bd < INFINITY);
    (dir ? idx1 : idx0)[at] = nothing ? -1 : (int)(unsigned)k;
    (dir ? d1 : d0)[at] = nothing ? INFINITY : bd;
}

// ------------------------------------------------- Chamfer loss and gradient
// From pc_nearest_pair's outputs: the loss (fp64 sums in a fixed order) in one launch
// or two, the gradient in two -- every point's own term stored, then the terms of
// the points that chose it added -- or three, where the elementwise operations of
// a framework took about 40 (30000 x 25001 points both ways, forward and gradients
// after the search: 130 -> 18 us of kernels).
struct ChDir { const float* p; const float* t; const int* idx; const float* d2; float* gp; float* gt; int n; };

// one workgroup: the loss; several: their sums to part[direction][workgroup], which
// k_ch_loss_sum adds
__global__ void __launch_bounds__(1024) k_ch_loss(const float* __restrict__ dx, int n, const float* __restrict__ dy, int m, int squared,
                                                  double* __restrict__ part, float* __restrict__ out) {
    __shared__ double s[2][16];
    double a[2] = {0.0, 0.0};
    for (int c = 0; c < 2; c++) {
        const float* d = c ? dy : dx;
        int k = d ? (c ? m : n) : 0;
        for (long long i0 = (long long)blockIdx.x * 8192 + threadIdx.x; i0 < k; i0 += (long long)gridDim.x * 8192) {
            float v[8];
#pragma unroll
            for (int u = 0; u < 8; u++) {
                long long i = i0 + u * 1024;
                v[u] = i < k ? d[i] : 0.f;
            }
#pragma unroll
            for (int u = 0; u < 8; u++) a[c] += squared ? v[u] : sqrtf(v[u]);
        }
        for (int o = 32; o > 0; o >>= 1) a[c] += __shfl_xor(a[c], o);
        if ((threadIdx.x & 63) == 0) s[c][threadIdx.x >> 6] = a[c];
    }
    __syncthreads();
    if (threadIdx.x != 0) return;
    a[0] = a[1] = 0.0;
    for (int w = 0; w < 16; w++) { a[0] += s[0][w]; a[1] += s[1][w]; }
    if (gridDim.x > 1) {
        part[blockIdx.x] = a[0];
        part[gridDim.x + blockIdx.x] = a[1];
        return;
    }
    float lx = (float)(a[0] / n);
    out[0] = dy ? lx + (float)(a[1] / m) : lx;
}
__global__ void __launch_bounds__(64) k_ch_loss_sum(const double* __restrict__ part, int groups, int n, int m, int both, float* __restrict__ out) {
    double a[2];
#pragma unroll
    for (int c = 0; c < 2; c++) {
        a[c] = (int)threadIdx.x < groups ? part[c * groups + threadIdx.x] : 0.0;
        for (int o = 32; o > 0; o >>= 1) a[c] += __shfl_xor(a[c], o);
    }
    if (threadIdx.x != 0) return;
    float lx = (float)(a[0] / n);
    out[0] = both ? lx + (float)(a[1] / m) : lx;
}
// Workgroups of the loss; up to 64, so that the second launch adds a value a lane.  One
// takes 4.7 us for 4000 distances, 12.0 for 65536, 147 for 1000000, several (with the
// second launch) 6.1 for 65536, 6.9 for 1000000.
int ch_loss_groups(int n, int m) {
    long long k = (long long)n + m;
    return k <= 49152 ? 1 : (int)std::min(64LL, k / 8192);
}

// component u of point i's own term; a point without a nearest target (no finite
// distance) gets NaN.  Its target's index, -1 for none.
DEV_PC int ch_term(const ChDir& c, int i, int u, int squared, const float* go, float& g) {
    int k = c.idx ? c.idx[i] : -1;
    g = 0.f;
    if (k >= 0) {
        float w = go[0] / (float)c.n;
        if (squared) w *= 2.f;
        else {
            float d = sqrtf(c.d2[i]);
            w = d > 0.f ? w * (1.f / fmaxf(d, 1e-30f)) : 0.f;
        }
        g = w * (c.p[(size_t)i * 3 + u] - c.t[(size_t)k * 3 + u]);
    } else if (c.idx) {
        g = NAN;
    }
    return k;
}
// lane t of a run of lanes from `first` on, a lane a component: its point (i) and component (u)
DEV_PC long long ch_lane(long long first, int t, int& u) {
    long long i0 = first / 3;   // (uniform)
    int r = (int)(first - 3 * i0) + t;
    u = r % 3;
    return i0 + r / 3;
}
// own = 1: the points' own terms; own = 0: the same, negated, to their targets.  A
// lane a component, so that a target's three meet in one line: 1000000 points to
// 40000 targets 171 us with a lane a point, 75 so.
__global__ void __launch_bounds__(PC_WG) k_ch_grad(ChDir d0, ChDir d1, int squared, const float* __restrict__ go, int own) {
    ChDir c = blockIdx.y ? d1 : d0;
    int u;
    long long i = ch_lane((long long)blockIdx.x * PC_WG, threadIdx.x, u);
    if (i >= c.n) return;
    float* dst = own ? c.gp : c.gt;
    if (!dst) return;
    float g;
    int k = ch_term(c, (int)i, u, squared, go, g);
    if (own) dst[i * 3 + u] = g;
    else if (k >= 0) atomicAdd(&dst[(size_t)k * 3 + u], -g);
}
// own = 0 for many points to a target: a workgroup adds its points' terms in LDS,
// 3 floats a target, and then those to memory, so that a target's address takes
// one atomic a workgroup instead of one a point.
extern __shared__ float ch_acc[];
__global__ void __launch_bounds__(1024) k_ch_share(ChDir c, int nt, int squared, const float* __restrict__ go) {
    for (int k = threadIdx.x; k < 3 * nt; k += 1024) ch_acc[k] = 0.f;
    __syncthreads();
    for (long long first = (long long)blockIdx.x * 1024; first < 3LL * c.n; first += (long long)gridDim.x * 1024) {
        int u;
        long long i = ch_lane(first, threadIdx.x, u);
        if (i >= c.n) break;
        float g;
        int k = ch_term(c, (int)i, u, squared, go, g);
        if (k >= 0) atomicAdd(&ch_acc[3 * k + u], -g);
    }
    __syncthreads();
    for (int k = threadIdx.x; k < 3 * nt; k += 1024)
        if (ch_acc[k] != 0.f) atomicAdd(&c.gt[k], ch_acc[k]);
}
// Whether k_ch_share takes a direction: targets that fit 60 KB of LDS, 32 points to
// each.  Both kernels of the gradient, every point's own atomics against the sums in
// LDS: 16000 points to 1000 targets 6.9, 7.5 us; 40000 to 3000 8.3, 8.8; 40000 to 1000
// 10.2, 8.1; 16000 to 300 11.2, 7.3; 40000 to 100 46, 7.7; 1000000 to 100 1050, 34.
constexpr int CH_SHARE_TARGETS = 5120;
bool ch_shares(int n, int nt) { return nt <= CH_SHARE_TARGETS && n / 32 >= nt; }
// (4000 points: 6.8 us with 7 workgroups, 9.4 with 3, 19.6 with 1)
int ch_share_groups(int n) { return std::max(1, std::min(256, n / 512)); }

// Scratch of pc_nearest_noalloc: the per-query (distance, index) words that
// pc_nearest takes from its workspace argument, as a file-scope device array
// (one copy per GPU, held until the process ends).  Host code reaches it only
// through the address hipGetSymbolAddress returns for the current device.
constexpr int PC_NOALLOC_MAX_QUERIES = 1 << 20;   // 8 MiB per GPU
static __device__ __align__(256) unsigned long long scratch[PC_NOALLOC_MAX_QUERIES];

int noalloc_scratch(unsigned long long** out) {
    int dev = -1;
    hipError_t e = hipGetDevice(&dev);
    if (e != hipSuccess) return pc_fail(std::string("pc_nearest_noalloc: hipGetDevice: ") + hipGetErrorString(e));
    if (dev < 0 || dev >= PC_MAX_DEVICES) return pc_fail("pc_nearest_noalloc: device index outside [0, 64)");
    std::lock_guard<std::mutex> lock(g_scratch_mu);
    if (!g_scratch_dev[dev]) {
        void* p = nullptr;
        e = hipGetSymbolAddress(&p, HIP_SYMBOL(scratch));
        if (e != hipSuccess || !p)
            return pc_fail(std::string("pc_nearest_noalloc: hipGetSymbolAddress(scratch): ") + hipGetErrorString(e));
        g_scratch_dev[dev] = static_cast<unsigned long long*>(p);
    }
    *out = g_scratch_dev[dev];
    return 0;
}

__global__ void __launch_bounds__(PC_WG) k_pc_unpack(const unsigned long long* __restrict__ best, int n, int* __restrict__ idx,
                                                    float* __restrict__ d2) {
    int i = blockIdx.x * PC_WG + threadIdx.x;
    if (i >= n) return;
    unsigned long long b = best[i];
    bool none = b == PC_EMPTY;
    idx[i] = none ? -1 : (int)(unsigned)(b & 0xffffffffull);
    d2[i] = none ? __int_as_float(0x7f800000) : __uint_as_float((unsigned)(b >> 32));
}

// ---------------------------------------------------------------- Sinkhorn
// The soft-min of the Sinkhorn divergence (geomloss SamplesLoss('sinkhorn'),
// the EMD loss of plb/engine/taichi_env.py:23-26) and the gradient of its
// transport plan, over all (row, column) pairs:
//   softmin_i = -eps log sum_j exp(h_j - C(x_i, y_j) / eps)
//   grad_i    = sum_j exp(h_j - C(x_i, y_j) / eps + r_i) dC/dx_i
// with C = |x - y| (p = 1) or |x - y|^2 / 2 (p = 2).  Base-2 arithmetic: the
// host passes h and r in log2 units (h * log2 e), the kernels scale the cost
// by log2(e) / eps and exponentiate with v_exp_f32.  A workgroup takes 256
// rows (one per lane) and one column range (a "split") staged through LDS;
// each lane keeps a running (max, scaled sum) per block of 4 columns, and the
// splits' partials are combined in split order by a second kernel, so the
// result does not depend on scheduling.
constexpr int SK_CHUNK = 2048;   // columns per LDS pass (32 KB)

DEV_PC float sk_cost(float dx, float dy, float dz, int p) {
    float d2 = fmaf(dz, dz, fmaf(dy, dy, dx * dx));
    return p == 1 ? sqrtf(d2) : 0.5f * d2;
}

__global__ void __launch_bounds__(PC_WG) k_sk_softmin(const float* __restrict__ x, int n, const float* __restrict__ y, int m,
                                                     const float* __restrict__ h2, float k2, int p, int per_split,
                                                     float2* __restrict__ part) {
    __shared__ float sx[SK_CHUNK], sy[SK_CHUNK], sz[SK_CHUNK], sh[SK_CHUNK];
    int i = blockIdx.x * PC_WG + threadIdx.x;
    int c0 = blockIdx.y * per_split, c1 = min(m, c0 + per_split);
    float xi = 0.f, yi = 0.f, zi = 0.f;
    if (i < n) { xi = x[(size_t)i * 3]; yi = x[(size_t)i * 3 + 1]; zi = x[(size_t)i * 3 + 2]; }
    float mx = -INFINITY, sm = 0.f;
    for (int b0 = c0; b0 < c1; b0 += SK_CHUNK) {
        int nc = min(SK_CHUNK, c1 - b0);
        __syncthreads();
        for (int k = threadIdx.x; k < nc; k += PC_WG) {
            const float* q = y + (size_t)(b0 + k) * 3;
            sx[k] = q[0]; sy[k] = q[1]; sz[k] = q[2]; sh[k] = h2[b0 + k];
        }
        __syncthreads();
        int k = 0;
        for (; k + 4 <= nc; k += 4) {
            float z[4];
#pragma unroll
            for (int u = 0; u < 4; u++) z[u] = sh[k + u] - k2 * sk_cost(xi - sx[k + u], yi - sy[k + u], zi - sz[k + u], p);
            float bm = fmaxf(fmaxf(z[0], z[1]), fmaxf(z[2], z[3]));
            float nm = fmaxf(mx, bm);
            float acc = 0.f;
#pragma unroll
            for (int u = 0; u < 4; u++) acc += __builtin_amdgcn_exp2f(z[u] - nm);
            sm = sm * __builtin_amdgcn_exp2f(mx - nm) + acc;
            mx = nm;
        }
        for (; k < nc; k++) {
            float z = sh[k] - k2 * sk_cost(xi - sx[k], yi - sy[k], zi - sz[k], p);
            float nm = fmaxf(mx, z);
            sm = sm * __builtin_amdgcn_exp2f(mx - nm) + __builtin_amdgcn_exp2f(z - nm);
            mx = nm;
        }
    }
    if (i < n) part[(size_t)blockIdx.y * n + i] = make_float2(mx, sm);
}

// combine the splits: softmin_i = -eps ln2 (M + log2 sum_s s_s 2^(m_s - M))
__global__ void __launch_bounds__(PC_WG) k_sk_softmin_combine(const float2* __restrict__ part, int n, int splits, float eps,
                                                             float* __restrict__ out) {
    int i = blockIdx.x * PC_WG + threadIdx.x;
    if (i >= n) return;
    float M = -INFINITY;
    for (int s = 0; s < splits; s++) M = fmaxf(M, part[(size_t)s * n + i].x);
    float S = 0.f;
    for (int s = 0; s < splits; s++) {
        float2 v = part[(size_t)s * n + i];
        S += v.y * __builtin_amdgcn_exp2f(v.x - M);
    }
    out[i] = -eps * 0.69314718055994531f * (M + __builtin_amdgcn_logf(S));
}

__global__ void __launch_bounds__(PC_WG) k_sk_plan_grad(const float* __restrict__ x, int n, const float* __restrict__ y, int m,
                                                       const float* __restrict__ h2, const float* __restrict__ r2, float k2, int p,
                                                       int per_split, float4* __restrict__ part) {
    __shared__ float sx[SK_CHUNK], sy[SK_CHUNK], sz[SK_CHUNK], sh[SK_CHUNK];
    int i = blockIdx.x * PC_WG + threadIdx.x;
    int c0 = blockIdx.y * per_split, c1 = min(m, c0 + per_split);
    float xi = 0.f, yi = 0.f, zi = 0.f, ri = 0.f;
    if (i < n) { xi = x[(size_t)i * 3]; yi = x[(size_t)i * 3 + 1]; zi = x[(size_t)i * 3 + 2]; ri = r2[i]; }
    float gx = 0.f, gy = 0.f, gz = 0.f;
    for (int b0 = c0; b0 < c1; b0 += SK_CHUNK) {
        int nc = min(SK_CHUNK, c1 - b0);
        __syncthreads();
        for (int k = threadIdx.x; k < nc; k += PC_WG) {
            const float* q = y + (size_t)(b0 + k) * 3;
            sx[k] = q[0]; sy[k] = q[1]; sz[k] = q[2]; sh[k] = h2[b0 + k];
        }
        __syncthreads();
        for (int k = 0; k < nc; k++) {
            float dx = xi - sx[k], dy = yi - sy[k], dz = zi - sz[k];
            float d2 = fmaf(dz, dz, fmaf(dy, dy, dx * dx));
            float c, w;
            if (p == 1) {
                float d = sqrtf(d2);
                c = d;
                w = d > 0.f ? 1.f / d : 0.f;   // dC/dx = (x - y) / |x - y|, 0 at coincident points
            } else {
                c = 0.5f * d2;
                w = 1.f;
            }
            float e = __builtin_amdgcn_exp2f(sh[k] + ri - k2 * c) * w;
            gx = fmaf(e, dx, gx); gy = fmaf(e, dy, gy); gz = fmaf(e, dz, gz);
        }
    }
    if (i < n) part[(size_t)blockIdx.y * n + i] = make_float4(gx, gy, gz, 0.f);
}

__global__ void __launch_bounds__(PC_WG) k_sk_grad_combine(const float4* __restrict__ part, int n, int splits, float* __restrict__ g) {
    int i = blockIdx.x * PC_WG + threadIdx.x;
    if (i >= n) return;
    float gx = 0.f, gy = 0.f, gz = 0.f;
    for (int s = 0; s < splits; s++) {
        float4 v = part[(size_t)s * n + i];
        gx += v.x; gy += v.y; gz += v.z;
    }
    g[(size_t)i * 3] = gx; g[(size_t)i * 3 + 1] = gy; g[(size_t)i * 3 + 2] = gz;
}

// One annealing step of the divergence: the four soft-mins in one launch.  The
// potentials are arrays pot = [a_x, b_x, a_y, b_y, pa_x, pb_x, pa_y, pb_y]
// (lengths n, n, m, m, n, n, m, m):
//   problem 0: a_y <- softmin over x of (log 1/n + b_x / eps)   rows y, cols x
//   problem 1: b_x <- softmin over y of (log 1/m + a_y / eps)   rows x, cols y
//   problem 2: a_x <- softmin over x of (log 1/n + a_x / eps)   rows x, cols x
//   problem 3: b_y <- softmin over y of (log 1/m + b_y / eps)   rows y, cols y
// mode 0 (first eps): the weights are 1/n, 1/m alone, the result replaces the
// potential; mode 1: symmetric update, (potential + result) / 2; mode 2 (last
// extrapolation): the potentials move to pa_x.. and the results replace them.
//
// Every problem has its columns packed as (x, y, z, log2 weight), SK_BATCH of
// them at a time read through the scalar cache: a lane holds one row, so a
// column's four numbers are the scalar operands of the wave's instructions, and
// neither LDS nor vector registers carry them.  A step reads one of two packed
// sets and its results write the other one's weights for the next eps; only the
// row itself reads or writes its potential.
//
// 64 rows and a share of the columns to a workgroup: its 4 waves take batches in
// turn, meet in LDS, and the last of a row group's workgroups (an arrival
// counter) joins the shares in order.  The shares (sk_splits_of) make up to
// 4096 workgroups, so that no compute unit is left with a whole row group more
// than the others, and small clouds fill the chip too.
// What bounds it: the VALU, 9.5 instructions and two transcendentals (four times
// the issue of an addition) a pair.  v_sqrt_f32 (one ulp) takes the place of
// sqrtf's 15 instructions; the weights lw + pot k2 use the costs' own scale k2,
// whose rounding then acts as one of eps, so that the results' errors against
// 64 bits are smaller than with sqrtf and 1 / eps (EMD gradients, 9001 x 8000:
// 2.3e-6 -> 1.8e-6).  The reference M of a row's sum moves up only when an exponent
// passes SK_LIFT.  The differences on the matrix cores (v_mfma_f32_32x32x2f32) were
// no faster: fp32 MFMA and the VALU do not overlap here.
// 9001 x 8000 points: 204.5 + 14.7 (256 columns a lane, a second launch to
// combine) -> 111.2 us a step; 500 x 500: 20.9 + 4.0 -> 6.9.
constexpr int SK_BATCH = 16;
constexpr int SK_WAVES = 4;
constexpr float SK_LIFT = 30.f;   // exponent that moves a row's reference
constexpr float LOG2E = 1.4426950408889634f;
typedef float f32x4 __attribute__((ext_vector_type(4)));

// where the packed columns of problem z start (in columns, of one set), padded
// to whole batches
struct SkSet { int np, mp; };
__host__ DEV_PC SkSet sk_set(int n, int m) {
    return SkSet{(n + SK_BATCH - 1) / SK_BATCH * SK_BATCH, (m + SK_BATCH - 1) / SK_BATCH * SK_BATCH};
}
// problem z: rows, columns, where its potential lies in pot, and which problem
// has its results as column weights
struct SkProb { const float* rows; int nr, nc; size_t cols, pot, next; };
DEV_PC SkProb sk_problem(int z, const float* x, int n, const float* y, int m) {
    SkSet t = sk_set(n, m);
    const size_t at[4] = {0, (size_t)t.np, (size_t)t.np + t.mp, 2 * (size_t)t.np + t.mp};   // columns x, y, x, y
    SkProb q;
    bool ry = z == 0 || z == 3, cy = z == 1 || z == 3;
    q.rows = ry ? y : x;
    q.nr = ry ? m : n;
    q.nc = cy ? m : n;
    q.cols = at[z];
    q.pot = z == 0 ? 2 * (size_t)n : (z == 1 ? (size_t)n : (z == 2 ? 0 : 2 * (size_t)n + m));
    q.next = z == 0 ? at[1] : (z == 1 ? at[0] : at[z]);
    return q;
}
// pack both sets (or one): weights from pot (null: 1/n, 1/m alone); clears the
// arrival counters
__global__ void __launch_bounds__(PC_WG) k_sk_pack(const float* __restrict__ x, int n, const float* __restrict__ y, int m,
                                                  const float* __restrict__ pot, float k2, f32x4* __restrict__ set0,
                                                  f32x4* __restrict__ set1, int* __restrict__ arrived, int groups) {
    int z = blockIdx.y, j = blockIdx.x * PC_WG + threadIdx.x;
    SkProb q = sk_problem(z, x, n, y, m);
    if (z == 0 && arrived)
        for (int k = j; k < groups; k += gridDim.x * PC_WG) arrived[k] = 0;
    int padded = (q.nc + SK_BATCH - 1) / SK_BATCH * SK_BATCH;
    if (j >= padded) return;
    // column weights: b_x, a_y, a_x, b_y
    const size_t src = z == 0 ? (size_t)n : (z == 1 ? 2 * (size_t)n : (z == 2 ? 0 : 2 * (size_t)n + m));
    f32x4 v = {0.f, 0.f, 0.f, -INFINITY};
    if (j < q.nc) {
        const float* c = (z == 1 || z == 3 ? y : x) + (size_t)j * 3;
        float lw = -logf((float)q.nc) * LOG2E;
        v = f32x4{c[0], c[1], c[2], pot ? fmaf(pot[src + j], k2, lw) : lw};
    }
    set0[q.cols + j] = v;
    if (set1) set1[q.cols + j] = v;
}

typedef const __attribute__((address_space(4))) float* SkScalar;
struct SkBatch { float v[4 * SK_BATCH]; };
DEV_PC void sk_fetch(const f32x4* cols, int j, SkBatch& b) {
    SkScalar p = (SkScalar)(uintptr_t)(cols + j);
#pragma unroll
    for (int u = 0; u < 4 * SK_BATCH; u++) b.v[u] = p[u];
}

// running reference and sum over the batches t0, t0 + step, ... below t1
template <int P>
DEV_PC void sk_scan(const f32x4* cols, int t0, int t1, int step, float xi, float yi, float zi, float k2, float& mref, float& sum) {
    float k = P == 1 ? -k2 : -0.5f * k2;
    asm("" : "+v"(k));   // in a vector register: an instruction has one scalar operand, the column's
    mref = -3.0e38f;
    sum = 0.f;
    for (int t = t0; t < t1; t += step) {
        SkBatch b;
        sk_fetch(cols, t * SK_BATCH, b);
        float z[SK_BATCH];
#pragma unroll
        for (int u = 0; u < SK_BATCH; u++) {
            float dx = xi - b.v[4 * u], dy = yi - b.v[4 * u + 1], dz = zi - b.v[4 * u + 2];
            float d2 = fmaf(dz, dz, fmaf(dy, dy, dx * dx));
            z[u] = fmaf(k, P == 1 ? __builtin_amdgcn_sqrtf(d2) : d2, b.v[4 * u + 3]);
        }
        float m = fmaxf(z[0], z[1]);
#pragma unroll
        for (int u = 2; u < SK_BATCH; u += 2) m = fmaxf(fmaxf(z[u], z[u + 1]), m);
        if (__any(m > mref + SK_LIFT)) {
            m = fmaxf(m, mref);
            asm volatile("" : "+v"(m));   // keeps the branch
            sum *= __builtin_amdgcn_exp2f(mref - m);
            mref = m;
        }
        float acc[2];
#pragma unroll
        for (int u = 0; u < SK_BATCH; u++) {
            float e = __builtin_amdgcn_exp2f(z[u] - mref);
            acc[u & 1] = u < 2 ? e : acc[u & 1] + e;
        }
        sum += acc[0] + acc[1];
    }
}
// (reference, sum) of two partial sums
DEV_PC void sk_join(float& m, float& s, float m2, float s2) {
    float nm = fmaxf(m, m2);
    s = s * __builtin_amdgcn_exp2f(m - nm) + s2 * __builtin_amdgcn_exp2f(m2 - nm);
    m = nm;
}

// Partials that pass between workgroups are stored and loaded past the caches
// that workgroups do not share (agent scope), by one wave of each; sk_last is
// called by that wave after its stores: whether it is the last of `count` to
// arrive, after which it may load the others'.  The wait lets the stores reach
// memory before the arrival counts (fences of agent scope would also write back
// and drop the whole L2: 100 us a step at 2048 workgroups).
template <typename T>
DEV_PC void sk_put(T* p, T v) { __hip_atomic_store(p, v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT); }
template <typename T>
DEV_PC T sk_get(T* p) { return __hip_atomic_load(p, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT); }
DEV_PC bool sk_last(int* arrived, int count) {
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
    int old = 0;
    if ((threadIdx.x & 63) == 0) old = __hip_atomic_fetch_add(arrived, 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    bool last = __builtin_amdgcn_readfirstlane(old) == count - 1;
    if (last) sk_put(arrived, 0);
    asm volatile("" ::: "memory");
    return last;
}

template <int P>
__global__ void __launch_bounds__(64 * SK_WAVES) k_sk_step(const float* __restrict__ x, int n, const float* __restrict__ y, int m,
                                                          float* __restrict__ pot, const f32x4* __restrict__ in, f32x4* __restrict__ out,
                                                          float k2, float k2_next, int mode, int splits, float* __restrict__ part,
                                                          int* __restrict__ arrived) {
    __shared__ float2 sp[SK_WAVES][64];
    SkProb q = sk_problem(blockIdx.z, x, n, y, m);
    if ((int)blockIdx.x * 64 >= q.nr) return;
    int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    int i = blockIdx.x * 64 + lane;
    const float* r3 = q.rows + (size_t)min(i, q.nr - 1) * 3;
    float xi = r3[0], yi = r3[1], zi = r3[2], M, S;
    int batches = (q.nc + SK_BATCH - 1) / SK_BATCH;
    sk_scan<P>(in + q.cols, blockIdx.y * SK_WAVES + wave, batches, splits * SK_WAVES, xi, yi, zi, k2, M, S);
    sp[wave][lane] = make_float2(M, S);
    __syncthreads();
    if (wave != 0) return;
#pragma unroll
    for (int w = 1; w < SK_WAVES; w++) sk_join(M, S, sp[w][lane].x, sp[w][lane].y);
    if (splits > 1) {
        // partials of this row group: [split][M, S][64]
        size_t group = (size_t)blockIdx.z * gridDim.x + blockIdx.x;
        float* pp = part + group * splits * 128 + lane;
        sk_put(pp + (size_t)blockIdx.y * 128, M);
        sk_put(pp + (size_t)blockIdx.y * 128 + 64, S);
        if (!sk_last(arrived + group, splits)) return;
        M = -3.0e38f;
        S = 0.f;
        for (int s = 0; s < splits; s++) sk_join(M, S, sk_get(pp + (size_t)s * 128), sk_get(pp + (size_t)s * 128 + 64));
    }
    if (i >= q.nr) return;
    float r = -(M + __builtin_amdgcn_logf(S)) / k2;
    float* pi = pot + q.pot + i;
    if (mode == 1) r = 0.5f * (*pi + r);
    if (mode == 2) pi[2 * ((size_t)n + m)] = *pi;
    *pi = r;
    if (out) out[q.next + i] = f32x4{xi, yi, zi, fmaf(r, k2_next, -logf((float)q.nr) * LOG2E)};
}

// Gradient of the divergence in one cloud's points (blockIdx.z: 0 x, 1 y), the
// transport plans' pulls towards the other cloud minus those within its own,
// scaled by *go / rows (1 / rows without go):
//   g_i = scale * (sum_j exp(h_j + r_i - C(a_i, b_j) / eps) dC/da_i - sum_k exp(...) dC(a_i, a_k)/da_i)
// with the column weights of the potentials before the last extrapolation and
// the rows' results of it.  Rows, columns and shares as in k_sk_step, both column
// sets in the same workgroup (four pairs of launches and their elementwise
// preparations before).  The distance takes the reciprocal root's estimate with one
// Newton step on the product and one on the reciprocal (half an ulp, 6
// instructions; sqrtf and the division took about 25); squared distances beyond
// fp32 turn that into NaN, and the wave scans again with sqrtf.
template <int P, bool FAR>
DEV_PC void sk_pull(const f32x4* cols, int t0, int t1, int step, float xi, float yi, float zi, float ri, float k2, float (&a)[3]) {
    float k = P == 1 ? -k2 : -0.5f * k2;
    asm("" : "+v"(k));
    a[0] = a[1] = a[2] = 0.f;
    for (int t = t0; t < t1; t += step) {
        SkBatch b;
        sk_fetch(cols, t * SK_BATCH, b);
        float g[3] = {0.f, 0.f, 0.f};
#pragma unroll
        for (int u = 0; u < SK_BATCH; u++) {
            float dx = xi - b.v[4 * u], dy = yi - b.v[4 * u + 1], dz = zi - b.v[4 * u + 2];
            float v = fmaf(dz, dz, fmaf(dy, dy, dx * dx)), w = 1.f;
            if (P == 1 && FAR) {
                v = sqrtf(v);
                w = v > 0.f ? 1.f / v : 0.f;
            } else if (P == 1) {
                // (coincident points: differences, and so pulls, of 0)
                v += 1e-37f;
                float rs = __builtin_amdgcn_rsqf(v), hr = 0.5f * rs, s = v * rs;
                v = fmaf(hr, fmaf(-s, s, v), s);
                w = fmaf(hr, fmaf(-v, rs, 1.f), rs);
            }
            float e = __builtin_amdgcn_exp2f(fmaf(k, v, b.v[4 * u + 3] + ri)) * w;
            g[0] = fmaf(e, dx, g[0]); g[1] = fmaf(e, dy, g[1]); g[2] = fmaf(e, dz, g[2]);
        }
#pragma unroll
        for (int u = 0; u < 3; u++) a[u] += g[u];
    }
}

template <int P>
__global__ void __launch_bounds__(64 * SK_WAVES) k_sk_grad(const float* __restrict__ x, int n, const float* __restrict__ y, int m,
                                                          const float* __restrict__ pot, const f32x4* __restrict__ set, float k2,
                                                          int splits, float* __restrict__ part, int* __restrict__ arrived,
                                                          const float* __restrict__ go, float* __restrict__ gx, float* __restrict__ gy) {
    __shared__ float sp[SK_WAVES][3][64];
    bool ry = blockIdx.z == 1;
    float* dst = ry ? gy : gx;
    int nr = ry ? m : n;
    if (!dst || (int)blockIdx.x * 64 >= nr) return;
    int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    int i = blockIdx.x * 64 + lane, row = min(i, nr - 1);
    const float* r3 = (ry ? y : x) + (size_t)row * 3;
    float xi = r3[0], yi = r3[1], zi = r3[2];
    float gs[3] = {0.f, 0.f, 0.f};
    for (int own = 0; own < 2; own++) {
        // rows x: problems 1, 2; rows y: problems 0, 3
        SkProb q = sk_problem(ry ? (own ? 3 : 0) : (own ? 2 : 1), x, n, y, m);
        float ri = pot[q.pot + row] * k2;
        int batches = (q.nc + SK_BATCH - 1) / SK_BATCH, t0 = blockIdx.y * SK_WAVES + wave;
        float a[3];
        sk_pull<P, false>(set + q.cols, t0, batches, splits * SK_WAVES, xi, yi, zi, ri, k2, a);
        if (P == 1 && __any(a[0] != a[0] || a[1] != a[1] || a[2] != a[2]))
            sk_pull<P, true>(set + q.cols, t0, batches, splits * SK_WAVES, xi, yi, zi, ri, k2, a);
#pragma unroll
        for (int d = 0; d < 3; d++) gs[d] = own ? gs[d] - a[d] : a[d];
    }
#pragma unroll
    for (int d = 0; d < 3; d++) sp[wave][d][lane] = gs[d];
    __syncthreads();
    if (wave != 0) return;
#pragma unroll
    for (int d = 0; d < 3; d++)
#pragma unroll
        for (int w = 1; w < SK_WAVES; w++) gs[d] += sp[w][d][lane];
    if (splits > 1) {
        size_t group = (size_t)blockIdx.z * gridDim.x + blockIdx.x;
        float* pp = part + group * splits * 192 + lane;
#pragma unroll
        for (int d = 0; d < 3; d++) sk_put(pp + ((size_t)blockIdx.y * 3 + d) * 64, gs[d]);
        if (!sk_last(arrived + group, splits)) return;
        gs[0] = gs[1] = gs[2] = 0.f;
        for (int s = 0; s < splits; s++)
#pragma unroll
            for (int d = 0; d < 3; d++) gs[d] += sk_get(pp + ((size_t)s * 3 + d) * 64);
    }
    if (i >= nr) return;
    float scale = (go ? go[0] : 1.f) / (float)nr;
#pragma unroll
    for (int d = 0; d < 3; d++) dst[(size_t)i * 3 + d] = gs[d] * scale;
}

// the divergence: mean(b_x - a_x) + mean(a_y - b_y), summed in fp64 by one
// workgroup in a fixed order
__global__ void __launch_bounds__(1024) k_sk_loss(const float* __restrict__ pot, int n, int m, float* __restrict__ out) {
    __shared__ double sx[16], sy[16];
    double ax = 0.0, ay = 0.0;
    for (int i = threadIdx.x; i < n; i += 1024) ax += (double)pot[n + i] - (double)pot[i];
    for (int i = threadIdx.x; i < m; i += 1024) ay += (double)pot[2 * n + i] - (double)pot[2 * n + m + i];
    for (int o = 32; o > 0; o >>= 1) { ax += __shfl_xor(ax, o); ay += __shfl_xor(ay, o); }
    if ((threadIdx.x & 63) == 0) { sx[threadIdx.x >> 6] = ax; sy[threadIdx.x >> 6] = ay; }
    __syncthreads();
    if (threadIdx.x != 0) return;
    ax = ay = 0.0;
    for (int w = 0; w < 16; w++) { ax += sx[w]; ay += sy[w]; }
    out[0] = (float)(ax / n + ay / m);
}
// extents of the bounding box of both clouds, by one workgroup; a NaN
// coordinate makes its extent NaN
DEV_PC float sk_min_nan(float a, float b) { return (b < a || b != b) ? b : a; }
__global__ void __launch_bounds__(1024) k_sk_extent(const float* __restrict__ x, int n, const float* __restrict__ y, int m,
                                                    float* __restrict__ out) {
    __shared__ float s[6][16];
    float v[6] = {INFINITY, INFINITY, INFINITY, INFINITY, INFINITY, INFINITY};   // min, -max
    for (int c = 0; c < 2; c++) {
        const float* p = c ? y : x;
        int k = c ? m : n;
#pragma unroll 4
        for (int i = threadIdx.x; i < k; i += 1024)
#pragma unroll
            for (int d = 0; d < 3; d++) {
                float u = p[(size_t)i * 3 + d];
                v[d] = sk_min_nan(v[d], u);
                v[3 + d] = sk_min_nan(v[3 + d], -u);
            }
    }
#pragma unroll
    for (int d = 0; d < 6; d++) {
        for (int o = 32; o > 0; o >>= 1) v[d] = sk_min_nan(v[d], __shfl_xor(v[d], o));
        if ((threadIdx.x & 63) == 0) s[d][threadIdx.x >> 6] = v[d];
    }
    __syncthreads();
    if (threadIdx.x >= 3) return;
    float lo = s[threadIdx.x][0], hi = s[3 + threadIdx.x][0];
    for (int w = 1; w < 16; w++) { lo = sk_min_nan(lo, s[threadIdx.x][w]); hi = sk_min_nan(hi, s[3 + threadIdx.x][w]); }
    out[threadIdx.x] = -hi - lo;
}

// column shares of a launch of `groups` row groups over `cols` columns: about
// 4096 workgroups, at least 4 batches a wave (us a step: 9001 x 8000 points 153.7
// with one share, 125.1, 109.8, 103.8 with 1024, 2048, 4096 workgroups; 1500 x
// 2000 points, 4096 asked for: 16.6 at 2 batches a wave, 13.4 at 4, 14.4 at 8)
int sk_splits_of(long long groups, int cols) {
    long long s = (4096 + groups - 1) / groups;
    return (int)std::max(1LL, std::min(s, (long long)((cols + SK_BATCH - 1) / SK_BATCH) / (4 * SK_WAVES)));
}
long long sk_groups(int n) { return (n + 63LL) / 64; }
// the workspace: two packed sets, the shares' partials (3 floats a row, for the
// gradient), the arrival counters
struct SkWork { f32x4* set[2]; float* part; int* arrived; long long groups, bytes; int splits_step, splits_grad; };
SkWork sk_work(int n, int m, void* work) {
    SkWork w;
    SkSet t = sk_set(n, m);
    long long cols = 2LL * t.np + 2LL * t.mp, gmax = std::max(sk_groups(n), sk_groups(m));
    w.splits_step = sk_splits_of(2 * (sk_groups(n) + sk_groups(m)), std::max(n, m));
    w.splits_grad = sk_splits_of(sk_groups(n) + sk_groups(m), std::max(n, m));
    w.groups = 4 * gmax;
    long long part = std::max(w.groups * w.splits_step * 128, 2 * gmax * w.splits_grad * 192);
    char* p = static_cast<char*>(work);
    w.set[0] = reinterpret_cast<f32x4*>(p);
    w.set[1] = w.set[0] + cols;
    w.part = reinterpret_cast<float*>(w.set[1] + cols);
    w.arrived = reinterpret_cast<int*>(w.part + part);
    w.bytes = 32 * cols + 4 * part + 4 * w.groups;
    return w;
}
bool sk_too_large(int n, int m) { return n > (1 << 28) || m > (1 << 28); }
void sk_pack(const float* x, int n, const float* y, int m, const float* pot, float k2, const SkWork& w, bool both, hipStream_t st) {
    hipLaunchKernelGGL(k_sk_pack, dim3((std::max(n, m) + SK_BATCH + PC_WG - 1) / PC_WG, 4), dim3(PC_WG), 0, st, x, n, y, m, pot, k2, w.set[0],
                       both ? w.set[1] : nullptr, w.arrived, (int)w.groups);
}
void sk_step(const float* x, int n, const float* y, int m, float* pot, const SkWork& w, int from, float eps, float eps_next, int p,
             int mode, bool more, hipStream_t st) {
    dim3 grid((unsigned)std::max(sk_groups(n), sk_groups(m)), w.splits_step, 4);
    auto kern = p == 1 ? k_sk_step<1> : k_sk_step<2>;
    hipLaunchKernelGGL(kern, grid, dim3(64 * SK_WAVES), 0, st, x, n, y, m, pot, (const f32x4*)w.set[from],
                       more ? w.set[from ^ 1] : (f32x4*)nullptr, LOG2E / eps, LOG2E / eps_next, mode, w.splits_step,
                       w.part, w.arrived);
}

// column splits: enough workgroups to fill the GPU (about 2048), at least
// 256 columns each
int sk_splits(int n, int m) {
    int gx = (n + PC_WG - 1) / PC_WG;
    int s = (2048 + gx - 1) / gx;
    s = std::min(s, (m + 255) / 256);
    return std::max(1, std::min(s, 65535));
}

// Which search takes a call: the times of both, us, as measured over 1 to 1000000
// points on either side.  Every pair: a workgroup passes over up to 2048 targets,
// 6.0e6 pairs a us once the chip is full.  Sorted: five launches, a term for each
// cloud's sort (targets more than queries: few queries leave few workgroups to
// go over many blocks' boxes) and one for the blocks' boxes, a pair of blocks each.
// One way, queries x targets, every pair against sorted: 300 x 300 15.4, 16.7;
// 300 x 1000 39.9, 20.5; 40000 x 600 27.9, 31.3; 40000 x 1000 42.9, 34.4; 1000 x
// 40000 83, 69; 300 x 100000 83, 118; 10000 x 100000 198, 84; 100 x 1000000 85, 792;
// 1000000 x 1000 187, 419; 1000000 x 4000 650, 521; 200000 x 150000 4566, 326.  Both
// ways: 300 x 100 25, 16.3; 200000 x 600 127, 181; 200000 x 4000 350, 199; 100 x
// 1000000 115, 808.
double nn_every_us(double nq, double nt) { return std::max(5.0 + 0.0375 * std::min(nt, (double)PC_CHUNK), nq * nt / 6.0e6); }
// (also without targets, or with more than the sorted search takes)
bool nn_brute(int n, int m, bool do_x, bool do_y) {
    if (n == 0 || m == 0 || n > 65535 * PC_CHUNK || m > 65535 * PC_CHUNK) return true;
    if (do_x && do_y) return nn_every_us(n, m) + nn_every_us(m, n) <= 16.5 + 0.8e-3 * ((double)n + m) + (double)n * m / 1.0e8;
    double nq = do_x ? n : m, nt = do_x ? m : n;
    return nn_every_us(nq, nt) <= 16.5 + 0.4e-3 * nq + 0.7e-3 * nt + nq * nt / 2.0e8;
}

}  // namespace

extern "C" {

long long pc_sinkhorn_work_bytes(int n, int m) {
    if (n < 0 || m < 0) return -1;
    return (long long)sk_splits(n, m) * std::max(n, 1) * (long long)sizeof(float4);
}

long long pc_sinkhorn_step_work_bytes(int n, int m) {
    if (n <= 0 || m <= 0 || sk_too_large(n, m)) return -1;
    return sk_work(n, m, nullptr).bytes;
}

int pc_sinkhorn_step(const float* x, int n, const float* y, int m, float* pot, float eps, int p, int mode, void* work, void* stream) {
    if (n <= 0 || m <= 0) return pc_fail("pc_sinkhorn_step: both clouds must be non-empty");
    if (sk_too_large(n, m)) return pc_fail("pc_sinkhorn_step: at most 2^28 points a cloud");
    if (!(eps > 0.f)) return pc_fail("pc_sinkhorn_step: eps must be positive");
    if (p != 1 && p != 2) return pc_fail("pc_sinkhorn_step: p must be 1 or 2");
    if (mode < 0 || mode > 2) return pc_fail("pc_sinkhorn_step: mode must be 0, 1 or 2");
    if (!x || !y || !pot || !work) return pc_fail("pc_sinkhorn_step: null argument");
    hipStream_t st = reinterpret_cast<hipStream_t>(stream);
    SkWork w = sk_work(n, m, work);
    sk_pack(x, n, y, m, mode == 0 ? nullptr : pot, LOG2E / eps, w, false, st);
    sk_step(x, n, y, m, pot, w, 0, eps, eps, p, mode, false, st);
    hipError_t e = hipGetLastError();
    if (e != hipSuccess) return pc_fail(std::string("pc_sinkhorn_step: ") + hipGetErrorString(e));
    return 0;
}

int pc_sinkhorn_solve(const float* x, int n, const float* y, int m, const float* eps, int n_eps, int p, float* pot, float* loss,
                      void* work, void* stream) {
    if (n <= 0 || m <= 0) return pc_fail("pc_sinkhorn_solve: both clouds must be non-empty");
    if (sk_too_large(n, m)) return pc_fail("pc_sinkhorn_solve: at most 2^28 points a cloud");
    if (n_eps <= 0 || !eps) return pc_fail("pc_sinkhorn_solve: no eps");
    for (int k = 0; k < n_eps; k++)
        if (!(eps[k] > 0.f)) return pc_fail("pc_sinkhorn_solve: eps must be positive");
    if (p != 1 && p != 2) return pc_fail("pc_sinkhorn_solve: p must be 1 or 2");
    if (!x || !y || !pot || !work) return pc_fail("pc_sinkhorn_solve: null argument");
    hipStream_t st = reinterpret_cast<hipStream_t>(stream);
    SkWork w = sk_work(n, m, work);
    // both sets get the points and the padding; each step writes the weights of
    // the set that the next one reads
    sk_pack(x, n, y, m, nullptr, 0.f, w, true, st);
    sk_step(x, n, y, m, pot, w, 0, eps[0], eps[0], p, 0, true, st);
    for (int k = 0; k < n_eps; k++) sk_step(x, n, y, m, pot, w, (k + 1) & 1, eps[k], eps[std::min(k + 1, n_eps - 1)], p, 1, true, st);
    sk_step(x, n, y, m, pot, w, (n_eps + 1) & 1, eps[n_eps - 1], eps[n_eps - 1], p, 2, false, st);
    if (loss) hipLaunchKernelGGL(k_sk_loss, dim3(1), dim3(1024), 0, st, (const float*)pot, n, m, loss);
    hipError_t e = hipGetLastError();
    if (e != hipSuccess) return pc_fail(std::string("pc_sinkhorn_solve: ") + hipGetErrorString(e));
    return 0;
}

int pc_sinkhorn_grad(const float* x, int n, const float* y, int m, const float* pot, float eps, int p, const float* go, float* gx,
                     float* gy, void* work, void* stream) {
    if (n <= 0 || m <= 0) return pc_fail("pc_sinkhorn_grad: both clouds must be non-empty");
    if (sk_too_large(n, m)) return pc_fail("pc_sinkhorn_grad: at most 2^28 points a cloud");
    if (!(eps > 0.f)) return pc_fail("pc_sinkhorn_grad: eps must be positive");
    if (p != 1 && p != 2) return pc_fail("pc_sinkhorn_grad: p must be 1 or 2");
    if (!x || !y || !pot || !work) return pc_fail("pc_sinkhorn_grad: null argument");
    if (!gx && !gy) return 0;
    hipStream_t st = reinterpret_cast<hipStream_t>(stream);
    SkWork w = sk_work(n, m, work);
    float k2 = LOG2E / eps;
    sk_pack(x, n, y, m, pot + 2 * ((size_t)n + m), k2, w, false, st);
    dim3 grid((unsigned)std::max(gx ? sk_groups(n) : 0, gy ? sk_groups(m) : 0), w.splits_grad, 2);
    auto kern = p == 1 ? k_sk_grad<1> : k_sk_grad<2>;
    hipLaunchKernelGGL(kern, grid, dim3(64 * SK_WAVES), 0, st, x, n, y, m, pot, (const f32x4*)w.set[0], k2, w.splits_grad, w.part,
                       w.arrived, go, gx, gy);
    hipError_t e = hipGetLastError();
    if (e != hipSuccess) return pc_fail(std::string("pc_sinkhorn_grad: ") + hipGetErrorString(e));
    return 0;
}

int pc_extent(const float* x, int n, const float* y, int m, float* out, void* stream) {
    if (n < 0 || m < 0 || (n == 0 && m == 0)) return pc_fail("pc_extent: no points");
    if ((n && !x) || (m && !y) || !out) return pc_fail("pc_extent: null argument");
    hipLaunchKernelGGL(k_sk_extent, dim3(1), dim3(1024), 0, reinterpret_cast<hipStream_t>(stream), x, n, y, m, out);
    hipError_t e = hipGetLastError();
    if (e != hipSuccess) return pc_fail(std::string("pc_extent: ") + hipGetErrorString(e));
    return 0;
}

int pc_softmin(const float* x, int n, const float* y, int m, const float* h2, float eps, int p, void* work, float* out, void* stream) {
    if (n < 0 || m <= 0) return pc_fail("pc_softmin: need n >= 0 rows and m > 0 columns");
    if (!(eps > 0.f)) return pc_fail("pc_softmin: eps must be positive");
    if (p != 1 && p != 2) return pc_fail("pc_softmin: p must be 1 or 2");
    if (n == 0) return 0;
    if (!x || !y || !h2 || !work || !out) return pc_fail("pc_softmin: null argument");
    hipStream_t st = reinterpret_cast<hipStream_t>(stream);
    int splits = sk_splits(n, m);
    int per = (m + splits - 1) / splits;
    int gx = (n + PC_WG - 1) / PC_WG;
    float k2 = 1.4426950408889634f / eps;
    hipLaunchKernelGGL(k_sk_softmin, dim3(gx, splits), dim3(PC_WG), 0, st, x, n, y, m, h2, k2, p, per, (float2*)work);
    hipLaunchKernelGGL(k_sk_softmin_combine, dim3(gx), dim3(PC_WG), 0, st, (const float2*)work, n, splits, eps, out);
    hipError_t e = hipGetLastError();
    if (e != hipSuccess) return pc_fail(std::string("pc_softmin: ") + hipGetErrorString(e));
    return 0;
}

int pc_plan_grad(const float* x, int n, const float* y, int m, const float* h2, const float* r2, float eps, int p, void* work,
                 float* g, void* stream) {
    if (n < 0 || m <= 0) return pc_fail("pc_plan_grad: need n >= 0 rows and m > 0 columns");
    if (!(eps > 0.f)) return pc_fail("pc_plan_grad: eps must be positive");
    if (p != 1 && p != 2) return pc_fail("pc_plan_grad: p must be 1 or 2");
    if (n == 0) return 0;
    if (!x || !y || !h2 || !r2 || !work || !g) return pc_fail("pc_plan_grad: null argument");
    hipStream_t st = reinterpret_cast<hipStream_t>(stream);
    int splits = sk_splits(n, m);
    int per = (m + splits - 1) / splits;
    int gx = (n + PC_WG - 1) / PC_WG;
    float k2 = 1.4426950408889634f / eps;
    hipLaunchKernelGGL(k_sk_plan_grad, dim3(gx, splits), dim3(PC_WG), 0, st, x, n, y, m, h2, r2, k2, p, per, (float4*)work);
    hipLaunchKernelGGL(k_sk_grad_combine, dim3(gx), dim3(PC_WG), 0, st, (const float4*)work, n, splits, g);
    hipError_t e = hipGetLastError();
    if (e != hipSuccess) return pc_fail(std::string("pc_plan_grad: ") + hipGetErrorString(e));
    return 0;
}


const char* pc_last_error(void) { return g_pc_err.c_str(); }

int pc_nearest(const float* q, int nq, const float* t, int nt, unsigned long long* work, int* idx, float* d2, void* stream) {
    if (nq < 0 || nt < 0) return pc_fail("pc_nearest: negative point count");
    if (nq == 0) return 0;
    if (!q || !work || !idx || !d2 || (nt > 0 && !t)) return pc_fail("pc_nearest: null argument");
    int gc = (nt + PC_CHUNK - 1) / PC_CHUNK;
    if (gc > 65535) return pc_fail("pc_nearest: too many targets (at most 65535 x 2048)");
    hipStream_t st = reinterpret_cast<hipStream_t>(stream);
    int gq = (nq + PC_WG - 1) / PC_WG;
    hipLaunchKernelGGL(k_pc_clear, dim3(gq), dim3(PC_WG), 0, st, work, nq);
    if (gc > 0) hipLaunchKernelGGL(k_pc_nearest, dim3(gq, gc), dim3(PC_WG), 0, st, q, nq, t, nt, work);
    hipLaunchKernelGGL(k_pc_unpack, dim3(gq), dim3(PC_WG), 0, st, (const unsigned long long*)work, nq, idx, d2);
    hipError_t e = hipGetLastError();
    if (e != hipSuccess) return pc_fail(std::string("pc_nearest: ") + hipGetErrorString(e));
    return 0;
}

long long pc_nearest_pair_work_bytes(int n, int m) {
    if (n < 0 || m < 0) return -1;
    long long b = 0;
    for (long long k : {n, m}) {
        long long blocks = (k + NN_BLOCK - 1) / NN_BLOCK;
        b += blocks * NN_BLOCK * 16 + blocks * 32 + k * 8 + 8 + NN_CELLS * 4 + NN_BOXES * 24;
    }
    return b;
}

int pc_nearest_pair(const float* x, int n, const float* y, int m, void* work, int* idx_x, float* d2_x, int* idx_y, float* d2_y,
                    void* stream) {
    if (n < 0 || m < 0) return pc_fail("pc_nearest_pair: negative point count");
    if (!idx_x != !d2_x || !idx_y != !d2_y) return pc_fail("pc_nearest_pair: indices and distances of a direction go together");
    if (!work || (n > 0 && !x) || (m > 0 && !y)) return pc_fail("pc_nearest_pair: null argument");
    bool do_x = idx_x && n > 0, do_y = idx_y && m > 0;
    if (!do_x && !do_y) return 0;
    if (nn_brute(n, m, do_x, do_y)) {
        unsigned long long* w = static_cast<unsigned long long*>(work);
        if (do_x && pc_nearest(x, n, y, m, w, idx_x, d2_x, stream)) return -1;
        return do_y ? pc_nearest(y, m, x, n, w, idx_y, d2_y, stream) : 0;
    }
    hipStream_t st = reinterpret_cast<hipStream_t>(stream);
    NnPair a;
    char* p = static_cast<char*>(work);
    for (int k = 0; k < 2; k++) {
        NnCloud& c = a.c[k];
        c.p = k ? y : x;
        c.n = k ? m : n;
        c.blocks = (int)(((long long)c.n + NN_BLOCK - 1) / NN_BLOCK);
        c.sorted = reinterpret_cast<nn4*>(p);
        c.box = c.sorted + (size_t)c.blocks * NN_BLOCK;
        c.at = reinterpret_cast<unsigned*>(c.box + 2 * (size_t)c.blocks);
        c.count = reinterpret_cast<int*>(c.at + 2 * (size_t)c.n);
        c.part = reinterpret_cast<float*>(c.count + NN_CELLS);
        p = reinterpret_cast<char*>(c.part + NN_BOXES * 6);
        p += (16 - (reinterpret_cast<uintptr_t>(p) & 15)) & 15;
    }
    int big = std::max(n, m), padded = std::max(a.c[0].blocks, a.c[1].blocks) * NN_BLOCK;
    hipLaunchKernelGGL(k_nn_box, dim3(NN_BOXES, 2), dim3(PC_WG), 0, st, a);
    hipLaunchKernelGGL(k_nn_count, dim3((big + PC_WG - 1) / PC_WG, 2), dim3(PC_WG), 0, st, a);
    hipLaunchKernelGGL(k_nn_sort, dim3((padded + 1023) / 1024, 2), dim3(1024), 0, st, a);
    hipLaunchKernelGGL(k_nn_blocks, dim3((padded + PC_WG - 1) / PC_WG, 2), dim3(PC_WG), 0, st, a);
    int first = do_x ? 0 : 1, rows = std::max(do_x ? n : 0, do_y ? m : 0);
    dim3 grid((rows + NN_BLOCK - 1) / NN_BLOCK, do_x && do_y ? 2 : 1);
    hipLaunchKernelGGL(k_nn_search, grid, dim3(NN_HALVES * NN_BLOCK), 0, st, a, first, idx_x, d2_x, idx_y, d2_y);
    hipError_t e = hipGetLastError();
    if (e != hipSuccess) return pc_fail(std::string("pc_nearest_pair: ") + hipGetErrorString(e));
    return 0;
}

int pc_chamfer_loss(const float* d2_x, int n, const float* d2_y, int m, int squared, float* out, void* stream) {
    if (n <= 0 || (d2_y && m <= 0)) return pc_fail("pc_chamfer_loss: no points");
    if (!d2_x || !out) return pc_fail("pc_chamfer_loss: null argument");
    hipLaunchKernelGGL(k_ch_loss, dim3(1), dim3(1024), 0, reinterpret_cast<hipStream_t>(stream), d2_x, n, d2_y, m, squared, (double*)nullptr, out);
    hipError_t e = hipGetLastError();
    if (e != hipSuccess) return pc_fail(std::string("pc_chamfer_loss: ") + hipGetErrorString(e));
    return 0;
}

int pc_chamfer(const float* x, int n, const float* y, int m, int squared, void* work, int* idx_x, float* d2_x, int* idx_y, float* d2_y,
               float* loss, void* stream) {
    if (n <= 0 || m <= 0) return pc_fail("pc_chamfer: both clouds must be non-empty");
    if (!idx_x || !loss) return pc_fail("pc_chamfer: null argument");
    if (pc_nearest_pair(x, n, y, m, work, idx_x, d2_x, idx_y, d2_y, stream)) return -1;
    hipStream_t st = reinterpret_cast<hipStream_t>(stream);
    int groups = ch_loss_groups(n, idx_y ? m : 0);
    double* part = static_cast<double*>(work);   // (the search is done with it)
    hipLaunchKernelGGL(k_ch_loss, dim3(groups), dim3(1024), 0, st, d2_x, n, d2_y, m, squared, part, loss);
    if (groups > 1) hipLaunchKernelGGL(k_ch_loss_sum, dim3(1), dim3(64), 0, st, (const double*)part, groups, n, m, idx_y ? 1 : 0, loss);
    hipError_t e = hipGetLastError();
    if (e != hipSuccess) return pc_fail(std::string("pc_chamfer: ") + hipGetErrorString(e));
    return 0;
}

int pc_chamfer_grad(const float* x, int n, const float* y, int m, const int* idx_x, const float* d2_x, const int* idx_y,
                    const float* d2_y, int squared, const float* go, float* gx, float* gy, void* stream) {
    if (n <= 0 || m <= 0) return pc_fail("pc_chamfer_grad: both clouds must be non-empty");
    if (!x || !y || !idx_x || !d2_x || !go || !idx_y != !d2_y) return pc_fail("pc_chamfer_grad: null argument");
    if (!gx && !gy) return 0;
    hipStream_t st = reinterpret_cast<hipStream_t>(stream);
    ChDir a{x, y, idx_x, d2_x, gx, gy, n}, b{y, x, idx_y, d2_y, gy, gx, m};
    dim3 grid((unsigned)((3LL * std::max(n, m) + PC_WG - 1) / PC_WG), 2);
    hipLaunchKernelGGL(k_ch_grad, grid, dim3(PC_WG), 0, st, a, b, squared, go, 1);
    // (a direction that k_ch_share takes leaves the others' launch)
    const ChDir dirs[2] = {a, b};
    const int nt[2] = {m, n};
    for (int k = 0; k < 2; k++) {
        if (!dirs[k].gt || !dirs[k].idx || !ch_shares(dirs[k].n, nt[k])) continue;
        hipLaunchKernelGGL(k_ch_share, dim3(ch_share_groups(dirs[k].n)), dim3(1024), 12 * nt[k], st, dirs[k], nt[k], squared, go);
        (k ? b : a).gt = nullptr;
    }
    if (a.gt || (b.gt && idx_y)) hipLaunchKernelGGL(k_ch_grad, grid, dim3(PC_WG), 0, st, a, b, squared, go, 0);
    hipError_t e = hipGetLastError();
    if (e != hipSuccess) return pc_fail(std::string("pc_chamfer_grad: ") + hipGetErrorString(e));
    return 0;
}

int pc_nearest_noalloc(const float* q, int nq, const float* t, int nt, int* idx, float* d2, void* stream) {
    if (nq < 0 || nt < 0) return pc_fail("pc_nearest_noalloc: negative point count");
    if (nq > PC_NOALLOC_MAX_QUERIES)
        return pc_fail("pc_nearest_noalloc: " + std::to_string(nq) + " queries exceed the static scratch of " +
                       std::to_string(PC_NOALLOC_MAX_QUERIES) + " (use pc_nearest with a workspace)");
    if (nq == 0) return 0;
    unsigned long long* work = nullptr;
    if (noalloc_scratch(&work)) return -1;
    // the scratch keeps the previous call's words; pc_nearest clears the
    // first nq of them (a fill kernel) before the search
    return pc_nearest(q, nq, t, nt, work, idx, d2, stream);
}

}  // extern "C"
