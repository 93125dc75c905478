// device_common.hpp -- device helpers shared by the beam and beamlet pipelines: XCD-aware work
// mapping, per-workgroup counters, the REV line table, and the collapsed-cone line walk.
#pragma once

#include <hip/hip_runtime.h>

#include <cstdint>

#include "cccs_internal.hpp"

namespace cccs {

// Workgroups are dispatched round-robin over the 8 XCDs of the part (workgroup b runs on XCD
// b % 8).  xcd_remap(b, nb) gives the workgroups of one XCD one contiguous range of work items,
// so neighbouring REV lines / voxel tiles share that XCD's L2.  A bijection on [0, nb).
__device__ __forceinline__ uint32_t xcd_remap(uint32_t b, uint32_t nb) {
    const uint32_t nx = 8;
    const uint32_t per = nb / nx, rem = nb % nx;
    const uint32_t x = b % nx, idx = b / nx;
    return x * per + (x < rem ? x : rem) + idx;
}

// The same with chunks of `chunk` consecutive work items going to the XCDs in turn: neighbours still
// share an L2, and work that is unevenly spread over the items (voxels outside the field, lines of
// different lengths) still reaches every XCD.  A bijection on [0, nb).  Against one range per XCD, chunks
// of 64: PVCS 276 -> 174 us per pass and cone kernel -4 % (thorax beam), beamlet gather 199 -> 187 us
// (thorax, 3 beams); chunks of 16 and 256 are within 2 %.
__device__ __forceinline__ uint32_t xcd_chunks(uint32_t b, uint32_t nb, uint32_t chunk) {
    const uint32_t super = 8 * chunk, s0 = b / super * super;
    if (super > nb - s0) return b;  // the incomplete last round
    const uint32_t r = b - s0;
    return s0 + (r % 8) * chunk + r / 8;
}

// Workgroups of 256 threads in one launch: the threads along a launch dimension are counted in 32 bits.
constexpr uint32_t kMaxGroups = (1u << 24) - 1;

// Sums one uint32 per lane over a 64-lane workgroup into part[slot] (no LDS).
__device__ __forceinline__ void wave_count(uint32_t v, uint32_t* __restrict__ part, size_t slot) {
    for (int o = 32; o > 0; o >>= 1) v += __shfl_xor(v, o, 64);
    if (threadIdx.x == 0) part[slot] = v;
}

// Sums one uint32 per thread over the workgroup (LDS tree, <= 256 threads) into part[slot].
__device__ __forceinline__ void block_count(uint32_t v, uint32_t* __restrict__ part, size_t slot) {
    __shared__ uint32_t s_cnt[256];
    const int t = threadIdx.x + threadIdx.y * blockDim.x + threadIdx.z * blockDim.x * blockDim.y;
    const int nt = blockDim.x * blockDim.y * blockDim.z;
    s_cnt[t] = v;
    __syncthreads();
    for (int w = 128; w > 0; w >>= 1) {
        if (t < w && t + w < nt) s_cnt[t] += s_cnt[t + w];
        __syncthreads();
    }
    if (t == 0) part[slot] = s_cnt[0];
}

// Read-only data at wave-uniform addresses, loaded through the scalar unit.
template <class T>
using uniform_ptr = const __attribute__((address_space(4))) T*;
template <class T>
__device__ __forceinline__ uniform_ptr<T> as_uniform(const T* p) {
    return (uniform_ptr<T>)p;
}

// Inclusive prefix sum over the 64 lanes of a wave.
__device__ __forceinline__ uint32_t wave_incl_u32(uint32_t v) {
    const int lane = threadIdx.x & 63;
    for (int o = 1; o < 64; o <<= 1) {
        const uint32_t u = __shfl_up(v, o, 64);
        if (lane >= o) v += u;
    }
    return v;
}

// One REV line of a cone grid in the compact store: samples [i0, i0 + len) of the line are kept at
// rev[off ...]; every other sample of the line is zero.
struct LineMeta {
    uint32_t off;  // first stored sample in the store
    int16_t i0;    // first stored sample index on the line (lines are <= 1024 samples)
    int16_t len;   // stored samples
};
static_assert(sizeof(LineMeta) == 8, "line table entries are 8 bytes");

// Entries kept before and after a line table and a REV store, so that a pair load at an end stays
// inside the allocation (128 bytes of the store: lines keep their alignment).
constexpr int kRevPad = 32;

// Two consecutive entries as one load (the address is a multiple of the entry, not of the pair).
typedef float pair_f32 __attribute__((ext_vector_type(2), aligned(4)));
typedef uint32_t pair_meta __attribute__((ext_vector_type(4), aligned(8)));

__device__ __forceinline__ LineMeta meta_of(uint32_t off, uint32_t w, bool in) {
    LineMeta r;
    r.off = off;
    r.i0 = (int16_t)(w & 0xffffu);
    r.len = in ? (int16_t)(w >> 16) : (int16_t)0;
    return r;
}

// Records of lines (j, k), (j+1, k), (j, k+1), (j+1, k+1) of a grid of ny x nz lines, j in [-1, ny-1],
// k in [-1, nz-1]; lines outside the grid get length 0.
__device__ __forceinline__ void meta_pairs(const LineMeta* __restrict__ meta, uint64_t line0, int ny, int nz, int j, int k,
                                           LineMeta m[4]) {
#pragma unroll
    for (int h = 0; h < 2; h++) {
        const int kk = k + h;
        const bool row = kk >= 0 && kk < nz;
        const LineMeta* p = meta + line0 + (uint64_t)(row ? kk : 0) * (uint64_t)ny + (int64_t)j;
        const pair_meta r = *reinterpret_cast<const pair_meta*>(p);
        m[2 * h] = meta_of(r.x, r.y, row && j >= 0);
        m[2 * h + 1] = meta_of(r.z, r.w, row && j + 1 < ny);
    }
}

// Samples i and i+1 of a stored line (zero outside its interval), interpolated at fraction a.
__device__ __forceinline__ float rev_lerp(const float* __restrict__ rev, const LineMeta& m, int i, float a) {
    const int d = i - m.i0;
    const bool vlo = d >= 0 && d < m.len, vhi = d + 1 >= 0 && d + 1 < m.len;
    const pair_f32 x = *reinterpret_cast<const pair_f32*>(rev + (vlo || vhi ? (int64_t)m.off + (int64_t)d : (int64_t)0));
    const float lo = vlo ? x.x : 0.f, hi = vhi ? x.y : 0.f;
    return lo + a * (hi - lo);
}

// Trilinear fetch from a compactly stored REV grid (nx samples per line, ny x nz lines) at texture
// coordinates (u, v, w) = (sample, line y, line z), texel centres at +0.5, border 0: the same
// operation sequence as tex3_border on the dense grid, so both give identical results.
//
// The loads are branch-free and issued in two rounds: the line records together, then the samples
// together, so a lane waits for two memory round trips instead of one per tap.  Neighbouring taps
// are neighbours in memory (lines j and j+1 of the table, samples i and i+1 of a line), so a pair is
// one load: two for the four records and four for the eight samples.  A gather of lanes on different
// lines costs the L1 one lookup per lane and load, so halving the loads halves the stage's bound
// (with the 4x4x4-voxel waves of pvcs_kernel: 472 -> 277 us per 4-cone pass of a 256x256x180 beam).  A
// tap outside the grid or outside its line's stored interval is replaced by zero; its pair may read
// one entry before or after the table or the store (kRevPad entries on both sides).
__device__ __forceinline__ float rev_fetch(const LineMeta* __restrict__ meta, const float* __restrict__ rev,
                                           uint64_t line0, int nx, int ny, int nz, float u, float v, float w) {
    if (ny <= 0 || nz <= 0) return 0.f;
    const float ub = u - 0.5f, vb = v - 0.5f, wb = w - 0.5f;
    if (!(ub > -1.f && vb > -1.f && wb > -1.f && ub < (float)nx && vb < (float)ny && wb < (float)nz)) return 0.f;
    const float fu = floorf(ub), fv = floorf(vb), fw = floorf(wb);
    const int i = (int)fu, j = (int)fv, k = (int)fw;
    const float a = ub - fu, b = vb - fv, c = wb - fw;
    LineMeta m[4];
    meta_pairs(meta, line0, ny, nz, j, k, m);
    float t[4];
#pragma unroll
    for (int q = 0; q < 4; q++) t[q] = rev_lerp(rev, m[q], i, a);
    const float e0 = t[0] + b * (t[1] - t[0]);
    const float e1 = t[2] + b * (t[3] - t[2]);
    return e0 + c * (e1 - e0);
}

// Zero samples kept before and behind every stored line, where a launch's `zeros` says so (a store of fewer
// than 2^30 samples; empty lines then have offset 0 and the store begins with as many zeros): a
// select on the index replaces one on each sample.
constexpr int kLineZeros = 2;

// The stored line of record (off, w) at sample i, interpolated at fraction x; rev0 is kLineZeros samples
// before the store.  Samples outside the line all read the store's first zeros: the load of a wave
// costs its different cache lines, so those lanes share one (clamped to their own line's zeros
// instead, two instructions less, the beamlet gather took 79 us a direction, not 70).
__device__ __forceinline__ float line_lerp(const char* __restrict__ rev0, uint32_t off, uint32_t w, int i, float x) {
    const int d = i - (int)(int16_t)(w & 0xffffu);
    const uint32_t at = (uint32_t)(d + 1) <= w >> 16 ? (uint32_t)(d + kLineZeros) + off : 0u;
    const pair_f32 p = *reinterpret_cast<const pair_f32*>(rev0 + at * 4u);
    return p.x + x * (p.y - p.x);
}

// The line's samples live in LDS as {half step, TERMA}: x = 0.5*delr*density (negative marks a
// sample outside the crop box or the calc_bbox), y = TERMA.
//
// walk_both runs the two walks of destination j (RowConvolve's do/while loops) back to back over
// the line's valid segment [vlo, vhi]: first toward lower indices with the forward kernel row,
// then toward higher indices with the backward row.  Every destination takes exactly vhi - vlo
// steps, so the trip count is the same on every lane of a wave (a scalar loop, no divergence);
// the direction switch and the reference's early exits (radiological depth beyond the last radius,
// reaching the last radial interval) become per-lane flags.  The cumulative kernel is linear
// between two radii, so a lane keeps its current interval in registers and reads the LDS tables
// only when the radiological depth crosses a radius.
CCCS_HD float walk_both(const float2* __restrict__ s, int j, int vlo, int vhi,
                                           const float* __restrict__ R, const float* __restrict__ IW,
                                           const float* __restrict__ rowF, const float* __restrict__ rowB, int nr,
                                           bool active, uint32_t& iters) {
    const float rmax = R[nr - 1];
    const int total = vhi - vlo;
    const int nfwd = j - vlo;
    const float* row = rowF;
    float r = 0.f, last = 0.f, lo = 0.f, hi = R[0], klo = 0.f, slope = rowF[0] * IW[0], sum = 0.f;
    int rs = 0, k = j, dir = -1;
    bool alive = active && nfwd > 0;
    for (int it = 0; it < total; ++it) {
        if (it == nfwd) {  // switch to the backward walk
            dir = 1;
            k = j;
            row = rowB;
            r = 0.f; last = 0.f; lo = 0.f; hi = R[0]; klo = 0.f; slope = rowB[0] * IW[0];
            rs = 0;
            alive = active;
        }
        k += dir;
        const float2 e = s[k];
        r += e.x;
        bool ok = alive && e.x >= 0.f && r <= rmax;
        if (ok && hi < r) {
            do {
                rs++;
                lo = hi;
                hi = R[rs];
                klo = row[rs - 1];
                slope = (row[rs] - klo) * IW[rs];
            } while (hi < r && rs < nr - 1);
        }
        const float cum = klo + (r - lo) * slope;
        sum += ok ? (cum - last) * e.y : 0.f;
        last = cum;
        r += e.x;
        iters += ok ? 1u : 0u;
        alive = ok && rs < nr - 1;
    }
    return sum;
}

// Narrows [t0, t1] to the parameters where o + t*d lies in [lo, hi) (widened by a margin that
// covers FP32 rounding; the exact per-sample test decides membership).
CCCS_HD void clip_slab(float o, float d, float lo, float hi, float& t0, float& t1) {
    if (fabsf(d) < 1e-3f) {
        // the coordinate moves by less than one index unit over a whole line (<= 1024 samples)
        if (!(o >= lo - 2.f && o < hi + 2.f)) { t0 = 1.f; t1 = 0.f; }
        return;
    }
    float ta = (lo - o) / d, tb = (hi - o) / d;
    t0 = fmaxf(t0, fminf(ta, tb));
    t1 = fminf(t1, fmaxf(ta, tb));
}

}  // namespace cccs
