// beam.hip -- resident context and the plain full-beam CCCS path on gfx950.
//
// Per beam (replacing radconvolveTexture, CCCS/dosecalc-beam/nvbbRayConvolve_host.cu:376-725):
//   1. terma_kernel      Siddon radiological path + poly-energetic TERMA per calc_bbox voxel
//                        (DoseCalcAlgo/cudaSiddon.cu:117-308)
//   2. crop_partial/final  BEV-rotated extent of non-zero TERMA, reduced on the GPU instead of the
//                        reference's D2H copy + host triple loop (:417-499); 28 bytes come back
//   3. host geometry     crop box + one REV grid per cone (findREV :75-155)
//   4. line_interval / class_scan / class_scatter_kernel  stored interval, offset and class-list entry of
//                        every REV line of every cone
//   5. cone_kernel       one workgroup per listed line, one launch per length class: resample density and
//                        TERMA along the line into LDS (cudaRaytrace, nvbbRayConvolve_device.cu:11-80)
//                        then the collapsed-cone walk in both directions from LDS (RowConvolve
//                        :87-218).  The REV grid is sized per cone; nothing is cleared per cone.
//   6. pvcs_kernel       passes over the PVCS voxels the crop box can reach, gathering their
//                        cones' REV dose trilinearly and adding the sum once (REV2XYZdose
//                        :222-261 per cone in the reference).
#include <hip/hip_runtime.h>

#include <algorithm>
#include <cfloat>
#include <cmath>
#include <cstdio>
#include <cstring>
#include <array>
#include <functional>
#include <limits>
#include <map>
#include <memory>
#include <mutex>
#include <string>
#include <vector>

#include "context.hpp"
#include "device_common.hpp"

namespace cccs {

BeamDev make_beam_dev(const cccs_beam& b) {
    BeamDev d;
    d.src = ld3(b.source);
    d.dir_n = norm3(ld3(b.direction));
    d.iso = ld3(b.isocenter);
    d.sad = b.sad;
    d.iso_dist = len3(d.iso - d.src);
    d.fmx = (int)b.fmap_size[0];
    d.fmy = (int)b.fmap_size[1];
    d.bsx = b.beamlet_size[0];
    d.bsy = b.beamlet_size[1];
    d.beam_fwd = rot2_beam_fwd(b.azimuth, b.zenith, b.coll);
    return d;
}

int check_beam(const cccs_ctx* ctx, const cccs_beam& b) {
    (void)ctx;
    if (b.fmap_size[0] == 0 || b.fmap_size[1] == 0 || b.fmap_size[0] > 4096 || b.fmap_size[1] > 4096)
        return set_error(CCCS_EINVAL, "fluence map dims must be in [1, 4096]");
    if (!(b.beamlet_size[0] > 0.f) || !(b.beamlet_size[1] > 0.f)) return set_error(CCCS_EINVAL, "beamlet size must be > 0");
    if (!(b.sad > 0.f)) return set_error(CCCS_EINVAL, "sad must be > 0");
    return CCCS_OK;
}

// ------------------------------------------------------------------------------------------------
// kernels

struct TermaArgs {
    float* terma;
    const float* fmap;
    const float* dens;
    VolDesc vd;
    BeamDev beam;
    SpecDev spec;
    int bx, by, bz;          // calc_bbox size
    int ox, oy, oz;          // calc_bbox start
    int ss;                  // supersampling factor
    float bhc;
    int beamletnum;
    int depth, far_first;     // axis along which the beam runs mostly; start at its high end
    float field2;             // squared tangent of a cone around the fluence map (infinite: unknown)
    uint32_t block0;          // first workgroup of this launch
    uint32_t* counts;         // per-block Siddon step counts (profiling) or nullptr
};

// Centre of calc_bbox voxel (X, Y, Z).
CCCS_HD v3 terma_point(const TermaArgs& a, int X, int Y, int Z) {
    return mk3(a.vd.start.x + ((float)a.ox + X) * a.vd.voxel.x, a.vd.start.y + ((float)a.oy + Y) * a.vd.voxel.y,
               a.vd.start.z + ((float)a.oz + Z) * a.vd.voxel.z);
}

// Voxel of a thread: a workgroup takes 16x4x4 voxels of the calc_bbox, each of its waves 4x4x4.  The
// march runs inside the field only, a part of the box, so the workgroups have to be small along x for
// their waves to be full or empty, and rows of them go to the XCDs in turn: with 64x4x1 workgroups
// dealt out one by one, a box of 4 or 8 workgroups along x left whole XCDs without field.  Thorax
// beam at 54 degrees 1133 -> 395 us, 128^3 water beam 217 -> 116 us.  A ray is a serial chain as long as
// its voxel is deep, so the deepest planes along the beam's main axis start first and the short
// rays fill the end; workgroups with and without field mix, so at most kTermaResident share a CU and
// the rest go where one ends.  Those two and the cheap test of the field below: thorax at 54, 90 and 3
// degrees 400, 220 and 243 -> 380, 176 and 182 us, 128^3 water 118 -> 95 us.  Four to eight a CU take 139,
// 137, 136, 138 and 144 us a beam over the 20 beams of a thorax plan, 85, 85, 94, 108 and 154 us for the 128^3
// water beam and 22 us each for a 32^3 one: six is the plan's best, by a hundredth, and water's runs of
// full workgroups would have fewer.
constexpr int kTermaResident = 6;
__device__ __forceinline__ void terma_voxel(const TermaArgs& a, int& X, int& Y, int& Z) {
    const uint32_t nx = (uint32_t)(a.bx + 15) / 16, ny = (uint32_t)(a.by + 3) / 4, nz = (uint32_t)(a.bz + 3) / 4;
    const uint32_t inner = a.depth == 0 ? ny : nx, middle = a.depth == 2 ? ny : nz;
    const uint32_t t = a.block0 + xcd_chunks(blockIdx.x, gridDim.x, inner), r = t / inner;
    // (the rows turn from plane to plane, or a multiple of 8 rows would keep each on one XCD)
    const uint32_t i = t - r * inner, w0 = r / middle, m0 = r - w0 * middle + (middle >= 8 ? 5 * w0 & 7u : 0u);
    const uint32_t m = m0 >= middle ? m0 - middle : m0;
    const uint32_t outer = a.depth == 0 ? nx : a.depth == 1 ? ny : nz, o = a.far_first ? outer - 1 - w0 : w0;
    const uint32_t bx = a.depth == 0 ? o : i, by = a.depth == 0 ? i : a.depth == 1 ? o : m, bz = a.depth == 2 ? o : m;
    const int l = threadIdx.x & 63, w = threadIdx.x >> 6;
    X = (int)bx * 16 + w * 4 + (l & 3);
    Y = (int)by * 4 + ((l >> 2) & 3);
    Z = (int)bz * 4 + (l >> 4);
}
// Point certainly outside the fluence map: farther from the beam's axis than the map's corners (by
// 0.5 %).  Most voxels of the box are, and the exact cell takes 200 instructions more.  (A point level
// with the source is left to the exact cell.)
__device__ __forceinline__ bool outside_field(const TermaArgs& a, v3 p) {
    const v3 d = p - a.beam.src;
    const float along = dot3(d, a.beam.dir_n), a2 = along * along;
    const v3 r = d - along * a.beam.dir_n;
    const float r2 = dot3(r, r);
    return r2 > a.field2 * a2 && a2 > 1e-6f * r2;
}
inline uint64_t terma_blocks(const TermaArgs& a) {
    return (uint64_t)((a.bx + 15) / 16) * (uint64_t)((a.by + 3) / 4) * (uint64_t)((a.bz + 3) / 4);
}

// The workgroups of a calc_bbox, in as many launches as their number takes (boxes beyond 2^32 voxels of
// whole workgroups: thin ones fill the last workgroup of a row badly).
template <class Launch>
void terma_launches(TermaArgs& a, Launch&& launch) {
    const uint64_t n = terma_blocks(a);
    for (uint64_t b = 0; b < n; b += kMaxGroups) {
        a.block0 = (uint32_t)b;
        launch(dim3((unsigned)std::min<uint64_t>(kMaxGroups, n - b)));
    }
}

// One lane per calc_bbox voxel (x fastest => coalesced store).  Each lane marches its own ray
// (the rpl-only march: same crossings and segments as cudaSiddon, fetch coordinates formed with
// reciprocal voxel sizes); neighbouring lanes follow near-parallel rays, so the density taps stay
// in L1/L2.
// Supersampling and the profiling counts have instances of their own: together they took 81 registers.
template <bool kSuper, bool kCount>
__global__ void __launch_bounds__(256) terma_kernel(TermaArgs a) {
    int X, Y, Z;
    terma_voxel(a, X, Y, Z);
    const bool in = (X < a.bx && Y < a.by && Z < a.bz);
    uint32_t steps = 0;
    float acc = 0.f;
    const v3 ivox = mk3(1.f / a.vd.voxel.x, 1.f / a.vd.voxel.y, 1.f / a.vd.voxel.z);
    int it = 0;
    int* const iters = kCount ? &it : nullptr;
    if (!in) {
    } else if (kSuper) {
        // supersampled: sub-voxel centres, summed in sub-voxel order then averaged
        const int nsub = a.ss * a.ss * a.ss;
        v3 subsz = mk3(a.vd.voxel.x / (float)a.ss, a.vd.voxel.y / (float)a.ss, a.vd.voxel.z / (float)a.ss);
        for (int s = 0; s < nsub; s++) {
            int sx = s % a.ss, sy = (s / a.ss) % a.ss, sz = s / (a.ss * a.ss);
            v3 p = mk3(a.vd.start.x + ((float)a.ox + X - 0.5f) * a.vd.voxel.x + (sx + 0.5f) * subsz.x,
                       a.vd.start.y + ((float)a.oy + Y - 0.5f) * a.vd.voxel.y + (sy + 0.5f) * subsz.y,
                       a.vd.start.z + ((float)a.oz + Z - 0.5f) * a.vd.voxel.z + (sz + 0.5f) * subsz.z);
            acc += point_terma_rpl(p, a.fmap, a.beam, a.spec, a.vd, ivox, a.dens, a.bhc, a.beamletnum, iters);
            if (kCount) steps += (uint32_t)it;
        }
        acc /= (float)nsub;
    } else {
        // fluence times the unit-fluence TERMA (the Siddon march only inside the field), the order
        // in which a resident unit-TERMA grid of the same source gives the same value
        const v3 p = terma_point(a, X, Y, Z);
        const float fl = outside_field(a, p) ? 0.f : point_fluence(p, a.fmap, a.beam, a.beamletnum);
        if (fl > 0.f) acc = fl * unit_point_terma(p, a.beam, a.spec, a.vd, ivox, a.dens, a.bhc, iters);
        if (kCount) steps = (uint32_t)it;
    }
    if (in) a.terma[(size_t)X + (size_t)a.bx * ((size_t)Y + (size_t)a.by * Z)] = acc;
    if (kCount) block_count(steps, a.counts, a.block0 + blockIdx.x);
}

// Unit-fluence TERMA of every calc_bbox voxel (the march runs for every voxel): one beam source's
// entry of the angle cache.
__global__ void __launch_bounds__(256) unit_terma_kernel(TermaArgs a, float* __restrict__ unit) {
    int X, Y, Z;
    terma_voxel(a, X, Y, Z);
    if (X >= a.bx || Y >= a.by || Z >= a.bz) return;
    const v3 ivox = mk3(1.f / a.vd.voxel.x, 1.f / a.vd.voxel.y, 1.f / a.vd.voxel.z);
    unit[(size_t)X + (size_t)a.bx * ((size_t)Y + (size_t)a.by * Z)] =
        unit_point_terma(terma_point(a, X, Y, Z), a.beam, a.spec, a.vd, ivox, a.dens, a.bhc, nullptr);
}

// TERMA from a resident unit-TERMA grid of the beam's source: the voxel's fluence times its entry.
__global__ void __launch_bounds__(256) terma_from_unit_kernel(TermaArgs a, const float* __restrict__ unit) {
    const int X = blockIdx.x * 64 + threadIdx.x;
    const int Y = blockIdx.y * 4 + threadIdx.y;
    const int Z = blockIdx.z;
    if (X >= a.bx || Y >= a.by || Z >= a.bz) return;
    const size_t v = (size_t)X + (size_t)a.bx * ((size_t)Y + (size_t)a.by * Z);
    const v3 p = terma_point(a, X, Y, Z);
    const float fl = outside_field(a, p) ? 0.f : point_fluence(p, a.fmap, a.beam, a.beamletnum);
    a.terma[v] = fl > 0.f ? fl * unit[v] : 0.f;
}

struct PathArgs {
    const float* dens;
    VolDesc vd;
    v3 src;
    const float* pts;
    int n, maxseg;
    int32_t* ijk;
    float* mid;
    float* len;
    int32_t* counts;
    float* rpl;
};

__global__ void __launch_bounds__(256) siddon_path_kernel(PathArgs a) {
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= a.n) return;
    int c = 0;
    v3 p = mk3(a.pts[3 * i], a.pts[3 * i + 1], a.pts[3 * i + 2]);
    float r = siddon_march(p, a.vd.start, a.vd.end, a.vd.voxel, a.src, a.dens, a.vd.nx, a.vd.ny, a.vd.nz,
                           [&](float fx, float fy, float fz, float l) {
                               if (c < a.maxseg) {
                                   size_t o = (size_t)i * a.maxseg + c;
                                   a.ijk[3 * o] = f2i_rd(fx + 0.5f);
                                   a.ijk[3 * o + 1] = f2i_rd(fy + 0.5f);
                                   a.ijk[3 * o + 2] = f2i_rd(fz + 0.5f);
                                   a.mid[3 * o] = fx;
                                   a.mid[3 * o + 1] = fy;
                                   a.mid[3 * o + 2] = fz;
                                   a.len[o] = l;
                               }
                               c++;
                           },
                           nullptr);
    a.counts[i] = c;
    a.rpl[i] = r;
}

// Crop box: min/max of the BEV-rotated bbox index of every voxel with non-zero TERMA.
// Pass 1 writes one partial (min xyz, max xyz, count) per workgroup.
constexpr int kCropBlocks = 1024;
__global__ void __launch_bounds__(256) crop_partial_kernel(const float* __restrict__ terma, int bx, int by, int bz,
                                                           Rot2 rot, float* __restrict__ part) {
    __shared__ float s[7][256];
    float mn0 = FLT_MAX, mn1 = FLT_MAX, mn2 = FLT_MAX, mx0 = -FLT_MAX, mx1 = -FLT_MAX, mx2 = -FLT_MAX, cnt = 0.f;
    const size_t n = (size_t)bx * by * bz;
    for (size_t v = (size_t)blockIdx.x * 256 + threadIdx.x; v < n; v += (size_t)gridDim.x * 256) {
        if (terma[v] != 0.f) {
            int x = (int)(v % bx);
            int y = (int)((v / bx) % by);
            int z = (int)(v / ((size_t)bx * by));
            v3 b = rot_fwd(rot, mk3((float)x, (float)y, (float)z));
            mn0 = fminf(mn0, b.x); mn1 = fminf(mn1, b.y); mn2 = fminf(mn2, b.z);
            mx0 = fmaxf(mx0, b.x); mx1 = fmaxf(mx1, b.y); mx2 = fmaxf(mx2, b.z);
            cnt += 1.f;
        }
    }
    const int t = threadIdx.x;
    s[0][t] = mn0; s[1][t] = mn1; s[2][t] = mn2; s[3][t] = mx0; s[4][t] = mx1; s[5][t] = mx2; s[6][t] = cnt;
    __syncthreads();
    for (int w = 128; w > 0; w >>= 1) {
        if (t < w) {
            for (int q = 0; q < 3; q++) s[q][t] = fminf(s[q][t], s[q][t + w]);
            for (int q = 3; q < 6; q++) s[q][t] = fmaxf(s[q][t], s[q][t + w]);
            s[6][t] += s[6][t + w];
        }
        __syncthreads();
    }
    if (t < 7) part[(size_t)blockIdx.x * 8 + t] = s[t][0];
}

__global__ void __launch_bounds__(256) crop_final_kernel(const float* __restrict__ part, int nblocks, float* __restrict__ out) {
    __shared__ float s[7][256];
    const int t = threadIdx.x;
    float v[7] = {FLT_MAX, FLT_MAX, FLT_MAX, -FLT_MAX, -FLT_MAX, -FLT_MAX, 0.f};
    for (int b = t; b < nblocks; b += 256) {
        for (int q = 0; q < 3; q++) v[q] = fminf(v[q], part[(size_t)b * 8 + q]);
        for (int q = 3; q < 6; q++) v[q] = fmaxf(v[q], part[(size_t)b * 8 + q]);
        v[6] += part[(size_t)b * 8 + 6];
    }
    for (int q = 0; q < 7; q++) s[q][t] = v[q];
    __syncthreads();
    for (int w = 128; w > 0; w >>= 1) {
        if (t < w) {
            for (int q = 0; q < 3; q++) s[q][t] = fminf(s[q][t], s[q][t + w]);
            for (int q = 3; q < 6; q++) s[q][t] = fmaxf(s[q][t], s[q][t + w]);
            s[6][t] += s[6][t + w];
        }
        __syncthreads();
    }
    if (t < 7) out[t] = s[t][0];
}

// A class-list entry: all that a workgroup needs of its line, as one 16-byte scalar load.  Samples
// [ja, jb] of the stored interval lie inside the crop box, the calc_bbox and the interpolation range
// by a margin that covers FP32 rounding (relative to i0; ja > jb: none); the others are tested one by
// one.
struct ConeLine {
    uint32_t off;   // first stored sample in the REV store
    uint32_t tyz;   // line of the cone's grid: ty | tz << ConeDev::tybits (a cone has < 2^31 lines)
    uint32_t seg;   // i0 | (len - 1) << 10 | ja << 20 (lines have at most 1024 samples)
    uint32_t last;  // jb + 1 | cone << 11
};
static_assert(kMaxLine <= 1024 && kMaxRays <= 64, "fields of a class-list entry");
static_assert(sizeof(ConeLine) == 16, "four dwords");

struct ConeArgs {
    const float2* dt;         // {density, TERMA (0 outside the calc_bbox)} over the CT grid
    const float* tables;      // kernel | radii | inverse widths
    const RampStep* steps;    // [ntheta/2][nradii]
    const ConeDev* cones;
    LineMeta* lines;          // one entry per REV line of every cone
    float* rev;               // compact REV dose store
    uint64_t nlines;
    int ncones;
    int ntheta, nradii, nphi;
    float delr;
    uint32_t* counts;         // per-workgroup walk step counts (profiling) or nullptr
    int ramp_min;             // valid segments at least this long use the segment-sum walk
    int maxn;                 // longest stored line of this launch (LDS sizing)
    const ConeLine* list;     // the lines of this launch, one workgroup each
    const uint32_t* count;    // their number, where the launch's grid is a bound (or nullptr)
    bool zeros;               // kLineZeros zero samples around every stored line
    VolDesc vd;
    m33 binv;                 // PVCS <- BEV rotation (index units)
    v3 off;                   // (bevStart - start) / voxel
    v3 bev_size;              // crop-box size (index units)
    v3 bb0, bb1;              // calc_bbox bounds (PVCS index)
};

__device__ __forceinline__ int cone_of_line(const ConeDev* __restrict__ cones, int ncones, uint64_t line) {
    int lo = 0, hi = ncones - 1;
    while (lo < hi) {  // last cone whose first line <= line
        int mid = (lo + hi + 1) >> 1;
        if (cones[mid].line0 <= line) lo = mid; else hi = mid - 1;
    }
    return lo;
}

// Sample interval [i0, i1) of REV line (tY, tZ) of cone c that can lie inside the crop box and the
// calc_bbox: the BEV and PVCS positions along a line are affine in the sample index, so each box
// clips the line to a slab interval.  Widened by 2/3 samples; the exact per-sample test of
// cudaRaytrace (nvbbRayConvolve_device.cu:50-70) still decides membership.
__device__ __forceinline__ void line_interval(const ConeArgs& a, const ConeDev& c, int tY, int tZ, int& i0,
                                              int& i1) {
    const int n = c.nx;
    const v3 p0 = mk3(c.rs.x + (float)tZ, c.rs.y, c.rs.z + (float)tY);
    const v3 b0 = c.kinv(p0);
    const v3 kd = mk3(c.kinv.m[1], c.kinv.m[4], c.kinv.m[7]);
    const v3 g0 = a.binv(b0) + a.off;
    const v3 gd = a.binv(kd);
    float t0 = 0.f, t1 = (float)n;
    clip_slab(b0.x, kd.x, 0.f, a.bev_size.x, t0, t1);
    clip_slab(b0.y, kd.y, 0.f, a.bev_size.y, t0, t1);
    clip_slab(b0.z, kd.z, 0.f, a.bev_size.z, t0, t1);
    clip_slab(g0.x, gd.x, a.bb0.x, a.bb1.x, t0, t1);
    clip_slab(g0.y, gd.y, a.bb0.y, a.bb1.y, t0, t1);
    clip_slab(g0.z, gd.z, a.bb0.z, a.bb1.z, t0, t1);
    i0 = 0;
    i1 = 0;
    if (t0 <= t1) {
        i0 = max(0, (int)floorf(t0) - 2);
        i1 = min(n, (int)ceilf(t1) + 3);
        if (i1 < i0) i1 = i0;
    }
}

// ---- segment-sum form of the two walks --------------------------------------------------------
// walk_both visits every sample of the segment for every destination (O(line^2) per line).  The
// same sums follow in O(nradii) per destination from three facts:
//  * the radiological distance from destination j to sample k is a difference of the line's
//    radiological coordinates: rho_k = P - c_k backward (P = boundary between j-1 and j, c_k the
//    centre of sample k) and c_k - P forward (P = boundary between j and j+1);
//  * summing by parts, sum_k T_k (C(rho_k) - C(rho_{k+1})) = sum_k (T_k - T_{k-1}) C(rho_k) + one
//    end term, with C the cumulative kernel;
//  * C is linear on each radial interval (R_{s-1}, R_s] with slope sigma_s and C(0) = 0, so it is a
//    sum of ramps: C(rho) = sum_s sigma_s (max(rho - R_{s-1}, 0) - max(rho - R_s, 0)).
// Hence the backward sum is sum_s sigma_s (F(P - R_{s-1}) - F(P - R_s)) with
// F(y) = sum_{c_k < y} (T_k - T_{k-1}) (y - c_k) = T_{q-1} y - E[q], q the first sample with c_q >= y
// and E the FP64 prefix sum of (T_k - T_{k-1}) c_k; the forward sum is its mirror image.  F is
// continuous, so a tie in the search for q does not matter, and one evaluation of F per radius is
// all that a destination costs: a lookup in a uniform table over the radiological coordinate, one
// probe of two centres, one multiply-add.  The walk's exits (distance beyond the last radius,
// entering the last interval) end the sum at one sample a: F(c_a) is then the constant that F
// starts from; a line that fits into the radii has no such end.  Same result as the sequential walk
// up to FP32 rounding of the accumulated distance.  The cone kernel issues VALU instructions in 92-98 %
// of its cycles, so a walk is as fast as its instructions are few: interval sums with a search loop per
// interval (about 55 per radius and direction) took 11.8 ms of a 256x256x180 request, this form with
// 28 8.9 ms, with 21 (no masks, no copies between the radii) 7.4 ms.
struct RampLine {
    const float* c;       // centres, radiological cm from the segment start; c[n..n+3] = +inf
    const double* E;      // E[k]  = sum_{m<k} (T_m - T_{m-1}) c_m   (T_{-1} = 0), k in [0, n]
    const double* E2;     // E2[k] = sum_{m<k} (T_m - T_{m+1}) c_m   (T_n = 0),    k in [0, n]
    const float2* s;      // {half step, TERMA} of the segment's samples
    const uint16_t* lb;   // lb[u] = first k with c_k >= c0 + u * D, u in [0, U + 1] (D = range / U)
    int n, U;
    float c0, cn, invD;
};

// The search for the first k with c_k >= y (kUpper: c_k > y), c_0 <= y <= c_{n-1}: a table lookup and
// two probes (one LDS load), no branch.  A cell holds at most one centre where the density is at
// least half the line's mean; `more` says that both probed centres lie below y, so that ramp_more has
// to go on from k.
CCCS_HD double max_f64(double a, double b) {
#ifdef __HIP_DEVICE_COMPILE__
    double r;  // (one instruction: the library form also quiets its operands)
    __asm__("v_max_f64 %0, %1, %2" : "=v"(r) : "v"(a), "v"(b));
    return r;
#else
    return a > b ? a : b;
#endif
}
struct RampPos {
    int u, k;
    bool more;
};
template <bool kUpper>
CCCS_HD bool ramp_below(float c, float y) { return kUpper ? c <= y : c < y; }
template <bool kUpper>
CCCS_HD RampPos ramp_probe(const RampLine& L, float y) {
    RampPos p;
    // biased by 2% of a cell so that the cell's threshold never exceeds y after rounding
    p.u = (int)fmaf(y, L.invD, -0.02f - L.c0 * L.invD);
    const int k = L.lb[p.u];
    const float ca = L.c[k], cb = L.c[k + 1];
    p.more = ramp_below<kUpper>(cb, y);
    p.k = k + (ramp_below<kUpper>(ca, y) ? 1 : 0) + (p.more ? 1 : 0);
    return p;
}
template <bool kUpper>
CCCS_HD int ramp_more(const RampLine& L, float y, const RampPos& p) {
    int k = min(p.k, L.n);
    if (L.lb[p.u + 1] - k > 8) {  // a crowded cell (low density): bisect up to the next cell's end
        int hi = L.lb[p.u + 2];
        while (k < hi) {
            const int mid = (k + hi) >> 1;
            if (ramp_below<kUpper>(L.c[mid], y)) k = mid + 1; else hi = mid;
        }
    }
    while (k < L.n && ramp_below<kUpper>(L.c[k], y)) k++;  // (bounded: y is infinite with an infinite density)
    return k;
}
template <bool kUpper>
CCCS_HD int ramp_find(const RampLine& L, float y) {
    if (y < L.c0) return 0;
    const RampPos p = ramp_probe<kUpper>(L, y);
    return p.more ? ramp_more<kUpper>(L, y, p) : p.k;
}
// Cells per cm over [c_0, c_{n-1}].  c_0 is half of the first sample and c_{n-1} at least all of it, so two samples
// or more span at least half of c_{n-1} and their 2n cells are never too fine for FP32 lookups; one sample, and a
// line without density, keep one cell (a margin of ten below that half).
CCCS_HD float ramp_cells(float c0, float cn, int U) { return cn - c0 > 0.05f * cn ? (float)U / (cn - c0) : 0.f; }

// Lanes of a wave leave the walk together, so that its body runs without masks.
struct RampWave {
    static __device__ __forceinline__ bool any(bool x) { return __any(x); }
};
struct RampAlone {
    static CCCS_HD bool any(bool x) { return x; }
};

// The backward (toward lower indices) and / or forward walk of destination j.  Both directions step
// through the radii together, so that their lookups (two dependent LDS trips each) overlap.  F starts
// at the boundary of the destination and ends, at Fa / Eb, at the centre ya / yb of the last sample
// that the walk reaches: there y is clamped (backward) or F taken as Eb (forward: the last cell may be
// crowded, so the lookup goes to the first), and F's differences are zero.  (Forward, F is taken
// without its constant: E2[q] + T_q y.)
template <bool kBack, bool kFwd, class Lanes>
CCCS_HD double ramp_walk(const RampLine& L, int j, const RampStep* steps, int nr, uint32_t& iters) {
    double Pb = L.c0, Pf = L.cn, Fb = 0.0, Ff = 0.0, Fa = 0.0, Eb = 0.0, ya = L.c0, yb = L.cn;
    const double rlast = steps[nr - 1].r, rprev = steps[nr - 2].r;
    const bool exits = (double)L.cn - (double)L.c0 > rprev;
    bool back = false, fwd = false;
    if (kBack && j > 0) {
        const float2 e = L.s[j - 1];
        Pb = (double)L.c[j - 1] + (double)e.x;
        const int a = exits ? max(ramp_find<false>(L, (float)(Pb - rlast)), ramp_find<false>(L, (float)(Pb - rprev)) - 1) : 0;
        back = a < j;
        if (back) {
            ya = (double)L.c[a];
            if (a > 0) Fa = fma((double)L.s[a - 1].y, ya, -L.E[a]);
            Fb = fma((double)e.y, Pb, -L.E[j]);
            // F rises where there is TERMA: a difference of rounding size means none in the walk's reach
            back = !exits || fabs(Fb - Fa) > 1e-14 * fabs(Fa);
        }
        if (!back) Pb = ya;
    }
    if (kFwd && j < L.n - 1) {
        const float2 e = L.s[j + 1];
        Pf = (double)L.c[j + 1] - (double)e.x;
        int b = L.n - 1;
        if (exits) {
            const float yl = (float)(Pf + rlast), yp = (float)(Pf + rprev);
            const int ml = yl < L.cn ? ramp_find<true>(L, yl) - 1 : b, mp = yp < L.cn ? ramp_find<true>(L, yp) - 1 : b;
            b = min(ml, mp + 1);
        }
        fwd = b > j;
        if (fwd) {
            yb = (double)L.c[b];
            Eb = L.E2[b + 1];
            if (b < L.n - 1) Eb = fma((double)L.s[b + 1].y, yb, Eb);
            Ff = fma((double)e.y, Pf, L.E2[j + 1]);
            fwd = !exits || fabs(Eb - Ff) > 1e-14 * fabs(Eb);
        }
        if (!fwd) Pf = yb;
    }
    const double span = fmax(Pb - ya, yb - Pf);
    double sb = 0.0, sf = 0.0;
    // one radius: F at distance r from the destination, gb and gf the slopes of the interval it ends
    auto step = [&](const RampStep& st, double Fb0, double Ff0, double& Fb1, double& Ff1) {
        const double y0 = max_f64(Pb - st.r, ya), y1 = Pf + st.r;
        const bool in1 = y1 < yb;
        const float z0 = (float)y0, z1 = in1 ? (float)y1 : L.c0;
        RampPos p0{0, 1, false}, p1{0, 0, false};
        if (kBack) p0 = ramp_probe<true>(L, z0);
        if (kFwd) p1 = ramp_probe<false>(L, z1);
        if (p0.more || p1.more) {
            if (p0.more) p0.k = ramp_more<true>(L, z0, p0);
            if (p1.more) p1.k = ramp_more<false>(L, z1, p1);
        }
        if (kBack) {
            Fb1 = fma((double)L.s[p0.k - 1].y, y0, -L.E[p0.k]);
            sb = fma(st.sigb, Fb0 - Fb1, sb);
        }
        if (kFwd) {
            const double Fs = fma((double)L.s[p1.k].y, y1, L.E2[p1.k]);
            Ff1 = in1 ? Fs : Eb;
            sf = fma(st.sigf, Ff1 - Ff0, sf);
        }
    };
    int s = 0;
    while (s < nr && Lanes::any(steps[s].r < span)) {  // two radii a round: no copies between them
        double Fb1 = 0.0, Ff1 = 0.0;
        step(steps[s], Fb, Ff, Fb1, Ff1);
        if (++s < nr && Lanes::any(steps[s].r < span)) {
            step(steps[s], Fb1, Ff1, Fb, Ff);
            s++;
        } else {
            Fb = Fb1;
            Ff = Ff1;
            break;
        }
    }
    if (s < nr) {  // the interval in which the last of the lanes ends
        if (kBack) sb = fma(steps[s].sigb, Fb - Fa, sb);
        if (kFwd) sf = fma(steps[s].sigf, Eb - Ff, sf);
    }
    iters += (uint32_t)s;
    return (back ? sb : 0.0) + (fwd ? sf : 0.0);
}

// One direction alone with a row's slopes in an array (the line checks).
template <bool kBack>
CCCS_HD double ramp_one(const RampLine& L, int j, const double* sig, const float* R, int nr, uint32_t& iters) {
    RampStep st[kMaxRadii];
    for (int q = 0; q < nr; q++) st[q] = RampStep{(double)R[q], sig[q], sig[q], 0.0};
    return ramp_walk<kBack, !kBack, RampAlone>(L, j, st, nr, iters);
}
CCCS_HD double ramp_back(const RampLine& L, int j, const double* sig, const double*, const float* R, int nr,
                         uint32_t& iters) {
    return ramp_one<true>(L, j, sig, R, nr, iters);
}
CCCS_HD double ramp_fwd(const RampLine& L, int j, const double* sig, const double*, const float* R, int nr,
                        uint32_t& iters) {
    return ramp_one<false>(L, j, sig, R, nr, iters);
}

// First cell u in [0, nu] whose threshold c0 + u * D exceeds v (nu when none does): an estimate
// from the cell width, corrected against the thresholds themselves (as the table defines them).
CCCS_HD int ramp_cell_after(float c0, float D, float invD, int nu, float v) {
    if (!(D > 0.f)) return v < c0 ? 0 : nu;
    const float g = fminf(fmaxf((v - c0) * invD, -1.f), (float)nu);
    int u = min(max((int)floorf(g) + 1, 0), nu);
    while (u > 0 && c0 + (float)(u - 1) * D > v) u--;
    while (u < nu && !(c0 + (float)u * D > v)) u++;
    return u;
}

// LDS bytes of the cone kernel for lines of up to maxn samples (with the segment-sum arrays).
inline size_t cone_lds_bytes(uint32_t maxn, bool ramp) {
    // (the sequential walk's rows take the place of the lookup table)
    const size_t rows = sizeof(float) * 4 * kMaxRadii;
    if (!ramp) return sizeof(float2) * maxn + rows;
    const size_t n1 = (size_t)maxn + 1, nc = ((size_t)maxn + 4 + 1) & ~(size_t)1;
    return 2 * sizeof(double) * n1 + sizeof(float) * nc + sizeof(float2) * maxn + std::max(sizeof(uint16_t) * (2 * (size_t)maxn + 4), rows);
}

// v moved across lanes by a DPP control; lanes outside the rows of the mask or without a source get 0.
template <int kCtrl, int kRows>
__device__ __forceinline__ double dpp_f64(double v) {
    const uint64_t b = (uint64_t)__double_as_longlong(v);
    const uint32_t lo = (uint32_t)__builtin_amdgcn_update_dpp(0, (int)(uint32_t)b, kCtrl, kRows, 0xf, false);
    const uint32_t hi = (uint32_t)__builtin_amdgcn_update_dpp(0, (int)(uint32_t)(b >> 32), kCtrl, kRows, 0xf, false);
    return __longlong_as_double((long long)(((uint64_t)hi << 32) | lo));
}
// Inclusive prefix sum over the 64 lanes of a wave: three instructions a step and no LDS trip.
__device__ __forceinline__ double wave_incl_sum(double x) {
    x += dpp_f64<0x111, 0xf>(x);  // row_shr 1, 2, 4, 8 (rows of 16 lanes)
    x += dpp_f64<0x112, 0xf>(x);
    x += dpp_f64<0x114, 0xf>(x);
    x += dpp_f64<0x118, 0xf>(x);
    x += dpp_f64<0x142, 0xa>(x);  // row_bcast 15 into rows 1 and 3
    x += dpp_f64<0x143, 0xc>(x);  // row_bcast 31 into rows 2 and 3
    return x;
}
// Workgroup-wide exclusive prefix sums of one or two doubles per thread (NT/64 waves; s_tot holds
// 2 * NT/64 doubles).  Contains barriers: every thread of the workgroup must call it.
template <int NT>
__device__ __forceinline__ void block_excl_sum2(double& v, double& w, double* s_tot) {
    const double x = wave_incl_sum(v), y = wave_incl_sum(w);
    v = dpp_f64<0x138, 0xf>(x);  // wave_shr 1
    w = dpp_f64<0x138, 0xf>(y);
    if (NT == 64) return;
    const int lane = threadIdx.x & 63, wid = threadIdx.x >> 6;
    if (lane == 63) {
        s_tot[2 * wid] = x;
        s_tot[2 * wid + 1] = y;
    }
    __syncthreads();
    for (int q = 0; q < wid; q++) {
        v += s_tot[2 * q];
        w += s_tot[2 * q + 1];
    }
    __syncthreads();
}

// Narrows [t0, t1] to the parameters where o + t*d lies in [lo, hi], for |t| <= 1024 (approximate
// reciprocal: the caller's bounds carry a margin).
__device__ __forceinline__ void keep_slab(float o, float d, float lo, float hi, float& t0, float& t1) {
    if (fabsf(d) < 1e-6f) {
        if (!(o >= lo && o <= hi)) { t0 = 1.f; t1 = 0.f; }
        return;
    }
    const float id = __builtin_amdgcn_rcpf(d), ta = (lo - o) * id, tb = (hi - o) * id;
    t0 = fmaxf(t0, fminf(ta, tb));
    t1 = fminf(t1, fmaxf(ta, tb));
}

// Interior samples [ja, jb] of a stored line (ConeLine).  The margin is far above the rounding of
// the exact per-sample chain and of the affine form (both a few 1e-4 index units at most), so inside it
// the exact test cannot fail and all eight taps exist.
__device__ __forceinline__ void line_interior(const ConeArgs& a, const ConeDev& c, int tY, int tZ, int i0, int len,
                                              int& ja, int& jb) {
    constexpr float m = 0.01f;
    const v3 b0 = c.kinv(mk3(c.rs.x + (float)tZ, c.rs.y, c.rs.z + (float)tY));
    const v3 kd = mk3(c.kinv.m[1], c.kinv.m[4], c.kinv.m[7]);
    const v3 g0 = c.g0 + (float)tY * c.gy + (float)tZ * c.gz;
    float t0 = (float)i0, t1 = (float)(i0 + len - 1);
    keep_slab(b0.x, kd.x, m, a.bev_size.x - m, t0, t1);
    keep_slab(b0.y, kd.y, m, a.bev_size.y - m, t0, t1);
    keep_slab(b0.z, kd.z, m, a.bev_size.z - m, t0, t1);
    keep_slab(g0.x, c.gx.x, a.bb0.x + m, fminf(a.bb1.x, (float)(a.vd.nx - 1)) - m, t0, t1);
    keep_slab(g0.y, c.gx.y, a.bb0.y + m, fminf(a.bb1.y, (float)(a.vd.ny - 1)) - m, t0, t1);
    keep_slab(g0.z, c.gx.z, a.bb0.z + m, fminf(a.bb1.z, (float)(a.vd.nz - 1)) - m, t0, t1);
    ja = len;
    jb = -1;
    // the interior's tap index is formed with 24-bit products: rows below 2^24
    if (!(t0 <= t1) || (int64_t)a.vd.ny * a.vd.nz >= (1 << 24) || a.vd.nx >= (1 << 24)) return;
    ja = (int)ceilf(t0) - i0;
    jb = (int)floorf(t1) - i0;
    if (ja > jb) {
        ja = len;
        jb = -1;
    }
}

__device__ __forceinline__ float lerp1(float a, float b, float t) { return fmaf(t, b - a, a); }

// {density, TERMA} at an interior point (all eight taps inside): four 16-byte loads.
__device__ __forceinline__ float2 interior_pair(const float2* __restrict__ dt, uint32_t nx, uint32_t ny, v3 g) {
    typedef float quad __attribute__((ext_vector_type(4), aligned(8)));
    const float fx = floorf(g.x), fy = floorf(g.y), fz = floorf(g.z);
    const float ax = g.x - fx, ay = g.y - fy, az = g.z - fz;
    const uint32_t row = __umul24((uint32_t)(int)fz, ny) + (uint32_t)(int)fy;
    const float2* p = dt + (__umul24(row, nx) + (uint32_t)(int)fx);
    const size_t sz = (size_t)nx * ny;
    const quad q0 = *reinterpret_cast<const quad*>(p), q1 = *reinterpret_cast<const quad*>(p + nx);
    const quad q2 = *reinterpret_cast<const quad*>(p + sz), q3 = *reinterpret_cast<const quad*>(p + sz + nx);
    float2 r;
    r.x = lerp1(lerp1(lerp1(q0.x, q0.z, ax), lerp1(q1.x, q1.z, ax), ay),
                lerp1(lerp1(q2.x, q2.z, ax), lerp1(q3.x, q3.z, ax), ay), az);
    r.y = lerp1(lerp1(lerp1(q0.y, q0.w, ax), lerp1(q1.y, q1.w, ax), ay),
                lerp1(lerp1(q2.y, q2.w, ax), lerp1(q3.y, q3.w, ax), ay), az);
    return r;
}

// Pass 2: one workgroup (one or more waves) per listed REV line of any cone, in XCD-aware order.  The
// stored interval of the line is resampled (density and TERMA, trilinear) into LDS; then every valid
// sample runs both collapsed-cone walks from LDS and the interval's cone dose is written to the
// compact REV store.  Interior samples take their position as one multiply-add per axis along the
// line and interpolate without tests; the few samples near a face of the crop box or the grid run
// the exact test of cudaRaytrace.  The line's entry, the cone's constants and the radial steps are
// scalar loads.
template <int NT>
__global__ void __launch_bounds__(NT) cone_kernel(ConeArgs a) {
    constexpr int NW = NT / 64;
    extern __shared__ double s_dyn[];
    __shared__ RampStep s_steps[kMaxRadii];
    __shared__ double s_tot[2 * NW];
    __shared__ int s_red[NW][3];
    __shared__ uint32_t s_cnt[NW];
    const uint32_t slot = xcd_chunks(blockIdx.x, gridDim.x, 64);
    if (a.zeros && blockIdx.x == 0 && threadIdx.x < 2 * kLineZeros) a.rev[(int)threadIdx.x - kLineZeros] = 0.f;
    if (a.count && slot >= *a.count) return;
    const uniform_ptr<ConeLine> en = as_uniform(a.list) + slot;
    const uint32_t off = en->off, tyz = en->tyz, seg = en->seg, last = en->last;
    const int i0 = (int)(seg & 1023u), m = (int)(seg >> 10 & 1023u) + 1, ja = (int)(seg >> 20);
    const int jb = (int)(last & 2047u) - 1;
    const uniform_ptr<ConeDev> c = as_uniform(a.cones) + (last >> 11);
    const int tY = (int)(tyz & ((1u << c->tybits) - 1u)), tZ = (int)(tyz >> c->tybits);
    const int rowf = c->rowf;
    const int tid = threadIdx.x, lane = tid & 63, wid = tid >> 6;
    const int nr = a.nradii;
    uint32_t iters = 0;
    // the radial steps go to LDS past the resample, so their latency overlaps the gathers
    const RampStep* my_step = a.steps + ((size_t)rowf * nr + min(tid, nr - 1));
    const double step_r = my_step->r, step_b = my_step->sigb, step_f = my_step->sigf;
    {
        const bool ramp_lds = a.ramp_min <= a.maxn;
        // LDS: [E | E2 | c | line | lb] with the segment-sum arrays, else [line]
        const int n1 = a.maxn + 1, nc = (a.maxn + 5) & ~1;
        double* rE = s_dyn;
        double* rE2 = rE + n1;
        float* rc = reinterpret_cast<float*>(rE2 + n1);
        float2* s_line = ramp_lds ? reinterpret_cast<float2*>(rc + nc) : reinterpret_cast<float2*>(s_dyn);
        uint16_t* rlb = reinterpret_cast<uint16_t*>(s_line + a.maxn);
        float* out = a.rev + off;
        if (a.zeros && tid < 2 * kLineZeros) out[tid < kLineZeros ? tid - kLineZeros : m + tid - kLineZeros] = 0.f;
        // interior (a negative or undefined density makes a sample invalid, as outside)
        bool bad = false;
        if (ja <= jb) {
            const float fY = (float)tY, fZ = (float)tZ;
            const v3 gx = mk3(c->gx.x, c->gx.y, c->gx.z);
            const v3 g0 = mk3(fmaf(fZ, c->gz.x, fmaf(fY, c->gy.x, c->g0.x)), fmaf(fZ, c->gz.y, fmaf(fY, c->gy.y, c->g0.y)),
                              fmaf(fZ, c->gz.z, fmaf(fY, c->gy.z, c->g0.z)));
            for (int j = ja + tid; j <= jb; j += NT) {
                const float t = (float)(i0 + j);
                const float2 dt = interior_pair(a.dt, (uint32_t)a.vd.nx, (uint32_t)a.vd.ny,
                                                mk3(fmaf(t, gx.x, g0.x), fmaf(t, gx.y, g0.y), fmaf(t, gx.z, g0.z)));
                const float h = 0.5f * (a.delr * dt.x);
                bad = bad || !(h >= 0.f);
                s_line[j] = make_float2(h, dt.y);
            }
        }
        const int nbad = __any(bad) ? 1 : 0;  // (per wave)
        // the other samples, exactly; the valid segment is the interior and the valid ones among these
        // (contiguous: the crop box and the calc_bbox are convex)
        int vlo = ja <= jb ? ja : m, vhi = jb, nvalid = 0;
        const int nhead = min(ja, m), nedge = m - (ja <= jb ? jb - ja + 1 : 0);
        if (nedge > 0) {
            m33 kinv;
            for (int q = 0; q < 9; q++) kinv.m[q] = c->kinv.m[q];
            const v3 rs = mk3(c->rs.x, c->rs.y, c->rs.z);
            for (int e0 = 64 * wid; e0 < nedge; e0 += NT) {
                const int e = e0 + lane;
                float2 v = make_float2(-1.f, 0.f);
                if (e < nedge) {
                    const int j = e < nhead ? e : jb + 1 + (e - nhead);
                    const v3 bev = kinv(mk3(rs.x + (float)tZ, rs.y + (float)(i0 + j), rs.z + (float)tY));
                    if (bev.x >= 0.f && bev.y >= 0.f && bev.z >= 0.f && bev.x < a.bev_size.x && bev.y < a.bev_size.y &&
                        bev.z < a.bev_size.z) {
                        const v3 g = a.binv(bev) + a.off;
                        if (g.x >= a.bb0.x && g.x < a.bb1.x && g.y >= a.bb0.y && g.y < a.bb1.y && g.z >= a.bb0.z &&
                            g.z < a.bb1.z) {
                            const float2 dt = tex3_pair(a.dt, a.vd.nx, a.vd.ny, a.vd.nz, g.x + 0.5f, g.y + 0.5f, g.z + 0.5f);
                            v.x = 0.5f * (a.delr * dt.x);
                            v.y = dt.y;
                        }
                    }
                    s_line[j] = v;
                }
                // (j rises with e, so the first and the last valid lane give the extremes)
                const uint64_t ok = __ballot(v.x >= 0.f);
                if (ok) {
                    const int ef = e0 + __builtin_ctzll(ok), el = e0 + 63 - __builtin_clzll(ok);
                    vlo = min(vlo, ef < nhead ? ef : jb + 1 + (ef - nhead));
                    vhi = max(vhi, el < nhead ? el : jb + 1 + (el - nhead));
                    nvalid += __popcll(ok);
                }
            }
        }
        nvalid -= nbad;
        if (tid < nr) {
            s_steps[tid].r = step_r;
            s_steps[tid].sigb = step_b;
            s_steps[tid].sigf = step_f;
        }
        if (NW > 1 && lane == 0) {
            s_red[wid][0] = vlo;
            s_red[wid][1] = vhi;
            s_red[wid][2] = nvalid;
        }
        __syncthreads();
        if (NW > 1) {
            vlo = s_red[0][0];
            vhi = s_red[0][1];
            nvalid = s_red[0][2];
            for (int w = 1; w < NW; w++) {
                vlo = min(vlo, s_red[w][0]);
                vhi = max(vhi, s_red[w][1]);
                nvalid += s_red[w][2];
            }
        }
        nvalid += m - nedge;  // (below the segment's length where the interior has an invalid sample)
        vlo = __builtin_amdgcn_readfirstlane(vlo);
        vhi = __builtin_amdgcn_readfirstlane(vhi);
        nvalid = __builtin_amdgcn_readfirstlane(nvalid);
        const float nphi_f = (float)a.nphi;
        for (int j = tid; j < m; j += NT)
            if (j < vlo || j > vhi) out[j] = 0.f;
        const int n = vhi - vlo + 1;
        if (n >= a.ramp_min && nvalid == n) {
            const float2* sv = s_line + vlo;
            // radiological centres (FP64 scan), then the two FP64 prefix sums and the lookup table, one
            // chunk of samples per thread; a sample's neighbours roll through registers
            const int per = (n + NT - 1) / NT;
            const int ca = min(n, tid * per), cb = min(n, ca + per);
            double P = 0.0, unused = 0.0;
            for (int k = ca; k < cb; k++) P += 2.0 * (double)sv[k].x;
            block_excl_sum2<NT>(P, unused, s_tot);
            double e1 = 0.0, e2 = 0.0;
            const float tfirst = ca > 0 && ca < cb ? sv[ca - 1].y : 0.f;
            {
                float tp = tfirst;
                float2 e = ca < cb ? sv[ca] : make_float2(0.f, 0.f);
                for (int k = ca; k < cb; k++) {
                    const float2 nx = k + 1 < n ? sv[k + 1] : make_float2(0.f, 0.f);
                    const float ck = (float)(P + (double)e.x);
                    rc[k] = ck;
                    P += 2.0 * (double)e.x;
                    e1 = fma((double)e.y - (double)tp, (double)ck, e1);
                    e2 = fma((double)e.y - (double)nx.y, (double)ck, e2);
                    tp = e.y;
                    e = nx;
                }
            }
            if (tid < 4) rc[n + tid] = INFINITY;  // lookups probe past n
            block_excl_sum2<NT>(e1, e2, s_tot);
            __syncthreads();
            // lookup table: lb[u] = first k with c_k >= c0 + u * D, U = 2n cells over [c0, c_{n-1}]
            RampLine L;
            L.c = rc;
            L.E = rE;
            L.E2 = rE2;
            L.s = sv;
            L.lb = rlb;
            L.n = n;
            L.U = 2 * n;
            L.c0 = rc[0];
            L.cn = rc[n - 1];
            const float range = L.cn - L.c0;
            L.invD = ramp_cells(L.c0, L.cn, L.U);
            const float D = L.invD > 0.f ? range / (float)L.U : 0.f;
            // sample k owns the cells whose threshold lies in (c_{k-1}, c_k] (c_{-1} = -inf, c_n =
            // +inf): each of the U + 2 entries is written by exactly one sample, the two past them by the
            // last chunk (a lookup may round one cell up)
            if (ca < cb) {
                float tp = tfirst;
                float2 e = sv[ca];
                int u = ca == 0 ? 0 : ramp_cell_after(L.c0, D, L.invD, L.U + 2, rc[ca - 1]);
                for (int k = ca; k < cb; k++) {
                    const float2 nx = k + 1 < n ? sv[k + 1] : make_float2(0.f, 0.f);
                    const float ck = rc[k];
                    rE[k] = e1;
                    rE2[k] = e2;
                    e1 = fma((double)e.y - (double)tp, (double)ck, e1);
                    e2 = fma((double)e.y - (double)nx.y, (double)ck, e2);
                    const int u1 = ramp_cell_after(L.c0, D, L.invD, L.U + 2, ck);
                    for (; u < u1; u++) rlb[u] = (uint16_t)k;
                    tp = e.y;
                    e = nx;
                }
                if (cb == n) {
                    rE[n] = e1;
                    rE2[n] = e2;
                    for (; u < L.U + 4; u++) rlb[u] = (uint16_t)n;
                }
            }
            __syncthreads();
            for (int j = tid; j < n; j += NT)
                out[vlo + j] = (float)ramp_walk<true, true, RampWave>(L, j, s_steps, nr, iters) / nphi_f;
        } else {
            // short segments: the sequential walk, its rows in LDS past the line
            float* sR = reinterpret_cast<float*>(s_line + a.maxn);
            float *sIW = sR + kMaxRadii, *sF = sIW + kMaxRadii, *sB = sF + kMaxRadii;
            if (tid < nr) {
                const float* K = a.tables;
                const float* R = a.tables + (size_t)a.ntheta * nr;
                sR[tid] = R[tid];
                sIW[tid] = R[nr + tid];
                sF[tid] = K[(size_t)rowf * nr + tid];
                sB[tid] = K[(size_t)(a.ntheta - 1 - rowf) * nr + tid];
            }
            __syncthreads();
            for (int base = vlo; base <= vhi; base += NT) {
                const int j = base + tid;
                const bool act = j <= vhi && s_line[min(j, vhi)].x >= 0.f;
                const float v = walk_both(s_line, min(j, vhi), vlo, vhi, sR, sIW, sF, sB, nr, act, iters);
                if (j <= vhi) out[j] = act ? v / nphi_f : 0.f;
            }
        }
    }
    // (empty lines' slots are zeroed by the class-list pass)
    if (a.counts) {
        const size_t line = (size_t)c->line0 + (uint32_t)tZ * (uint32_t)c->ny + (uint32_t)tY;
        for (int o = 32; o > 0; o >>= 1) iters += __shfl_xor(iters, o, 64);
        if (NW == 1) {
            if (tid == 0) a.counts[line] = iters;
        } else {
            if (lane == 0) s_cnt[wid] = iters;
            __syncthreads();
            if (tid == 0) {
                uint32_t t = 0;
                for (int w = 0; w < NW; w++) t += s_cnt[w];
                a.counts[line] = t;
            }
        }
    }
}

constexpr int kPvcsGroup = 4;

struct PvcsArgs {
    const ConeDev* cones;
    const LineMeta* lines;
    const float* rev;
    float* dose;
    int q0, q1;                 // cones of this pass
    int nx, ny;                 // full volume dims (x, y)
    int x0, y0, z0, sx, sy, sz; // PVCS index box
    int tx, ty, tz;             // tiles per axis
    m33 bfwd;                   // BEV <- PVCS rotation (index units)
    v3 off;                     // BEV origin in PVCS index units
    v3 bev_lo, bev_hi;          // dilated crop box (BEV index units)
};

// One lane per PVCS voxel, 16x4x4 voxel tiles in XCD-aware order, each wave a 4x4x4 cube of the
// tile: the gathers are bound by the number of different cache lines per load, and the cones run in
// every direction, so the shape with the least projected area (24 voxels on average, against 42 for a
// 16x4x1 slab) touches the fewest REV lines.  Voxels outside the dilated
// crop box receive nothing from any cone and leave at once; the others sum every cone's trilinear
// REV dose (compact store, REV2XYZdose's fetch) in a register and add it to the dose volume once.
template <bool kZeros>
__global__ void __launch_bounds__(256) pvcs_kernel(PvcsArgs a) {
    const int tid = threadIdx.x;
    const uint32_t tile = xcd_chunks(blockIdx.x, gridDim.x, 64);
    const int txi = (int)(tile % (uint32_t)a.tx);
    const int tyi = (int)((tile / (uint32_t)a.tx) % (uint32_t)a.ty);
    const int tzi = (int)(tile / ((uint32_t)a.tx * (uint32_t)a.ty));
    const int X = txi * 16 + (tid >> 6) * 4 + (tid & 3), Y = tyi * 4 + ((tid >> 2) & 3), Z = tzi * 4 + ((tid >> 4) & 3);
    if (X >= a.sx || Y >= a.sy || Z >= a.sz) return;
    const int gx = a.x0 + X, gy = a.y0 + Y, gz = a.z0 + Z;
    const v3 g = mk3((float)gx, (float)gy, (float)gz);
    const v3 bv = a.bfwd(g - a.off);
    if (!(bv.x >= a.bev_lo.x && bv.y >= a.bev_lo.y && bv.z >= a.bev_lo.z && bv.x < a.bev_hi.x && bv.y < a.bev_hi.y &&
          bv.z < a.bev_hi.z))
        return;
    // Cones in groups of kPvcsGroup: the line-table loads of a group are issued together, then its
    // REV loads (branch-free: taps outside a line's stored interval read sample 0 of the store and
    // are replaced by zero), so each lane keeps several dependent gathers in flight.  The
    // arithmetic per cone is rev_fetch's and the sum runs in cone order.  The voxel's dose is read
    // first so that its latency overlaps the gathers (this lane alone writes the voxel).
    float* dst = a.dose + ((size_t)gx + (size_t)a.nx * ((size_t)gy + (size_t)a.ny * gz));
    const float old = *dst;
    float sum = 0.f;
    if constexpr (kZeros) {
        // Lines end in zeros: no test of a sample against its line, and of the lines only the upper
        // neighbours may lie outside the grid (the voxel does not lie below it).  Half the instructions
        // of the general form below; per pass 174 -> 152 us (thorax beam), 118 -> 107 us (128^3 water),
        // 206 -> 200 us (256x256x180 request) and 12 -> 7 us (32^3 water).
        const char* rev0 = reinterpret_cast<const char*>(a.rev - kLineZeros);
        for (int q0 = a.q0; q0 < a.q1; q0 += kPvcsGroup) {
            pair_meta m0[kPvcsGroup], m1[kPvcsGroup];
            float fa[kPvcsGroup], fb[kPvcsGroup], fc[kPvcsGroup];
            int di[kPvcsGroup];
            bool ok[kPvcsGroup], row[kPvcsGroup], plane[kPvcsGroup];
#pragma unroll
            for (int u = 0; u < kPvcsGroup; u++) {
                const uniform_ptr<ConeDev> c = as_uniform(a.cones) + min(q0 + u, a.q1 - 1);
                m33 ca;
                for (int w = 0; w < 9; w++) ca.m[w] = c->a.m[w];
                const int nx = c->nx, ny = c->ny, nz = c->nz;
                const v3 r = ca(g) + mk3(c->t.x, c->t.y, c->t.z);
                const float ub = (r.y + 0.5f) - 0.5f, vb = (r.z + 0.5f) - 0.5f, wb = (r.x + 0.5f) - 0.5f;
                ok[u] = q0 + u < a.q1 && r.x >= 0.f && r.y >= 0.f && r.z >= 0.f && r.y < (float)nx && r.z < (float)ny &&
                        r.x < (float)nz && ub < (float)nx && vb < (float)ny && wb < (float)nz;
                const float fu = floorf(ub), fv = floorf(vb), fw = floorf(wb);
                di[u] = (int)fu;
                fa[u] = ub - fu;
                fb[u] = vb - fv;
                fc[u] = wb - fw;
                // (lanes outside the cone's grid load its first records with the others)
                const int j = ok[u] ? (int)fv : 0, k = ok[u] ? (int)fw : 0;
                row[u] = j + 1 < ny;
                plane[u] = k + 1 < nz;
                const char* base = reinterpret_cast<const char*>(a.lines + c->line0);
                const uint32_t l = mad24((uint32_t)k, (uint32_t)ny, (uint32_t)j) * (uint32_t)sizeof(LineMeta);
                m0[u] = *reinterpret_cast<const pair_meta*>(base + l);
                m1[u] = *reinterpret_cast<const pair_meta*>(base + (l + (plane[u] ? (uint32_t)ny * (uint32_t)sizeof(LineMeta) : 0u)));
            }
#pragma unroll
            for (int u = 0; u < kPvcsGroup; u++) {
                if (!ok[u]) continue;
                if (!row[u]) m0[u].z = m0[u].w = m1[u].z = m1[u].w = 0u;  // (an empty line)
                const float t0 = line_lerp(rev0, m0[u].x, m0[u].y, di[u], fa[u]);
                const float t1 = line_lerp(rev0, m0[u].z, m0[u].w, di[u], fa[u]);
                const float t2 = line_lerp(rev0, m1[u].x, m1[u].y, di[u], fa[u]);
                const float t3 = line_lerp(rev0, m1[u].z, m1[u].w, di[u], fa[u]);
                const float e0 = t0 + fb[u] * (t1 - t0), e1 = t2 + fb[u] * (t3 - t2);
                sum += e0 + fc[u] * ((plane[u] ? e1 : 0.f) - e0);
            }
        }
        if (sum != 0.f) *dst = old + sum;
        return;
    }
    for (int q0 = a.q0; q0 < a.q1; q0 += kPvcsGroup) {
        LineMeta mt[kPvcsGroup][4];
        float fa[kPvcsGroup], fb[kPvcsGroup], fc[kPvcsGroup];
        int di[kPvcsGroup];
        bool ok[kPvcsGroup];
#pragma unroll
        for (int u = 0; u < kPvcsGroup; u++) {
            ok[u] = false;
            di[u] = 0;
            fa[u] = fb[u] = fc[u] = 0.f;
#pragma unroll
            for (int t = 0; t < 4; t++) mt[u][t] = LineMeta{0u, 0, 0};
            const int q = q0 + u;
            if (q >= a.q1) continue;
            const uniform_ptr<ConeDev> c = as_uniform(a.cones) + q;
            m33 ca;
            for (int w = 0; w < 9; w++) ca.m[w] = c->a.m[w];
            const int nx = c->nx, ny = c->ny, nz = c->nz;
            const v3 r = ca(g) + mk3(c->t.x, c->t.y, c->t.z);
            if (r.y >= (float)nx || r.z >= (float)ny || r.x >= (float)nz || r.x < 0.f || r.y < 0.f || r.z < 0.f)
                continue;
            const float ub = (r.y + 0.5f) - 0.5f, vb = (r.z + 0.5f) - 0.5f, wb = (r.x + 0.5f) - 0.5f;
            if (!(ub > -1.f && vb > -1.f && wb > -1.f && ub < (float)nx && vb < (float)ny && wb < (float)nz))
                continue;
            const float fu = floorf(ub), fv = floorf(vb), fw = floorf(wb);
            ok[u] = true;
            di[u] = (int)fu;
            fa[u] = ub - fu;
            fb[u] = vb - fv;
            fc[u] = wb - fw;
            meta_pairs(a.lines, c->line0, ny, nz, (int)fv, (int)fw, mt[u]);
        }
#pragma unroll
        for (int u = 0; u < kPvcsGroup; u++) {
            if (!ok[u]) continue;
            float tv[4];
#pragma unroll
            for (int t = 0; t < 4; t++) tv[t] = rev_lerp(a.rev, mt[u][t], di[u], fa[u]);
            const float e0 = tv[0] + fb[u] * (tv[1] - tv[0]);
            const float e1 = tv[2] + fb[u] * (tv[3] - tv[2]);
            sum += e0 + fc[u] * (e1 - e0);
        }
    }
    if (sum != 0.f) *dst = old + sum;
}

// Interleaves density and TERMA over the CT grid for the cone kernel's paired fetch; TERMA is 0
// outside the calc_bbox, which is what the bbox-bounded TERMA fetch returns there.
__global__ void __launch_bounds__(256) pack_dt_kernel(const float* __restrict__ dens, const float* __restrict__ terma,
                                                      int nx, int ny, int nz, int bx0, int by0, int bz0, int bx, int by,
                                                      int bz, float2* __restrict__ out) {
    const int x = blockIdx.x * 64 + threadIdx.x, y = blockIdx.y * 4 + threadIdx.y, z = blockIdx.z;
    if (x >= nx || y >= ny) return;
    const size_t v = (size_t)x + (size_t)nx * ((size_t)y + (size_t)ny * z);
    const int tx = x - bx0, ty = y - by0, tz = z - bz0;
    const float t = (tx >= 0 && ty >= 0 && tz >= 0 && tx < bx && ty < by && tz < bz)
                        ? terma[(size_t)tx + (size_t)bx * ((size_t)ty + (size_t)by * tz)]
                        : 0.f;
    out[v] = make_float2(dens[v], t);
}

// ---- structure projection onto fluence maps (preprocess: findFluenceProjection + cudaRaycast,
// dosecalc-preprocess/cudaMemFunctions.cu:308-393, kernels.cuh:136-224) ---------------------------
struct ProjBeam {
    v3 src, iso;
    Rot2 inv;         // FCS -> PVCS (inverseRotateBeamAtOriginRHS)
    int fx, fy;       // fluence map size
    float bsx, bsy;   // beamlet size [cm]
    uint32_t off;     // first beamlet of this beam in the output
};

// Mask bytes to floats, and the index box {lo xyz, hi xyz} of the non-zero voxels (initialised by the
// caller to {INT_MAX, -1}).  Four voxels per thread and step.
__global__ void __launch_bounds__(256) mask_to_float_kernel(const uint8_t* __restrict__ m, float* __restrict__ f, size_t n,
                                                            int nx, int ny, int* __restrict__ box) {
    int lo[3] = {INT32_MAX, INT32_MAX, INT32_MAX}, hi[3] = {-1, -1, -1};
    const size_t n4 = (n + 3) / 4;
    for (size_t q = (size_t)blockIdx.x * 256 + threadIdx.x; q < n4; q += (size_t)gridDim.x * 256) {
        uint32_t w = 0;
        if (4 * q + 4 <= n) {
            w = reinterpret_cast<const uint32_t*>(m)[q];
            reinterpret_cast<float4*>(f)[q] =
                make_float4((float)(w & 255u), (float)(w >> 8 & 255u), (float)(w >> 16 & 255u), (float)(w >> 24));
        } else {
            for (size_t i = 4 * q; i < n; i++) {
                f[i] = (float)m[i];
                w |= (uint32_t)m[i] << (8 * (i - 4 * q));
            }
        }
        for (int e = 0; w != 0u; e++, w >>= 8) {
            if (!(w & 255u)) continue;
            const size_t i = 4 * q + (size_t)e, row = i / (size_t)nx;
            const int c[3] = {(int)(i - row * (size_t)nx), (int)(row % (size_t)ny), (int)(row / (size_t)ny)};
            for (int k = 0; k < 3; k++) {
                lo[k] = min(lo[k], c[k]);
                hi[k] = max(hi[k], c[k]);
            }
        }
    }
    for (int k = 0; k < 3; k++) {
        for (int o = 32; o > 0; o >>= 1) {
            lo[k] = min(lo[k], __shfl_xor(lo[k], o, 64));
            hi[k] = max(hi[k], __shfl_xor(hi[k], o, 64));
        }
        // (only what moves the box: thousands of waves would queue at six words, 46 us against 32)
        if ((threadIdx.x & 63) == 0 && hi[k] >= 0) {
            if (lo[k] < __hip_atomic_load(box + k, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT)) atomicMin(box + k, lo[k]);
            if (hi[k] > __hip_atomic_load(box + 3 + k, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT)) atomicMax(box + 3 + k, hi[k]);
        }
    }
}

// True if the path integral of a ray over the mask is positive: siddon_march's segments (its planes in
// its order), ended at the first segment with a positive contribution.  The mask is not negative and
// neither is its interpolation, so the sum of the segments can only grow.  A segment's taps can be
// non-zero only if its midpoint lies within half a voxel cell of the mask's box; the midpoint
// parameters for which it does form one interval [t0, t1] (widened far beyond the rounding of the
// coordinates), so the others cost no fetch, and the march ends behind the interval.
__device__ __forceinline__ bool mask_ray_hit(v3 sink, const VolDesc& vd, v3 ivoxel, v3 src, const float* __restrict__ mask,
                                             const int* __restrict__ box) {
    const v3 diff = sink - src, startdiff = vd.start - src, enddiff = vd.end - src;
    const float ax0 = (startdiff.x - 0.5f * vd.voxel.x) / diff.x, ax1 = (enddiff.x + 0.5f * vd.voxel.x) / diff.x;
    const float ay0 = (startdiff.y - 0.5f * vd.voxel.y) / diff.y, ay1 = (enddiff.y + 0.5f * vd.voxel.y) / diff.y;
    const float az0 = (startdiff.z - 0.5f * vd.voxel.z) / diff.z, az1 = (enddiff.z + 0.5f * vd.voxel.z) / diff.z;
    const float a_min = fmaxf(0.f, fmaxf(fmaxf(fminf(ax0, ax1), fminf(ay0, ay1)), fminf(az0, az1)));
    const float a_max = fminf(1.f, fminf(fminf(fmaxf(ax0, ax1), fmaxf(ay0, ay1)), fmaxf(az0, az1)));
    if (a_min >= a_max) return false;
    float t0 = 0.f, t1 = 1.f;
    const v3 o = (src - vd.start) * ivoxel, dd = diff * ivoxel;
    const float oc[3] = {o.x, o.y, o.z}, dc[3] = {dd.x, dd.y, dd.z};
    for (int k = 0; k < 3; k++) {
        const float m = 0.05f + 4e-6f * (fabsf(oc[k]) + fabsf(dc[k]));
        const float ta = ((float)box[k] - 0.5f - m - oc[k]) / dc[k], tb = ((float)box[3 + k] + 1.5f + m - oc[k]) / dc[k];
        t0 = fmaxf(t0, fminf(ta, tb));
        t1 = fminf(t1, fmaxf(ta, tb));
    }
    if (t0 > t1) return false;
    const float d12 = len3(diff);
    const float step_x = fabsf(vd.voxel.x / diff.x), step_y = fabsf(vd.voxel.y / diff.y), step_z = fabsf(vd.voxel.z / diff.z);
    float alpha = a_min, ax = a_min, ay = a_min, az = a_min;
    int iter = 0;
    while (alpha < a_max && !(alpha > t1) && ++iter < 5000) {
        // (the planes of one step: siddon_rpl)
        const float m0 = fminf(fminf(ax, ay), az);
        if (!(m0 < 1.0f)) break;
        if (ax == m0) ax += step_x;
        const float m1 = fminf(fminf(ax, ay), az);
        const bool ty = ay == m1 && m1 < 1.0f;
        if (ty) ay += step_y;
        const float m2 = fminf(fminf(ax, ay), az);
        const bool tz = az == m2 && m2 < 1.0f;
        if (tz) az += step_z;
        const float nextalpha = tz ? m2 : (ty ? m1 : m0);
        const float inter = fabsf(d12 * (nextalpha - alpha));
        const float am = (nextalpha + alpha) * 0.5f;
        if (inter >= 0.001f && am >= t0 && am <= t1) {
            const v3 f = div_by(mk3(src.x + am * diff.x - vd.start.x, src.y + am * diff.y - vd.start.y,
                                    src.z + am * diff.z - vd.start.z), vd.voxel, ivoxel);
            if (inter * tex3_border(mask, vd.nx, vd.ny, vd.nz, f.x, f.y, f.z) > 0.f) return true;
        }
        alpha = nextalpha;
    }
    return false;
}

// Nine sub-rays per beamlet of any beam (offsets -1/0/+1 half beamlets along each fluence axis) run
// from the source to three times the source-to-cell distance through the trilinearly sampled mask with
// the TERMA path's Siddon planes; the beamlet is 1 when any sub-ray accumulates a positive path
// integral.  A workgroup takes 64 beamlets, each of its nine waves one sub-ray of them: with one lane
// per beamlet the rays ran one after another and a 64-beam set filled one wave per SIMD.  With the
// fetches and the march held to the mask's box: 5270 -> 145 us (64 beams of 40x40 beamlets, 200x200x160
// mask).  What is left is the planes of the rays up to the box, a serial chain.
constexpr int kSubRays = 9;
__global__ void __launch_bounds__(64 * kSubRays) projection_kernel(const float* __restrict__ mask, VolDesc vd, v3 ivoxel,
                                                        const int* __restrict__ box, const ProjBeam* __restrict__ beams,
                                                        int nbeams, uint32_t block0, uint32_t total,
                                                        float* __restrict__ out) {
    __shared__ uint32_t s_hit[64];
    const int lane = threadIdx.x & 63, sr = threadIdx.x >> 6;
    const uint32_t t = (block0 + blockIdx.x) * 64 + lane;
    if (sr == 0) s_hit[lane] = 0u;
    __syncthreads();
    if (t < total && box[3] >= 0) {
        int lo = 0, hi = nbeams - 1;
        while (lo < hi) {
            const int mid = (lo + hi + 1) >> 1;
            if (beams[mid].off <= t) lo = mid; else hi = mid - 1;
        }
        const ProjBeam& b = beams[lo];
        const int pix = (int)(t - b.off);
        const int rx = pix % b.fx, rz = pix / b.fx;
        const int sx = sr % 3 - 1, sz = sr / 3 - 1;
        const v3 fcs = mk3(b.bsx * ((float)rx + 0.5f * (float)sx - (float)b.fx * 0.5f + 0.5f), 0.f,
                           b.bsy * ((float)rz + 0.5f * (float)sz - (float)b.fy * 0.5f + 0.5f));
        v3 ctr = rot_inv(b.inv, fcs) + b.iso;
        ctr = ctr + 1e-9f;
        const v3 sd = ctr - b.src;
        const v3 sink = b.src + 3.f * sd;
        if (mask_ray_hit(sink, vd, ivoxel, b.src, mask, box)) s_hit[lane] = 1u;
    }
    __syncthreads();
    if (sr == 0 && t < total) out[t] = s_hit[lane] ? 1.f : 0.f;
}

// ---- fluence-map convolution (the FCBB lateral step; no reference source) --------------------
// out[y][x] = sum_j sum_i K[j][i] * F[y - (j - kh/2)][x - (i - kw/2)], zero outside the map, the
// terms added j outer, i inner.  One lane per output of a 16x16 tile; the tile plus its halo and
// the kernel sit in LDS.  The sum is one chain per lane, in order, so a row of the kernel is unrolled
// (KW taps, every odd width up to 31): its LDS reads are under way together instead of one round trip
// per tap (20 maps of 64x64, 15x15 kernel: 12.8 -> 7.9 us).
constexpr int kConvTile = 16, kConvMaxK = 31;

template <int KW>
__global__ void __launch_bounds__(256) fluence_conv_kernel(const float* __restrict__ f, int w, int h,
                                                           const float* __restrict__ k, int kh, float* __restrict__ out) {
    constexpr int kw = KW;
    __shared__ float s_k[kConvMaxK * kConvMaxK];
    // rows 48 apart: a wave's four rows of 16 outputs then read 64 different banks
    constexpr int stride = 48;
    static_assert(kConvTile + kConvMaxK - 1 <= stride, "row of the tile");
    __shared__ float s_f[(kConvTile + kConvMaxK - 1) * stride];
    const int map = blockIdx.z;
    const float* F = f + (size_t)map * w * h;
    const int x0 = blockIdx.x * kConvTile, y0 = blockIdx.y * kConvTile;
    const int rx = kw / 2, ry = kh / 2;
    const int sw = kConvTile + kw - 1, sh = kConvTile + kh - 1;
    const int tid = threadIdx.x;
    // s_f[v][u] = F[y0 + ry - v][x0 + rx - u]: the flipped window, so output (tx, ty) reads
    // s_f[ty + j][tx + i] for kernel tap (i, j); four loads of a lane are under way together, with the
    // kernel's
    const float k0 = tid < kw * kh ? k[tid] : 0.f;
    for (int q0 = 0; q0 < sw * sh; q0 += 4 * 256) {
        float r[4];
#pragma unroll
        for (int e = 0; e < 4; e++) {
            const int q = q0 + 256 * e + tid, v = q / sw, u = q - v * sw;
            const int xx = x0 + (kConvTile - 1) - u + rx, yy = y0 + (kConvTile - 1) - v + ry;
            r[e] = (q < sw * sh && xx >= 0 && yy >= 0 && xx < w && yy < h) ? F[(size_t)yy * w + xx] : 0.f;
        }
#pragma unroll
        for (int e = 0; e < 4; e++)
            if (const int q = q0 + 256 * e + tid; q < sw * sh) s_f[q / sw * stride + q % sw] = r[e];
    }
    if (tid < kw * kh) s_k[tid] = k0;
    for (int q = 256 + tid; q < kw * kh; q += 256) s_k[q] = k[q];
    __syncthreads();
    const int tx = tid % kConvTile, ty = tid / kConvTile;
    const int x = x0 + tx, y = y0 + ty;
    if (x >= w || y >= h) return;
    // output (x, y) needs F[y - j + ry][x - i + rx] = s_f[(kConvTile-1-ty) + j][(kConvTile-1-tx) + i]
    const int bu = kConvTile - 1 - tx, bv = kConvTile - 1 - ty;
    float acc = 0.f;
    for (int j = 0; j < kh; j++) {
        float a[KW], b[KW];
#pragma unroll
        for (int i = 0; i < KW; i++) {
            a[i] = s_k[j * kw + i];
            b[i] = s_f[(bv + j) * stride + bu + i];
        }
#pragma unroll
        for (int i = 0; i < KW; i++) acc += a[i] * b[i];
    }
    out[(size_t)map * w * h + (size_t)y * w + x] = acc;
}

template <int KW>
void launch_conv(int kw, dim3 grid, hipStream_t st, const float* f, int w, int h, const float* k, int kh, float* out) {
    if constexpr (KW <= kConvMaxK) {
        if (kw == KW) hipLaunchKernelGGL(fluence_conv_kernel<KW>, grid, dim3(256), 0, st, f, w, h, k, kh, out);
        else launch_conv<KW + 2>(kw, grid, st, f, w, h, k, kh, out);
    }
}

__global__ void add_kernel(float* __restrict__ dst, const float* __restrict__ src, size_t n) {
    for (size_t i = (size_t)blockIdx.x * blockDim.x + threadIdx.x; i < n; i += (size_t)gridDim.x * blockDim.x) dst[i] += src[i];
}

// ------------------------------------------------------------------------------------------------
// host pipeline

namespace {

inline size_t bbox_voxels(const cccs_ctx* ctx) {
    return (size_t)ctx->prob.bbox_size[0] * ctx->prob.bbox_size[1] * ctx->prob.bbox_size[2];
}
inline size_t vol_voxels(const cccs_ctx* ctx) {
    return (size_t)ctx->prob.size[0] * ctx->prob.size[1] * ctx->prob.size[2];
}

TermaArgs terma_args(cccs_ctx* ctx, const cccs_beam& b, const float* d_fmap, float* d_terma, int beamletnum) {
    TermaArgs a;
    a.terma = d_terma;
    a.fmap = d_fmap;
    a.dens = ctx->d_dens;
    a.vd = ctx->vol;
    a.beam = make_beam_dev(b);
    a.spec = ctx->spec;
    a.bx = (int)ctx->prob.bbox_size[0]; a.by = (int)ctx->prob.bbox_size[1]; a.bz = (int)ctx->prob.bbox_size[2];
    a.ox = (int)ctx->prob.bbox_start[0]; a.oy = (int)ctx->prob.bbox_start[1]; a.oz = (int)ctx->prob.bbox_start[2];
    a.ss = std::max(1u, ctx->prob.ss_factor);
    a.bhc = ctx->prob.beamhard_correct;
    a.beamletnum = beamletnum;
    a.counts = nullptr;
    a.block0 = 0;
    const v3 dir = a.beam.iso - a.beam.src;
    const float dc[3] = {dir.x, dir.y, dir.z};
    a.depth = 2;
    for (int k = 1; k >= 0; k--)
        if (std::fabs(dc[k]) > std::fabs(dc[a.depth])) a.depth = k;
    a.far_first = dc[a.depth] > 0.f;
    // the map's cone, where the beam's direction is the y axis of its frame as for beams made here
    const v3 y = rot2(a.beam.beam_fwd, a.beam.dir_n);
    const float hx = 0.5f * (float)a.beam.fmx * a.beam.bsx, hz = 0.5f * (float)a.beam.fmy * a.beam.bsy;
    a.field2 = std::fabs(y.x) < 1e-3f && std::fabs(y.z) < 1e-3f && a.beam.iso_dist > 0.f
                   ? 1.01f * (hx * hx + hz * hz) / (a.beam.iso_dist * a.beam.iso_dist)
                   : INFINITY;
    return a;
}

int launch_terma(cccs_ctx* ctx, const TermaArgs& a0) {
    const uint64_t blocks = terma_blocks(a0);
    if (blocks > 0x7fffffffULL) return set_error(CCCS_EGEOM, "calc_bbox too large");
    TermaArgs a = a0;
    a.counts = prof_counter(ctx, blocks);
    const double nbb = (double)a.bx * a.by * a.bz;
    const double nct = (double)a.vd.nx * a.vd.ny * a.vd.nz;
    int tok = prof_begin(ctx, K_TERMA);
    const auto kernel = a.ss > 1 ? (a.counts ? terma_kernel<true, true> : terma_kernel<true, false>)
                                 : (a.counts ? terma_kernel<false, true> : terma_kernel<false, false>);
    // (LDS it does not use bounds the workgroups of a CU)
    const size_t lds = (size_t)(160 * 1024 / kTermaResident - 256);
    terma_launches(a, [&](dim3 grid) { hipLaunchKernelGGL(kernel, grid, dim3(256), lds, ctx->stream, a); });
    prof_end(ctx, tok, 4.0 * nct + 4.0 * nbb, 0.0, (uint64_t)nbb);
    CCCS_HIP(hipGetLastError());
    return CCCS_OK;
}

const float* angle_cache_lookup(const cccs_ctx* ctx, const cccs_beam& b);

// TERMA from the resident unit-TERMA grid of the beam's source (angle cache).
int launch_terma_from_unit(cccs_ctx* ctx, const TermaArgs& a, const float* unit) {
    dim3 blk(64, 4, 1), grd((a.bx + 63) / 64, (a.by + 3) / 4, a.bz);
    const double nbb = (double)a.bx * a.by * a.bz;
    int tok = prof_begin(ctx, K_TERMA_CACHED);
    hipLaunchKernelGGL(terma_from_unit_kernel, grd, blk, 0, ctx->stream, a, unit);
    prof_end(ctx, tok, 8.0 * nbb, 0.0, (uint64_t)nbb);
    CCCS_HIP(hipGetLastError());
    return CCCS_OK;
}

// Crop box + REV grids (nvbbRayConvolve_host.cu:429-587), from the reduced extent.
int beam_geometry(cccs_ctx* ctx, const cccs_beam& b, const float* red, BeamGeom& g) {
    const cccs_problem& p = ctx->prob;
    // the reference starts max at FLT_MIN and min at FLT_MAX (:436-437)
    v3 bmin = mk3(std::min(red[0], FLT_MAX), std::min(red[1], FLT_MAX), std::min(red[2], FLT_MAX));
    v3 bmax = mk3(std::max(red[3], FLT_MIN), std::max(red[4], FLT_MIN), std::max(red[5], FLT_MIN));
    if (red[6] < 0.5f) return set_error(CCCS_EGEOM, "beam has no non-zero TERMA inside the calc_bbox");
    bmin.x -= p.penumbra / p.rev_latspacing;
    bmin.y -= p.penumbra / p.rev_longspacing;
    bmin.z -= p.penumbra / p.rev_latspacing;
    bmax.x += p.penumbra / p.rev_latspacing;
    bmax.y += p.penumbra / p.rev_longspacing;
    bmax.z += p.penumbra / p.rev_latspacing;
    float sx = std::ceil(std::fabs(bmax.x - bmin.x)), sy = std::ceil(std::fabs(bmax.y - bmin.y)),
          sz = std::ceil(std::fabs(bmax.z - bmin.z));
    if (!(sx >= 1.f && sx < 1000.f && sy >= 1.f && sy < 1000.f && sz >= 1.f && sz < 1000.f))
        return set_error(CCCS_EGEOM, "BEV crop box size out of range (0, 1000)");
    g.bev_size[0] = (uint32_t)sx; g.bev_size[1] = (uint32_t)sy; g.bev_size[2] = (uint32_t)sz;
    g.bev_min = bmin;
    g.bev_max = bmax;
    dm33 binv = dm_beam_inv(b.azimuth, b.zenith, b.coll);
    v3 tmin = rot2(rot2_beam_inv(b.azimuth, b.zenith, b.coll), bmin);
    g.lim_min = mk3(p.start[0] + (tmin.x + (float)p.bbox_start[0]) * p.voxel[0],
                    p.start[1] + (tmin.y + (float)p.bbox_start[1]) * p.voxel[1],
                    p.start[2] + (tmin.z + (float)p.bbox_start[2]) * p.voxel[2]);
    // REV grid per cone: bounding box of the rotated crop box (cm), sized in spacing units
    v3 lim = mk3(sx * p.rev_latspacing, sy * p.rev_longspacing, sz * p.rev_latspacing);
    g.nrays = ctx->nrays;
    g.total_lines = 0;
    g.total_rev = 0;
    for (int r = 0; r < ctx->nrays; r++) {
        float th = ctx->theta[r] * 3.14159265358979323846f / 180.f;
        float ph = ctx->phi[r] * 3.14159265358979323846f / 180.f;
        Rot2 kf = rot2_kernel_fwd(th, ph);
        v3 mn = mk3(FLT_MAX, FLT_MAX, FLT_MAX), mx = mk3(FLT_MIN, FLT_MIN, FLT_MIN);
        for (int c = 0; c < 8; c++) {
            v3 in = mk3(lim.x * (float)(c & 1), lim.y * (float)((c >> 1) & 1), lim.z * (float)((c >> 2) & 1));
            v3 o = rot2(kf, in);
            if (o.x < mn.x) mn.x = o.x;
            if (o.y < mn.y) mn.y = o.y;
            if (o.z < mn.z) mn.z = o.z;
            if (o.x > mx.x) mx.x = o.x;
            if (o.y > mx.y) mx.y = o.y;
            if (o.z > mx.z) mx.z = o.z;
        }
        uint32_t n0 = (uint32_t)std::ceil(std::fabs(mx.y - mn.y) / p.rev_longspacing);
        uint32_t n1 = (uint32_t)std::ceil(std::fabs(mx.z - mn.z) / p.rev_latspacing);
        uint32_t n2 = (uint32_t)std::ceil(std::fabs(mx.x - mn.x) / p.rev_latspacing);
        if (n0 > ctx->max_rev_beam[0] || n1 > ctx->max_rev_beam[1] || n2 > ctx->max_rev_beam[2])
            return set_error(CCCS_EGEOM, "REV grid exceeds max_rev_size (ArraySizeError)");
        if (n0 > (uint32_t)kMaxLine) return set_error(CCCS_EGEOM, "REV line longer than 1024 samples");
        g.rev_min[r] = mn;
        g.rev_size[r][0] = n0; g.rev_size[r][1] = n1; g.rev_size[r][2] = n2;
        g.total_lines += (uint64_t)n1 * n2;
        g.total_rev += (uint64_t)n0 * n1 * n2;
    }
    // PVCS index box reachable from the crop box dilated by 2 index units (trilinear support of
    // a REV sample is within sqrt(3) of it), clamped to the calc_bbox
    v3 off = mk3((g.lim_min.x - p.start[0]) / p.voxel[0], (g.lim_min.y - p.start[1]) / p.voxel[1],
                 (g.lim_min.z - p.start[2]) / p.voxel[2]);
    double lo[3] = {1e30, 1e30, 1e30}, hi[3] = {-1e30, -1e30, -1e30};
    for (int c = 0; c < 8; c++) {
        v3 cb = mk3((c & 1) ? sx + 2.f : -2.f, ((c >> 1) & 1) ? sy + 2.f : -2.f, ((c >> 2) & 1) ? sz + 2.f : -2.f);
        v3 q = dm_apply_f(binv, cb) + off;
        lo[0] = std::min(lo[0], (double)q.x); lo[1] = std::min(lo[1], (double)q.y); lo[2] = std::min(lo[2], (double)q.z);
        hi[0] = std::max(hi[0], (double)q.x); hi[1] = std::max(hi[1], (double)q.y); hi[2] = std::max(hi[2], (double)q.z);
    }
    for (int k = 0; k < 3; k++) {
        long l0 = (long)std::floor(lo[k]) - 1, h0 = (long)std::ceil(hi[k]) + 2;
        long b0 = (long)p.bbox_start[k], b1 = b0 + (long)p.bbox_size[k];
        g.pvcs_lo[k] = (int)std::max(b0, std::min(b1, l0));
        g.pvcs_hi[k] = (int)std::max(b0, std::min(b1, h0));
    }
    return CCCS_OK;
}

// Device and host scratch of one full-beam dose computation: the context's grow-only buffers, or,
// for the no-allocation entry point, consecutive 256-byte aligned pieces of the library's fixed
// device array with host staging on the caller's stack.
struct BeamScratch {
    cccs_ctx* ctx = nullptr;
    char* arena = nullptr;          // fixed device array, or nullptr: the context's buffers
    size_t cap = 0, used = 0;
    float* host_small = nullptr;    // >= 64 bytes of host staging
    ConeDev* host_cones = nullptr;  // kMaxRays entries of host staging
    int get(DevBuf& buf, size_t bytes, void** out) {
        if (!arena) {
            CCCS_TRY(buf.ensure(bytes));
            *out = buf.p;
            return CCCS_OK;
        }
        const size_t at = (used + 255) & ~size_t(255);
        if (bytes > cap || at > cap - bytes)
            return set_error(CCCS_ENOMEM, "beam needs more than the " + std::to_string(cap >> 20) +
                                              " MiB fixed scratch of the no-allocation entry point");
        used = at + bytes;
        *out = arena + at;
        return CCCS_OK;
    }
    template <class T>
    int get(DevBuf& buf, size_t count, T** out) {
        void* v = nullptr;
        CCCS_TRY(get(buf, sizeof(T) * std::max<size_t>(1, count), &v));
        *out = static_cast<T*>(v);
        return CCCS_OK;
    }
};

// Scratch from the context's own (allocating) buffers.
int context_scratch(cccs_ctx* ctx, BeamScratch& S) {
    S = BeamScratch();
    S.ctx = ctx;
    CCCS_TRY(ctx->h_small.ensure(64));
    CCCS_TRY(ctx->h_cones.ensure(sizeof(ConeDev) * kMaxRays));
    S.host_small = ctx->h_small.as<float>();
    S.host_cones = ctx->h_cones.as<ConeDev>();
    return CCCS_OK;
}

// `before_wait` (may be empty) enqueues work that needs the TERMA alone, before the host waits.
int run_crop(BeamScratch& S, const float* d_terma, const cccs_beam& b, float* red_host,
             const std::function<int()>& before_wait) {
    cccs_ctx* ctx = S.ctx;
    float* part = nullptr;
    const size_t used = S.used;
    CCCS_TRY(S.get(ctx->partial, kCropBlocks * 8 + 8, &part));
    S.used = used;  // the partials are read back below: what follows in a fixed array takes their place
    Rot2 rot = rot2_beam_fwd(b.azimuth, b.zenith, b.coll);
    const cccs_problem& p = ctx->prob;
    size_t n = bbox_voxels(ctx);
    int blocks = (int)std::min<size_t>(kCropBlocks, (n + 255) / 256);
    // the result goes straight to pinned host memory (the fixed array's caller has none)
    float* out = S.arena ? part + kCropBlocks * 8 : S.host_small;
    int tok = prof_begin(ctx, K_CROP);
    hipLaunchKernelGGL(crop_partial_kernel, dim3(blocks), dim3(256), 0, ctx->stream, d_terma, (int)p.bbox_size[0],
                       (int)p.bbox_size[1], (int)p.bbox_size[2], rot, part);
    hipLaunchKernelGGL(crop_final_kernel, dim3(1), dim3(256), 0, ctx->stream, part, blocks, out);
    prof_end(ctx, tok, 4.0 * (double)n, 0.0, n);
    CCCS_HIP(hipGetLastError());
    if (S.arena)
        CCCS_HIP(hipMemcpyAsync(S.host_small, out, 7 * sizeof(float), hipMemcpyDeviceToHost, ctx->stream));
    if (before_wait) CCCS_TRY(before_wait());
    CCCS_HIP(hipStreamSynchronize(ctx->stream));
    std::memcpy(red_host, S.host_small, 7 * sizeof(float));
    return CCCS_OK;
}

// ---- line table and per-class line lists ---------------------------------------------------------
// The cone kernel runs one launch per stored-length class (LDS sized for the class's longest line).
// Each launch takes the list of its own lines, in line order, so that no workgroup is spent on an
// empty line or on a line of another class.  Three passes: the stored interval of every line with the
// stored samples and class counts of every 1024 lines, one workgroup that turns those into offsets
// (seven passes, of 3 to 23 us each, when intervals, offsets and lists had their own), and the
// lines' offsets and list entries.
constexpr int kClassBlock = 1024;
constexpr int kClassCols = kConeClasses + 1;  // lines per class, stored samples

struct ClassArgs {
    int hi[kConeClasses];  // longest stored line of each class (ascending)
    int ncls;
    uint32_t* bcnt;        // [blocks][kClassCols]: counts, then the blocks' offsets (classes: in their list)
    uint32_t* tot;         // [kClassCols]: lines per class, stored samples
    uint32_t* host;        // the same in pinned host memory, or nullptr
    ConeLine* list;        // the lines' entries, class by class
    uint32_t* counts;      // profiling: the slots of empty lines are zeroed here (or nullptr)
};

__device__ __forceinline__ int class_of_line(const ClassArgs& a, int len) {
    if (len <= 0) return -1;
    for (int c = 0; c < a.ncls - 1; c++)
        if (len <= a.hi[c]) return c;
    return a.ncls - 1;
}

__global__ void __launch_bounds__(kClassBlock) line_interval_kernel(ConeArgs ca, ClassArgs a) {
    __shared__ uint32_t s[kClassBlock / 64][kClassCols];
    const uint64_t i = (uint64_t)blockIdx.x * kClassBlock + threadIdx.x;
    int len = 0;
    if (i < ca.nlines) {
        const ConeDev& c = ca.cones[cone_of_line(ca.cones, ca.ncones, i)];
        const uint32_t l = (uint32_t)(i - c.line0), tz = l / (uint32_t)c.ny, ty = l - tz * (uint32_t)c.ny;
        int i0, i1;
        line_interval(ca, c, (int)ty, (int)tz, i0, i1);
        len = (int)(int16_t)(i1 - i0);
        ca.lines[i] = LineMeta{0u, (int16_t)i0, (int16_t)len};
    }
    const int cls = class_of_line(a, len);
    if (a.counts && i < ca.nlines && cls < 0) a.counts[i] = 0;
    const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
    for (int c = 0; c < kConeClasses; c++) {
        const uint64_t m = __ballot(cls == c);
        if (lane == 0) s[w][c] = (uint32_t)__popcll(m);
    }
    uint32_t sum = (uint32_t)len + (ca.zeros && len > 0 ? (uint32_t)kLineZeros : 0u);
    for (int o = 32; o > 0; o >>= 1) sum += __shfl_xor(sum, o, 64);
    if (lane == 0) s[w][kConeClasses] = sum;
    __syncthreads();
    if (threadIdx.x < kClassCols) {
        uint32_t t = 0;
        for (int q = 0; q < kClassBlock / 64; q++) t += s[q][threadIdx.x];
        a.bcnt[(size_t)blockIdx.x * kClassCols + threadIdx.x] = t;
    }
}

// One workgroup: exclusive scan of the block counts, column by column.
__global__ void __launch_bounds__(kClassBlock) class_scan_kernel(ClassArgs a, uint32_t nb) {
    __shared__ uint32_t s[kClassCols][kClassBlock / 64];
    const int t = threadIdx.x, lane = t & 63, w = t >> 6;
    uint32_t carry[kClassCols] = {};
    for (uint32_t b0 = 0; b0 < nb; b0 += kClassBlock) {
        uint32_t* row = a.bcnt + (size_t)(b0 + t) * kClassCols;
        uint32_t v[kClassCols], inc[kClassCols];
#pragma unroll
        for (int q = 0; q < kClassCols; q++) v[q] = b0 + t < nb ? row[q] : 0u;
#pragma unroll
        for (int q = 0; q < kClassCols; q++) {
            inc[q] = wave_incl_u32(v[q]);
            if (lane == 63) s[q][w] = inc[q];
        }
        __syncthreads();
#pragma unroll
        for (int q = 0; q < kClassCols; q++) {
            uint32_t before = 0, total = 0;
            for (int k = 0; k < kClassBlock / 64; k++) {
                before += k < w ? s[q][k] : 0u;
                total += s[q][k];
            }
            if (b0 + t < nb) row[q] = carry[q] + before + inc[q] - v[q];
            carry[q] += total;
        }
        __syncthreads();
    }
#pragma unroll
    for (int q = 0; q < kClassCols; q++)
        if (t == q) {
            a.tot[q] = carry[q];
            if (a.host) a.host[q] = carry[q];
        }
}

__global__ void __launch_bounds__(kClassBlock) class_scatter_kernel(ClassArgs a, ConeArgs ca) {
    __shared__ uint32_t s[kClassBlock / 64][kClassCols];
    const uint64_t i = (uint64_t)blockIdx.x * kClassBlock + threadIdx.x;
    LineMeta meta{};
    if (i < ca.nlines) meta = ca.lines[i];
    const int cls = class_of_line(a, meta.len);
    const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
    const uint64_t below = (uint64_t(1) << lane) - 1;
    const uint32_t pad = ca.zeros && meta.len > 0 ? (uint32_t)kLineZeros : 0u, take = (uint32_t)meta.len + pad;
    const uint32_t inc = wave_incl_u32(take);
    if (lane == 63) s[w][kConeClasses] = inc;
    uint32_t rank = 0;
    for (int c = 0; c < kConeClasses; c++) {
        const uint64_t m = __ballot(cls == c);
        if (lane == 0) s[w][c] = (uint32_t)__popcll(m);
        if (cls == c) rank = (uint32_t)__popcll(m & below);
    }
    __syncthreads();
    const uint32_t* block = a.bcnt + (size_t)blockIdx.x * kClassCols;
    meta.off = block[kConeClasses] + inc - take + pad;
    for (int q = 0; q < w; q++) meta.off += s[q][kConeClasses];
    if (ca.zeros && meta.len <= 0) meta.off = 0u;
    if (i < ca.nlines) ca.lines[i] = meta;
    if (cls >= 0) {
        uint32_t off = block[cls] + rank;
        for (int c = 0; c < cls; c++) off += a.tot[c];
        for (int q = 0; q < w; q++) off += s[q][cls];
        const int q = cone_of_line(ca.cones, ca.ncones, i);
        const ConeDev& c = ca.cones[q];
        const uint32_t l = (uint32_t)(i - c.line0), tz = l / (uint32_t)c.ny, ty = l - tz * (uint32_t)c.ny;
        int ja, jb;
        line_interior(ca, c, (int)ty, (int)tz, meta.i0, meta.len, ja, jb);
        ConeLine e;
        e.off = meta.off;
        e.tyz = ty | tz << c.tybits;
        e.seg = (uint32_t)meta.i0 | (uint32_t)(meta.len - 1) << 10 | (uint32_t)ja << 20;
        e.last = (uint32_t)(jb + 1) | (uint32_t)q << 11;
        a.list[off] = e;
    }
}

void launch_cone(int threads, dim3 grid, size_t lds, hipStream_t st, const ConeArgs& ca) {
    switch (threads) {
        case 256: hipLaunchKernelGGL(cone_kernel<256>, grid, dim3(256), lds, st, ca); break;
        case 128: hipLaunchKernelGGL(cone_kernel<128>, grid, dim3(128), lds, st, ca); break;
        default: hipLaunchKernelGGL(cone_kernel<64>, grid, dim3(64), lds, st, ca); break;
    }
}

// Everything after TERMA: geometry, cones, PVCS accumulation into d_dose.
int run_cones(BeamScratch& S, const cccs_beam& b, const float* d_terma, float* d_dose, BeamGeom* gout) {
    cccs_ctx* ctx = S.ctx;
    float red[7];
    const size_t nvox = vol_voxels(ctx);
    float2* d_dt = nullptr;
    auto pack = [&]() -> int {
        const cccs_problem& p = ctx->prob;
        dim3 blk(64, 4, 1), grd((unsigned)((p.size[0] + 63) / 64), (unsigned)((p.size[1] + 3) / 4), p.size[2]);
        hipLaunchKernelGGL(pack_dt_kernel, grd, blk, 0, ctx->stream, (const float*)ctx->d_dens, d_terma,
                           (int)p.size[0], (int)p.size[1], (int)p.size[2], (int)p.bbox_start[0],
                           (int)p.bbox_start[1], (int)p.bbox_start[2], (int)p.bbox_size[0], (int)p.bbox_size[1],
                           (int)p.bbox_size[2], d_dt);
        CCCS_HIP(hipGetLastError());
        return CCCS_OK;
    };
    // the interleaved volume needs the TERMA alone: it is packed while the host waits for the crop box
    // (the fixed array's pieces keep their order)
    const bool pack_early = d_dose && !S.arena && nvox < (size_t(1) << 31);
    if (pack_early) CCCS_TRY(S.get(ctx->dt, nvox, &d_dt));
    CCCS_TRY(run_crop(S, d_terma, b, red, pack_early ? std::function<int()>(pack) : std::function<int()>()));
    BeamGeom g;
    CCCS_TRY(beam_geometry(ctx, b, red, g));
    if (gout) *gout = g;
    if (!d_dose) return CCCS_OK;
    const cccs_problem& p = ctx->prob;
    if (g.total_lines > 0x7fffffffULL || g.total_rev > 0xffffffffULL)
        return set_error(CCCS_EGEOM, "REV grids exceed 2^32 samples");
    ConeDev* d_cones = nullptr;
    LineMeta* d_lines = nullptr;
    CCCS_TRY(S.get(ctx->cones, kMaxRays, &d_cones));
    CCCS_TRY(S.get(ctx->lines, g.total_lines + 2 * kRevPad, &d_lines));
    d_lines += kRevPad;
    ConeDev* hc = S.host_cones;
    dm33 bfwd = dm_beam_fwd(b.azimuth, b.zenith, b.coll);
    dm33 binv = dm_beam_inv(b.azimuth, b.zenith, b.coll);
    v3 rv = mk3(p.rev_latspacing, p.rev_longspacing, p.rev_latspacing);
    v3 off = mk3((g.lim_min.x - p.start[0]) / p.voxel[0], (g.lim_min.y - p.start[1]) / p.voxel[1],
                 (g.lim_min.z - p.start[2]) / p.voxel[2]);
    uint64_t line0 = 0;
    const int half = (int)p.ntheta / 2;
    for (int r = 0; r < g.nrays; r++) {
        float th = ctx->theta[r] * 3.14159265358979323846f / 180.f;
        float ph = ctx->phi[r] * 3.14159265358979323846f / 180.f;
        dm33 kf = dm_kernel_fwd(th, ph), ki = dm_kernel_inv(th, ph);
        ConeDev& c = hc[r];
        c.kinv = to_f(ki);
        dm33 a = dm_mul(kf, bfwd);
        c.a = to_f(a);
        c.rs = mk3(g.rev_min[r].x / rv.x, g.rev_min[r].y / rv.y, g.rev_min[r].z / rv.z);
        // REV coordinate of PVCS index 0: a * (-off) - rs
        v3 t0 = dm_apply_f(a, mk3(-off.x, -off.y, -off.z));
        c.t = mk3(t0.x - c.rs.x, t0.y - c.rs.y, t0.z - c.rs.z);
        c.nx = (int)g.rev_size[r][0];
        c.ny = (int)g.rev_size[r][1];
        c.nz = (int)g.rev_size[r][2];
        c.rowf = r % half;
        c.line0 = line0;
        c.tybits = 0;
        while ((uint64_t(1) << c.tybits) < (uint64_t)c.ny) c.tybits++;
        line0 += (uint64_t)c.ny * c.nz;
        // PVCS index along the grid's axes (lines run along REV y, tY counts along z, tZ along x)
        dm33 gm = dm_mul(binv, ki);
        c.g0 = dm_apply_f(gm, c.rs) + off;
        c.gx = mk3((float)gm.m[1], (float)gm.m[4], (float)gm.m[7]);
        c.gy = mk3((float)gm.m[2], (float)gm.m[5], (float)gm.m[8]);
        c.gz = mk3((float)gm.m[0], (float)gm.m[3], (float)gm.m[6]);
    }
    CCCS_HIP(hipMemcpyAsync(d_cones, hc, sizeof(ConeDev) * g.nrays, hipMemcpyHostToDevice, ctx->stream));
    // the host staging may be the caller's stack (no-allocation entry point): the copy completes first
    if (S.arena) CCCS_HIP(hipStreamSynchronize(ctx->stream));
    if (nvox >= (size_t(1) << 31)) return set_error(CCCS_EGEOM, "CT grid beyond 2^31 voxels");
    if (!pack_early) CCCS_TRY(S.get(ctx->dt, nvox, &d_dt));
    ConeArgs ca;
    ca.list = nullptr;
    ca.dt = d_dt;
    ca.tables = ctx->d_tables;
    ca.steps = ctx->d_steps;
    ca.cones = d_cones;
    ca.lines = d_lines;
    ca.rev = nullptr;
    // (the zeros take two samples a line: not from the fixed array, and not where indices would overflow)
    ca.zeros = !S.arena && g.total_rev + (uint64_t)kLineZeros * g.total_lines + 2 * kRevPad < (uint64_t(1) << 30);
    for (int r = 0; r < g.nrays; r++)
        ca.zeros = ca.zeros && g.rev_size[r][1] < (1u << 20) && g.rev_size[r][2] < (1u << 20) &&
                   (uint64_t)g.rev_size[r][1] * g.rev_size[r][2] < (uint64_t(1) << 28);
    ca.nlines = g.total_lines;
    ca.ncones = g.nrays;
    ca.ntheta = (int)p.ntheta;
    ca.nradii = (int)p.nradii;
    ca.nphi = (int)p.nphi;
    ca.delr = p.rev_longspacing;
    ca.counts = nullptr;
    ca.vd = ctx->vol;
    ca.binv = to_f(binv);
    ca.off = off;
    ca.bev_size = mk3((float)g.bev_size[0], (float)g.bev_size[1], (float)g.bev_size[2]);
    ca.bb0 = ldu3(p.bbox_start);
    ca.bb1 = ca.bb0 + ldu3(p.bbox_size);
    if (g.total_lines == 0) return CCCS_OK;
    if (!pack_early) CCCS_TRY(pack());
    // stored-length classes: one launch each, with LDS for the class's longest line, so that the
    // many short lines are not held to the occupancy of the longest
    uint32_t maxn = 1;
    for (int r = 0; r < g.nrays; r++) maxn = std::max(maxn, g.rev_size[r][0]);
    int cls_hi[kConeClasses], cls_threads[kConeClasses], ncls = 0;
    for (int ci = 0, lo = 1; ci < kConeClasses && lo <= (int)maxn; ci++) {
        const int hi = ci == kConeClasses - 1 ? (int)maxn : std::min<int>(ctx->sched.cone_class_len[ci], (int)maxn);
        if (hi < lo) continue;
        cls_hi[ncls] = hi;
        cls_threads[ncls] = ctx->sched.cone_class_threads[ci];
        ncls++;
        lo = hi + 1;
    }
    ca.counts = prof_counter(ctx, g.total_lines);
    ClassArgs cl;
    for (int c = 0; c < kConeClasses; c++) cl.hi[c] = c < ncls ? cls_hi[c] : 0;
    cl.ncls = ncls;
    cl.counts = ca.counts;
    const uint64_t ncb = (g.total_lines + kClassBlock - 1) / kClassBlock;
    CCCS_TRY(S.get(ctx->cls_cnt, (size_t)ncb * kClassCols + kClassCols, &cl.bcnt));
    cl.tot = cl.bcnt + (size_t)ncb * kClassCols;
    // The launches and the store are sized from the totals on the host.  Small beams take the bounds
    // instead; their cone launch reads its count on the device.  The wait costs 10 to 12 us at every size
    // measured (8 to 48 cones on grids of 16^3 to 64^3, 2500 to 115000 lines of up to 96 samples: 97 against 87 us
    // the smallest, 338 against 327 the largest); the bounds below keep the empty workgroups below 32768 and the
    // store, dense, at 64 MiB.
    const bool wait = S.arena || ctx->prof.on || ncls != 1 || g.total_lines > 32768 || g.total_rev > (uint64_t(1) << 24);
    uint32_t* totals = reinterpret_cast<uint32_t*>(S.host_small + 8);
    cl.host = wait && !S.arena ? totals : nullptr;
    CCCS_TRY(S.get(ctx->cls_list, g.total_lines, &cl.list));
    hipLaunchKernelGGL(line_interval_kernel, dim3((unsigned)ncb), dim3(kClassBlock), 0, ctx->stream, ca, cl);
    hipLaunchKernelGGL(class_scan_kernel, dim3(1), dim3(kClassBlock), 0, ctx->stream, cl, (uint32_t)ncb);
    hipLaunchKernelGGL(class_scatter_kernel, dim3((unsigned)ncb), dim3(kClassBlock), 0, ctx->stream, cl, ca);
    CCCS_HIP(hipGetLastError());
    uint32_t cls_n[kConeClasses] = {};
    uint64_t stored = g.total_rev + (ca.zeros ? (uint64_t)kLineZeros * g.total_lines : 0);
    ca.count = nullptr;
    if (wait) {
        if (S.arena)
            CCCS_HIP(hipMemcpyAsync(totals, cl.tot, sizeof(uint32_t) * kClassCols, hipMemcpyDeviceToHost, ctx->stream));
        CCCS_HIP(hipStreamSynchronize(ctx->stream));
        std::memcpy(cls_n, totals, sizeof(cls_n));
        stored = totals[kConeClasses];
    } else {
        cls_n[0] = (uint32_t)g.total_lines;
        ca.count = cl.tot;
    }
    CCCS_TRY(S.get(ctx->rev, stored + 2 * kRevPad, &ca.rev));
    ca.rev += kRevPad;
    // pass 2: per-line resample + walks into the compact store, one workgroup per listed line
    ca.ramp_min = ctx->sched.cone_ramp_min;
    int tok = prof_begin(ctx, K_CONE);
    uint64_t list_off = 0;
    for (int c = 0; c < ncls; c++) {
        if (cls_n[c] == 0) continue;
        ca.maxn = cls_hi[c];
        ca.list = cl.list + list_off;
        list_off += cls_n[c];
        const size_t lds = cone_lds_bytes((uint32_t)ca.maxn, ca.ramp_min <= ca.maxn);
        launch_cone(cls_threads[c], dim3(cls_n[c]), lds, ctx->stream, ca);
        CCCS_HIP(hipGetLastError());
    }
    const uint64_t lines = (uint64_t)cls_n[0] + cls_n[1] + cls_n[2] + cls_n[3];
    if (ca.zeros) stored -= (uint64_t)kLineZeros * lines;
    // algorithmic traffic: density + TERMA in, cone dose out, per stored sample
    prof_end(ctx, tok, 12.0 * (double)stored, 0.0, stored);
    if (ca.zeros && lines == 0) return CCCS_OK;  // (nothing wrote the zeros that the short form reads)
    PvcsArgs pa;
    pa.cones = d_cones;
    pa.lines = ca.lines;
    pa.rev = ca.rev;
    pa.dose = d_dose;
    pa.nx = (int)p.size[0];
    pa.ny = (int)p.size[1];
    pa.x0 = g.pvcs_lo[0]; pa.y0 = g.pvcs_lo[1]; pa.z0 = g.pvcs_lo[2];
    pa.sx = g.pvcs_hi[0] - g.pvcs_lo[0]; pa.sy = g.pvcs_hi[1] - g.pvcs_lo[1]; pa.sz = g.pvcs_hi[2] - g.pvcs_lo[2];
    if (pa.sx > 0 && pa.sy > 0 && pa.sz > 0) {
        pa.tx = (pa.sx + 15) / 16;
        pa.ty = (pa.sy + 3) / 4;
        pa.tz = (pa.sz + 3) / 4;
        pa.bfwd = to_f(bfwd);
        pa.off = off;
        // a voxel gets dose only within the trilinear support (< sqrt(3) index units) of a stored
        // sample, and stored samples lie inside the crop box
        pa.bev_lo = mk3(-2.f, -2.f, -2.f);
        pa.bev_hi = mk3((float)g.bev_size[0] + 2.f, (float)g.bev_size[1] + 2.f, (float)g.bev_size[2] + 2.f);
        const uint64_t tiles = (uint64_t)pa.tx * pa.ty * pa.tz;
        if (tiles > 0xffffffffULL) return set_error(CCCS_EGEOM, "PVCS box too large");
        const double nbox = (double)pa.sx * pa.sy * pa.sz;
        // cones in passes: the REV data the resident tiles gather at a time then belongs to fewer
        // cones (better L2 / Infinity Cache reuse); each pass adds its cones' dose to the volume.
        // Automatic (0): as many cones per pass as keep a pass's REV data within 128 MB (measured
        // on the 256x256x180 serving requests, ~31 MB per cone: 4 cones per pass -20 %; small plans
        // stay in one pass, where extra passes only add launches)
        int per = ctx->sched.pvcs_pass_cones;
        if (per <= 0) {
            const double cone_bytes = 4.0 * (double)stored / std::max(1, g.nrays);
            per = (int)std::min<double>(g.nrays, std::max(1.0, std::floor(128.0 * 1048576.0 / std::max(cone_bytes, 1.0))));
        }
        // (LDS that the short form does not use bounds the waves whose lines share a CU's cache: 152
        // against 178 us a pass for the thorax beam)
        const size_t lds = ca.zeros ? (size_t)(160 * 1024 / 6 - 256) : 0;
        int tk = prof_begin(ctx, K_PVCS);
        for (pa.q0 = 0; pa.q0 < g.nrays; pa.q0 += per) {
            pa.q1 = std::min(g.nrays, pa.q0 + per);
            hipLaunchKernelGGL(ca.zeros ? pvcs_kernel<true> : pvcs_kernel<false>, dim3((unsigned)tiles), dim3(256), lds,
                               ctx->stream, pa);
        }
        // algorithmic traffic: every stored sample read once, the box's dose read and written once
        prof_end(ctx, tk, 4.0 * (double)stored + 8.0 * nbox, 0.0, (uint64_t)nbox);
        CCCS_HIP(hipGetLastError());
    }
    return CCCS_OK;
}

int upload_fmap(cccs_ctx* ctx, const cccs_beam& b, const float* host_fmap, const float** d_out) {
    size_t n = (size_t)b.fmap_size[0] * b.fmap_size[1];
    CCCS_TRY(ctx->fmap.ensure(n * sizeof(float)));
    // synchronous copy: the host buffer may be reused by the caller right after the call
    CCCS_HIP(hipStreamSynchronize(ctx->stream));
    CCCS_HIP(hipMemcpy(ctx->fmap.p, host_fmap, n * sizeof(float), hipMemcpyHostToDevice));
    *d_out = ctx->fmap.as<float>();
    return CCCS_OK;
}

}  // namespace

int beam_dose_scratch(BeamScratch& S, const cccs_beam& b, const float* d_fmap, float* d_dose) {
    cccs_ctx* ctx = S.ctx;
    CCCS_TRY(check_beam(ctx, b));
    float* d_terma = nullptr;
    CCCS_TRY(S.get(ctx->terma, bbox_voxels(ctx), &d_terma));
    TermaArgs ta = terma_args(ctx, b, d_fmap, d_terma, -1);
    if (const float* unit = angle_cache_lookup(ctx, b)) CCCS_TRY(launch_terma_from_unit(ctx, ta, unit));
    else CCCS_TRY(launch_terma(ctx, ta));
    return run_cones(S, b, d_terma, d_dose, nullptr);
}

// Shared by the C-ABI entry points below and by the beamlet path.
int beam_dose_one(cccs_ctx* ctx, const cccs_beam& b, const float* d_fmap, float* d_dose) {
    BeamScratch S;
    CCCS_TRY(context_scratch(ctx, S));
    return beam_dose_scratch(S, b, d_fmap, d_dose);
}

}  // namespace cccs

// ---- angle cache: resident unit TERMA per beam source -------------------------------------------
// The unit-fluence TERMA of a full-beam dose depends on the beam's source and SAD (the Siddon
// march and the inverse square) and on the problem (density, spectrum, grids), not on the fluence
// map or the collimator.  An optimiser asks for beams from a fixed candidate set, so each
// candidate source's unit TERMA over the calc_bbox can stay in HBM; a request's TERMA is then the
// voxel's fluence times that entry, bit-identical to the march (the direct path multiplies in the
// same order).
struct cccs_angle_cache {
    int device = 0;
    uint32_t size[3] = {0, 0, 0}, bbox_start[3] = {0, 0, 0}, bbox_size[3] = {0, 0, 0};
    float voxel[3] = {0, 0, 0}, start[3] = {0, 0, 0};
    float bhc = 1.f;
    uint64_t dens_hash = 0;
    cccs::SpecDev spec{};
    size_t nbbox = 0;
    float* data = nullptr;  // one calc_bbox grid per entry
    std::map<std::array<uint32_t, 4>, size_t> index;  // (source bits, SAD bits) -> entry
};

namespace cccs {
namespace {
std::array<uint32_t, 4> angle_key(const cccs_beam& b) {
    std::array<uint32_t, 4> k;
    std::memcpy(&k[0], &b.source[0], 4);
    std::memcpy(&k[1], &b.source[1], 4);
    std::memcpy(&k[2], &b.source[2], 4);
    std::memcpy(&k[3], &b.sad, 4);
    return k;
}

bool cache_fits(const cccs_ctx* ctx, const cccs_angle_cache* c) {
    const cccs_problem& p = ctx->prob;
    for (int k = 0; k < 3; k++)
        if (c->size[k] != p.size[k] || c->bbox_start[k] != p.bbox_start[k] || c->bbox_size[k] != p.bbox_size[k] ||
            c->voxel[k] != p.voxel[k] || c->start[k] != p.start[k])
            return false;
    if (c->bhc != p.beamhard_correct || c->dens_hash != ctx->dens_hash || c->device != ctx->device) return false;
    return std::memcmp(&c->spec, &ctx->spec, sizeof(SpecDev)) == 0;
}

const float* angle_cache_lookup(const cccs_ctx* ctx, const cccs_beam& b) {
    const cccs_angle_cache* c = ctx->angle_cache;
    if (!c || ctx->prob.ss_factor > 1) return nullptr;
    auto it = c->index.find(angle_key(b));
    return it == c->index.end() ? nullptr : c->data + it->second * c->nbbox;
}
}  // namespace

// ---- fixed scratch of the no-allocation entry point ----------------------------------------------
// The full-beam path's device scratch (TERMA, interleaved density/TERMA, line table, scan partials,
// cone constants, compact REV store) for callers that cannot allocate: one array per GPU, held
// until the process ends.  Host code uses the per-device address from hipGetSymbolAddress, never
// the array's name.
constexpr size_t kNoAllocScratchBytes = size_t(256) << 20;
static __device__ __align__(256) unsigned char scratch[kNoAllocScratchBytes];

namespace {
constexpr int kMaxDevices = 64;
std::mutex g_scratch_mu;
void* g_scratch_ptr[kMaxDevices] = {};
}  // namespace

int noalloc_scratch_init(int device) {
    if (device < 0 || device >= kMaxDevices) return set_error(CCCS_EINVAL, "device ordinal beyond 64");
    std::lock_guard<std::mutex> lk(g_scratch_mu);
    if (g_scratch_ptr[device]) return CCCS_OK;
    void* ptr = nullptr;
    const hipError_t e = hipGetSymbolAddress(&ptr, HIP_SYMBOL(scratch));
    if (e != hipSuccess || !ptr)
        return set_error(CCCS_EDEVICE, std::string("hipGetSymbolAddress(scratch): ") + hipGetErrorString(e));
    g_scratch_ptr[device] = ptr;
    return CCCS_OK;
}

}  // namespace cccs

using namespace cccs;

// =================================================================================================
// C-ABI

extern "C" int cccs_angle_cache_create(cccs_ctx* ctx, const cccs_beam* beams, int nbeams, uint64_t max_bytes,
                                      cccs_angle_cache** out) {
    clear_error();
    if (!ctx || !out || (!beams && nbeams > 0) || nbeams < 0) return set_error(CCCS_EINVAL, "null argument");
    *out = nullptr;
    if (ctx->prob.ss_factor > 1) return set_error(CCCS_EINVAL, "the angle cache needs ss_factor 1");
    CCCS_HIP(hipSetDevice(ctx->device));
    std::unique_ptr<cccs_angle_cache> c(new cccs_angle_cache());
    const cccs_problem& p = ctx->prob;
    for (int k = 0; k < 3; k++) {
        c->size[k] = p.size[k];
        c->bbox_start[k] = p.bbox_start[k];
        c->bbox_size[k] = p.bbox_size[k];
        c->voxel[k] = p.voxel[k];
        c->start[k] = p.start[k];
    }
    c->bhc = p.beamhard_correct;
    c->dens_hash = ctx->dens_hash;
    c->spec = ctx->spec;
    c->device = ctx->device;
    c->nbbox = bbox_voxels(ctx);
    const uint64_t per = sizeof(float) * (uint64_t)c->nbbox;
    std::vector<int> keep;
    for (int i = 0; i < nbeams; i++) {
        // only the source and SAD enter the unit TERMA; the fluence-map fields are not used
        const cccs_beam& b = beams[i];
        if (!(b.sad > 0.f) || !std::isfinite(b.source[0]) || !std::isfinite(b.source[1]) || !std::isfinite(b.source[2]))
            return set_error(CCCS_EINVAL, "angle cache: beam " + std::to_string(i) + " needs a finite source and sad > 0");
        const auto k = angle_key(beams[i]);
        if (c->index.count(k)) continue;
        if ((uint64_t)(keep.size() + 1) * per > max_bytes) break;
        c->index[k] = keep.size();
        keep.push_back(i);
    }
    if (!keep.empty()) {
        if (hipMalloc(&c->data, per * keep.size()) != hipSuccess) {
            (void)hipGetLastError();
            return set_error(CCCS_ENOMEM, "angle cache of " + std::to_string(per * keep.size()) + " bytes");
        }
        for (size_t e = 0; e < keep.size(); e++) {
            TermaArgs a = terma_args(ctx, beams[keep[e]], nullptr, nullptr, -1);
            const uint64_t blocks = terma_blocks(a);
            if (blocks <= 0x7fffffffULL)
                terma_launches(a, [&](dim3 grid) {
                    hipLaunchKernelGGL(unit_terma_kernel, grid, dim3(256), 0, ctx->stream, a, c->data + e * c->nbbox);
                });
            const hipError_t err = blocks <= 0x7fffffffULL ? hipGetLastError() : hipErrorInvalidValue;
            if (err != hipSuccess) {
                (void)hipStreamSynchronize(ctx->stream);
                (void)hipFree(c->data);
                return set_error(CCCS_EDEVICE, std::string("unit TERMA kernel: ") + hipGetErrorString(err));
            }
        }
        if (hipStreamSynchronize(ctx->stream) != hipSuccess) {
            (void)hipFree(c->data);
            return set_error(CCCS_EDEVICE, "angle cache build");
        }
    }
    *out = c.release();
    return CCCS_OK;
}

extern "C" int cccs_angle_cache_info(const cccs_angle_cache* cache, int* nangles, uint64_t* bytes) {
    clear_error();
    if (!cache) return set_error(CCCS_EINVAL, "null argument");
    if (nangles) *nangles = (int)cache->index.size();
    if (bytes) *bytes = sizeof(float) * (uint64_t)cache->nbbox * cache->index.size();
    return CCCS_OK;
}

extern "C" int cccs_ctx_use_angle_cache(cccs_ctx* ctx, const cccs_angle_cache* cache) {
    clear_error();
    if (!ctx) return set_error(CCCS_EINVAL, "null argument");
    if (cache && !cache_fits(ctx, cache))
        return set_error(CCCS_EINVAL, "angle cache built for another problem, density or device");
    ctx->angle_cache = cache;
    return CCCS_OK;
}

extern "C" int cccs_angle_cache_destroy(cccs_angle_cache* cache) {
    clear_error();
    if (!cache) return CCCS_OK;
    if (cache->data) {
        CCCS_HIP(hipSetDevice(cache->device));
        CCCS_HIP(hipFree(cache->data));
    }
    delete cache;
    return CCCS_OK;
}

extern "C" int cccs_beam_dose_device_noalloc(cccs_ctx* ctx, const cccs_beam* beams, int nbeams,
                                             const float* d_fluence, float* d_dose) {
    clear_error();
    if (!ctx || (!beams && nbeams > 0) || nbeams < 0 || !d_dose || (!d_fluence && nbeams > 0))
        return set_error(CCCS_EINVAL, "null argument");
    if (ctx->prof.on) return set_error(CCCS_EINVAL, "per-kernel profiling allocates: turn it off for this call");
    CCCS_HIP(hipSetDevice(ctx->device));
    void* base = nullptr;
    {
        std::lock_guard<std::mutex> lk(g_scratch_mu);
        if (ctx->device >= 0 && ctx->device < kMaxDevices) base = g_scratch_ptr[ctx->device];
    }
    if (!base) return set_error(CCCS_EDEVICE, "fixed scratch not resolved for this device");
    float host_small[16];
    ConeDev host_cones[kMaxRays];
    size_t fo = 0;
    for (int i = 0; i < nbeams; i++) {
        BeamScratch S;
        S.ctx = ctx;
        S.arena = static_cast<char*>(base);
        S.cap = kNoAllocScratchBytes;
        S.host_small = host_small;
        S.host_cones = host_cones;
        CCCS_TRY(beam_dose_scratch(S, beams[i], d_fluence + fo, d_dose));
        fo += (size_t)beams[i].fmap_size[0] * beams[i].fmap_size[1];
    }
    return CCCS_OK;
}

extern "C" int cccs_beam_dose_device(cccs_ctx* ctx, const cccs_beam* beams, int nbeams, const float* d_fluence,
                                     float* d_dose) {
    clear_error();
    if (!ctx || (!beams && nbeams > 0) || nbeams < 0 || !d_dose || (!d_fluence && nbeams > 0))
        return set_error(CCCS_EINVAL, "null argument");
    CCCS_HIP(hipSetDevice(ctx->device));
    size_t fo = 0;
    for (int i = 0; i < nbeams; i++) {
        CCCS_TRY(beam_dose_one(ctx, beams[i], d_fluence + fo, d_dose));
        fo += (size_t)beams[i].fmap_size[0] * beams[i].fmap_size[1];
    }
    return CCCS_OK;
}

extern "C" int cccs_beam_dose(cccs_ctx* ctx, const cccs_beam* beams, int nbeams, const float* const* fluence,
                              float* dose) {
    clear_error();
    if (!ctx || (!beams && nbeams > 0) || nbeams < 0 || !dose || (!fluence && nbeams > 0))
        return set_error(CCCS_EINVAL, "null argument");
    CCCS_HIP(hipSetDevice(ctx->device));
    size_t nv = vol_voxels(ctx);
    CCCS_TRY(ctx->dose.ensure(nv * sizeof(float)));
    float* d = ctx->dose.as<float>();
    CCCS_HIP(hipMemsetAsync(d, 0, nv * sizeof(float), ctx->stream));
    for (int i = 0; i < nbeams; i++) {
        if (!fluence[i]) return set_error(CCCS_EINVAL, "null fluence map");
        const float* dfm = nullptr;
        CCCS_TRY(upload_fmap(ctx, beams[i], fluence[i], &dfm));
        CCCS_TRY(beam_dose_one(ctx, beams[i], dfm, d));
    }
    return download_staged(ctx, dose, d, nv * sizeof(float), true);
}

extern "C" int cccs_beam_terma(cccs_ctx* ctx, const cccs_beam* beam, const float* fluence, int beamletnum,
                               float* terma_bbox) {
    clear_error();
    if (!ctx || !beam || !fluence || !terma_bbox) return set_error(CCCS_EINVAL, "null argument");
    CCCS_HIP(hipSetDevice(ctx->device));
    CCCS_TRY(check_beam(ctx, *beam));
    const float* dfm = nullptr;
    CCCS_TRY(upload_fmap(ctx, *beam, fluence, &dfm));
    size_t n = bbox_voxels(ctx);
    CCCS_TRY(ctx->terma.ensure(n * sizeof(float)));
    TermaArgs ta = terma_args(ctx, *beam, dfm, ctx->terma.as<float>(), beamletnum);
    CCCS_TRY(launch_terma(ctx, ta));
    CCCS_HIP(hipStreamSynchronize(ctx->stream));
    CCCS_HIP(hipMemcpy(terma_bbox, ctx->terma.p, n * sizeof(float), hipMemcpyDeviceToHost));
    return CCCS_OK;
}

extern "C" int cccs_beam_geometry_of(cccs_ctx* ctx, const cccs_beam* beam, const float* fluence,
                                     cccs_beam_geometry* geom) {
    clear_error();
    if (!ctx || !beam || !fluence || !geom) return set_error(CCCS_EINVAL, "null argument");
    CCCS_HIP(hipSetDevice(ctx->device));
    CCCS_TRY(check_beam(ctx, *beam));
    const float* dfm = nullptr;
    CCCS_TRY(upload_fmap(ctx, *beam, fluence, &dfm));
    CCCS_TRY(ctx->terma.ensure(sizeof(float) * bbox_voxels(ctx)));
    TermaArgs ta = terma_args(ctx, *beam, dfm, ctx->terma.as<float>(), -1);
    CCCS_TRY(launch_terma(ctx, ta));
    BeamGeom g;
    BeamScratch S;
    CCCS_TRY(context_scratch(ctx, S));
    CCCS_TRY(run_cones(S, *beam, ctx->terma.as<float>(), nullptr, &g));
    std::memset(geom, 0, sizeof(*geom));
    geom->lim_min[0] = g.lim_min.x; geom->lim_min[1] = g.lim_min.y; geom->lim_min[2] = g.lim_min.z;
    for (int k = 0; k < 3; k++) geom->bev_size[k] = g.bev_size[k];
    geom->bev_min[0] = g.bev_min.x; geom->bev_min[1] = g.bev_min.y; geom->bev_min[2] = g.bev_min.z;
    geom->bev_max[0] = g.bev_max.x; geom->bev_max[1] = g.bev_max.y; geom->bev_max[2] = g.bev_max.z;
    geom->nrays = g.nrays;
    for (int r = 0; r < g.nrays; r++) {
        geom->rev_min[r][0] = g.rev_min[r].x; geom->rev_min[r][1] = g.rev_min[r].y; geom->rev_min[r][2] = g.rev_min[r].z;
        for (int k = 0; k < 3; k++) geom->rev_size[r][k] = g.rev_size[r][k];
    }
    return CCCS_OK;
}

extern "C" int cccs_fluence_projection(cccs_ctx* ctx, const uint8_t* mask, const cccs_beam* beams, int nbeams,
                                       float* fluence) {
    clear_error();
    if (!ctx || !mask || (!beams && nbeams > 0) || nbeams < 0 || (!fluence && nbeams > 0))
        return set_error(CCCS_EINVAL, "null argument");
    if (nbeams == 0) return CCCS_OK;
    CCCS_HIP(hipSetDevice(ctx->device));
    std::vector<ProjBeam> pb((size_t)nbeams);
    uint64_t total = 0;
    for (int i = 0; i < nbeams; i++) {
        const cccs_beam& b = beams[i];
        if (b.fmap_size[0] == 0 || b.fmap_size[1] == 0) return set_error(CCCS_EINVAL, "empty fluence map");
        if (!(b.beamlet_size[0] > 0.f) || !(b.beamlet_size[1] > 0.f)) return set_error(CCCS_EINVAL, "beamlet size");
        ProjBeam& o = pb[(size_t)i];
        o.src = ld3(b.source);
        o.iso = ld3(b.isocenter);
        o.inv = rot2_beam_inv(b.azimuth, b.zenith, b.coll);
        o.fx = (int)b.fmap_size[0];
        o.fy = (int)b.fmap_size[1];
        o.bsx = b.beamlet_size[0];
        o.bsy = b.beamlet_size[1];
        o.off = (uint32_t)total;
        total += (uint64_t)b.fmap_size[0] * b.fmap_size[1];
        if (total > 0x7fffffffULL) return set_error(CCCS_EINVAL, "too many beamlets");
    }
    const size_t nv = vol_voxels(ctx);
    // scratch: the mask (bytes, then float), the beam table and the maps; released on every return
    DevBuf mb, mf, tb, ob;
    struct Release {
        DevBuf* b[4];
        ~Release() {
            for (DevBuf* x : b) x->release();
        }
    } release{{&mb, &mf, &tb, &ob}};
    CCCS_TRY(mb.ensure(nv));
    CCCS_TRY(mf.ensure(nv * sizeof(float)));
    // beam table, then the mask's index box
    const size_t box_at = (sizeof(ProjBeam) * pb.size() + 15) & ~size_t(15);
    std::vector<uint8_t> tab(box_at + 6 * sizeof(int), 0);
    std::memcpy(tab.data(), pb.data(), sizeof(ProjBeam) * pb.size());
    const int box0[6] = {INT32_MAX, INT32_MAX, INT32_MAX, -1, -1, -1};
    std::memcpy(tab.data() + box_at, box0, sizeof(box0));
    CCCS_TRY(tb.ensure(tab.size()));
    CCCS_TRY(ob.ensure(sizeof(float) * total));
    CCCS_HIP(hipStreamSynchronize(ctx->stream));
    CCCS_HIP(hipMemcpy(mb.p, mask, nv, hipMemcpyHostToDevice));
    CCCS_HIP(hipMemcpy(tb.p, tab.data(), tab.size(), hipMemcpyHostToDevice));
    int* box = reinterpret_cast<int*>(tb.as<uint8_t>() + box_at);
    hipLaunchKernelGGL(mask_to_float_kernel, dim3(1024), dim3(256), 0, ctx->stream, (const uint8_t*)mb.p,
                       mf.as<float>(), nv, ctx->vol.nx, ctx->vol.ny, box);
    CCCS_HIP(hipGetLastError());
    const v3 vox = ctx->vol.voxel;
    // (a launch holds kMaxGroups workgroups of 256 threads; these have 576)
    const uint32_t groups = (uint32_t)((total + 63) / 64), per = kMaxGroups / 3;
    for (uint32_t b0 = 0; b0 < groups; b0 += per)
        hipLaunchKernelGGL(projection_kernel, dim3(std::min(per, groups - b0)), dim3(64 * kSubRays), 0, ctx->stream,
                           (const float*)mf.as<float>(), ctx->vol, mk3(1.f / vox.x, 1.f / vox.y, 1.f / vox.z),
                           (const int*)box, (const ProjBeam*)tb.as<ProjBeam>(), nbeams, b0, (uint32_t)total, ob.as<float>());
    CCCS_HIP(hipGetLastError());
    CCCS_HIP(hipStreamSynchronize(ctx->stream));
    CCCS_HIP(hipMemcpy(fluence, ob.p, sizeof(float) * total, hipMemcpyDeviceToHost));
    return CCCS_OK;
}

extern "C" int cccs_fluence_convolve(cccs_ctx* ctx, const float* fluence, int nmaps, int width, int height,
                                     const float* kernel, int kw, int kh, float* out) {
    clear_error();
    if (!ctx || (nmaps > 0 && (!fluence || !kernel || !out))) return set_error(CCCS_EINVAL, "null argument");
    if (nmaps < 0 || width < 1 || height < 1 || width > 4096 || height > 4096) return set_error(CCCS_EINVAL, "map size");
    if (kw < 1 || kh < 1 || kw > kConvMaxK || kh > kConvMaxK || !(kw & 1) || !(kh & 1))
        return set_error(CCCS_EINVAL, "kernel dims must be odd and at most 31");
    if (nmaps == 0) return CCCS_OK;
    if (nmaps > 65535) return set_error(CCCS_EINVAL, "at most 65535 maps per call");
    CCCS_HIP(hipSetDevice(ctx->device));
    const size_t n = (size_t)nmaps * width * height;
    DevBuf fb, kb, ob;
    struct Release {
        DevBuf* b[3];
        ~Release() {
            for (DevBuf* x : b) x->release();
        }
    } release{{&fb, &kb, &ob}};
    CCCS_TRY(fb.ensure(sizeof(float) * n));
    CCCS_TRY(kb.ensure(sizeof(float) * (size_t)kw * kh));
    CCCS_TRY(ob.ensure(sizeof(float) * n));
    CCCS_HIP(hipStreamSynchronize(ctx->stream));
    CCCS_HIP(hipMemcpy(fb.p, fluence, sizeof(float) * n, hipMemcpyHostToDevice));
    CCCS_HIP(hipMemcpy(kb.p, kernel, sizeof(float) * (size_t)kw * kh, hipMemcpyHostToDevice));
    const dim3 grid((unsigned)((width + kConvTile - 1) / kConvTile), (unsigned)((height + kConvTile - 1) / kConvTile),
                    (unsigned)nmaps);
    launch_conv<1>(kw, grid, ctx->stream, fb.as<float>(), width, height, kb.as<float>(), kh, ob.as<float>());
    CCCS_HIP(hipGetLastError());
    CCCS_HIP(hipStreamSynchronize(ctx->stream));
    CCCS_HIP(hipMemcpy(out, ob.p, sizeof(float) * n, hipMemcpyDeviceToHost));
    return CCCS_OK;
}

extern "C" int cccs_siddon_paths(cccs_ctx* ctx, const float* source, const float* points, int npoints,
                                 int max_segments, int32_t* ijk, float* mid, float* len, int32_t* counts, float* rpl) {
    clear_error();
    if (!ctx || !source || !points || npoints < 0 || max_segments < 0 || !ijk || !mid || !len || !counts || !rpl)
        return set_error(CCCS_EINVAL, "null argument");
    if (npoints == 0) return CCCS_OK;
    CCCS_HIP(hipSetDevice(ctx->device));
    const size_t ns = (size_t)npoints * std::max(1, max_segments);
    DevBuf b;
    size_t bytes = sizeof(float) * 3 * npoints + ns * (3 * sizeof(int32_t) + 3 * sizeof(float) + sizeof(float)) +
                   (size_t)npoints * (sizeof(int32_t) + sizeof(float));
    CCCS_TRY(b.ensure(bytes));
    char* base = b.as<char>();
    float* d_pts = (float*)base;
    int32_t* d_ijk = (int32_t*)(d_pts + 3 * npoints);
    float* d_mid = (float*)(d_ijk + 3 * ns);
    float* d_len = d_mid + 3 * ns;
    int32_t* d_cnt = (int32_t*)(d_len + ns);
    float* d_rpl = (float*)(d_cnt + npoints);
    int st = CCCS_OK;
    do {
        if (hipMemcpy(d_pts, points, sizeof(float) * 3 * npoints, hipMemcpyHostToDevice) != hipSuccess) { st = set_error(CCCS_EDEVICE, "copy"); break; }
        // slots past a point's segment count are returned as zeros
        if (hipMemset(d_ijk, 0, bytes - sizeof(float) * 3 * npoints) != hipSuccess) { st = set_error(CCCS_EDEVICE, "memset"); break; }
        PathArgs a;
        a.dens = ctx->d_dens;
        a.vd = ctx->vol;
        a.src = ld3(source);
        a.pts = d_pts;
        a.n = npoints;
        a.maxseg = max_segments;
        a.ijk = d_ijk; a.mid = d_mid; a.len = d_len; a.counts = d_cnt; a.rpl = d_rpl;
        hipLaunchKernelGGL(siddon_path_kernel, dim3((npoints + 255) / 256), dim3(256), 0, ctx->stream, a);
        if (hipGetLastError() != hipSuccess || hipStreamSynchronize(ctx->stream) != hipSuccess) { st = set_error(CCCS_EDEVICE, "siddon kernel"); break; }
        if (max_segments > 0) {
            if (hipMemcpy(ijk, d_ijk, ns * 3 * sizeof(int32_t), hipMemcpyDeviceToHost) != hipSuccess ||
                hipMemcpy(mid, d_mid, ns * 3 * sizeof(float), hipMemcpyDeviceToHost) != hipSuccess ||
                hipMemcpy(len, d_len, ns * sizeof(float), hipMemcpyDeviceToHost) != hipSuccess) { st = set_error(CCCS_EDEVICE, "copy back"); break; }
        }
        if (hipMemcpy(counts, d_cnt, npoints * sizeof(int32_t), hipMemcpyDeviceToHost) != hipSuccess ||
            hipMemcpy(rpl, d_rpl, npoints * sizeof(float), hipMemcpyDeviceToHost) != hipSuccess) { st = set_error(CCCS_EDEVICE, "copy back"); break; }
    } while (false);
    b.release();
    return st;
}

