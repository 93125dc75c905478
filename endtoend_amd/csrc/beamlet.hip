// beamlet.hip -- beamlet dose coefficients (dosecalc-beamlet: nvbbRayConvolve_host.cu:444-1409,
// nvbbRayConvolve_device.cu:19-521) on gfx950.
//
// Every active beamlet of a beam becomes a pillar (its beamlet's path through the calc_bbox plus a
// kernel_extent margin and a wall), and the pillars of a batch are tiled side by side in one packed
// BEV grid.  For each cone direction, every REV line of every batch in the job is resampled into
// LDS (pillar mapping, per-beamlet TERMA, density), walked inside its pillar segment, and the cone
// dose is gathered into the packed grid.  Each beamlet's pillar is then resampled back onto the
// calc_bbox and compacted on the device into a sparse column.
//
// A job is a list of batches, possibly from several beams: one launch of each kernel covers every
// batch of the job, so small beams and large beams share launches.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <cfloat>
#include <cmath>
#include <cstring>
#include <functional>
#include <limits>
#include <thread>
#include <vector>

#include "context.hpp"
#include "device_common.hpp"

namespace cccs {

constexpr int kWall = 2;        // pillar wall, REV samples (PILLAR_GRID, io_data_structs.h:139-160)
constexpr int kBuffer = 2;      // pillar rim excluded from unpacking (same struct)
constexpr int kMaxBatches = 100;  // batch-count retry limit of the reference (host.cu:692-834)
constexpr uint32_t kSubQueues = 64;  // TERMA sub-queues per cone direction
constexpr uint32_t kCntStride = 32;  // a sub-queue counter per 128-byte line: no two share one
constexpr uint32_t kPillarBits = 4096;  // batches up to this many pillars track footprint pillars per line

// One Rodrigues rotation with host-evaluated sine/cosine.
struct Rot1 {
    v3 a;
    float s, c;
};
// invRotateBeamlet / rotateBeamlet (CudaUtilities/geometry.cu:99-115): a rotation about
// (sin(-phi), 0, cos(-phi)) by -theta (beamlet frame -> BEV) or +theta (BEV -> beamlet frame).
// Both axes lie in the x-z plane.
CCCS_HD v3 rot1(const Rot1& R, v3 p) { return rot_xz(p, R.a.x, R.a.z, R.s, R.c); }
static Rot1 beamlet_rot(float theta, float phi, bool to_bev) {
    Rot1 r;
    float s, c;
    sincosf(-phi, &s, &c);
    r.a = mk3(s, 0.f, c);
    sincosf(to_bev ? -theta : theta, &r.s, &r.c);
    return r;
}

struct BeamletDev {
    v3 pst;          // pillar origin [cm]
    Rot1 inv;        // beamlet frame -> BEV
    Rot1 fwd;        // BEV -> beamlet frame
    int fidx;        // fluence-map index of the beamlet
    int batch;       // batch of the job
    int pix, piy;    // pillar column / row inside the batch grid
    int box0[3];     // calc_bbox-relative voxel box that can receive its dose
    int boxn[3];
    uint64_t arena;  // first element of its box in the column arena (i outer, k inner)
    uint32_t row0;   // first of its box's (i, j) rows in the job's row counts
    m33 fwd_m;       // PVCS -> beamlet frame (beamlet forward * beam forward), matrix form
};

struct BatchDev {
    BeamDev beam;
    Rot2 beam_inv;         // BEV -> PVCS
    const float* fmap;     // fluence map of the beam (device)
    int n, npx, npy;       // beamlets, pillars per row, rows
    int gd[3];             // packed grid dims (pX, pY, pZ)
    int pd[3];             // pillar dims
    int beamlet0;          // first beamlet of the batch in the job's beamlet table
    uint64_t pdose;        // float offset of its packed dose grid ([pX][pZ][pY], pY fastest)
    uint32_t tile0;        // first gather tile
    int tiles[3];          // gather tiles along pY (16), pZ (4), pX (4)
    uint32_t tdiv[2];      // t / tiles[k] == umulhi(t, tdiv[k]) for the batch's tiles (0: divide)
    float ipd[3];          // 1 / pd
    float fc[2];           // beamlet axis in pillar sample coordinates (x, z)
    float fw;              // bound on the footprint half-width [samples]: farther samples get no TERMA
    float cb[8];           // footprint bounds linear in depth (footprint_cull): x lo, x hi, z lo, z hi
    float gw;              // largest footprint distance from the axis over the grid's depth (<= fw)
};

// A footprint sample whose TERMA needs a Siddon march.
constexpr uint32_t kNoSlot = 0xffffffffu;  // a reserved queue entry that carries no request

struct TermaReq {
    uint32_t slot;     // position in the REV store of the cone direction, or kNoSlot
    uint32_t beamlet;  // job beamlet index
    float x, y, z;     // TERMA point [cm]
};

// One (cone, batch) REV grid.
struct BlConeDev {
    Rot2 kinv;       // REV -> packed BEV (invRotateKernel)
    Rot2 kfwd;       // packed BEV -> REV (rotateKernel)
    m33 kinv_m;      // matrix form of kinv, for line intervals only
    m33 kfwd_m;      // matrix form of kfwd, for the packed-BEV gather
    v3 minc;         // REV grid origin [cm]
    int nx, ny, nz;  // line length, lines along y, lines along z
    int batch;
    float hx, hz, hb;  // gather: |dx hz - dz hx| <= hb for a pillar axis that the voxel's lines can reach
    uint64_t line0;  // first line of this grid among the launch's lines
};

struct BlArgs {
    const float* dens;
    const float* tables;        // kernel rows | radii | 1/width | mean radii | 1/width of mean radii
    const BatchDev* batches;
    const BlConeDev* cones;     // the grids of one cone direction, one per batch
    const BeamletDev* beamlets;
    LineMeta* lines;
    float* rev;
    float* pdose;
    int nbatch;
    uint64_t nlines;
    int ntheta, nradii, nphi, rowf, rowb;
    float delr;
    v3 rvs, rrv;                // REV spacings (lat, long, lat) and reciprocals
    VolDesc vd;
    v3 ivoxel;                  // 1 / vd.voxel
    SpecDev spec;
    float bhc;
    uint32_t* line_cone;        // grid (= batch) of every line, written by the interval pass
    uint32_t* blocks;           // stored samples of every kLineBlock lines, or their exclusive scan
    uint32_t* counts;
    const uint32_t* tile_batch; // batch of every gather tile (nullptr: a single batch)
    // stored lines have kLineZeros zero samples on both sides, empty lines' offset points at zeros, and
    // the store has fewer than 2^30 samples: the gather's short form applies
    bool zeros;
};

CCCS_HD int find_cone(const BlConeDev* __restrict__ c, int n, uint64_t line) {
    int lo = 0, hi = n - 1;
    while (lo < hi) {
        int mid = (lo + hi + 1) >> 1;
        if (c[mid].line0 <= line) lo = mid; else hi = mid - 1;
    }
    return lo;
}

// REV sample (tX, tY, tZ) of a grid -> packed-BEV coordinate (cudaBeamletRaytrace,
// nvbbRayConvolve_device.cu:33-41).
CCCS_HD v3 rev_to_packed(const BlConeDev& c, v3 rrv, int tX, int tY, int tZ) {
    v3 q = mk3(fmaf(c.minc.x, rrv.x, (float)tZ), fmaf(c.minc.y, rrv.y, (float)tX), fmaf(c.minc.z, rrv.z, (float)tY));
    return rot_inv(c.kinv, q) + 0.5f;
}

// Interval of stored samples of every line of one cone direction: the line clipped to the packed
// grid box (packed coordinates are affine in the sample index), widened by 2/3 samples.
CCCS_HD LineMeta line_interval(const BlArgs& a, const BlConeDev& c, const BatchDev& B, uint64_t line) {
    const uint64_t l = line - c.line0;
    const int tY = (int)(l % (uint64_t)c.ny), tZ = (int)(l / (uint64_t)c.ny);
    v3 q0 = mk3(fmaf(c.minc.x, a.rrv.x, (float)tZ), c.minc.y * a.rrv.y, fmaf(c.minc.z, a.rrv.z, (float)tY));
    v3 p0 = c.kinv_m(q0) + 0.5f;
    v3 d = mk3(c.kinv_m.m[1], c.kinv_m.m[4], c.kinv_m.m[7]);
    float t0 = 0.f, t1 = (float)c.nx;
    clip_slab(p0.x, d.x, 0.f, (float)B.gd[0], t0, t1);
    clip_slab(p0.y, d.y, 0.f, (float)B.gd[1], t0, t1);
    clip_slab(p0.z, d.z, 0.f, (float)B.gd[2], t0, t1);
    LineMeta m;
    m.i0 = 0;
    m.len = 0;
    m.off = 0;
    if (t0 <= t1) {
        const int i0 = max(0, (int)floorf(t0) - 2);
        const int i1 = min(c.nx, (int)ceilf(t1) + 3);
        m.i0 = (int16_t)i0;
        m.len = (int16_t)max(0, i1 - i0);
    }
    return m;
}

// Offsets into the REV store: every stored line is preceded by kLineZeros samples of its own where
// BlArgs::zeros holds, and empty lines get offset 0 there.  The interval pass leaves offsets within
// blocks of kLineBlock lines and the blocks' totals; the sample stage, which reads every record first
// and writes it back, adds the blocks before, from the totals themselves up to 64 blocks and from their
// scan beyond (three scan launches of their own cost a 32^3 job a tenth of its time).
constexpr int kLineBlock = 256;
constexpr uint32_t kWaveBlocks = 64;  // blocks whose totals one wave scans
// Samples of the store before a line's own, beside the lines before it.
CCCS_HD uint32_t line_pad(bool zeros, int len) { return zeros && len > 0 ? (uint32_t)kLineZeros : 0u; }

__global__ void __launch_bounds__(kLineBlock) bl_interval_kernel(BlArgs a) {
    __shared__ uint32_t s_w[kLineBlock / 64];
    const uint64_t line = (uint64_t)blockIdx.x * kLineBlock + threadIdx.x;
    const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
    // what empty lines (offset 0) read; the walk writes the zeros around the others
    if (a.zeros && line < 2 * kLineZeros) a.rev[(int64_t)line - kLineZeros] = 0.f;
    LineMeta m{};
    int ci = 0;
    if (line < a.nlines) {
        ci = find_cone(a.cones, a.nbatch, line);
        m = line_interval(a, a.cones[ci], a.batches[ci], line);
    }
    const uint32_t pad = line_pad(a.zeros, m.len), take = (uint32_t)m.len + pad;
    const uint32_t inc = wave_incl_u32(take);
    if (lane == 63) s_w[w] = inc;
    __syncthreads();
    uint32_t before = inc - take;
    for (int q = 0; q < w; q++) before += s_w[q];
    m.off = m.len > 0 ? before + pad : 0u;
    if (line < a.nlines) {
        a.line_cone[line] = (uint32_t)ci;
        a.lines[line] = m;
    }
    if (threadIdx.x == kLineBlock - 1) a.blocks[blockIdx.x] = before + take;
}

// One workgroup: exclusive scan of the block totals.
__global__ void __launch_bounds__(kLineBlock) bl_block_scan_kernel(uint32_t* __restrict__ blocks, uint32_t nb) {
    __shared__ uint32_t s_w[kLineBlock / 64];
    const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
    uint32_t carry = 0;
    for (uint32_t b0 = 0; b0 < nb; b0 += kLineBlock) {
        const uint32_t b = b0 + threadIdx.x, v = b < nb ? blocks[b] : 0u, inc = wave_incl_u32(v);
        if (lane == 63) s_w[w] = inc;
        __syncthreads();
        uint32_t before = carry;
        for (int q = 0; q < kLineBlock / 64; q++) {
            before += q < w ? s_w[q] : 0u;
            carry += s_w[q];
        }
        if (b < nb) blocks[b] = before + inc - v;
        __syncthreads();
    }
}

// fmodf(x, y) for 0 <= x < 2^24 and a positive integer y <= 2^20: n*y is exact, x - n*y is exact,
// and the fix-ups absorb a quotient rounded across an integer.  Equal to fmodf bit for bit there.
CCCS_HD float fmod_pos(float x, float y) {
    const float n = truncf(x / y);
    float r = fmaf(-n, y, x);
    if (r < 0.f) r += y;
    if (r >= y) r -= y;
    return r;
}

// floorf(x / y) of the correctly rounded quotient, for 0 <= x < 2^24 and a positive integer
// y <= 2^20, with iy = 1 / y rounded.  q = x * iy lies within q * 2^-22 of the rounded quotient (two
// roundings of 2^-24 relative, plus half an ulp of the quotient), so the two have the same floor
// unless q lies within that distance of an integer; there the division decides.  Lanes near a
// multiple of y are rare, so most waves skip the IEEE division.
CCCS_HD float floor_quot(float x, float y, float iy) {
    const float q = x * iy;
    const float fq = floorf(q);
    const float m = q * 4.76837158e-7f;  // 2^-21: twice the bound
    if (q - fq > m && (fq + 1.f) - q > m) return fq;
    return floorf(x / y);
}

// fmod_pos(x, y) given the floor n of its quotient (the same n fmod_pos computes).
CCCS_HD float fmod_pos_n(float x, float y, float n) {
    float r = fmaf(-n, y, x);
    if (r < 0.f) r += y;
    if (r >= y) r -= y;
    return r;
}

// Pillar mapping of one REV sample (cudaBeamletRaytrace, nvbbRayConvolve_device.cu:33-68):
// false for a wall, a sample outside the packed grid or past the last pillar; otherwise the
// beamlet (pidx, batch-local) and the pillar-local coordinate inp (already shifted by -0.5).
// ipd holds the reciprocals of the pillar dimensions; the pillar index and the in-pillar
// coordinate are those of the IEEE quotients pb / pd (floor_quot).
CCCS_HD bool bl_locate(const BlArgs& a, const BlConeDev& c, const BatchDev& B, v3 ipd, int tX, int tY, int tZ,
                       int& pidx, v3& inp) {
    const v3 pb = rev_to_packed(c, a.rrv, tX, tY, tZ);
    const v3 gdf = mk3((float)B.gd[0], (float)B.gd[1], (float)B.gd[2]);
    if (pb.x < 0.f || pb.y < 0.f || pb.z < 0.f || pb.x >= gdf.x || pb.y >= gdf.y || pb.z >= gdf.z) return false;
    const v3 pdf = mk3((float)B.pd[0], (float)B.pd[1], (float)B.pd[2]);
    const float nx = floor_quot(pb.x, pdf.x, ipd.x), ny = floor_quot(pb.y, pdf.y, ipd.y),
                nz = floor_quot(pb.z, pdf.z, ipd.z);
    pidx = (int)nx + (int)nz * B.npx;
    if (pidx >= B.n) return false;
    inp = mk3(fmod_pos_n(pb.x, pdf.x, nx), fmod_pos_n(pb.y, pdf.y, ny), fmod_pos_n(pb.z, pdf.z, nz));
    if (inp.x < (float)kWall || inp.y < (float)kWall || inp.z < (float)kWall) return false;
    inp = inp - 0.5f;
    return true;
}

// What a REV sample's density and TERMA points need of its beamlet (the head of BeamletDev).
struct PillarRec {
    v3 pst;
    Rot1 inv;
    int fidx;
};
CCCS_HD PillarRec pillar_rec(const BeamletDev& d) {
    PillarRec r;
    r.pst = d.pst;
    r.inv = d.inv;
    r.fidx = d.fidx;
    return r;
}

// PVCS point [cm] where the sample's TERMA is evaluated (device.cu:170-180).
CCCS_HD v3 bl_terma_point(const BlArgs& a, const BatchDev& B, const PillarRec& bl, v3 inp) {
    const v3 g = rot_inv(B.beam_inv, rot1(bl.inv, inp));
    return mk3(fmaf(g.x, a.rvs.x, bl.pst.x), fmaf(g.y, a.rvs.y, bl.pst.y), fmaf(g.z, a.rvs.z, bl.pst.z));
}

// Density at the sample (device.cu:213-223): trilinear, border 0.
__device__ __forceinline__ float bl_density(const BlArgs& a, const MarchVol& vol, const BatchDev& B, const PillarRec& bl,
                                            v3 inp) {
    const v3 g2 = rot_inv(B.beam_inv, rot1(bl.inv, inp * a.rvs)) + bl.pst;
    const v3 gi = div_by(g2 - a.vd.start, a.vd.voxel, a.ivoxel);
    const float s = gi.x + gi.y + gi.z;  // (div_by makes an infinite quotient NaN: outside, as the quotient)
    return s == s ? tex3_march(vol, gi.x + 0.5f, gi.y + 0.5f, gi.z + 0.5f) : 0.f;
}

// The affine form of the mapping, in the sample stage: the packed coordinate of sample t of line (tY, tZ) is
// line_start + t * line_step (matrix rotation).  It only skips samples that are far from every footprint or
// inside pillars without footprint samples, with margins far above its rounding; the exact mapping decides
// every other sample.
CCCS_HD v3 line_start(const BlArgs& a, const BlConeDev& c, int tY, int tZ) {
    return c.kinv_m(mk3(fmaf(c.minc.x, a.rrv.x, (float)tZ), c.minc.y * a.rrv.y, fmaf(c.minc.z, a.rrv.z, (float)tY))) + 0.5f;
}
CCCS_HD v3 line_step(const BlConeDev& c) { return mk3(c.kinv_m.m[1], c.kinv_m.m[4], c.kinv_m.m[7]); }

// Pass A.1's cull of one sample.  First the distance from the nearest beamlet axis, in pillars with the axis at
// 0.5 (cx, cz: the second test's half-width and 0.05 samples).
CCCS_HD bool near_axis(bool in, float ux, float uz, float cx, float cz) {
    return in && fabsf((ux - floorf(ux)) - 0.5f) <= cx && fabsf((uz - floorf(uz)) - 0.5f) <= cz;
}
// Then the footprint half-width fw (cull: 0.05 samples wider) and the batch's depth-linear footprint bounds (cb).
CCCS_HD bool in_foot_bounds(bool near, const BatchDev& B, float px, float py, float pz, float pdx, float pdz, float ipdx,
                            float ipdz, float cull) {
    const float xl = px - floorf(px * ipdx) * pdx, zl = pz - floorf(pz * ipdz) * pdz;
    return near && fabsf(xl - B.fc[0]) <= cull && fabsf(zl - B.fc[1]) <= cull && xl >= B.cb[0] + B.cb[1] * py &&
           xl <= B.cb[2] + B.cb[3] * py && zl >= B.cb[4] + B.cb[5] * py && zl <= B.cb[6] + B.cb[7] * py;
}

// Pass B.1: whether a sample at (ux, uz), in pillars, needs the exact mapping: not where it certainly lies in a
// pillar without a bit in `pil` or outside the grid's pillars (by 0.05 samples; hx, hz: half a pillar less that).
CCCS_HD bool may_take_dose(bool in, const BatchDev& B, float ux, float uz, float hx, float hz, const uint32_t* pil) {
    const float fx = floorf(ux), fz = floorf(uz);
    if (fabsf((ux - fx) - 0.5f) < hx && fabsf((uz - fz) - 0.5f) < hz) {
        const int px = (int)fx, pa = px + (int)fz * B.npx;
        const bool grid = (uint32_t)px < (uint32_t)B.npx && fz >= 0.f && pa < B.n;
        in = in && grid && (pil[grid ? pa >> 5 : 0] >> (pa & 31)) & 1u;
    }
    return in;
}

// Cumulative kernel of one row, linear between radii (the reference's clamped linear texture
// lookup, nvbbRayConvolve_device.cu:330-352).  Interval s of a row is {lo, K(lo), slope, hi}: the
// value at r in (lo, hi] is K(lo) + (r - lo) * slope.  s tracks the first radius >= r and r must
// not decrease between calls.
__device__ __forceinline__ float kc_at(float r, const float4* __restrict__ tab, int nr, int& s, float4& iv) {
    while (s < nr - 1 && iv.w < r) iv = tab[++s];
    return iv.y + (r - iv.x) * iv.z;
}

// Footprint pillars of a line beyond which the host's index audit counts a line apart (the stage has no such limit).
constexpr int kStagePillars = 64;

__device__ __forceinline__ int lane_i(int v, int lane) { return __builtin_amdgcn_readlane(v, lane); }
__device__ __forceinline__ float lane_f(float v, int lane) {
    return __int_as_float(__builtin_amdgcn_readlane(__float_as_int(v), lane));
}

// A record at a wave-uniform address, through the scalar unit; only the fields that are used load.
template <class T>
__device__ __forceinline__ T uniform_copy(const T* p) {
    static_assert(sizeof(T) % 4 == 0, "whole dwords");
    uint32_t w[sizeof(T) / 4];
    const uniform_ptr<uint32_t> s = as_uniform(reinterpret_cast<const uint32_t*>(p));
#pragma unroll
    for (int i = 0; i < (int)(sizeof(T) / 4); i++) w[i] = s[i];
    T r;
    __builtin_memcpy(&r, w, sizeof(T));
    return r;
}

// Stage 1 of a cone direction, one wave per stride of REV lines: pillar mapping of every stored sample
// and the beamlet-footprint test (fluence cell of the sample == its beamlet).  A line without footprint
// samples carries no TERMA, so all its cone dose is zero: it is marked empty.  Otherwise the half
// steps (0.5 * delr * density, -1 for walls) go to H, TERMA slots are zeroed, and the footprint
// samples are queued for their Siddon TERMA.
//
// Most stored samples are far from every footprint (1 to 2 % are candidates, 7 to 15 % reach the exact
// mapping), and most lines have a handful of candidates, so the kernel's time is its instructions per
// line.  A wave takes the records of 64 lines at once, one per lane (line record, grid indices and
// affine start cost once per 64 lines), culls the samples line by line (pass A.1: one multiply-add, a
// fraction and a compare per axis and sample), and collects the candidates of consecutive lines
// until the list is full, so that the exact test (pass A.2) runs on full waves.  Lines with footprint
// samples then take passes B.1 and B.2.  The grid's and batch's fields come through the scalar
// unit.
__global__ void __launch_bounds__(64) bl_sample_kernel(BlArgs a, float* __restrict__ H, TermaReq* __restrict__ q,
                                                       uint32_t subcap, uint32_t* __restrict__ qcnt) {
    __shared__ uint16_t s_cand[kMaxLine];         // candidates: lane of the line << 10 | sample
    __shared__ uint16_t s_cpil[kMaxLine];         // footprint samples among them: their pillar, else kNoPil
    __shared__ uint16_t s_list[kMaxLine];         // one line's samples for pass B.2
    __shared__ uint32_t s_foot[kMaxLine / 32];    // one line's footprint samples
    __shared__ uint64_t s_exact[kMaxLine / 64];   // one line's samples on s_list
    __shared__ uint32_t s_pil[kPillarBits / 32];  // pillars with footprint samples on the line
    constexpr uint16_t kNoPil = 0xffff;
    const int tid = threadIdx.x;
    const uint64_t lt = (1ull << tid) - 1ull;
    const MarchVol vol = march_vol(a.dens, a.vd.nx, a.vd.ny, a.vd.nz);
    uint32_t stored = 0;
    const uint64_t G = gridDim.x;
    for (uint64_t base = xcd_remap(blockIdx.x, gridDim.x); base < a.nlines; base += 64 * G) {
    // this lane's line
    const uint64_t my_line = base + (uint64_t)tid * G;
    LineMeta mine{};
    // (the totals of up to kWaveBlocks blocks are scanned here)
    const uint32_t nblocks = (uint32_t)((a.nlines + kLineBlock - 1) / kLineBlock);
    uint32_t total = (uint32_t)tid < nblocks && nblocks <= kWaveBlocks ? a.blocks[tid] : 0u;
    total = wave_incl_u32(total) - total;
    int my_ci = 0, my_y = 0, my_z = 0;
    v3 my_p0 = mk3(0.f, 0.f, 0.f);
    if (my_line < a.nlines) {
        mine = a.lines[my_line];
        my_ci = (int)a.line_cone[my_line];
        const BlConeDev& c = a.cones[my_ci];
        const uint64_t l = my_line - c.line0;
        my_z = (int)(l / (uint64_t)c.ny);
        my_y = (int)(l - (uint64_t)my_z * (uint64_t)c.ny);
        my_p0 = line_start(a, c, my_y, my_z);
        if (mine.len > 0) stored += (uint32_t)mine.len;  // summed over the wave's lanes by wave_count
    }
    {
        const uint32_t b = (uint32_t)(my_line / kLineBlock);
        const uint32_t before = nblocks <= kWaveBlocks ? (uint32_t)__shfl((int)total, (int)(b & 63u), 64)
                                                       : (mine.len > 0 ? a.blocks[b] : 0u);
        mine.off += before;
    }
    uint64_t todo = __ballot(mine.len > 0);
    while (todo) {
        // pass A.1: affine cull of consecutive lines of one grid, candidates to s_cand
        const int ci = lane_i(my_ci, __builtin_ctzll(todo));
        const BlConeDev* pc = a.cones + ci;
        const BatchDev* pB = a.batches + ci;  // grid ci of a direction belongs to batch ci
        uint64_t lines_in = 0, with_cand = 0;
        int my_c0 = 0, my_c1 = 0, ncand = 0;
        {
            const BlConeDev c = uniform_copy(pc);
            const BatchDev B = uniform_copy(pB);
            const v3 dl = line_step(c);
            const float pdx = (float)B.pd[0], pdz = (float)B.pd[2], ipdx = B.ipd[0], ipdz = B.ipd[2];
            const float cull = B.fw + 0.05f;
            const float dux = dl.x * ipdx, duz = dl.z * ipdz, cx = (cull + 0.05f) * ipdx, cz = (cull + 0.05f) * ipdz;
            while (todo) {
                const int k = __builtin_ctzll(todo);
                const int m = lane_i((int)mine.len, k);
                if (lane_i(my_ci, k) != ci || ncand + m > kMaxLine) break;
                todo &= todo - 1ull;
                lines_in |= 1ull << k;
                const float px0 = lane_f(my_p0.x, k), py0 = lane_f(my_p0.y, k), pz0 = lane_f(my_p0.z, k);
                const float t0 = (float)(lane_i((int)mine.i0, k) + tid);
                const float ux0 = fmaf(px0 - B.fc[0], ipdx, 0.5f), uz0 = fmaf(pz0 - B.fc[1], ipdz, 0.5f);
                const int c0 = ncand;
                for (int j0 = 0; j0 < m; j0 += 64) {
                    const float t = t0 + (float)j0;
                    const float ux = fmaf(t, dux, ux0), uz = fmaf(t, duz, uz0);
                    bool cand = near_axis(tid < m - j0, ux, uz, cx, cz);
                    if (!__ballot(cand)) continue;
                    cand = in_foot_bounds(cand, B, px0 + t * dl.x, py0 + t * dl.y, pz0 + t * dl.z, pdx, pdz, ipdx, ipdz, cull);
                    const uint64_t mask = __ballot(cand);
                    if (cand) s_cand[ncand + __popcll(mask & lt)] = (uint16_t)(k << 10 | (j0 + tid));
                    ncand += __popcll(mask);
                }
                if (ncand > c0) {
                    with_cand |= 1ull << k;
                    if (tid == k) {
                        my_c0 = c0;
                        my_c1 = ncand;
                    }
                }
            }
        }
        if ((lines_in & ~with_cand) >> tid & 1ull) a.lines[my_line] = LineMeta{0u, 0, 0};
        __syncthreads();
        // pass A.2: exact pillar mapping and fluence-cell test of the candidates, full waves
        if (ncand > 0) {
            const BlConeDev c = uniform_copy(pc);
            const BatchDev B = uniform_copy(pB);
            const v3 ipd = mk3(B.ipd[0], B.ipd[1], B.ipd[2]);
            for (int r = 0; r < ncand; r += 64) {
                const bool in = r + tid < ncand;
                const int e = in ? (int)s_cand[r + tid] : 0, k = e >> 10;
                const int i = __shfl((int)mine.i0, k, 64) + (e & 1023), y = __shfl(my_y, k, 64), z = __shfl(my_z, k, 64);
                if (in) {
                    int pidx;
                    v3 inp;
                    bool fp = false;
                    if (bl_locate(a, c, B, ipd, i, y, z, pidx, inp) && fabsf(inp.x - B.fc[0]) <= B.fw &&
                        fabsf(inp.z - B.fc[1]) <= B.fw) {
                        // point_fluence(...) > 0 without its map load: a job beamlet's own cell has a
                        // positive weight (plan_beam keeps only those), so the cell test decides alone
                        const PillarRec bl = pillar_rec(a.beamlets[B.beamlet0 + pidx]);
                        fp = fluence_cell(bl_terma_point(a, B, bl, inp), B.beam) == bl.fidx;
                    }
                    s_cpil[r + tid] = !fp ? kNoPil : (uint16_t)(B.n <= (int)kPillarBits ? pidx : 0);
                }
            }
        }
        __syncthreads();
        while (with_cand) {
            const int k = __builtin_ctzll(with_cand);
            with_cand &= with_cand - 1ull;
            const uint64_t line = base + (uint64_t)k * G;
            const int c0 = lane_i(my_c0, k), c1 = lane_i(my_c1, k);
            uint32_t nfoot = 0;  // footprint samples of the line: exactly its TERMA requests below
            for (int e = c0; e < c1; e += 64)
                nfoot += (uint32_t)__popcll(__ballot(e + tid < c1 && s_cpil[e + tid] != kNoPil));
            if (nfoot == 0) {
                if (tid == 0) a.lines[line] = LineMeta{0u, 0, 0};
                continue;
            }
            // a line's TERMA requests go to one of kSubQueues queues, chosen by its run of 64
            // consecutive lines: the Siddon stage then marches neighbouring lines' rays side by side
            // (shared cache lines; -26 % stage time against one queue per wave), and the lines in
            // flight still spread over every counter.  One reservation per line (its latency overlaps
            // pass B.1): every footprint sample, and no other, queues one TERMA request in pass B.2
            const uint32_t sq = (uint32_t)((line >> 6) % kSubQueues);
            TermaReq* qs = q + (size_t)sq * subcap;
            uint32_t qres = 0;
            if (tid == 0) qres = atomicAdd(qcnt + sq * kCntStride, nfoot);
            const BatchDev B = uniform_copy(pB);
            const BlConeDev c = uniform_copy(pc);
            const bool track = B.n <= (int)kPillarBits;
            if (tid < kMaxLine / 32) s_foot[tid] = 0u;
            s_pil[tid] = 0u;
            s_pil[tid + 64] = 0u;
            __syncthreads();
            for (int e = c0 + tid; e < c1; e += 64) {
                const uint32_t pil = s_cpil[e], j = s_cand[e] & 1023u;
                if (pil == kNoPil) continue;
                atomicOr(&s_foot[j >> 5], 1u << (j & 31u));
                if (track) atomicOr(&s_pil[pil >> 5], 1u << (pil & 31u));
            }
            __syncthreads();
            // pass B.1: a pillar without footprint samples on this line gets no dose on it, so its
            // samples act as walls (a pillar crossing is exactly one segment of the walk).  Samples
            // confidently in such pillars (or outside the grid's pillars) are walls; the others go to
            // the list.  Only the walls between the first and the last listed sample are written: the
            // line is trimmed to its non-wall span below, so no stage reads the others.
            const int i0 = lane_i((int)mine.i0, k), m = lane_i((int)mine.len, k);
            const uint32_t moff = (uint32_t)lane_i((int)mine.off, k);
            float* T = a.rev + moff;
            float* Hl = H + moff;
            int nex = 0;
            {
                const float ipdx = B.ipd[0], ipdz = B.ipd[2];
                const float ux0 = lane_f(my_p0.x, k) * ipdx, uz0 = lane_f(my_p0.z, k) * ipdz;
                const float dux = c.kinv_m.m[1] * ipdx, duz = c.kinv_m.m[7] * ipdz;
                // (inside the pillar by 0.05 samples on each side)
                const float hx = 0.5f - 0.05f * ipdx, hz = 0.5f - 0.05f * ipdz;
                for (int j0 = 0; j0 < m; j0 += 64) {
                    const int j = j0 + tid;
                    bool exact = j < m;
                    if (track) {
                        const float t = (float)(i0 + j);
                        exact = may_take_dose(exact, B, fmaf(t, dux, ux0), fmaf(t, duz, uz0), hx, hz, s_pil);
                    }
                    const uint64_t mask = __ballot(exact);
                    if (tid == 0) s_exact[j0 >> 6] = mask;
                    if (exact) s_list[nex + __popcll(mask & lt)] = (uint16_t)j;
                    nex += __popcll(mask);
                }
            }
            const uint32_t qbase = (uint32_t)lane_i((int)qres, 0);
            if (nex == 0) {  // every sample is a wall: no dose on this line, and the reservation stays empty
                if (tid == 0) a.lines[line] = LineMeta{0u, 0, 0};
                for (uint32_t e = (uint32_t)tid; e < nfoot; e += 64)
                    if (qbase + e < subcap) qs[qbase + e].slot = kNoSlot;
                __syncthreads();
                continue;
            }
            __syncthreads();
            {
                const int elo = s_list[0], ehi = s_list[nex - 1];
                for (int j0 = elo & ~63; j0 <= ehi; j0 += 64) {
                    const int j = j0 + tid;
                    if (j > elo && j < ehi && !(s_exact[j0 >> 6] >> tid & 1ull)) {
                        Hl[j] = -1.f;
                        T[j] = 0.f;
                    }
                }
            }
            // pass B.2: exact mapping, density and TERMA request of the listed samples, full waves
            int first = -1, last = -1;  // first and last listed sample that is not a wall
            uint32_t qdone = 0;
            const int tY = lane_i(my_y, k), tZ = lane_i(my_z, k);
            const v3 ipd = mk3(B.ipd[0], B.ipd[1], B.ipd[2]);
            for (int r = 0; r < nex; r += 64) {
                bool ok = false, need = false;
                int j = 0, pidx = 0;
                v3 inp;
                PillarRec bl;
                if (r + tid < nex) {
                    j = s_list[r + tid];
                    if (bl_locate(a, c, B, ipd, i0 + j, tY, tZ, pidx, inp) &&
                        (!track || ((s_pil[pidx >> 5] >> (pidx & 31)) & 1u))) {
                        ok = true;
                        bl = pillar_rec(a.beamlets[B.beamlet0 + pidx]);
                        need = (s_foot[j >> 5] >> (j & 31)) & 1u;
                    }
                }
                // the TERMA requests first, then the density: the two rotations are not live together
                const uint64_t mask = __ballot(need);
                if (mask) {
                    if (need) {
                        const uint32_t pos = qbase + qdone + (uint32_t)__popcll(mask & lt);
                        const v3 gcs = bl_terma_point(a, B, bl, inp);
                        TermaReq rq;
                        rq.slot = moff + (uint32_t)j;
                        rq.beamlet = (uint32_t)(B.beamlet0 + pidx);
                        rq.x = gcs.x; rq.y = gcs.y; rq.z = gcs.z;
                        if (pos < subcap) qs[pos] = rq;
                    }
                    qdone += (uint32_t)__popcll(mask);
                }
                float h = -1.f;
                if (r + tid < nex) {
                    if (ok) h = 0.5f * (a.delr * bl_density(a, vol, B, bl, inp));
                    Hl[j] = h;
                    T[j] = 0.f;
                }
                const uint64_t open = __ballot(h >= 0.f);
                if (open) {
                    if (first < 0) first = r + __builtin_ctzll(open);
                    last = r + 63 - __builtin_clzll(open);
                }
            }
            // The reservation counted footprint samples of pass A.2; pass B.2 requests TERMA for those of
            // them it maps to the same pillar again, so any shortfall is closed with empty entries.
            for (uint32_t e = qdone + (uint32_t)tid; e < nfoot; e += 64) {
                const uint32_t pos = qbase + e;
                if (pos < subcap) qs[pos].slot = kNoSlot;
            }
            // Walls before the first and after the last non-wall sample bound no segment and receive no
            // dose: the line's stored interval shrinks to the span between, so the walk and the gather
            // skip them (the gather reads samples outside a line's interval as zero, the dose the walk
            // gives a wall).
            const int nlo = first < 0 ? m : (int)s_list[first], nhi = last < 0 ? -1 : (int)s_list[last];
            if (tid == 0) {
                a.lines[line] = nhi < nlo ? LineMeta{0u, 0, 0}
                                          : LineMeta{moff + (uint32_t)nlo, (int16_t)(i0 + nlo), (int16_t)(nhi - nlo + 1)};
            }
            __syncthreads();  // the next line reuses the LDS arrays
        }
        __syncthreads();  // the next lines reuse the candidate list
    }
    }
    if (a.counts) wave_count(stored, a.counts, blockIdx.x);
}

// Stage 2: the queued samples' TERMA (cudaSiddon_device with the beamlet filter), one sample per
// lane, grid-stride over the queue.
__global__ void __launch_bounds__(256) bl_siddon_kernel(BlArgs a, const TermaReq* __restrict__ q, uint32_t subcap,
                                                        const uint32_t* __restrict__ qcnt, uint32_t* counts) {
    // workgroup b serves sub-queue b % kSubQueues
    const uint32_t sq = blockIdx.x % kSubQueues, per = gridDim.x / kSubQueues;
    const uint32_t n = min(qcnt[sq * kCntStride], subcap);
    const TermaReq* qs = q + (size_t)sq * subcap;
    uint32_t steps = 0;
    for (uint32_t i = (blockIdx.x / kSubQueues) * 256 + threadIdx.x; i < n; i += per * 256) {
        const TermaReq r = qs[i];
        if (r.slot == kNoSlot) continue;
        const BeamletDev& bl = a.beamlets[r.beamlet];
        const BatchDev& B = a.batches[bl.batch];
        // (the request's point lies in its beamlet's cell: the sample stage tested it)
        const float fluence = B.fmap[bl.fidx];
        const v3 p = mk3(r.x, r.y, r.z);
        float v = 0.f;
        if (fluence <= 0.f) {
        } else if (counts) {
            int it = 0;
            v = fluence_terma_rpl(p, fluence, B.beam, a.spec, a.vd, a.ivoxel, a.dens, a.bhc, &it);
            steps += (uint32_t)it;
        } else {
            v = fluence_terma_rpl(p, fluence, B.beam, a.spec, a.vd, a.ivoxel, a.dens, a.bhc, nullptr);
        }
        a.rev[r.slot] = v;
    }
    if (counts) block_count(steps, counts, blockIdx.x);
}

// A 64-bit value from lane addr / 4 (ds_bpermute on both halves).
__device__ __forceinline__ double bperm_f64(int addr, double v) {
    const uint64_t b = (uint64_t)__double_as_longlong(v);
    const uint32_t lo = (uint32_t)__builtin_amdgcn_ds_bpermute(addr, (int)(uint32_t)b);
    const uint32_t hi = (uint32_t)__builtin_amdgcn_ds_bpermute(addr, (int)(uint32_t)(b >> 32));
    return __longlong_as_double((long long)(((uint64_t)hi << 32) | lo));
}

// Stage 3, one wave per non-empty REV line: PackRowConvolve (nvbbRayConvolve_device.cu:284-417)
// for every sample.  Both walks of destination j run inside the pillar segment holding j, start at
// j itself (the self sample adds only its first half step) and stop when the radiological
// distance passes the last radius or enters the last radial interval.  Only samples with TERMA
// contribute, and the distance from j to sample k is the difference of the line's radiological
// prefix sums (FP64), so each destination visits just the footprint samples of its segment, in the
// reference's walk order, instead of every sample.
//
// A line has some 40 samples and 4 footprint samples, so the time is the instructions around the
// walks: the segment bounds and the place in the footprint list come from one ballot of the walls and
// one of the footprint samples per 64 samples (bit scans instead of three wave scans and a search), and
// a footprint sample next to the one before it takes its inner cumulative value from that one.
//
// Dynamic LDS: for up to maxn samples the radiological centre (FP64), {half step, TERMA} (8 B) and the
// footprint list (2 B).
__global__ void __launch_bounds__(64) bl_walk_kernel(BlArgs a, const float* __restrict__ H, int maxn, int len_lo) {
    extern __shared__ double s_dyn[];
    __shared__ float4 sTab[2][kMaxRadii];
    __shared__ uint64_t s_wall[kMaxLine / 64], s_foot[kMaxLine / 64];  // walls and footprint samples
    __shared__ int s_first[kMaxLine / 64];                             // footprint samples before each 64
    const int tid = threadIdx.x;
    const int nr = a.nradii;
    if (tid < nr) {
        const float* K = a.tables;
        const float* MR = a.tables + (size_t)a.ntheta * nr + 2 * nr;
        for (int d = 0; d < 2; d++) {
            const float* row = K + (size_t)(d == 0 ? a.rowf : a.rowb) * nr;
            const float lo = tid == 0 ? 0.f : MR[tid - 1];
            const float klo = tid == 0 ? 0.f : row[tid - 1];
            sTab[d][tid] = make_float4(lo, klo, (row[tid] - klo) * MR[nr + tid], MR[tid]);
        }
    }
    double* sC = s_dyn;
    float2* sL = reinterpret_cast<float2*>(s_dyn + maxn);
    short* s_fp = reinterpret_cast<short*>(sL + maxn);
    __syncthreads();
    const float rmax = sTab[0][nr - 1].w, rlast = sTab[0][nr - 2].w;
    const float nphi_f = (float)a.nphi;
    uint32_t iters = 0;
    // a wave walks lines base, base + G, base + 2G, ..., so that neighbouring waves work on neighbouring
    // lines at the same time, and takes the records of its next 64 lines at once, one per lane
    const uint64_t G = gridDim.x;
    for (uint64_t base = xcd_remap(blockIdx.x, gridDim.x); base < a.nlines; base += 64 * G) {
    LineMeta mine{};
    if (base + (uint64_t)tid * G < a.nlines) mine = a.lines[base + (uint64_t)tid * G];
    // empty lines and other launches' lines are skipped here
    uint64_t todo = __ballot(mine.len >= len_lo && mine.len <= maxn);
    while (todo) {
        const int kl = __builtin_ctzll(todo);
        todo &= todo - 1ull;
        const uint32_t moff = (uint32_t)lane_i((int)mine.off, kl);
        const int m = lane_i((int)mine.len, kl);
        // the scans' lane arithmetic is redone per line from an opaque lane id: hoisted out of
        // the line loop, it held some 20 VGPRs for the whole kernel
        int ln = tid;
        __asm__ volatile("" : "+v"(ln));
        const uint64_t upto = (2ull << ln) - 1ull, below = upto >> 1;  // lanes up to and below this one
        float* T = a.rev + moff;
        const float* Hl = H + moff;
        int nfoot = 0;
        for (int c = 0; 64 * c < m; c++) {
            const int j = 64 * c + tid;
            float2 e = make_float2(-1.f, 0.f);  // (behind the line: a wall)
            if (j < m) {
                e = make_float2(Hl[j], T[j]);
                sL[j] = e;
            }
            const uint64_t W = __ballot(e.x < 0.f), F = __ballot(e.y != 0.f);
            if (e.y != 0.f) s_fp[nfoot + __popcll(F & below)] = (short)j;
            if (tid == 0) {
                s_wall[c] = W;
                s_foot[c] = F;
                s_first[c] = nfoot;
            }
            nfoot += __popcll(F);
        }
        __syncthreads();
        // radiological centres: a lane sums its run of samples, a wave scan carries the sums over
        const int per = (m + 63) / 64;
        const int ca = min(m, tid * per), cb = min(m, ca + per);
        double csum = 0.0;
        for (int k = ca; k < cb; k++) {
            const float h = sL[k].x;
            if (!(h < 0.f)) csum += 2.0 * (double)h;
        }
        double pc = csum;
        for (int o = 1; o < 64 && o * per < m; o <<= 1) {  // (lanes behind the line's end add nothing)
            const double uc = bperm_f64(max(ln - o, 0) << 2, pc);
            if (tid >= o) pc += uc;
        }
        double cacc = pc - csum;
        for (int k = ca; k < cb; k++) {
            const float h = sL[k].x;
            const double hh = h < 0.f ? 0.0 : (double)h;
            sC[k] = cacc + hh;
            cacc += 2.0 * hh;
        }
        __syncthreads();
        int wall_before = -1;  // last wall of the samples before the current 64
        for (int c = 0; 64 * c < m; c++) {
            const int j = 64 * c + tid;
            const uint64_t W = s_wall[c], F = s_foot[c];
            int wall_behind = m;  // first wall of the samples behind the current 64
            for (int n = c + 1; 64 * n < m; n++)
                if (const uint64_t v = s_wall[n]) {
                    wall_behind = 64 * n + __builtin_ctzll(v);
                    break;
                }
            if (j < m) {
                const float2 ej = sL[j];
                float sum = 0.f;
                if (ej.x >= 0.f && nfoot > 0) {
                    const uint64_t wl = W & below, wr = W & ~upto;
                    const int slo = (wl ? 64 * c + 63 - __builtin_clzll(wl) : wall_before) + 1;
                    const int shi = (wr ? 64 * c + __builtin_ctzll(wr) : wall_behind) - 1;
                    const double cj = sC[j];
                    const int p = s_first[c] + __popcll(F & below);  // first footprint entry >= j
                    const float r0 = ej.x;
                    for (int d = 0; d < 2; d++) {
                        const float4* tab = sTab[d];
                        int s = 0;
                        float4 iv = tab[0];
                        if (!(r0 <= rmax)) continue;
                        float klast = kc_at(r0, tab, nr, s, iv);
                        sum += klast * ej.y;  // the self sample
                        iters++;
                        if (r0 > rlast) continue;
                        float rl = r0;  // distance to the outer face of the last sample, whose value is klast
                        int kl2 = j;
                        if (d == 0) {
                            for (int q = p - 1; q >= 0; q--) {
                                const int k = s_fp[q];
                                if (k < slo) break;
                                const bool next = k + 1 == kl2;
                                if (!next) rl = (float)(cj - sC[k + 1]);
                                if (rl > rlast) break;
                                const float rk = (float)(cj - sC[k]);
                                if (rk > rmax) break;
                                if (!next) klast = kc_at(rl, tab, nr, s, iv);
                                const float kk = kc_at(rk, tab, nr, s, iv);
                                sum += (kk - klast) * sL[k].y;
                                klast = kk;
                                rl = rk;
                                kl2 = k;
                                iters++;
                            }
                        } else {
                            for (int q = p + (int)(F >> ln & 1ull); q < nfoot; q++) {
                                const int k = s_fp[q];
                                if (k > shi) break;
                                const bool next = k - 1 == kl2;
                                if (!next) rl = (float)(sC[k - 1] - cj);
                                if (rl > rlast) break;
                                const float rk = (float)(sC[k] - cj);
                                if (rk > rmax) break;
                                if (!next) klast = kc_at(rl, tab, nr, s, iv);
                                const float kk = kc_at(rk, tab, nr, s, iv);
                                sum += (kk - klast) * sL[k].y;
                                klast = kk;
                                rl = rk;
                                kl2 = k;
                                iters++;
                            }
                        }
                    }
                }
                T[j] = ej.x >= 0.f ? sum / nphi_f : 0.f;
            }
            if (W) wall_before = 64 * c + 63 - __builtin_clzll(W);
        }
        if (a.zeros && tid < 2 * kLineZeros) T[tid < kLineZeros ? tid - kLineZeros : m + tid - kLineZeros] = 0.f;
        __syncthreads();  // the next line reuses the LDS arrays
    }
    }
    if (a.counts) wave_count(iters, a.counts, blockIdx.x);
}

// Only REV lines with footprint samples in a pillar carry dose in it, and those lines pass within
// sqrt(2)*gw of that pillar's beamlet axis (footprint samples satisfy |x-fc|,|z-fc| <= gw, the
// farthest reach of the footprint bounds, itself <= fw).  The four lines a voxel reads lie within
// sqrt(2) of the line through it, so if that line passes farther than sqrt(2)*(gw + 1) + 0.5 from
// the axes of the voxel's pillar and of the neighbouring pillars it touches, the fetch is zero and
// is skipped.  Depends on pX and pZ only.  The distance times the length of the line's direction in
// the x-z plane, (hx, hz), is a cross product; a neighbour's differs from it by a pillar's width
// (past the grid's last pillar the test is made all the same: the fetch is zero there).
void gather_bound(const BatchDev& B, BlConeDev& c) {
    const float wx = c.kinv_m.m[1], wz = c.kinv_m.m[7];
    const float wn = std::sqrt(wx * wx + wz * wz);
    c.hx = wx;
    c.hz = wz;
    const float bound = 1.41421356f * (B.gw + 1.f) + 0.5f;
    // (negative: a line along the pillars, with the voxel's own distance)
    c.hb = !(B.fw < 1e29f) ? INFINITY : wn > 1e-6f ? bound * wn * (1.f + 1e-5f) + 1e-4f : -bound;
}
__device__ __forceinline__ bool bl_gather_hit(const BatchDev& B, const BlConeDev& c, int pX, int pZ) {
    const float pdx = (float)B.pd[0], pdz = (float)B.pd[2];
    // (exact: pX and pZ are small integers, half a step away from the multiples of the pillar)
    const float rx = (float)pX - floorf(((float)pX + 0.5f) * B.ipd[0]) * pdx;
    const float rz = (float)pZ - floorf(((float)pZ + 0.5f) * B.ipd[2]) * pdz;
    const float dx = rx - B.fc[0], dz = rz - B.fc[1], cross = dx * c.hz - dz * c.hx;
    const float sx = rx < 2.f ? -pdx : (rx >= pdx - 2.f ? pdx : 0.f);
    const float sz = rz < 2.f ? -pdz : (rz >= pdz - 2.f ? pdz : 0.f);
    if (c.hb < 0.f) {
        const float mx = fminf(fabsf(dx), fabsf(dx - sx)), mz = fminf(fabsf(dz), fabsf(dz - sz));
        return sqrtf(mx * mx + mz * mz) <= -c.hb * (1.f + 1e-5f);
    }
    const float nx = sx * c.hz, nz = sz * c.hx;
    return fminf(fminf(fabsf(cross), fabsf(cross - nx)), fminf(fabsf(cross + nz), fabsf(cross - nx + nz))) <= c.hb;
}

// PackedREVtoBEVdose (nvbbRayConvolve_device.cu:427-452) for one cone direction over every batch's
// packed grid: dose += cone dose where it is positive.  One wave per 16x4x4 voxel tile (pY
// fastest), as four 4x4x4 cubes along pY: a load of a cube touches the fewest different REV lines
// over all cone directions (projected area 24 against 42 voxels for a 16x4x1 slab), which is what
// bounds the gather, and a lane keeps one (pX, pZ) for its four voxels, so the pillar test runs once
// per lane instead of once per voxel.  The four voxels' loads are all issued before any of their
// stores, so a lane has four fetches in flight.  One 5 mm beam, 128^3 water, per direction alone on
// the device: 140 us with single-tap loads, 133 with pair loads, 91 with the cubes, 77 with lines that
// end in zeros (half the instructions), 70 with one cache line for the lanes outside their lines.
constexpr int kGatherX = 4;  // the tile's depth along pX
constexpr int kGatherY = 4;  // pY voxels per lane

__global__ void __launch_bounds__(64) bl_gather_kernel(BlArgs a, uint32_t ntiles) {
    const uint32_t tile = xcd_chunks(blockIdx.x, gridDim.x, 64);
    if (tile >= ntiles) return;
    const int lo = a.tile_batch ? (int)a.tile_batch[tile] : 0;
    const BatchDev& B = a.batches[lo];
    const BlConeDev& c = a.cones[lo];
    const uint32_t t = tile - B.tile0;
    const uint32_t row = B.tdiv[0] ? __umulhi(t, B.tdiv[0]) : t / (uint32_t)B.tiles[0];
    const uint32_t plane = B.tdiv[1] ? __umulhi(row, B.tdiv[1]) : row / (uint32_t)B.tiles[1];
    const int ty = (int)(t - row * (uint32_t)B.tiles[0]), tz = (int)(row - plane * (uint32_t)B.tiles[1]), tx = (int)plane;
    const int tid = threadIdx.x;
    const int pY0 = ty * 16 + (tid & 3), pZ = tz * 4 + ((tid >> 2) & 3), pX = tx * kGatherX + (tid >> 4);
    if (pY0 >= B.gd[1] || pZ >= B.gd[2] || pX >= B.gd[0] || !bl_gather_hit(B, c, pX, pZ)) return;
    float old[kGatherY], dc[kGatherY];
    float* dst = a.pdose + B.pdose + (size_t)pY0 + (size_t)B.gd[1] * ((size_t)pZ + (size_t)B.gd[2] * pX);
    v3 at[kGatherY];
    bool inner = true;
#pragma unroll
    for (int s = 0; s < kGatherY; s++) {
        const int pY = pY0 + 4 * s;
        // continuous resampling: the matrix form of rotateKernel (the Rodrigues form differs only
        // in the last bits of the fetch coordinate)
        const v3 rk = c.kfwd_m(mk3((float)pX, (float)pY, (float)pZ));
        // (sample, line y, line z), texel centres at +0.5 (rev_fetch)
        at[s] = mk3(fmaf(-c.minc.y, a.rrv.y, rk.y) + 0.5f - 0.5f, fmaf(-c.minc.z, a.rrv.z, rk.z) + 0.5f - 0.5f,
                    fmaf(-c.minc.x, a.rrv.x, rk.x) + 0.5f - 0.5f);
        // the voxel's packed dose is read before the fetch so that its latency overlaps the
        // fetch's (this lane alone writes the voxel in this launch)
        old[s] = pY < B.gd[1] ? dst[4 * s] : 0.f;
        inner = inner && (pY >= B.gd[1] || (at[s].y >= 0.f && at[s].z >= 0.f && at[s].y < (float)(c.ny - 1) &&
                                            at[s].z < (float)(c.nz - 1)));
    }
    if (a.zeros && __all(inner) && c.ny < (1 << 12) && c.nz < (1 << 12)) {
        // every voxel of the tile has its four lines inside the grid: no test on lines or samples
        const char* m0 = reinterpret_cast<const char*>(a.lines + c.line0);
        const char* m1 = m0 + (size_t)c.ny * sizeof(LineMeta);
        const char* rev0 = reinterpret_cast<const char*>(a.rev - kLineZeros);
        pair_meta q0[kGatherY], q1[kGatherY];
#pragma unroll
        for (int s = 0; s < kGatherY; s++) {
            // (rows past the grid's pY range stay inside the line table: their lane's own records)
            const float y = fminf(fmaxf(at[s].y, 0.f), (float)(c.ny - 2)), z = fminf(fmaxf(at[s].z, 0.f), (float)(c.nz - 2));
            const uint32_t l = mad24((uint32_t)(int)z, (uint32_t)c.ny, (uint32_t)(int)y) * (uint32_t)sizeof(LineMeta);
            q0[s] = *reinterpret_cast<const pair_meta*>(m0 + l);
            q1[s] = *reinterpret_cast<const pair_meta*>(m1 + l);
        }
#pragma unroll
        for (int s = 0; s < kGatherY; s++) {
            const float fu = floorf(at[s].x), x = at[s].x - fu, y = at[s].y - floorf(at[s].y), z = at[s].z - floorf(at[s].z);
            const int i = (int)fu;
            const float t0 = line_lerp(rev0, q0[s].x, q0[s].y, i, x), t1 = line_lerp(rev0, q0[s].z, q0[s].w, i, x);
            const float t2 = line_lerp(rev0, q1[s].x, q1[s].y, i, x), t3 = line_lerp(rev0, q1[s].z, q1[s].w, i, x);
            const float e0 = t0 + y * (t1 - t0), e1 = t2 + y * (t3 - t2);
            dc[s] = pY0 + 4 * s < B.gd[1] ? e0 + z * (e1 - e0) : 0.f;
        }
    } else {
#pragma unroll
        for (int s = 0; s < kGatherY; s++)
            dc[s] = pY0 + 4 * s < B.gd[1]
                        ? rev_fetch(a.lines, a.rev, c.line0, c.nx, c.ny, c.nz, at[s].x + 0.5f, at[s].y + 0.5f, at[s].z + 0.5f)
                        : 0.f;
    }
#pragma unroll
    for (int s = 0; s < kGatherY; s++)
        if (dc[s] > 0.f) dst[4 * s] = old[s] + dc[s];
}

// The batch of every gather tile of a job (one fill per batch range).
__global__ void __launch_bounds__(256) bl_tile_batch_kernel(const BatchDev* __restrict__ batches,
                                                            uint32_t* __restrict__ tb) {
    const int b = blockIdx.y;
    const BatchDev& B = batches[b];
    const uint32_t n = (uint32_t)B.tiles[0] * (uint32_t)B.tiles[1] * (uint32_t)B.tiles[2];
    for (uint32_t t = blockIdx.x * 256 + threadIdx.x; t < n; t += gridDim.x * 256) tb[B.tile0 + t] = (uint32_t)b;
}

// A job's tables from pinned host memory.  (An upload would wait for its copy engine behind the columns of the job
// before, some 6 ms of copies for 27 million entries, and the whole job behind it.)
__global__ void __launch_bounds__(256) bl_table_kernel(uint4* __restrict__ dst, const uint4* __restrict__ src, uint32_t n) {
    for (uint32_t i = blockIdx.x * 256 + threadIdx.x; i < n; i += gridDim.x * 256) dst[i] = src[i];
}

__global__ void __launch_bounds__(256) bl_fill_kernel(float* __restrict__ p, uint64_t n, float v) {
    for (uint64_t i = (uint64_t)blockIdx.x * 256 + threadIdx.x; i < n; i += (uint64_t)gridDim.x * 256) p[i] = v;
}

struct UnpackArgs {
    const BatchDev* batches;
    const BeamletDev* beamlets;
    const float* pdose;
    float* arena;
    int nbeamlets;
    uint64_t narena;
    v3 start, voxel, rvs, rrv;  // (rrv: 1 / rvs)
    int bbs[3];   // calc_bbox start
};

// UnpackBEVDosePillar (nvbbRayConvolve_device.cu:459-521) over each beamlet's voxel box: the
// calc_bbox voxel goes to its pillar (beam then beamlet rotation), rim and walls read nothing, and
// the packed dose is fetched trilinearly.  Arena order inside a box: i outer, j, k inner.
__global__ void __launch_bounds__(256) bl_unpack_kernel(UnpackArgs a) {
    const uint64_t e = (uint64_t)blockIdx.x * 256 + threadIdx.x;
    if (e >= a.narena) return;
    int lo = 0, hi = a.nbeamlets - 1;
    while (lo < hi) {
        int mid = (lo + hi + 1) >> 1;
        if (a.beamlets[mid].arena <= e) lo = mid; else hi = mid - 1;
    }
    const BeamletDev& bl = a.beamlets[lo];
    const BatchDev& B = a.batches[bl.batch];
    const uint64_t le = e - bl.arena;
    const int k = (int)(le % (uint64_t)bl.boxn[2]);
    const int j = (int)((le / (uint64_t)bl.boxn[2]) % (uint64_t)bl.boxn[1]);
    const int i = (int)(le / ((uint64_t)bl.boxn[2] * bl.boxn[1]));
    const int tX = bl.box0[0] + i, tY = bl.box0[1] + j, tZ = bl.box0[2] + k;
    const v3 gc = mk3(((float)tX + (float)a.bbs[0]) * a.voxel.x + a.start.x,
                      ((float)tY + (float)a.bbs[1]) * a.voxel.y + a.start.y,
                      ((float)tZ + (float)a.bbs[2]) * a.voxel.z + a.start.z);
    v3 pidx = div_by(rot1(bl.fwd, rot_fwd(B.beam.beam_fwd, gc - bl.pst)), a.rvs, a.rrv) + 0.5f;
    float v = 0.f;
    const float lo_f = (float)(kWall + kBuffer);
    if (!(pidx.x < lo_f || pidx.y < lo_f || pidx.z < lo_f || pidx.x >= (float)(B.pd[0] - kBuffer) ||
          pidx.y >= (float)(B.pd[1] - kBuffer) || pidx.z >= (float)(B.pd[2] - kBuffer))) {
        pidx = mk3(pidx.x + (float)(bl.pix * B.pd[0]), pidx.y, pidx.z + (float)(bl.piy * B.pd[2]));
        const float dc = tex3_border(a.pdose + B.pdose, B.gd[1], B.gd[2], B.gd[0], pidx.y, pidx.z, pidx.x);
        if (dc > 0.f) v = dc;
    }
    a.arena[e] = v;
}

// ---- sparse columns without an arena -------------------------------------------------------------
// Workgroups walk the calc_bbox rows (i, j) of a beamlet's box in the emission order of _sparsify (i
// outer, j, k inner), 256 rows each.  The pillar's voxels along a row form one interval of k (the
// pillar is a box in its own frame and the frame is affine in k), found by clipping the row
// against the pillar's three slabs (matrix form, widened); inside it the exact unpack test and
// fetch of UnpackBEVDosePillar decide each value.  Nothing is stored between passes: the values
// are recomputed for the max, the counts and the emission.
//
// One workgroup per beamlet left most of the device idle (a job has some 400 beamlets, their boxes up
// to 150 chunks of rows each) and made every pass a chain of its chunks; the three passes took 0.93 ms
// (one 5 mm beam, 128^3 water), 4.1 ms (thorax, 3 beams) and 110 us (32^3 water), by chunks 0.35 ms, 1.4 ms and
// 36 us.  The max and count passes issue VALU in all of their cycles, the emission in 0.77 (one beam) and 0.68
// (thorax).  The emission's launch lasts no less than its longest row, a serial chain of one lane, so a job emits
// all its columns in one launch: by parts of the columns, as they go to the host, it took 1.76 ms of eight
// launches (0.23 of VALU issue) instead of 0.17 ms (one beam), 3.5 instead of 0.56 ms (thorax) and 6.1 instead of
// 0.88 ms (two fine 4pi beams).

struct ColArgs {
    const BatchDev* batches;
    const BeamletDev* beamlets;
    const float* pdose;
    v3 start, voxel, rvs, rrv;  // (rrv: 1 / rvs)
    int bbs[3];        // calc_bbox start
    int nx, ny;        // full volume dims (keys)
    float thresh;
    uint32_t* stat;    // per beamlet {kept, dropped, max bits, 0}
    uint16_t* rowcnt;  // kept entries of every (i, j) row of every beamlet's box
    uint32_t* chunkcnt;  // [beamlet][chunks]: kept entries of every chunk of 256 rows
    int chunks;        // chunks of the largest box
    int beamlet0;      // first beamlet of this launch
    const uint64_t* off;
    uint64_t* keys;
    float* vals;
};

// UnpackBEVDosePillar (nvbbRayConvolve_device.cu:459-521) at one calc_bbox voxel.
__device__ __forceinline__ float pillar_value(const ColArgs& a, const BeamletDev& bl, const BatchDev& B, int tX, int tY,
                                              int tZ) {
    const v3 gc = mk3(((float)tX + (float)a.bbs[0]) * a.voxel.x + a.start.x,
                      ((float)tY + (float)a.bbs[1]) * a.voxel.y + a.start.y,
                      ((float)tZ + (float)a.bbs[2]) * a.voxel.z + a.start.z);
    v3 pidx = div_by(rot1(bl.fwd, rot_fwd(B.beam.beam_fwd, gc - bl.pst)), a.rvs, a.rrv) + 0.5f;
    const float lo_f = (float)(kWall + kBuffer);
    if (pidx.x < lo_f || pidx.y < lo_f || pidx.z < lo_f || pidx.x >= (float)(B.pd[0] - kBuffer) ||
        pidx.y >= (float)(B.pd[1] - kBuffer) || pidx.z >= (float)(B.pd[2] - kBuffer))
        return 0.f;
    pidx = mk3(pidx.x + (float)(bl.pix * B.pd[0]), pidx.y, pidx.z + (float)(bl.piy * B.pd[2]));
    const float dc = tex3_border(a.pdose + B.pdose, B.gd[1], B.gd[2], B.gd[0], pidx.y, pidx.z, pidx.x);
    return dc > 0.f ? dc : 0.f;
}

// k range [k0, k1) of row (tX, tY) that can lie inside the pillar's unpacked region.
__device__ __forceinline__ void pillar_row(const ColArgs& a, const BeamletDev& bl, const BatchDev& B, int tX, int tY,
                                           int& k0, int& k1) {
    const v3 g0 = mk3(((float)tX + (float)a.bbs[0]) * a.voxel.x + a.start.x,
                      ((float)tY + (float)a.bbs[1]) * a.voxel.y + a.start.y,
                      ((float)bl.box0[2] + (float)a.bbs[2]) * a.voxel.z + a.start.z);
    const v3 q0 = bl.fwd_m(g0 - bl.pst) / a.rvs + 0.5f;
    const v3 dq = mk3(bl.fwd_m.m[2] * a.voxel.z / a.rvs.x, bl.fwd_m.m[5] * a.voxel.z / a.rvs.y,
                      bl.fwd_m.m[8] * a.voxel.z / a.rvs.z);
    float t0 = 0.f, t1 = (float)bl.boxn[2];
    const float lo_f = (float)(kWall + kBuffer);
    clip_slab(q0.x, dq.x, lo_f, (float)(B.pd[0] - kBuffer), t0, t1);
    clip_slab(q0.y, dq.y, lo_f, (float)(B.pd[1] - kBuffer), t0, t1);
    clip_slab(q0.z, dq.z, lo_f, (float)(B.pd[2] - kBuffer), t0, t1);
    k0 = 0;
    k1 = 0;
    if (t0 <= t1) {
        k0 = max(0, (int)floorf(t0) - 1);
        k1 = min(bl.boxn[2], (int)ceilf(t1) + 2);
        if (k1 < k0) k1 = k0;
    }
}

// The chunk of rows of a workgroup: its beamlet (of the launch's), and the chunk's place in the box.
// Chunks of a beamlet are neighbours, so they share an L2.
__device__ __forceinline__ int row_chunk(const ColArgs& a, int& chunk) {
    const uint32_t item = xcd_chunks(blockIdx.x, gridDim.x, 64);
    const int q = (int)(item / (uint32_t)a.chunks);
    chunk = (int)(item - (uint32_t)q * (uint32_t)a.chunks);
    return a.beamlet0 + q;
}

// Per-beamlet column statistics of _sparsify (DoseCalcIO/sparse_io.cpp:22-58): max over the
// column (zeros outside the pillar count), kept (v > t * max) and dropped (0 < v <= t * max).  Pass 1:
// the maximum (the bits of a non-negative float order as integers).
__global__ void __launch_bounds__(256) bl_colmax_kernel(ColArgs a) {
    int chunk;
    const int b = row_chunk(a, chunk);
    const BeamletDev& bl = a.beamlets[b];
    const BatchDev& B = a.batches[bl.batch];
    const int rows = bl.boxn[0] * bl.boxn[1], r = chunk * 256 + (int)threadIdx.x;
    float mx = 0.f;
    if (r < rows) {
        const int i = r / bl.boxn[1], j = r - i * bl.boxn[1];
        int k0, k1;
        pillar_row(a, bl, B, bl.box0[0] + i, bl.box0[1] + j, k0, k1);
        for (int k = k0; k < k1; k++)
            mx = fmaxf(mx, pillar_value(a, bl, B, bl.box0[0] + i, bl.box0[1] + j, bl.box0[2] + k));
    }
    for (int o = 32; o > 0; o >>= 1) mx = fmaxf(mx, __shfl_xor(mx, o, 64));
    if ((threadIdx.x & 63) == 0 && mx > 0.f) atomicMax(a.stat + 4 * b + 2, __float_as_uint(mx));
}

// Pass 2: the counts, of every row, chunk and beamlet.
__global__ void __launch_bounds__(256) bl_colcount_kernel(ColArgs a) {
    __shared__ uint32_t s_k[4], s_d[4];
    int chunk;
    const int b = row_chunk(a, chunk);
    const BeamletDev& bl = a.beamlets[b];
    const BatchDev& B = a.batches[bl.batch];
    const int rows = bl.boxn[0] * bl.boxn[1], r = chunk * 256 + (int)threadIdx.x;
    if (chunk * 256 >= rows) return;
    const float cut = a.thresh * __uint_as_float(a.stat[4 * b + 2]);
    uint32_t kept = 0, dropped = 0;
    if (r < rows) {
        const int i = r / bl.boxn[1], j = r - i * bl.boxn[1];
        int k0, k1;
        pillar_row(a, bl, B, bl.box0[0] + i, bl.box0[1] + j, k0, k1);
        for (int k = k0; k < k1; k++) {
            const float v = pillar_value(a, bl, B, bl.box0[0] + i, bl.box0[1] + j, bl.box0[2] + k);
            if (v > cut) kept++;
            else if (v > 0.f) dropped++;
        }
        a.rowcnt[(size_t)bl.row0 + (size_t)r] = (uint16_t)kept;
    }
    for (int o = 32; o > 0; o >>= 1) {
        kept += __shfl_xor(kept, o, 64);
        dropped += __shfl_xor(dropped, o, 64);
    }
    const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
    if (lane == 0) { s_k[w] = kept; s_d[w] = dropped; }
    __syncthreads();
    if (threadIdx.x == 0) {
        const uint32_t tk = s_k[0] + s_k[1] + s_k[2] + s_k[3], td = s_d[0] + s_d[1] + s_d[2] + s_d[3];
        a.chunkcnt[(size_t)b * a.chunks + chunk] = tk;
        if (tk) atomicAdd(a.stat + 4 * b + 0, tk);
        if (td) atomicAdd(a.stat + 4 * b + 1, td);
    }
}

// Exclusive scan of the kept counts over the job's beamlets (one workgroup; n is small).
__global__ void __launch_bounds__(1024) bl_offsets_kernel(uint32_t* __restrict__ stat, int n, uint64_t* __restrict__ off) {
    __shared__ uint64_t s[1024];
    uint64_t carry = 0;
    for (int base = 0; base < n; base += 1024) {
        const int i = base + threadIdx.x;
        const uint64_t v = i < n ? stat[4 * i] : 0;
        s[threadIdx.x] = v;
        __syncthreads();
        for (int o = 1; o < 1024; o <<= 1) {
            const uint64_t add = threadIdx.x >= (unsigned)o ? s[threadIdx.x - o] : 0;
            __syncthreads();
            s[threadIdx.x] += add;
            __syncthreads();
        }
        if (i < n) off[i] = carry + s[threadIdx.x] - v;
        carry += s[1023];
        __syncthreads();
    }
    if (threadIdx.x == 0) off[n] = carry;
}

// Writes each beamlet's kept entries at its offset, key = full-volume linear index, value = dose, in the
// emission order of _sparsify.  A workgroup takes one chunk of 256 rows, one per thread, with their
// kept counts from the count pass; each wave's 64 rows form one contiguous range of the output.  A wave
// fills that range window by window: every lane evaluates its row's values once, in k order, and stages
// the kept entries that fall in the window in LDS; then the wave copies the window out with
// whole-wave, contiguous stores.
constexpr uint32_t kEmitWindow = 512;  // staged entries per wave and round (6 KB)
__global__ void __launch_bounds__(256) bl_emit_kernel(ColArgs a) {
    __shared__ uint64_t s_key[4][kEmitWindow];
    __shared__ float s_val[4][kEmitWindow];
    __shared__ uint32_t s_w[4], s_b[4];
    int chunk;
    const int b = row_chunk(a, chunk);
    const BeamletDev& bl = a.beamlets[b];
    const BatchDev& B = a.batches[bl.batch];
    const uint32_t* cc = a.chunkcnt + (size_t)b * a.chunks;
    const int rows = bl.boxn[0] * bl.boxn[1];
    if (chunk * 256 >= rows || cc[chunk] == 0u) return;
    const int t = threadIdx.x, lane = t & 63, w = t >> 6;
    const float cut = a.thresh * __uint_as_float(a.stat[4 * b + 2]);
    // entries of the beamlet's earlier chunks
    uint32_t earlier = 0;
    for (int c = t; c < chunk; c += 256) earlier += cc[c];
    for (int o = 32; o > 0; o >>= 1) earlier += __shfl_xor(earlier, o, 64);
    const int r = chunk * 256 + t;
    const uint32_t n = r < rows ? (uint32_t)a.rowcnt[(size_t)bl.row0 + (size_t)r] : 0u;
    // inclusive scan of n over the wave, and the waves' totals
    uint32_t inc = n;
    for (int o = 1; o < 64; o <<= 1) {
        const uint32_t u = __shfl_up(inc, o, 64);
        if (lane >= o) inc += u;
    }
    if (lane == 63) s_w[w] = inc;
    if (lane == 0) s_b[w] = earlier;
    __syncthreads();
    uint64_t wout = a.off[b];
    uint32_t most = 0;
    for (int q = 0; q < 4; q++) {
        wout += s_b[q] + (q < w ? s_w[q] : 0u);
        most = max(most, s_w[q]);
    }
    const uint32_t W = s_w[w];
    int X = 0, Y = 0, k = 0, k1 = 0;
    if (n) {
        const int i = r / bl.boxn[1], j = r - i * bl.boxn[1];
        pillar_row(a, bl, B, bl.box0[0] + i, bl.box0[1] + j, k, k1);
        X = bl.box0[0] + i;
        Y = bl.box0[1] + j;
    }
    uint32_t p = inc - n;  // next output of this lane, relative to the wave's range
    // the same number of rounds in every wave (the barriers), enough for the fullest wave
    for (uint32_t wb = 0; wb < most; wb += kEmitWindow) {
        const uint32_t we = min(W, wb + kEmitWindow);
        while (p < inc && p < we && k < k1) {
            const float v = pillar_value(a, bl, B, X, Y, bl.box0[2] + k);
            if (v > cut) {
                s_key[w][p - wb] = ((uint64_t)(bl.box0[2] + k + a.bbs[2]) * (uint64_t)a.ny +
                                    (uint64_t)(Y + a.bbs[1])) * (uint64_t)a.nx + (uint64_t)(X + a.bbs[0]);
                s_val[w][p - wb] = v;
                p++;
            }
            k++;
        }
        __syncthreads();
        for (uint32_t e = wb + (uint32_t)lane; e < we; e += 64) {
            a.keys[wout + e] = s_key[w][e - wb];
            a.vals[wout + e] = s_val[w][e - wb];
        }
        __syncthreads();
    }
}

// ------------------------------------------------------------------------------------------------
// plain path: the reference dataflow on HIP, kept as the baseline the batched path is measured
// against (dosecalc-beamlet/nvbbRayConvolve_host.cu:692-1409): one batch at a time; per cone a
// raytrace over the whole REV grid, PackRowConvolve with one thread per sample, and the
// packed-BEV gather; then per beamlet a full calc_bbox unpack, a device-to-host copy of the
// dense column and a host sparsify.

// cudaBeamletRaytrace (nvbbRayConvolve_device.cu:19-242), one thread per REV sample: density
// (-1e-12 for walls and outside) and the Siddon TERMA of the sample's beamlet.
__global__ void __launch_bounds__(256) plain_ray_kernel(BlArgs a, float* __restrict__ dens, float* __restrict__ terma) {
    const BlConeDev& c = a.cones[0];
    const BatchDev& B = a.batches[c.batch];
    const uint64_t n = (uint64_t)c.nx * c.ny * c.nz;
    const uint64_t i = (uint64_t)blockIdx.x * 256 + threadIdx.x;
    if (i >= n) return;
    const int tX = (int)(i % (uint64_t)c.nx);
    const uint64_t l = i / (uint64_t)c.nx;
    const int tY = (int)(l % (uint64_t)c.ny), tZ = (int)(l / (uint64_t)c.ny);
    float d = -1e-12f, t = 0.f;
    int pidx;
    v3 inp;
    const v3 ipd = mk3(B.ipd[0], B.ipd[1], B.ipd[2]);
    if (bl_locate(a, c, B, ipd, tX, tY, tZ, pidx, inp)) {
        const PillarRec bl = pillar_rec(a.beamlets[B.beamlet0 + pidx]);
        t = point_terma(bl_terma_point(a, B, bl, inp), B.fmap, B.beam, a.spec, a.vd, a.dens, a.bhc, bl.fidx, nullptr);
        d = bl_density(a, march_vol(a.dens, a.vd.nx, a.vd.ny, a.vd.nz), B, bl, inp);
    }
    dens[i] = d;
    terma[i] = t;
}

// PackRowConvolve body for one destination (nvbbRayConvolve_device.cu:284-417): two walks that
// stop at a wall, past the last radius, or after entering the last radial interval.
__device__ float plain_walk(const float* __restrict__ d, const float* __restrict__ T, int n, int tx,
                            const float* __restrict__ R, const float* __restrict__ IW, const float* __restrict__ rowF,
                            const float* __restrict__ rowB, int nr, float delr) {
    if (d[tx] < 0.f) return 0.f;
    float sum = 0.f;
    for (int dir = -1; dir <= 1; dir += 2) {
        const float* row = dir < 0 ? rowF : rowB;
        int k = tx, s = 0;
        float r = 0.f, last = 0.f;
        do {
            if (k < 0 || k >= n || d[k] < 0.f) break;
            const float h = 0.5f * (delr * d[k]);
            r += h;
            if (r > R[nr - 1]) break;
            while (R[s] < r) s++;
            const float lo = s == 0 ? 0.f : R[s - 1];
            const float klo = s == 0 ? 0.f : row[s - 1];
            const float cum = klo + (r - lo) * ((row[s] - klo) * IW[s]);
            sum += (cum - last) * T[k];
            last = cum;
            if (k != tx) r += h;
            k += dir;
        } while (s < nr - 1);
    }
    return sum;
}

// One workgroup per REV line, the line's density and TERMA in LDS.
__global__ void __launch_bounds__(256) plain_conv_kernel(BlArgs a, const float* __restrict__ dens,
                                                         const float* __restrict__ terma, float* __restrict__ out) {
    extern __shared__ float s_pl[];
    __shared__ float sR[kMaxRadii], sIW[kMaxRadii], sF[kMaxRadii], sB[kMaxRadii];
    const BlConeDev& c = a.cones[0];
    const int n = c.nx, tid = threadIdx.x, nr = a.nradii;
    const uint64_t base = (uint64_t)blockIdx.x * n;
    for (int j = tid; j < n; j += 256) {
        s_pl[j] = dens[base + j];
        s_pl[n + j] = terma[base + j];
    }
    if (tid < nr) {
        const float* MR = a.tables + (size_t)a.ntheta * nr + 2 * nr;
        sR[tid] = MR[tid];
        sIW[tid] = MR[nr + tid];
        sF[tid] = a.tables[(size_t)a.rowf * nr + tid];
        sB[tid] = a.tables[(size_t)a.rowb * nr + tid];
    }
    __syncthreads();
    for (int j = tid; j < n; j += 256)
        out[base + j] = plain_walk(s_pl, s_pl + n, n, j, sR, sIW, sF, sB, nr, a.delr) / (float)a.nphi;
}

// Line table of a dense REV grid (every sample stored), so the packed-BEV gather reads it too.
__global__ void __launch_bounds__(256) plain_meta_kernel(LineMeta* __restrict__ lines, uint64_t nlines, int nx) {
    const uint64_t l = (uint64_t)blockIdx.x * 256 + threadIdx.x;
    if (l >= nlines) return;
    LineMeta m;
    m.i0 = 0;
    m.len = (int16_t)nx;
    m.off = (uint32_t)(l * (uint64_t)nx);
    lines[l] = m;
}

// ------------------------------------------------------------------------------------------------
// host planning

namespace {

struct Rev {
    v3 minc;
    uint32_t size[3];
};

// findREV (dosecalc-beamlet/nvbbRayConvolve_host.cu:104-173): REV grid holding the rotated box
// [0, lim]; false when it exceeds max_rev (the reference's ArraySizeError).
bool find_rev(const cccs_problem& p, const uint32_t* max_rev, v3 lim, float theta, float phi, Rev& out) {
    Rot2 kf = rot2_kernel_fwd(theta, phi);
    v3 mn = mk3(FLT_MAX, FLT_MAX, FLT_MAX), mx = mk3(FLT_MIN, FLT_MIN, FLT_MIN);
    for (int c = 0; c < 8; c++) {
        v3 in = mk3(lim.x * (float)(c >> 2 & 1), lim.y * (float)(c >> 1 & 1), lim.z * (float)(c & 1));
        v3 o = rot2(kf, in);
        mn.x = std::min(mn.x, o.x); mn.y = std::min(mn.y, o.y); mn.z = std::min(mn.z, o.z);
        mx.x = std::max(mx.x, o.x); mx.y = std::max(mx.y, o.y); mx.z = std::max(mx.z, o.z);
    }
    out.size[0] = (uint32_t)std::ceil(std::fabs(mx.y - mn.y) / p.rev_longspacing);
    out.size[1] = (uint32_t)std::ceil(std::fabs(mx.z - mn.z) / p.rev_latspacing);
    out.size[2] = (uint32_t)std::ceil(std::fabs(mx.x - mn.x) / p.rev_latspacing);
    out.minc = mn;
    return !(out.size[0] > max_rev[0] || out.size[1] > max_rev[1] || out.size[2] > max_rev[2]);
}

float comp(v3 v, int i) { return i == 0 ? v.x : (i == 1 ? v.y : v.z); }

// One active beamlet of a beam.
struct BeamletPlan {
    int fidx;
    v3 start, end;
    float theta, phi;  // divergence angles of the beamlet axis
    float len;
    v3 pst;
};

struct BeamPlan {
    int beam;                     // position in the request
    const cccs_beam* b;
    std::vector<BeamletPlan> bl;
    int pd[3];
    v3 psize;                     // pillar size [cm]
    float max_bs;                 // largest divergent beamlet width at a beamlet's exit [cm]
    float min_exit;               // smallest source-to-exit distance [cm]
    std::vector<int> bsizes;      // beamlets per batch
};

// calcBeamletAnchors (dosecalc-beamlet/nvbbRayConvolve_host.cu:180-280): beamlet isocentre,
// divergence angles and the entry/exit points of the beamlet axis through the calc_bbox.
bool beamlet_anchor(const cccs_problem& p, const cccs_beam& b, int idx, BeamletPlan& o, v3& biso) {
    const v3 src = ld3(b.source), iso = ld3(b.isocenter);
    const int fx = (int)b.fmap_size[0], fy = (int)b.fmap_size[1];
    const int bx = idx % fx, by = idx / fx;
    const v3 bdiff = mk3(b.beamlet_size[0] * (-0.5f * (float)fx + (float)bx + 0.5f), 0.f,
                         b.beamlet_size[1] * (-0.5f * (float)fy + (float)by + 0.5f));
    biso = iso + rot2(rot2_beam_inv(b.azimuth, b.zenith, b.coll), bdiff);
    o.theta = std::acos(len3(iso - src) / len3(biso - src));
    o.phi = std::atan2(bdiff.z, bdiff.x);
    const v3 voxel = ld3(p.voxel), dstart = ld3(p.start);
    const v3 bb_begin = dstart + voxel * ldu3(p.bbox_start);
    const v3 bb_end = bb_begin + voxel * ldu3(p.bbox_size);
    const double buffer = 0.05;
    const v3 d = biso - src;
    v3 hits[6];
    for (int ax = 0; ax < 3; ax++) {
        const double den = (double)comp(d, ax) + 1e-12;
        const double a1 = (double)(comp(bb_begin, ax) - comp(src, ax)) / den;
        const double a2 = (double)(comp(bb_end, ax) - comp(src, ax)) / den;
        hits[2 * ax] = src + (float)a1 * d;
        hits[2 * ax + 1] = src + (float)a2 * d;
    }
    double dmin = std::numeric_limits<double>::max(), dmax = std::numeric_limits<double>::min();
    o.start = mk3(FLT_MAX, FLT_MAX, FLT_MAX);
    o.end = mk3(FLT_MIN, FLT_MIN, FLT_MIN);
    for (int ax = 0; ax < 3; ax++)
        for (int s = 0; s < 2; s++) {
            const v3 h = hits[2 * ax + s];
            const int a1 = (ax + 1) % 3, a2 = (ax + 2) % 3;
            if (comp(h, a1) + buffer >= comp(bb_begin, a1) && comp(h, a1) - buffer <= comp(bb_end, a1) &&
                comp(h, a2) + buffer >= comp(bb_begin, a2) && comp(h, a2) - buffer <= comp(bb_end, a2)) {
                const float dist = len3(h - src);
                if (dist < dmin) { o.start = h; dmin = len3(o.start - src); }
                if (dist > dmax) { o.end = h; dmax = len3(o.end - src); }
            }
        }
    return dmin < (double)std::numeric_limits<float>::max() && dmax > (double)std::numeric_limits<float>::min();
}

// Pillar sizes, origins and batch sizes of one beam (host.cu:575-834).
int plan_beam(const cccs_ctx* ctx, const cccs_beam& b, const float* fmap, int beam_index, BeamPlan& P) {
    const cccs_problem& p = ctx->prob;
    P.beam = beam_index;
    P.b = &b;
    P.bl.clear();
    P.bsizes.clear();
    const int nf = (int)(b.fmap_size[0] * b.fmap_size[1]);
    const v3 rvs = mk3(p.rev_latspacing, p.rev_longspacing, p.rev_latspacing);
    const v3 src = ld3(b.source);
    float max_len = 0.f, mbx = 0.f, mby = 0.f, min_exit = FLT_MAX;
    for (int i = 0; i < nf; i++) {
        if (!(fmap[i] > 0.f)) continue;
        BeamletPlan o;
        o.fidx = i;
        v3 biso;
        if (!beamlet_anchor(p, b, i, o, biso)) return set_error(CCCS_EGEOM, "beamlet axis misses the calc_bbox");
        o.len = len3(o.end - o.start);
        max_len = std::max(max_len, o.len);
        const float num = len3(o.end - src), den = len3(biso - src);
        mbx = std::max(mbx, b.beamlet_size[0] * num / den);
        mby = std::max(mby, b.beamlet_size[1] * num / den);
        min_exit = std::min(min_exit, num);
        P.bl.push_back(o);
    }
    const int n = (int)P.bl.size();
    if (n == 0) return CCCS_OK;
    const float ke = p.kernel_extent;
    const float plong = max_len + 2.f * ke + (float)kWall * rvs.y;
    const float ptx = mbx + 2.f * ke + (float)kWall * rvs.x;
    const float pty = mby + 2.f * ke + (float)kWall * rvs.x;
    const v3 expand = rvs - mk3(std::fmod(ptx, rvs.x), std::fmod(plong, rvs.y), std::fmod(pty, rvs.z));
    const v3 psize = mk3(ptx, plong, pty) + expand + 2.f * (float)kBuffer * rvs;
    const v3 pdf = psize / rvs;
    P.pd[0] = (int)pdf.x; P.pd[1] = (int)pdf.y; P.pd[2] = (int)pdf.z;
    P.psize = psize;
    P.max_bs = std::max(mbx, mby);
    P.min_exit = min_exit;
    const Rot2 binv = rot2_beam_inv(b.azimuth, b.zenith, b.coll);
    for (BeamletPlan& o : P.bl) {
        v3 go = mk3(-0.5f * (psize.x + (float)kWall * rvs.x), -0.5f * (psize.y - o.len + (float)kWall * rvs.y),
                    -0.5f * (psize.z + (float)kWall * rvs.z));
        go = rot2(binv, rot1(beamlet_rot(o.theta, o.phi, true), go));
        o.pst = o.start + go;
    }
    uint32_t mr[3] = {p.max_rev_size[0], p.max_rev_size[1], p.max_rev_size[2]};
    if (mr[0] == 0) mr[0] = mr[1] = mr[2] = 500;  // dosecalc-preprocess/argparser.h:29
    for (int nb = 1;; nb++) {
        if (nb > kMaxBatches) return set_error(CCCS_ENOMEM, "beamlets do not fit max_rev_size in 100 batches");
        P.bsizes.assign(nb, n / nb);
        for (int r = 0, rem = n - (n / nb) * nb; rem > 0; r++, rem--) P.bsizes[r % nb]++;
        bool ok = true;
        for (int bi = 0; bi < nb && ok; bi++) {
            const int m = P.bsizes[bi];
            const int npx = (int)std::ceil(std::sqrt((float)m));
            const int npy = (int)std::ceil((float)m / (float)npx);
            const v3 gsize = mk3((float)(npx * P.pd[0] + kWall), (float)(P.pd[1] + kWall), (float)(npy * P.pd[2] + kWall)) * rvs;
            for (int r = 0; r < ctx->nrays && ok; r++) {
                Rev rv;
                const float th = ctx->theta[r] * 3.14159265358979323846f / 180.f;
                const float ph = ctx->phi[r] * 3.14159265358979323846f / 180.f;
                if (!find_rev(p, mr, gsize, th, ph, rv)) ok = false;
                else if (rv.size[0] > (uint32_t)kMaxLine) return set_error(CCCS_EGEOM, "REV line longer than 1024 samples");
            }
        }
        if (ok) break;
    }
    return CCCS_OK;
}

struct BatchRef {
    int plan;   // index into the beam plans
    int first;  // first beamlet of the plan in this batch
    int n;
};

// Linear-in-depth bounds of a batch's footprint in the pillar frame, for the sample stage's cull.
// A sample is a footprint sample when its TERMA point lies in its beamlet's fluence cell, i.e.
// inside the pyramid from the source through the cell's corners at the isocentre plane
// (fluence_cell projects centrally from the source).  The pillar frame is a rotation of PVCS
// scaled by 1/rvs (isotropic spacing), so the pyramid stays a pyramid there, and its section at
// pillar depth y has the four corner rays' points as corners, whose x and z are linear in y.  The
// lowest corner x over the batch's beamlets is a minimum of linear functions (concave in y), the
// highest a maximum (convex), so the chords between the depths -0.5 and pd[1] - 0.5 bound them
// from below and above.  (A point on the beam's central axis has no defined cell and takes cell
// 0; the beamlet of cell 0 therefore also counts the axis line.)  out[0..3]: x lower and upper
// bounds of the local packed coordinate (pillar frame + 0.5) as c + s * py, py the packed depth
// coordinate, as {c_lo, s_lo, c_hi, s_hi}; out[4..7] the same for z; widened by `margin` samples.
void footprint_cull(const BatchDev& B, const BeamletDev* bl, v3 rvs, float margin, float out[8]) {
    const BeamDev& bm = B.beam;
    const double y0 = -0.5, y1 = (double)B.pd[1] - 0.5;
    double lo[2][2] = {{1e300, 1e300}, {1e300, 1e300}}, hi[2][2] = {{-1e300, -1e300}, {-1e300, -1e300}};  // [x|z][end]
    for (int q = 0; q < B.n; q++) {
        const BeamletDev& d = bl[q];
        // pillar frame of a PVCS point: fwd_m (p - pst) / rvs
        auto frame = [&](double px, double py, double pz, double f[3]) {
            const double r[3] = {px - d.pst.x, py - d.pst.y, pz - d.pst.z};
            for (int i = 0; i < 3; i++)
                f[i] = ((double)d.fwd_m.m[3 * i] * r[0] + (double)d.fwd_m.m[3 * i + 1] * r[1] +
                        (double)d.fwd_m.m[3 * i + 2] * r[2]) / (double)rvs.x;
        };
        double S[3];
        frame(bm.src.x, bm.src.y, bm.src.z, S);
        const int ix = d.fidx % bm.fmx, iz = d.fidx / bm.fmx;
        const double cx0 = (double)bm.src.x + (double)bm.iso_dist * bm.dir_n.x,
                     cy0 = (double)bm.src.y + (double)bm.iso_dist * bm.dir_n.y,
                     cz0 = (double)bm.src.z + (double)bm.iso_dist * bm.dir_n.z;
        const int ncorner = d.fidx == 0 ? 5 : 4;
        for (int k = 0; k < ncorner; k++) {
            v3 lat = mk3(0.f, 0.f, 0.f);
            if (k < 4) {
                const float ax = (float)(ix + (k & 1)) - 0.5f * (float)bm.fmx;
                const float az = (float)(iz + (k >> 1)) - 0.5f * (float)bm.fmy;
                lat = rot2(B.beam_inv, mk3(ax * bm.bsx, 0.f, az * bm.bsy));  // BEV -> PVCS
            }
            double C[3];
            frame(cx0 + lat.x, cy0 + lat.y, cz0 + lat.z, C);
            for (int e = 0; e < 2; e++) {
                const double y = e == 0 ? y0 : y1;
                const double u = (y - S[1]) / (C[1] - S[1]);
                const double x = S[0] + u * (C[0] - S[0]), z = S[2] + u * (C[2] - S[2]);
                lo[0][e] = std::min(lo[0][e], x); hi[0][e] = std::max(hi[0][e], x);
                lo[1][e] = std::min(lo[1][e], z); hi[1][e] = std::max(hi[1][e], z);
            }
        }
    }
    // local coordinate = frame + 0.5, and depth y = py - 0.5: bound(py) = v(y0) + 0.5 + slope * py
    for (int a = 0; a < 2; a++) {
        const double sl = (lo[a][1] - lo[a][0]) / (y1 - y0), sh = (hi[a][1] - hi[a][0]) / (y1 - y0);
        out[4 * a + 0] = (float)(lo[a][0] + 0.5 - margin);
        out[4 * a + 1] = (float)sl;
        out[4 * a + 2] = (float)(hi[a][0] + 0.5 + margin);
        out[4 * a + 3] = (float)sh;
    }
}

// Device tables and sizes of one job.
struct Job {
    std::vector<BatchDev> batches;
    std::vector<BeamletDev> beamlets;
    std::vector<BlConeDev> cones;          // [ray][batch]
    std::vector<uint64_t> ray_lines;       // lines per ray
    uint64_t max_lines = 0, max_rev = 0, pdose = 0, arena = 0, rows = 0;
    uint64_t pvox = 0;                     // pillar voxels of all beamlets (bounds the sparse output)
    uint32_t tiles = 0;
};

// Calc_bbox-relative voxel box of one pillar's unpacked region (rim excluded), widened by 2.
void pillar_box(const cccs_problem& p, const cccs_beam& b, const BeamletPlan& o, const int* pd, int* box0, int* boxn) {
    const v3 rvs = mk3(p.rev_latspacing, p.rev_longspacing, p.rev_latspacing);
    const Rot2 binv = rot2_beam_inv(b.azimuth, b.zenith, b.coll);
    const Rot1 r = beamlet_rot(o.theta, o.phi, true);
    const float lo = (float)(kWall + kBuffer) - 0.5f;
    double mn[3] = {1e30, 1e30, 1e30}, mx[3] = {-1e30, -1e30, -1e30};
    for (int c = 0; c < 8; c++) {
        v3 q = mk3((c & 1) ? (float)(pd[0] - kBuffer) - 0.5f : lo, (c & 2) ? (float)(pd[1] - kBuffer) - 0.5f : lo,
                   (c & 4) ? (float)(pd[2] - kBuffer) - 0.5f : lo);
        v3 g = rot2(binv, rot1(r, q * rvs)) + o.pst;
        for (int k = 0; k < 3; k++) {
            const double idx = ((double)comp(g, k) - p.start[k]) / p.voxel[k] - (double)p.bbox_start[k];
            mn[k] = std::min(mn[k], idx);
            mx[k] = std::max(mx[k], idx);
        }
    }
    for (int k = 0; k < 3; k++) {
        const long a = std::max(0L, (long)std::floor(mn[k]) - 2);
        const long e = std::min((long)p.bbox_size[k], (long)std::ceil(mx[k]) + 3);
        box0[k] = (int)a;
        boxn[k] = (int)std::max(0L, e - a);
    }
}

// A finished job's sparse columns in pinned host memory, and the event that marks them copied.
struct Delivery {
    bool live = false;
    int nparts = 0;
    hipEvent_t ev[kColParts] = {};  // the copy of each part's columns
    size_t end[kColParts] = {};     // one past the last column of each part
    uint64_t* keys = nullptr;
    float* vals = nullptr;
    const uint32_t* stat = nullptr;  // per column: kept, dropped, (two unused)
    const uint32_t* rcnt = nullptr;  // per column and ROI: kept entries (ROI reduction)
    int nroi = 0;
    std::vector<std::pair<int, int>> cols;  // (request beam, fluence index) per column
};

int build_job(cccs_ctx* ctx, const std::vector<BeamPlan>& plans, const std::vector<BatchRef>& refs,
              const std::vector<const float*>& d_fmaps, Job& J) {
    const cccs_problem& p = ctx->prob;
    const v3 rvs = mk3(p.rev_latspacing, p.rev_longspacing, p.rev_latspacing);
    const int nb = (int)refs.size(), nrays = ctx->nrays;
    J = Job();
    J.batches.resize(nb);
    J.cones.resize((size_t)nrays * nb);
    J.ray_lines.assign(nrays, 0);
    std::vector<uint64_t> ray_rev(nrays, 0);
    uint32_t mr[3] = {p.max_rev_size[0], p.max_rev_size[1], p.max_rev_size[2]};
    if (mr[0] == 0) mr[0] = mr[1] = mr[2] = 500;
    for (int bi = 0; bi < nb; bi++) {
        const BatchRef& R = refs[bi];
        const BeamPlan& P = plans[R.plan];
        const cccs_beam& b = *P.b;
        BatchDev& B = J.batches[bi];
        B.beam = make_beam_dev(b);
        B.beam_inv = rot2_beam_inv(b.azimuth, b.zenith, b.coll);
        B.fmap = d_fmaps[R.plan];
        B.n = R.n;
        B.npx = (int)std::ceil(std::sqrt((float)R.n));
        B.npy = (int)std::ceil((float)R.n / (float)B.npx);
        for (int k = 0; k < 3; k++) B.pd[k] = P.pd[k];
        B.gd[0] = B.npx * P.pd[0] + kWall;
        B.gd[1] = P.pd[1] + kWall;
        B.gd[2] = B.npy * P.pd[2] + kWall;
        B.beamlet0 = (int)J.beamlets.size();
        B.pdose = J.pdose;
        J.pdose += (uint64_t)B.gd[0] * B.gd[1] * B.gd[2];
        B.tiles[0] = (B.gd[1] + 15) / 16;
        B.tiles[1] = (B.gd[2] + 3) / 4;
        B.tiles[2] = (B.gd[0] + kGatherX - 1) / kGatherX;
        for (int k = 0; k < 2; k++) {  // (t * (d * ceil(2^32 / d) - 2^32) < 2^32 for every t below)
            const uint64_t d = (uint64_t)B.tiles[k], n = (uint64_t)B.tiles[0] * B.tiles[1] * B.tiles[2];
            B.tdiv[k] = d >= 2 && n * d < (uint64_t(1) << 32) ? (uint32_t)(((uint64_t(1) << 32) + d - 1) / d) : 0u;
        }
        for (int k = 0; k < 3; k++) B.ipd[k] = 1.f / (float)B.pd[k];
        B.tile0 = J.tiles;
        // footprint prefilter: the beamlet axis runs along the pillar's y axis through its x/z
        // centre; a sample farther from it than half the widest divergent beamlet (at the far end
        // of the pillar, with a 1.2x allowance for the tilt of the cell boundaries) plus one sample
        // cannot project into its beamlet's fluence cell
        B.fc[0] = 0.5f * (P.psize.x / rvs.x + (float)kWall);
        B.fc[1] = 0.5f * (P.psize.z / rvs.z + (float)kWall);
        B.fw = 0.5f * P.max_bs * 1.2f * (1.f + P.psize.y / P.min_exit) / std::min(rvs.x, rvs.z) + 1.f;
        if (std::fabs(rvs.x - rvs.y) > 1e-6f * rvs.x) B.fw = 1e30f;  // the bound assumes isotropic spacing
        const uint64_t nt = (uint64_t)J.tiles + (uint64_t)B.tiles[0] * B.tiles[1] * B.tiles[2];
        if (nt > 0xffffffffULL) return set_error(CCCS_EGEOM, "packed grids too large for one job");
        J.tiles = (uint32_t)nt;
        for (int q = 0; q < R.n; q++) {
            const BeamletPlan& o = P.bl[R.first + q];
            BeamletDev d;
            d.pst = o.pst;
            d.inv = beamlet_rot(o.theta, o.phi, true);
            d.fwd = beamlet_rot(o.theta, o.phi, false);
            d.fwd_m = to_f(dm_mul(dm_beamlet_fwd(o.theta, o.phi), dm_beam_fwd(b.azimuth, b.zenith, b.coll)));
            d.fidx = o.fidx;
            d.batch = bi;
            d.pix = q % B.npx;
            d.piy = q / B.npx;
            pillar_box(p, b, o, P.pd, d.box0, d.boxn);
            d.arena = J.arena;
            J.arena += (uint64_t)d.boxn[0] * d.boxn[1] * d.boxn[2];
            // row counts are 16-bit and row offsets 32-bit
            if (d.boxn[2] > 65535 || J.rows + (uint64_t)d.boxn[0] * d.boxn[1] > 0xffffffffULL)
                return set_error(CCCS_EGEOM, "column boxes too large for one job");
            d.row0 = (uint32_t)J.rows;
            J.rows += (uint64_t)d.boxn[0] * d.boxn[1];
            J.pvox += (uint64_t)P.pd[0] * P.pd[1] * P.pd[2];
            J.beamlets.push_back(d);
        }
        B.gw = B.fw;
        if (B.fw < 1e29f) {
            footprint_cull(B, J.beamlets.data() + B.beamlet0, rvs, 0.05f, B.cb);
            // the bounds' farthest reach from the axis (local frame: axis at fc + 0.5) at either end
            // of the grid's depth range; the bounds are linear, so the ends hold the maximum
            for (int e = 0; e < 2; e++) {
                const float py = e == 0 ? 0.f : (float)B.gd[1];
                for (int ax = 0; ax < 2; ax++) {
                    const float ctr = B.fc[ax] + 0.5f;
                    const float lo = B.cb[4 * ax] + B.cb[4 * ax + 1] * py, hi = B.cb[4 * ax + 2] + B.cb[4 * ax + 3] * py;
                    B.gw = e == 0 && ax == 0 ? std::max(ctr - lo, hi - ctr) : std::max(B.gw, std::max(ctr - lo, hi - ctr));
                }
            }
            B.gw = std::min(B.gw, B.fw);
        } else {  // anisotropic spacing: no bound
            const float nb_[8] = {-1e30f, 0.f, 1e30f, 0.f, -1e30f, 0.f, 1e30f, 0.f};
            std::copy(nb_, nb_ + 8, B.cb);
        }
        const v3 gsize = mk3((float)B.gd[0], (float)B.gd[1], (float)B.gd[2]) * rvs;
        for (int r = 0; r < nrays; r++) {
            const float th = ctx->theta[r] * 3.14159265358979323846f / 180.f;
            const float ph = ctx->phi[r] * 3.14159265358979323846f / 180.f;
            Rev rv;
            if (!find_rev(p, mr, gsize, th, ph, rv)) return set_error(CCCS_EGEOM, "REV grid exceeds max_rev_size");
            if (rv.size[0] > (uint32_t)kMaxLine) return set_error(CCCS_EGEOM, "REV line longer than 1024 samples");
            BlConeDev& c = J.cones[(size_t)r * nb + bi];
            c.kinv = rot2_kernel_inv(th, ph);
            c.kfwd = rot2_kernel_fwd(th, ph);
            c.kinv_m = to_f(dm_kernel_inv(th, ph));
            c.kfwd_m = to_f(dm_kernel_fwd(th, ph));
            c.minc = rv.minc;
            c.nx = (int)rv.size[0];
            c.ny = (int)rv.size[1];
            c.nz = (int)rv.size[2];
            c.batch = bi;
            gather_bound(B, c);
            c.line0 = J.ray_lines[r];
            J.ray_lines[r] += (uint64_t)c.ny * c.nz;
            ray_rev[r] += (uint64_t)c.nx * c.ny * c.nz;
        }
    }
    for (int r = 0; r < nrays; r++) {
        J.max_lines = std::max(J.max_lines, J.ray_lines[r]);
        J.max_rev = std::max(J.max_rev, ray_rev[r]);
    }
    if (J.max_lines > 0x7fffffffULL || J.max_rev > 0xffffffffULL)
        return set_error(CCCS_EGEOM, "REV grids of one cone exceed 2^32 samples in one job");
    return CCCS_OK;
}

BlArgs base_args(cccs_ctx* ctx) {
    const cccs_problem& p = ctx->prob;
    BlArgs a;
    std::memset(&a, 0, sizeof(a));
    a.dens = ctx->d_dens;
    a.tables = ctx->d_tables;
    a.ntheta = (int)p.ntheta;
    a.nradii = (int)p.nradii;
    a.nphi = (int)p.nphi;
    a.delr = p.rev_longspacing;
    a.rvs = mk3(p.rev_latspacing, p.rev_longspacing, p.rev_latspacing);
    a.rrv = mk3(1.f / a.rvs.x, 1.f / a.rvs.y, 1.f / a.rvs.z);
    a.vd = ctx->vol;
    a.ivoxel = mk3(1.f / a.vd.voxel.x, 1.f / a.vd.voxel.y, 1.f / a.vd.voxel.z);
    a.spec = ctx->spec;
    a.bhc = p.beamhard_correct;
    return a;
}

// Line table and REV store with the pads of rev_fetch's pair loads.
inline size_t line_bytes(uint64_t n) { return sizeof(LineMeta) * (size_t)(n + 2 * kRevPad); }
inline size_t rev_bytes(uint64_t n) { return sizeof(float) * (size_t)(n + 2 * kRevPad); }
// Whether a store of `rev` samples in `lines` lines keeps the zeros around its lines, and the samples that it
// then has.
inline bool line_zeros(uint64_t rev, uint64_t lines) {
    return rev + (uint64_t)kLineZeros * lines + 2 * kRevPad < (uint64_t(1) << 30);
}
inline uint64_t store_samples(uint64_t rev, uint64_t lines) {
    return rev + (line_zeros(rev, lines) ? (uint64_t)kLineZeros * lines : 0);
}
// Device bytes of one cone direction in flight: REV store, half steps, line table and the lines' grids (the
// pads apart).
inline uint64_t direction_bytes(uint64_t rev, uint64_t lines) {
    return 2 * sizeof(float) * store_samples(rev, lines) + (sizeof(LineMeta) + sizeof(uint32_t)) * lines;
}

inline unsigned grid_for(uint64_t n, unsigned block) { return (unsigned)std::min<uint64_t>((n + block - 1) / block, 1u << 20); }

// `while_busy` (may be empty) runs on the host once every launch of the job's first pass is
// enqueued, before the host waits for them: host work there overlaps the job on the device.
int run_job_cones(cccs_ctx* ctx, const Job& J, const std::function<int()>& while_busy) {
    const cccs_problem& p = ctx->prob;
    const int nb = (int)J.batches.size(), nrays = ctx->nrays;
    // device tables: batches | beamlets | cones
    const size_t sz_b = sizeof(BatchDev) * nb, sz_l = sizeof(BeamletDev) * J.beamlets.size(),
                 sz_c = sizeof(BlConeDev) * J.cones.size();
    const size_t o_l = (sz_b + 255) & ~size_t(255), o_c = (o_l + sz_l + 255) & ~size_t(255);
    const size_t total = (o_c + sz_c + 15) & ~size_t(15);
    CCCS_TRY(ctx->bl_tab.ensure(total));
    CCCS_HIP(hipStreamSynchronize(ctx->stream));  // the pinned staging buffer may still be in use
    CCCS_TRY(ctx->h_bl.ensure(total));
    uint8_t* h = ctx->h_bl.as<uint8_t>();
    std::memcpy(h, J.batches.data(), sz_b);
    std::memcpy(h + o_l, J.beamlets.data(), sz_l);
    std::memcpy(h + o_c, J.cones.data(), sz_c);
    uint8_t* d = ctx->bl_tab.as<uint8_t>();
    hipLaunchKernelGGL(bl_table_kernel, dim3((unsigned)std::min<size_t>(1024, (total / 16 + 255) / 256)), dim3(256), 0,
                       ctx->stream, reinterpret_cast<uint4*>(d), reinterpret_cast<const uint4*>(h), (uint32_t)(total / 16));
    CCCS_HIP(hipGetLastError());
    CCCS_TRY(ctx->bl_pdose.ensure(sizeof(float) * std::max<uint64_t>(1, J.pdose)));
    CCCS_TRY(ctx->lines.ensure(line_bytes(J.max_lines)));
    // (the zeros around every line count as samples of the store)
    const bool zeros = line_zeros(J.max_rev, J.max_lines);
    const uint64_t max_rev = store_samples(J.max_rev, J.max_lines);
    CCCS_TRY(ctx->rev.ensure(rev_bytes(max_rev)));
    CCCS_TRY(ctx->bl_h.ensure(sizeof(float) * std::max<uint64_t>(1, max_rev)));
    CCCS_TRY(ctx->bl_qcnt.ensure(sizeof(uint32_t) * (size_t)std::max(1, nrays)));
    CCCS_TRY(ctx->h_small.ensure(sizeof(uint32_t) * kMaxRays + 64));
    // TERMA queue: footprint samples are a few percent of the stored samples; the counts are
    // checked after the pass and the pass reruns with larger queues if one overflowed
    uint64_t subcap = std::max<uint64_t>(uint64_t(1) << 14, J.max_rev / 8 / kSubQueues);
    CCCS_TRY(ctx->bl_qcnt.ensure(sizeof(uint32_t) * kSubQueues * kCntStride * (size_t)std::max(1, nrays)));
    CCCS_TRY(ctx->h_small.ensure(sizeof(uint32_t) * kSubQueues * kCntStride * kMaxRays));
    BlArgs a = base_args(ctx);
    a.batches = reinterpret_cast<const BatchDev*>(d);
    a.beamlets = reinterpret_cast<const BeamletDev*>(d + o_l);
    a.lines = ctx->lines.as<LineMeta>() + kRevPad;
    a.rev = ctx->rev.as<float>() + kRevPad;
    a.pdose = ctx->bl_pdose.as<float>();
    a.nbatch = nb;
    a.zeros = zeros;
    CCCS_TRY(ctx->bl_tiles.ensure(sizeof(uint32_t) * std::max<uint32_t>(1, J.tiles)));
    hipLaunchKernelGGL(bl_tile_batch_kernel, dim3(64, (unsigned)nb), dim3(256), 0, ctx->stream, a.batches,
                       ctx->bl_tiles.as<uint32_t>());
    CCCS_HIP(hipGetLastError());
    a.tile_batch = ctx->bl_tiles.as<uint32_t>();
    const int half = (int)p.ntheta / 2;
    // Several cone directions in flight (bl_streams = n): direction r runs on stream r % n with its
    // own line table, REV store, half steps, TERMA queue and scan partials, so consecutive
    // directions' sample, Siddon and walk overlap.  The gathers read-modify-write the shared packed
    // grids, so gather r waits for gather r-1 (an event).  A set is reused by direction r+n on the
    // same stream, after direction r's gather in stream order.
    const int nset = std::min(std::max(ctx->sched.bl_streams, 1), kRaySets);
    hipStream_t S[kRaySets];
    DevBuf *set_lines[kRaySets], *set_rev[kRaySets], *set_h[kRaySets], *set_q[kRaySets], *set_scan[kRaySets];
    S[0] = ctx->stream;
    set_lines[0] = &ctx->lines; set_rev[0] = &ctx->rev; set_h[0] = &ctx->bl_h; set_q[0] = &ctx->bl_queue;
    set_scan[0] = &ctx->scan;
    DevBuf* set_cone[kRaySets];
    set_cone[0] = &ctx->bl_lcone;
    for (int k = 1; k < kRaySets; k++) {
        S[k] = ctx->xstream[k - 1];
        set_lines[k] = &ctx->xlines[k - 1]; set_rev[k] = &ctx->xrev[k - 1]; set_h[k] = &ctx->xh[k - 1];
        set_q[k] = &ctx->xqueue[k - 1]; set_scan[k] = &ctx->xscan[k - 1]; set_cone[k] = &ctx->xlcone[k - 1];
    }
    for (int k = 0; k < nset; k++) CCCS_TRY(set_cone[k]->ensure(sizeof(uint32_t) * std::max<uint64_t>(1, J.max_lines)));
    for (int k = 1; k < nset; k++) {
        CCCS_TRY(set_lines[k]->ensure(line_bytes(J.max_lines)));
        CCCS_TRY(set_rev[k]->ensure(rev_bytes(max_rev)));
        CCCS_TRY(set_h[k]->ensure(sizeof(float) * std::max<uint64_t>(1, max_rev)));
    }
    for (int attempt = 0; attempt < 3; attempt++) {
        subcap = std::min<uint64_t>(subcap, 0xffffffffULL / kSubQueues);
        for (int k = 0; k < nset; k++) CCCS_TRY(set_q[k]->ensure(sizeof(TermaReq) * subcap * kSubQueues));
        uint32_t* qcnt = ctx->bl_qcnt.as<uint32_t>();
        hipLaunchKernelGGL(bl_fill_kernel, dim3(grid_for(J.pdose, 256)), dim3(256), 0, ctx->stream, a.pdose, J.pdose, 0.f);
        hipLaunchKernelGGL(bl_fill_kernel, dim3(grid_for((uint64_t)kSubQueues * kCntStride * nrays, 256)), dim3(256), 0,
                           ctx->stream,
                           reinterpret_cast<float*>(qcnt), (uint64_t)kSubQueues * kCntStride * nrays, 0.f);
        CCCS_HIP(hipGetLastError());
        if (nset > 1) {  // the other streams start after the tables, fills and earlier work
            CCCS_HIP(hipEventRecord(ctx->ray_ev[kRaySets], S[0]));
            for (int k = 1; k < nset; k++) CCCS_HIP(hipStreamWaitEvent(S[k], ctx->ray_ev[kRaySets], 0));
        }
        int last = -1;  // set of the last gather enqueued
        int rc = CCCS_OK;
        for (int r = 0; r < nrays && rc == CCCS_OK; r++) {
            a.cones = reinterpret_cast<const BlConeDev*>(d + o_c) + (size_t)r * nb;
            a.nlines = J.ray_lines[r];
            a.rowf = r % half;
            a.rowb = (int)p.ntheta - 1 - (r % half);
            a.counts = nullptr;
            if (a.nlines == 0) continue;
            const int k = r % nset;
            // the profiling events enqueue on ctx->stream, and the block totals sit in ctx->scan
            ctx->stream = S[k];
            std::swap(ctx->scan, *set_scan[k]);
            a.lines = set_lines[k]->as<LineMeta>() + kRevPad;
            a.line_cone = set_cone[k]->as<uint32_t>();
            a.rev = set_rev[k]->as<float>() + kRevPad;
            float* H = set_h[k]->as<float>();
            TermaReq* q = set_q[k]->as<TermaReq>();
            do {
                const uint32_t nblocks = (uint32_t)((a.nlines + kLineBlock - 1) / kLineBlock);
                if ((rc = ctx->scan.ensure(sizeof(uint32_t) * nblocks)) != CCCS_OK) break;
                a.blocks = ctx->scan.as<uint32_t>();
                hipLaunchKernelGGL(bl_interval_kernel, dim3(nblocks), dim3(kLineBlock), 0, ctx->stream, a);
                if (nblocks > kWaveBlocks)
                    hipLaunchKernelGGL(bl_block_scan_kernel, dim3(1), dim3(kLineBlock), 0, ctx->stream, a.blocks, nblocks);
                if (hipGetLastError() != hipSuccess) { rc = set_error(CCCS_EDEVICE, "interval kernel"); break; }
                uint32_t maxn = 1;
                for (int bi = 0; bi < nb; bi++) maxn = std::max(maxn, (uint32_t)J.cones[(size_t)r * nb + bi].nx);
                const unsigned lw = (unsigned)std::min<uint64_t>(a.nlines, (uint64_t)ctx->sched.bl_sample_waves);
                const unsigned ww = (unsigned)std::min<uint64_t>(a.nlines, (uint64_t)ctx->sched.bl_walk_waves);
                a.counts = prof_counter(ctx, lw);
                int tok = prof_begin(ctx, K_BL_SAMPLE);
                hipLaunchKernelGGL(bl_sample_kernel, dim3(lw), dim3(64), 0, ctx->stream, a, H, q, (uint32_t)subcap,
                                   qcnt + (size_t)kSubQueues * kCntStride * r);
                prof_end(ctx, tok, 0.0, 0.0, a.nlines);
                if (hipGetLastError() != hipSuccess) { rc = set_error(CCCS_EDEVICE, "sample kernel"); break; }
                {
                    const unsigned sb = kSubQueues * 64;
                    uint32_t* cnt = prof_counter(ctx, sb);
                    int ts = prof_begin(ctx, K_BL_SIDDON);
                    hipLaunchKernelGGL(bl_siddon_kernel, dim3(sb), dim3(256), 0, ctx->stream, a, q, (uint32_t)subcap,
                                       (const uint32_t*)(qcnt + (size_t)kSubQueues * kCntStride * r), cnt);
                    prof_end(ctx, ts, 0.0, 0.0, 0);
                    if (hipGetLastError() != hipSuccess) { rc = set_error(CCCS_EDEVICE, "siddon kernel"); break; }
                }
                // length classes (bl_walk_split, twice that, ...; the last ends at the longest
                // line): each launch sizes its LDS for its own longest line, so the short lines,
                // the bulk after trimming, run with more waves per CU
                const uint32_t split = (uint32_t)ctx->sched.bl_walk_split;
                uint32_t bounds[12];
                int nclass = 0;
                for (uint32_t hi = split; split > 0 && hi < maxn && nclass < 11; hi *= 2) bounds[nclass++] = hi;
                bounds[nclass++] = maxn;
                const size_t per = sizeof(double) + sizeof(float2) + sizeof(short);
                uint32_t* wc = prof_counter(ctx, (size_t)nclass * ww);
                int tw = prof_begin(ctx, K_BL_WALK);
                for (int ci = 0; ci < nclass; ci++) {
                    a.counts = wc ? wc + (size_t)ci * ww : nullptr;
                    hipLaunchKernelGGL(bl_walk_kernel, dim3(ww), dim3(64), per * bounds[ci], ctx->stream, a,
                                       (const float*)H, (int)bounds[ci], ci == 0 ? 1 : (int)bounds[ci - 1] + 1);
                }
                prof_end(ctx, tw, 0.0, 0.0, a.nlines);
                if (hipGetLastError() != hipSuccess) { rc = set_error(CCCS_EDEVICE, "walk kernel"); break; }
                a.counts = nullptr;
                if (nset > 1 && last >= 0 && last != k &&
                    hipStreamWaitEvent(ctx->stream, ctx->ray_ev[last], 0) != hipSuccess) {
                    rc = set_error(CCCS_EDEVICE, "stream wait");
                    break;
                }
                int tk = prof_begin(ctx, K_BL_GATHER);
                hipLaunchKernelGGL(bl_gather_kernel, dim3(J.tiles), dim3(64), 0, ctx->stream, a, J.tiles);
                prof_end(ctx, tk, 8.0 * (double)J.pdose, 0.0, J.pdose);
                if (hipGetLastError() != hipSuccess) { rc = set_error(CCCS_EDEVICE, "gather kernel"); break; }
                if (nset > 1 && hipEventRecord(ctx->ray_ev[k], ctx->stream) != hipSuccess) {
                    rc = set_error(CCCS_EDEVICE, "event");
                    break;
                }
                last = k;
            } while (false);
            std::swap(ctx->scan, *set_scan[k]);
            ctx->stream = S[0];
        }
        // join: the first stream continues after every direction's work (the gathers are chained,
        // and no stream has work after its last gather)
        if (nset > 1 && last > 0) CCCS_HIP(hipStreamWaitEvent(S[0], ctx->ray_ev[last], 0));
        if (rc != CCCS_OK) {
            for (int k = 0; k < nset; k++) (void)hipStreamSynchronize(S[k]);
            return rc;
        }
        if (attempt == 0 && while_busy) {
            const int hr = while_busy();
            if (hr != CCCS_OK) {
                for (int k = 0; k < nset; k++) (void)hipStreamSynchronize(S[k]);
                return hr;
            }
        }
        uint32_t* hc = ctx->h_small.as<uint32_t>();
        CCCS_HIP(hipMemcpyAsync(hc, qcnt, sizeof(uint32_t) * kSubQueues * kCntStride * nrays, hipMemcpyDeviceToHost,
                                ctx->stream));
        CCCS_HIP(hipStreamSynchronize(ctx->stream));
        uint64_t need = 0;
        for (int r = 0; r < kSubQueues * nrays; r++) need = std::max<uint64_t>(need, hc[(size_t)r * kCntStride]);
        if (need <= subcap) return CCCS_OK;
        subcap = need + need / 4;
    }
    return set_error(CCCS_ENOMEM, "TERMA queue overflow");
}

int run_job_unpack(cccs_ctx* ctx, const Job& J) {
    const cccs_problem& p = ctx->prob;
    CCCS_TRY(ctx->bl_arena.ensure(sizeof(float) * std::max<uint64_t>(1, J.arena)));
    const size_t sz_b = sizeof(BatchDev) * J.batches.size();
    const size_t o_l = (sz_b + 255) & ~size_t(255);
    UnpackArgs u;
    u.batches = ctx->bl_tab.as<BatchDev>();
    u.beamlets = reinterpret_cast<const BeamletDev*>(ctx->bl_tab.as<uint8_t>() + o_l);
    u.pdose = ctx->bl_pdose.as<float>();
    u.arena = ctx->bl_arena.as<float>();
    u.nbeamlets = (int)J.beamlets.size();
    u.narena = J.arena;
    u.start = ld3(p.start);
    u.voxel = ld3(p.voxel);
    u.rvs = mk3(p.rev_latspacing, p.rev_longspacing, p.rev_latspacing);
    u.rrv = mk3(1.f / u.rvs.x, 1.f / u.rvs.y, 1.f / u.rvs.z);
    for (int k = 0; k < 3; k++) u.bbs[k] = (int)p.bbox_start[k];
    if (J.arena == 0) return CCCS_OK;
    const uint64_t blocks = (J.arena + 255) / 256;
    if (blocks > 0x7fffffffULL) return set_error(CCCS_EGEOM, "column arena too large for one job");
    int tok = prof_begin(ctx, K_BL_UNPACK);
    hipLaunchKernelGGL(bl_unpack_kernel, dim3((unsigned)blocks), dim3(256), 0, ctx->stream, u);
    prof_end(ctx, tok, 8.0 * (double)J.arena, 0.0, J.arena);
    CCCS_HIP(hipGetLastError());
    return CCCS_OK;
}

// Keeps v > t * max(column) in the reference's emission order (_sparsify, sparse_io.cpp:22-58) for a
// column stored i outer, k inner over the whole calc_bbox.
void sparsify_host(const float* col, const cccs_problem& p, float thresh, std::vector<uint64_t>& keys,
                   std::vector<float>& vals, uint64_t& dropped) {
    const uint64_t bx = p.bbox_size[0], by = p.bbox_size[1], bz = p.bbox_size[2], n = bx * by * bz;
    float mx = 0.f;
    for (uint64_t e = 0; e < n; e++) mx = std::max(mx, col[e]);
    const float cut = thresh * mx;
    keys.clear();
    vals.clear();
    dropped = 0;
    uint64_t e = 0;
    for (uint64_t i = 0; i < bx; i++)
        for (uint64_t j = 0; j < by; j++)
            for (uint64_t k = 0; k < bz; k++, e++) {
                const float v = col[e];
                if (v <= cut) {
                    if (v > 0.f) dropped++;
                    continue;
                }
                keys.push_back(((k + p.bbox_start[2]) * p.size[1] + (j + p.bbox_start[1])) * p.size[0] +
                               (i + p.bbox_start[0]));
                vals.push_back(v);
            }
}

// The plain path for one batch (see plain_ray_kernel): per cone raytrace / convolve / gather
// launches, then per beamlet a full calc_bbox unpack copied to the host and sparsified there by
// worker threads while the device unpacks the next group.
int run_plain_batch(cccs_ctx* ctx, const std::vector<BeamPlan>& plans, const BatchRef& R,
                    const std::vector<const float*>& d_fmaps, float thresh, cccs_sparse_sink sink, void* user) {
    const cccs_problem& p = ctx->prob;
    Job J;
    CCCS_TRY(build_job(ctx, plans, std::vector<BatchRef>{R}, d_fmaps, J));
    const uint64_t nbb = (uint64_t)p.bbox_size[0] * p.bbox_size[1] * p.bbox_size[2];
    for (BeamletDev& d : J.beamlets) {
        for (int k = 0; k < 3; k++) { d.box0[k] = 0; d.boxn[k] = (int)p.bbox_size[k]; }
        d.arena = 0;
    }
    J.arena = nbb;
    const int nrays = ctx->nrays;
    const size_t sz_b = sizeof(BatchDev), sz_l = sizeof(BeamletDev) * J.beamlets.size(),
                 sz_c = sizeof(BlConeDev) * J.cones.size();
    const size_t o_l = (sz_b + 255) & ~size_t(255), o_c = (o_l + sz_l + 255) & ~size_t(255);
    CCCS_TRY(ctx->bl_tab.ensure(o_c + sz_c));
    CCCS_HIP(hipStreamSynchronize(ctx->stream));
    CCCS_TRY(ctx->h_bl.ensure(o_c + sz_c));
    uint8_t* h = ctx->h_bl.as<uint8_t>();
    std::memcpy(h, J.batches.data(), sz_b);
    std::memcpy(h + o_l, J.beamlets.data(), sz_l);
    std::memcpy(h + o_c, J.cones.data(), sz_c);
    uint8_t* d = ctx->bl_tab.as<uint8_t>();
    CCCS_HIP(hipMemcpyAsync(d, h, o_c + sz_c, hipMemcpyHostToDevice, ctx->stream));
    uint64_t max_rev = 0, max_lines = 0;
    for (const BlConeDev& c : J.cones) {
        max_rev = std::max<uint64_t>(max_rev, (uint64_t)c.nx * c.ny * c.nz);
        max_lines = std::max<uint64_t>(max_lines, (uint64_t)c.ny * c.nz);
    }
    if (max_rev > 0xffffffffULL) return set_error(CCCS_EGEOM, "REV grid exceeds 2^32 samples");
    CCCS_TRY(ctx->bl_pdose.ensure(sizeof(float) * std::max<uint64_t>(1, J.pdose)));
    CCCS_TRY(ctx->lines.ensure(line_bytes(max_lines)));
    CCCS_TRY(ctx->rev.ensure(rev_bytes(max_rev)));
    CCCS_TRY(ctx->bl_h.ensure(sizeof(float) * 2 * std::max<uint64_t>(1, max_rev)));
    BlArgs a = base_args(ctx);
    a.batches = reinterpret_cast<const BatchDev*>(d);
    a.beamlets = reinterpret_cast<const BeamletDev*>(d + o_l);
    a.lines = ctx->lines.as<LineMeta>() + kRevPad;
    a.rev = ctx->rev.as<float>() + kRevPad;
    a.pdose = ctx->bl_pdose.as<float>();
    a.nbatch = 1;
    float* dd = ctx->bl_h.as<float>();
    float* dt = dd + max_rev;
    hipLaunchKernelGGL(bl_fill_kernel, dim3(grid_for(J.pdose, 256)), dim3(256), 0, ctx->stream, a.pdose, J.pdose, 0.f);
    const int half = (int)p.ntheta / 2;
    for (int r = 0; r < nrays; r++) {
        const BlConeDev& c = J.cones[r];
        a.cones = reinterpret_cast<const BlConeDev*>(d + o_c) + r;
        a.nlines = (uint64_t)c.ny * c.nz;
        a.rowf = r % half;
        a.rowb = (int)p.ntheta - 1 - (r % half);
        const uint64_t nrev = (uint64_t)c.nx * c.ny * c.nz;
        if (nrev == 0) continue;
        int t0 = prof_begin(ctx, K_PL_RAY);
        hipLaunchKernelGGL(plain_ray_kernel, dim3((unsigned)((nrev + 255) / 256)), dim3(256), 0, ctx->stream, a, dd, dt);
        prof_end(ctx, t0, 8.0 * (double)nrev, 0.0, nrev);
        int t1 = prof_begin(ctx, K_PL_CONV);
        hipLaunchKernelGGL(plain_conv_kernel, dim3((unsigned)a.nlines), dim3(256), sizeof(float) * 2 * c.nx, ctx->stream,
                           a, (const float*)dd, (const float*)dt, a.rev);
        prof_end(ctx, t1, 12.0 * (double)nrev, 0.0, nrev);
        hipLaunchKernelGGL(plain_meta_kernel, dim3((unsigned)((a.nlines + 255) / 256)), dim3(256), 0, ctx->stream, a.lines,
                           a.nlines, c.nx);
        int t2 = prof_begin(ctx, K_BL_GATHER);
        hipLaunchKernelGGL(bl_gather_kernel, dim3(J.tiles), dim3(64), 0, ctx->stream, a, J.tiles);
        prof_end(ctx, t2, 8.0 * (double)J.pdose, 0.0, J.pdose);
        CCCS_HIP(hipGetLastError());
    }
    // per beamlet: dense unpack -> host -> sparsify (groups of G, two pinned slot sets)
    const int G = 8, nbl = (int)J.beamlets.size();
    CCCS_TRY(ctx->bl_arena.ensure(sizeof(float) * nbb * G));
    CCCS_HIP(hipStreamSynchronize(ctx->stream));
    CCCS_TRY(ctx->h_bl_out.ensure(sizeof(float) * nbb * 2 * G));
    float* pin = ctx->h_bl_out.as<float>();
    std::vector<std::vector<uint64_t>> keys(2 * G);
    std::vector<std::vector<float>> vals(2 * G);
    std::vector<uint64_t> drop(2 * G);
    std::vector<std::thread> workers;
    struct Joiner {  // no early return leaves a worker running
        std::vector<std::thread>& w;
        ~Joiner() {
            for (std::thread& t : w)
                if (t.joinable()) t.join();
        }
    } joiner{workers};
    int pending0 = -1;  // first beamlet of the group being sparsified
    auto emit = [&](int g0) -> int {
        for (std::thread& t : workers) t.join();
        workers.clear();
        const int set = (g0 / G) % 2;
        for (int q = g0; q < std::min(nbl, g0 + G); q++) {
            const int sl = set * G + (q - g0);
            cccs_sparse_column col{};
            col.beam_index = plans[R.plan].beam;
            col.beamlet_index = J.beamlets[q].fidx;
            col.nnz = keys[sl].size();
            col.keys = keys[sl].data();
            col.values = vals[sl].data();
            col.perc_nonzero = (float)(100.0 * (double)keys[sl].size() / (double)nbb);
            col.perc_dropped = (float)(100.0 * (double)drop[sl] / (double)nbb);
            if (sink(user, &col) != 0) return set_error(CCCS_EIO, "sparse sink aborted the call");
        }
        return CCCS_OK;
    };
    UnpackArgs u;
    u.batches = reinterpret_cast<const BatchDev*>(d);
    u.pdose = a.pdose;
    u.nbeamlets = 1;
    u.narena = nbb;
    u.start = ld3(p.start);
    u.voxel = ld3(p.voxel);
    u.rvs = a.rvs;
    u.rrv = a.rrv;
    for (int k = 0; k < 3; k++) u.bbs[k] = (int)p.bbox_start[k];
    for (int g0 = 0; g0 < nbl; g0 += G) {
        const int set = (g0 / G) % 2;
        for (int q = g0; q < std::min(nbl, g0 + G); q++) {
            u.beamlets = reinterpret_cast<const BeamletDev*>(d + o_l) + q;
            u.arena = ctx->bl_arena.as<float>() + nbb * (size_t)(q - g0);
            int tk = prof_begin(ctx, K_BL_UNPACK);
            hipLaunchKernelGGL(bl_unpack_kernel, dim3((unsigned)((nbb + 255) / 256)), dim3(256), 0, ctx->stream, u);
            prof_end(ctx, tk, 8.0 * (double)nbb, 0.0, nbb);
            CCCS_HIP(hipMemcpyAsync(pin + nbb * (size_t)(set * G + (q - g0)), u.arena, sizeof(float) * nbb,
                                    hipMemcpyDeviceToHost, ctx->stream));
        }
        CCCS_HIP(hipStreamSynchronize(ctx->stream));
        if (pending0 >= 0) CCCS_TRY(emit(pending0));
        for (int q = g0; q < std::min(nbl, g0 + G); q++) {
            const int sl = set * G + (q - g0);
            const float* col = pin + nbb * (size_t)sl;
            workers.emplace_back([&, col, sl] { sparsify_host(col, p, thresh, keys[sl], vals[sl], drop[sl]); });
        }
        pending0 = g0;
    }
    if (pending0 >= 0) CCCS_TRY(emit(pending0));
    return CCCS_OK;
}

// One batch's share of a job's device footprint: REV samples and lines per cone direction, and
// the packed grid plus the sparse-output bound (12 B per pillar voxel) in bytes.
int batch_footprint(const cccs_ctx* ctx, const std::vector<BeamPlan>& plans, const BatchRef& R,
                    std::vector<uint64_t>& rev, std::vector<uint64_t>& lines, uint64_t& fixed) {
    const cccs_problem& p = ctx->prob;
    const BeamPlan& P = plans[R.plan];
    const v3 rvs = mk3(p.rev_latspacing, p.rev_longspacing, p.rev_latspacing);
    uint32_t mr[3] = {p.max_rev_size[0], p.max_rev_size[1], p.max_rev_size[2]};
    if (mr[0] == 0) mr[0] = mr[1] = mr[2] = 500;
    const int npx = (int)std::ceil(std::sqrt((float)R.n));
    const int npy = (int)std::ceil((float)R.n / (float)npx);
    const uint64_t gd0 = (uint64_t)npx * P.pd[0] + kWall, gd1 = (uint64_t)P.pd[1] + kWall,
                   gd2 = (uint64_t)npy * P.pd[2] + kWall;
    const v3 gsize = mk3((float)gd0, (float)gd1, (float)gd2) * rvs;
    rev.assign(ctx->nrays, 0);
    lines.assign(ctx->nrays, 0);
    for (int r = 0; r < ctx->nrays; r++) {
        const float th = ctx->theta[r] * 3.14159265358979323846f / 180.f;
        const float ph = ctx->phi[r] * 3.14159265358979323846f / 180.f;
        Rev rv;
        if (!find_rev(p, mr, gsize, th, ph, rv)) return set_error(CCCS_EGEOM, "REV grid exceeds max_rev_size");
        rev[r] = (uint64_t)rv.size[0] * rv.size[1] * rv.size[2];
        lines[r] = (uint64_t)rv.size[1] * rv.size[2];
    }
    fixed = sizeof(float) * gd0 * gd1 * gd2 + 12ull * (uint64_t)R.n * P.pd[0] * P.pd[1] * P.pd[2];
    return CCCS_OK;
}


}  // namespace

}  // namespace cccs

using namespace cccs;

// =================================================================================================
// C-ABI

namespace {

// Uploads the fluence maps of the plans (one device block, pinned staging).
int upload_fmaps(cccs_ctx* ctx, const std::vector<BeamPlan>& plans, const float* const* fluence,
                 std::vector<const float*>& d_fmaps) {
    size_t total = 0;
    std::vector<size_t> off(plans.size());
    for (size_t i = 0; i < plans.size(); i++) {
        off[i] = total;
        total += (size_t)plans[i].b->fmap_size[0] * plans[i].b->fmap_size[1];
    }
    CCCS_TRY(ctx->bl_fmap.ensure(sizeof(float) * std::max<size_t>(1, total)));
    CCCS_HIP(hipStreamSynchronize(ctx->stream));
    CCCS_TRY(ctx->h_bl_out.ensure(sizeof(float) * std::max<size_t>(1, total)));
    float* h = ctx->h_bl_out.as<float>();
    for (size_t i = 0; i < plans.size(); i++)
        std::memcpy(h + off[i], fluence[plans[i].beam],
                    sizeof(float) * plans[i].b->fmap_size[0] * plans[i].b->fmap_size[1]);
    CCCS_HIP(hipMemcpyAsync(ctx->bl_fmap.p, h, sizeof(float) * total, hipMemcpyHostToDevice, ctx->stream));
    d_fmaps.resize(plans.size());
    for (size_t i = 0; i < plans.size(); i++) d_fmaps[i] = ctx->bl_fmap.as<float>() + off[i];
    return CCCS_OK;
}

// Runs the cone passes and the unpack of one job (the arena then holds every beamlet's box).
int run_job(cccs_ctx* ctx, const std::vector<BeamPlan>& plans, const std::vector<BatchRef>& refs,
            const std::vector<const float*>& d_fmaps, Job& J) {
    CCCS_TRY(build_job(ctx, plans, refs, d_fmaps, J));
    CCCS_TRY(run_job_cones(ctx, J, std::function<int()>()));
    return run_job_unpack(ctx, J);
}

std::vector<BatchRef> all_batches(const std::vector<BeamPlan>& plans) {
    std::vector<BatchRef> refs;
    for (size_t i = 0; i < plans.size(); i++) {
        int first = 0;
        for (int n : plans[i].bsizes) {
            refs.push_back(BatchRef{(int)i, first, n});
            first += n;
        }
    }
    return refs;
}

}  // namespace

namespace {

// ---- ROI reduction (_reduce_by_roi, DoseCalcIO/sparse_io.cpp:62-158) ------------------------------
constexpr int kMaxRoi = 64;

struct RoiDev {
    int c0[3], cs[3];    // crop box start and size on the CT grid
    uint64_t rank_off;   // first rank entry (crop box, x fastest; -1 outside the mask)
    uint64_t mark;       // voxels of all earlier ROIs (first key of this block)
};

struct RoiArgs {
    const RoiDev* rois;
    const int32_t* rank;
    int nroi;
    int nx, ny;                  // CT grid
    const uint64_t* keys;        // the job's kept entries, column after column
    const float* vals;
    const uint64_t* off;         // first entry of each column (nbl + 1)
    uint32_t* cnt;               // [column][roi] reduced counts
    const uint64_t* roff;        // [column][roi] first reduced entry (exclusive scan of cnt)
    uint64_t* rkeys;
    float* rvals;
};

// ROI rank of CT voxel `key` in ROI r (or -1).
__device__ __forceinline__ int32_t roi_rank(const RoiArgs& a, const RoiDev& R, int x, int y, int z) {
    const int lx = x - R.c0[0], ly = y - R.c0[1], lz = z - R.c0[2];
    if (lx < 0 || ly < 0 || lz < 0 || lx >= R.cs[0] || ly >= R.cs[1] || lz >= R.cs[2]) return -1;
    return a.rank[R.rank_off + (uint64_t)lx + (uint64_t)R.cs[0] * ((uint64_t)ly + (uint64_t)R.cs[1] * lz)];
}

// Pass 1: per column and ROI, the number of kept entries inside the ROI (one LDS add per wave,
// chunk and ROI).
__global__ void __launch_bounds__(256) roi_count_kernel(RoiArgs a) {
    __shared__ uint32_t s_c[kMaxRoi];
    const int q = (int)blockIdx.x, tid = threadIdx.x, lane = tid & 63;
    for (int r = tid; r < a.nroi; r += 256) s_c[r] = 0u;
    __syncthreads();
    const uint64_t e0 = a.off[q], e1 = a.off[q + 1];
    const uint64_t plane = (uint64_t)a.nx * (uint64_t)a.ny;
    for (uint64_t base = e0; base < e1; base += 256) {
        const uint64_t e = base + tid;
        int x = -1, y = -1, z = -1;
        if (e < e1) {
            const uint64_t key = a.keys[e];
            z = (int)(key / plane);
            const int rem = (int)(key - (uint64_t)z * plane);
            y = rem / a.nx;
            x = rem - y * a.nx;
        }
        for (int r = 0; r < a.nroi; r++) {
            const uint64_t m = __ballot(e < e1 && roi_rank(a, a.rois[r], x, y, z) >= 0);
            if (lane == 0 && m) atomicAdd(&s_c[r], (uint32_t)__popcll(m));
        }
    }
    __syncthreads();
    for (int r = tid; r < a.nroi; r += 256) a.cnt[(size_t)q * a.nroi + r] = s_c[r];
}

// Pass 2: ROI by ROI, the column's entries inside the ROI in the column's order (an
// order-preserving compaction per 256-entry chunk), keyed mark + rank.
__global__ void __launch_bounds__(256) roi_emit_kernel(RoiArgs a) {
    __shared__ uint32_t s_w[4];
    const int q = (int)blockIdx.x, tid = threadIdx.x, lane = tid & 63, wid = tid >> 6;
    const uint64_t e0 = a.off[q], e1 = a.off[q + 1];
    const uint64_t plane = (uint64_t)a.nx * (uint64_t)a.ny;
    const uint64_t lt = (1ull << lane) - 1ull;
    for (int r = 0; r < a.nroi; r++) {
        const RoiDev R = a.rois[r];
        uint64_t pos = a.roff[(size_t)q * a.nroi + r];
        for (uint64_t base = e0; base < e1; base += 256) {
            const uint64_t e = base + tid;
            int32_t rk = -1;
            if (e < e1) {
                const uint64_t key = a.keys[e];
                const int z = (int)(key / plane), rem = (int)(key - (uint64_t)z * plane);
                const int y = rem / a.nx, x = rem - y * a.nx;
                rk = roi_rank(a, R, x, y, z);
            }
            const uint64_t m = __ballot(rk >= 0);
            if (lane == 0) s_w[wid] = (uint32_t)__popcll(m);
            __syncthreads();
            uint32_t before = 0, total = 0;
            for (int w = 0; w < 4; w++) {
                before += w < wid ? s_w[w] : 0u;
                total += s_w[w];
            }
            if (rk >= 0) {
                const uint64_t o = pos + before + (uint32_t)__popcll(m & lt);
                a.rkeys[o] = R.mark + (uint64_t)rk;
                a.rvals[o] = a.vals[e];
            }
            pos += total;
            __syncthreads();
        }
    }
}

// Exclusive scan of n uint32 counts into n+1 uint64 offsets (one workgroup, serial chunks).
__global__ void __launch_bounds__(1024) roi_scan_kernel(const uint32_t* __restrict__ cnt, size_t n,
                                                        uint64_t* __restrict__ out) {
    __shared__ uint64_t s_p[1024];
    const int tid = threadIdx.x;
    const size_t per = (n + 1023) / 1024;
    const size_t c0 = std::min(n, (size_t)tid * per), c1 = std::min(n, c0 + per);
    uint64_t loc = 0;
    for (size_t i = c0; i < c1; i++) loc += cnt[i];
    s_p[tid] = loc;
    __syncthreads();
    for (int o = 1; o < 1024; o <<= 1) {
        const uint64_t v = tid >= o ? s_p[tid - o] : 0;
        __syncthreads();
        s_p[tid] += v;
        __syncthreads();
    }
    uint64_t run = s_p[tid] - loc;
    for (size_t i = c0; i < c1; i++) {
        out[i] = run;
        run += cnt[i];
    }
    if (tid == 1023) out[n] = s_p[1023];
}

}  // namespace

extern "C" int cccs_set_roi_masks(cccs_ctx* ctx, int nroi, const uint8_t* const* masks, const uint32_t* crop_start,
                                  const uint32_t* crop_size) {
    clear_error();
    if (!ctx || nroi < 0 || (nroi > 0 && (!masks || !crop_start || !crop_size))) return set_error(CCCS_EINVAL, "null argument");
    if (nroi > kMaxRoi) return set_error(CCCS_EINVAL, "at most " + std::to_string(kMaxRoi) + " ROIs");
    CCCS_HIP(hipSetDevice(ctx->device));
    ctx->nroi = 0;
    if (nroi == 0) return CCCS_OK;
    const cccs_problem& p = ctx->prob;
    std::vector<RoiDev> tab((size_t)nroi);
    std::vector<int32_t> rank;
    uint64_t mark = 0;
    for (int r = 0; r < nroi; r++) {
        RoiDev& R = tab[(size_t)r];
        for (int k = 0; k < 3; k++) {
            R.c0[k] = (int)crop_start[3 * r + k];
            R.cs[k] = (int)crop_size[3 * r + k];
            if (crop_start[3 * r + k] + (uint64_t)crop_size[3 * r + k] > p.size[k])
                return set_error(CCCS_EINVAL, "ROI crop box outside the CT grid");  // sparse_io.cpp:111-113
        }
        if (!masks[r]) return set_error(CCCS_EINVAL, "null ROI mask");
        R.rank_off = rank.size();
        R.mark = mark;
        const size_t n = (size_t)R.cs[0] * R.cs[1] * R.cs[2];
        rank.resize(rank.size() + n, -1);
        int32_t* rk = rank.data() + R.rank_off;
        int32_t elem = 0;
        // the reference's iteration: ii (x) outer, jj (y), kk (z) inner over the crop box
        for (int ii = 0; ii < R.cs[0]; ii++)
            for (int jj = 0; jj < R.cs[1]; jj++)
                for (int kk = 0; kk < R.cs[2]; kk++) {
                    const size_t ck = ((size_t)kk * R.cs[1] + jj) * R.cs[0] + ii;
                    if (masks[r][ck]) rk[ck] = elem++;
                }
        mark += (uint64_t)elem;
    }
    CCCS_TRY(ctx->roi_tab.ensure(sizeof(RoiDev) * tab.size()));
    CCCS_TRY(ctx->roi_rank.ensure(sizeof(int32_t) * std::max<size_t>(1, rank.size())));
    CCCS_HIP(hipStreamSynchronize(ctx->stream));
    CCCS_HIP(hipMemcpy(ctx->roi_tab.p, tab.data(), sizeof(RoiDev) * tab.size(), hipMemcpyHostToDevice));
    if (!rank.empty())
        CCCS_HIP(hipMemcpy(ctx->roi_rank.p, rank.data(), sizeof(int32_t) * rank.size(), hipMemcpyHostToDevice));
    ctx->nroi = nroi;
    return CCCS_OK;
}

extern "C" int cccs_beamlet_footprint(const cccs_ctx* ctx, const cccs_beam* beam, const float* fluence, uint64_t* bytes) {
    clear_error();
    if (!ctx || !beam || !fluence || !bytes) return set_error(CCCS_EINVAL, "null argument");
    *bytes = 0;
    CCCS_TRY(check_beam(ctx, *beam));
    std::vector<BeamPlan> plans(1);
    CCCS_TRY(plan_beam(ctx, *beam, fluence, 0, plans[0]));
    if (plans[0].bl.empty()) return CCCS_OK;
    const std::vector<BatchRef> refs = all_batches(plans);
    std::vector<uint64_t> rev(ctx->nrays, 0), lines(ctx->nrays, 0), r1, l1;
    uint64_t fixed = 0, f1 = 0;
    for (const BatchRef& R : refs) {
        CCCS_TRY(batch_footprint(ctx, plans, R, r1, l1, f1));
        for (int r = 0; r < ctx->nrays; r++) { rev[r] += r1[r]; lines[r] += l1[r]; }
        fixed += f1;
    }
    uint64_t mr = 0, ml = 0;
    for (int r = 0; r < ctx->nrays; r++) { mr = std::max(mr, rev[r]); ml = std::max(ml, lines[r]); }
    *bytes = fixed + direction_bytes(mr, ml);
    return CCCS_OK;
}

extern "C" int cccs_sink_count(void* user, const cccs_sparse_column* column) {
    if (!user || !column) return 1;
    cccs_sink_totals* t = static_cast<cccs_sink_totals*>(user);
    t->columns++;
    t->nnz += column->nnz;
    double s = 0.0;
    for (uint64_t i = 0; i < column->nnz; i++) s += column->values[i];
    t->value_sum += s;
    return 0;
}

extern "C" int cccs_beamlet_dense(cccs_ctx* ctx, const cccs_beam* beam, const float* fluence, int mode, float* out,
                                  int max_beamlets, int* nactive) {
    clear_error();
    if (!ctx || !beam || !fluence || !out) return set_error(CCCS_EINVAL, "null argument");
    if (mode != CCCS_BEAMLET_FAITHFUL) return set_error(CCCS_EINVAL, "unknown beamlet mode");
    CCCS_HIP(hipSetDevice(ctx->device));
    CCCS_TRY(check_beam(ctx, *beam));
    std::vector<BeamPlan> plans(1);
    CCCS_TRY(plan_beam(ctx, *beam, fluence, 0, plans[0]));
    const int n = (int)plans[0].bl.size();
    if (nactive) *nactive = n;
    if (n == 0) return CCCS_OK;
    if (n > max_beamlets) return set_error(CCCS_EINVAL, "more active beamlets than max_beamlets");
    const cccs_problem& p = ctx->prob;
    const size_t nbb = (size_t)p.bbox_size[0] * p.bbox_size[1] * p.bbox_size[2];
    std::memset(out, 0, sizeof(float) * nbb * n);
    std::vector<const float*> d_fmaps;
    const float* fl[1] = {fluence};
    CCCS_TRY(upload_fmaps(ctx, plans, fl, d_fmaps));
    // one job per batch, as the reference processes its batches
    int done = 0;
    for (const BatchRef& R : all_batches(plans)) {
        Job J;
        CCCS_TRY(run_job(ctx, plans, std::vector<BatchRef>{R}, d_fmaps, J));
        std::vector<float> arena(J.arena);
        CCCS_HIP(hipStreamSynchronize(ctx->stream));
        if (J.arena) CCCS_HIP(hipMemcpy(arena.data(), ctx->bl_arena.p, sizeof(float) * J.arena, hipMemcpyDeviceToHost));
        for (int q = 0; q < R.n; q++) {
            const BeamletDev& d = J.beamlets[q];
            float* col = out + (size_t)(done + q) * nbb;
            const float* src = arena.data() + d.arena;
            for (int i = 0; i < d.boxn[0]; i++)
                for (int j = 0; j < d.boxn[1]; j++)
                    for (int k = 0; k < d.boxn[2]; k++) {
                        const size_t X = (size_t)(d.box0[0] + i), Y = (size_t)(d.box0[1] + j), Z = (size_t)(d.box0[2] + k);
                        col[X + p.bbox_size[0] * (Y + p.bbox_size[1] * Z)] =
                            src[((size_t)i * d.boxn[1] + j) * d.boxn[2] + k];
                    }
        }
        done += R.n;
    }
    return CCCS_OK;
}

extern "C" int cccs_beamlet_dose(cccs_ctx* ctx, const cccs_beam* beams, int nbeams, const float* const* fluence,
                                 float threshold, int mode, cccs_sparse_sink sink, void* user) {
    clear_error();
    if (!ctx || (!beams && nbeams > 0) || nbeams < 0 || (!fluence && nbeams > 0))
        return set_error(CCCS_EINVAL, "null argument");
    if (!sink && mode == CCCS_BEAMLET_PLAIN) return set_error(CCCS_EINVAL, "the plain path needs a sink");
    if (ctx && ctx->nroi > 0 && mode == CCCS_BEAMLET_PLAIN)
        return set_error(CCCS_EINVAL, "ROI reduction runs in the batched modes");
    if (mode != CCCS_BEAMLET_FAITHFUL && mode != CCCS_BEAMLET_PLAIN)
        return set_error(CCCS_EINVAL, "unknown beamlet mode");
    if (!(threshold >= 0.f)) return set_error(CCCS_EINVAL, "threshold must be >= 0");
    CCCS_HIP(hipSetDevice(ctx->device));
    const cccs_problem& p = ctx->prob;
    std::vector<BeamPlan> plans;
    plans.reserve(nbeams);
    for (int i = 0; i < nbeams; i++) {
        if (!fluence[i]) return set_error(CCCS_EINVAL, "null fluence map");
        CCCS_TRY(check_beam(ctx, beams[i]));
        BeamPlan P;
        CCCS_TRY(plan_beam(ctx, beams[i], fluence[i], i, P));
        if (!P.bl.empty()) plans.push_back(std::move(P));
    }
    if (plans.empty()) return CCCS_OK;
    CCCS_TRY(ctx->h_small.ensure(64));
    std::vector<const float*> d_fmaps;
    CCCS_TRY(upload_fmaps(ctx, plans, fluence, d_fmaps));
    const std::vector<BatchRef> refs = all_batches(plans);
    if (mode == CCCS_BEAMLET_PLAIN) {
        for (const BatchRef& R : refs) CCCS_TRY(run_plain_batch(ctx, plans, R, d_fmaps, threshold, sink, user));
        return CCCS_OK;
    }
    const size_t nvox = (size_t)p.bbox_size[0] * p.bbox_size[1] * p.bbox_size[2];
    const uint64_t budget_max = uint64_t(ctx->sched.bl_job_gb) << 30;  // device bytes per job
    const int nset = std::min(std::max(ctx->sched.bl_streams, 1), kRaySets);
    size_t next = 0;
    // device footprint of each batch, additive per cone direction: a job needs its batches' packed
    // grids and sparse-output bounds, plus one direction's REV store, half steps and line table
    // (summed over its batches per direction, maximised over directions)
    const int nrays = ctx->nrays;
    std::vector<std::vector<uint64_t>> b_rev(refs.size()), b_lines(refs.size());
    std::vector<uint64_t> b_fixed(refs.size());
    for (size_t i = 0; i < refs.size(); i++)
        CCCS_TRY(batch_footprint(ctx, plans, refs[i], b_rev[i], b_lines[i], b_fixed[i]));
    // device bytes of the batches [k0, k1) as one job: every direction in flight holds its own REV
    // store, half steps and line table
    auto job_bytes = [&](size_t k0, size_t k1) {
        uint64_t mr = 0, ml = 0, fixed = 0;
        for (int r = 0; r < nrays; r++) {
            uint64_t rev = 0, lines = 0;
            for (size_t i = k0; i < k1; i++) { rev += b_rev[i][r]; lines += b_lines[i][r]; }
            mr = std::max(mr, rev);
            ml = std::max(ml, lines);
        }
        for (size_t i = k0; i < k1; i++) fixed += b_fixed[i];
        return fixed + (uint64_t)nset * direction_bytes(mr, ml);
    };
    constexpr uint64_t kMinJob = uint64_t(1) << 30;
    constexpr uint64_t kPartEntries = 1 << 18;  // entries a part of the columns is worth (3 MiB, 60 us of copy)
    // columns of the last finished job, waiting in pinned host memory for the sink
    if (sink) {
        if (!ctx->cstream) CCCS_HIP(hipStreamCreateWithFlags(&ctx->cstream, hipStreamNonBlocking));
        for (hipEvent_t& e : ctx->col_ev)
            if (!e) CCCS_HIP(hipEventCreateWithFlags(&e, hipEventDisableTiming));
    }
    hipEvent_t copy_done = nullptr;  // the last job's last column copy (its buffers are rewritten after it)
    // No return leaves a column copy on its way: the next call's fluence maps are staged in the buffer that
    // the copies write.
    struct Drain {
        hipStream_t s;
        bool queued;
        ~Drain() {
            if (queued) (void)hipStreamSynchronize(s);
        }
    } drain{ctx->cstream, false};
    Delivery pending;
    int njob = 0;
    auto deliver = [&]() -> int {
        if (!pending.live) return CCCS_OK;
        pending.live = false;
        const int nroi = pending.nroi;
        std::vector<uint64_t> blocks((size_t)nroi);
        uint64_t pos = 0;
        int part = -1;
        for (size_t q = 0; q < pending.cols.size(); q++) {
            while (part < 0 || q >= pending.end[part]) CCCS_HIP(hipEventSynchronize(pending.ev[++part]));
            const uint32_t* st = pending.stat + 4 * q;
            cccs_sparse_column col{};
            col.beam_index = pending.cols[q].first;
            col.beamlet_index = pending.cols[q].second;
            col.nnz = st[0];
            col.perc_nonzero = (float)(100.0 * (double)st[0] / (double)nvox);
            col.perc_dropped = (float)(100.0 * (double)st[1] / (double)nvox);
            if (nroi > 0) {
                // _reduce_by_roi's statistics (sparse_io.cpp:150-156)
                uint64_t kept = 0;
                for (int r = 0; r < nroi; r++) kept += blocks[(size_t)r] = pending.rcnt[q * (size_t)nroi + (size_t)r];
                const double pn = 100.0 * (double)kept / (double)nvox;
                col.perc_reducedrop = (float)((double)col.perc_nonzero - pn);
                col.perc_nonzero = (float)pn;
                col.nnz = kept;
                col.nblocks = nroi;
                col.row_block_sizes = blocks.data();
            }
            col.keys = pending.keys + pos;
            col.values = pending.vals + pos;
            pos += col.nnz;
            if (sink(user, &col) != 0) return set_error(CCCS_EIO, "sparse sink aborted the call");
        }
        return CCCS_OK;
    };
    while (next < refs.size()) {
        // grow the job batch by batch while it fits the budget and, where columns go to a sink, seven
        // tenths of what is left: the sink takes a job's columns while the next job computes, so the
        // last job, whose columns nothing hides, should be small, and the one before it about as long
        // as the sink takes over its predecessor (a third of the compute time or less).  Jobs below
        // kMinJob do not fill the device, so a rest of that size stays whole.  Whole calls with the
        // 12 GiB budget alone and with this rule: 63.8 and 55.3 ms (two fine 4pi beams), 54.5 and
        // 49.2 ms (thorax, 3 beams).
        std::vector<uint64_t> rev(nrays, 0), lines(nrays, 0);
        uint64_t fixed = 0;
        size_t k = next;
        const uint64_t left = job_bytes(next, refs.size());
        const uint64_t budget = !sink ? budget_max : std::min<uint64_t>(budget_max, std::max(kMinJob, left / 10 * 7));
        while (k < refs.size()) {
            uint64_t mr = 0, ml = 0;
            for (int r = 0; r < nrays; r++) {
                mr = std::max(mr, rev[r] + b_rev[k][r]);
                ml = std::max(ml, lines[r] + b_lines[k][r]);
            }
            // every direction in flight holds its own REV store, half steps and line table
            const uint64_t bytes = fixed + b_fixed[k] + (uint64_t)nset * direction_bytes(mr, ml);
            if (k > next && bytes > budget) break;
            for (int r = 0; r < nrays; r++) {
                rev[r] += b_rev[k][r];
                lines[r] += b_lines[k][r];
            }
            fixed += b_fixed[k];
            k++;
        }
        std::vector<BatchRef> sel(refs.begin() + (long)next, refs.begin() + (long)k);
        Job J;
        CCCS_TRY(build_job(ctx, plans, sel, d_fmaps, J));
        next = k;
        // the previous job's columns reach the sink while this job's cone passes run on the device
        CCCS_TRY(run_job_cones(ctx, J, deliver));
        const int nbl = (int)J.beamlets.size();
        int max_rows = 1;
        for (const BeamletDev& bl : J.beamlets) max_rows = std::max(max_rows, bl.boxn[0] * bl.boxn[1]);
        const int chunks = (max_rows + 255) / 256;
        const uint64_t units = (uint64_t)nbl * (uint64_t)chunks;
        const size_t o_off = (sizeof(uint32_t) * 4 * nbl + 255) & ~size_t(255);
        const size_t o_chunk = (o_off + sizeof(uint64_t) * (nbl + 1) + 255) & ~size_t(255);
        CCCS_TRY(ctx->bl_cnt.ensure(o_chunk + sizeof(uint32_t) * units));
        uint32_t* stat = ctx->bl_cnt.as<uint32_t>();
        uint64_t* offs = reinterpret_cast<uint64_t*>(ctx->bl_cnt.as<uint8_t>() + o_off);
        const size_t sz_b = sizeof(BatchDev) * J.batches.size();
        ColArgs ca;
        ca.batches = ctx->bl_tab.as<BatchDev>();
        ca.beamlets = reinterpret_cast<const BeamletDev*>(ctx->bl_tab.as<uint8_t>() + ((sz_b + 255) & ~size_t(255)));
        ca.pdose = ctx->bl_pdose.as<float>();
        ca.start = ld3(p.start);
        ca.voxel = ld3(p.voxel);
        ca.rvs = mk3(p.rev_latspacing, p.rev_longspacing, p.rev_latspacing);
        ca.rrv = mk3(1.f / ca.rvs.x, 1.f / ca.rvs.y, 1.f / ca.rvs.z);
        for (int k = 0; k < 3; k++) ca.bbs[k] = (int)p.bbox_start[k];
        ca.nx = (int)p.size[0];
        ca.ny = (int)p.size[1];
        ca.thresh = threshold;
        ca.stat = stat;
        CCCS_TRY(ctx->bl_rowcnt.ensure(sizeof(uint16_t) * std::max<uint64_t>(1, J.rows)));
        ca.rowcnt = ctx->bl_rowcnt.as<uint16_t>();
        ca.chunkcnt = reinterpret_cast<uint32_t*>(ctx->bl_cnt.as<uint8_t>() + o_chunk);
        ca.chunks = chunks;
        ca.beamlet0 = 0;
        ca.off = offs;
        ca.keys = nullptr;
        ca.vals = nullptr;
        if (copy_done) CCCS_HIP(hipStreamWaitEvent(ctx->stream, copy_done, 0));
        int tok = prof_begin(ctx, K_BL_UNPACK);
        hipLaunchKernelGGL(bl_fill_kernel, dim3(grid_for(4 * (uint64_t)nbl, 256)), dim3(256), 0, ctx->stream,
                           reinterpret_cast<float*>(stat), 4 * (uint64_t)nbl, 0.f);
        // one launch takes as many beamlets as its workgroups allow: jobs of many small boxes and a few huge
        // ones have more than kMaxGroups chunks (a single box never does: it has fewer than 2^32 rows)
        auto over = [&](void (*kernel)(ColArgs)) {
            const int per = (int)std::max<uint32_t>(1, kMaxGroups / (uint32_t)chunks);
            for (int b = 0; b < nbl; b += per) {
                ca.beamlet0 = b;
                hipLaunchKernelGGL(kernel, dim3((unsigned)(std::min(per, nbl - b) * chunks)), dim3(256), 0, ctx->stream, ca);
            }
        };
        over(bl_colmax_kernel);
        over(bl_colcount_kernel);
        prof_end(ctx, tok, 0.0, 0.0, (uint64_t)nbl);
        hipLaunchKernelGGL(bl_offsets_kernel, dim3(1), dim3(1024), 0, ctx->stream, stat, nbl, offs);
        CCCS_HIP(hipGetLastError());
        // totals decide the output size; the counts and offsets of every column follow them to the host
        // (two sets in turn: the sink may still read the last job's)
        HostBuf& hst = ctx->h_bl_st[njob & 1];
        const int nroi = ctx->nroi;
        const size_t ncr = (size_t)nbl * (size_t)nroi;
        const size_t cbytes = (sizeof(uint32_t) * ncr + 255) & ~size_t(255);
        CCCS_TRY(hst.ensure(o_chunk + cbytes + sizeof(uint64_t) * (ncr + 1)));
        uint8_t* hs = hst.as<uint8_t>();
        const uint64_t* hoff = reinterpret_cast<const uint64_t*>(hs + o_off);
        CCCS_HIP(hipMemcpyAsync(hs, stat, o_off + sizeof(uint64_t) * (nbl + 1), hipMemcpyDeviceToHost, ctx->stream));
        CCCS_HIP(hipStreamSynchronize(ctx->stream));
        const uint64_t nnz_total = hoff[nbl];
        CCCS_TRY(ctx->bl_keys.ensure(sizeof(uint64_t) * std::max<uint64_t>(1, nnz_total)));
        CCCS_TRY(ctx->bl_vals.ensure(sizeof(float) * std::max<uint64_t>(1, nnz_total)));
        ca.keys = ctx->bl_keys.as<uint64_t>();
        ca.vals = ctx->bl_vals.as<float>();
        // ROI reduction of the job's columns (count, scan, order-preserving emit)
        RoiArgs ra;
        const uint64_t* out_off = hoff;  // first output entry of every column
        std::vector<uint64_t> roi_off;
        if (nroi > 0) {
            int tk = prof_begin(ctx, K_BL_COMPACT);
            over(bl_emit_kernel);
            // algorithmic traffic: the kept entries (8 B key + 4 B value)
            prof_end(ctx, tk, 12.0 * (double)nnz_total, 0.0, nnz_total);
            CCCS_HIP(hipGetLastError());
            CCCS_TRY(ctx->roi_cnt.ensure(cbytes + sizeof(uint64_t) * (ncr + 1)));
            uint32_t* rcnt = ctx->roi_cnt.as<uint32_t>();
            uint64_t* roff = reinterpret_cast<uint64_t*>(ctx->roi_cnt.as<uint8_t>() + cbytes);
            ra.rois = ctx->roi_tab.as<RoiDev>();
            ra.rank = ctx->roi_rank.as<int32_t>();
            ra.nroi = nroi;
            ra.nx = (int)p.size[0];
            ra.ny = (int)p.size[1];
            ra.keys = ctx->bl_keys.as<uint64_t>();
            ra.vals = ctx->bl_vals.as<float>();
            ra.off = offs;
            ra.cnt = rcnt;
            ra.roff = roff;
            ra.rkeys = nullptr;
            ra.rvals = nullptr;
            hipLaunchKernelGGL(roi_count_kernel, dim3(nbl), dim3(256), 0, ctx->stream, ra);
            hipLaunchKernelGGL(roi_scan_kernel, dim3(1), dim3(1024), 0, ctx->stream, (const uint32_t*)rcnt, ncr, roff);
            CCCS_HIP(hipGetLastError());
            CCCS_HIP(hipMemcpyAsync(hs + o_chunk, rcnt, cbytes + sizeof(uint64_t) * (ncr + 1), hipMemcpyDeviceToHost,
                                    ctx->stream));
            CCCS_HIP(hipStreamSynchronize(ctx->stream));
            const uint64_t* hroff = reinterpret_cast<const uint64_t*>(hs + o_chunk + cbytes);
            roi_off.resize((size_t)nbl + 1);
            for (int q = 0; q <= nbl; q++) roi_off[(size_t)q] = hroff[(size_t)q * (size_t)nroi];
            out_off = roi_off.data();
            CCCS_TRY(ctx->roi_keys.ensure(sizeof(uint64_t) * std::max<uint64_t>(1, out_off[nbl])));
            CCCS_TRY(ctx->roi_vals.ensure(sizeof(float) * std::max<uint64_t>(1, out_off[nbl])));
            ra.rkeys = ctx->roi_keys.as<uint64_t>();
            ra.rvals = ctx->roi_vals.as<float>();
        }
        const uint64_t nout = out_off[nbl];
        // All columns in one launch: a launch lasts as long as its longest row, one lane's serial chain, however
        // few columns it has.
        int tk = nroi > 0 ? -1 : prof_begin(ctx, K_BL_COMPACT);
        if (nroi > 0) hipLaunchKernelGGL(roi_emit_kernel, dim3(nbl), dim3(256), 0, ctx->stream, ra);
        else over(bl_emit_kernel);
        if (nroi == 0) prof_end(ctx, tk, 12.0 * (double)nnz_total, 0.0, nnz_total);
        CCCS_HIP(hipGetLastError());
        if (!sink) continue;  // columns stay on the device (overwritten by the next job)
        // Columns to pinned host memory (full PCIe rate, one of two buffers in turn); the sink sees them in
        // place, during the next job or at the end of the call.  They go in parts of about equal size: while
        // the sink takes one part, the next ones are copied.  The copies run on their own stream: the next
        // job's cone passes, queued behind this compaction, do not wait for them; the next compaction waits
        // before rewriting the buffers.
        const int nparts = (int)std::min<uint64_t>(kColParts, std::max<uint64_t>(1, nout / kPartEntries));
        const size_t kbytes = sizeof(uint64_t) * nout;
        HostBuf& hbuf = (njob & 1) ? ctx->h_bl_out2 : ctx->h_bl_out;
        CCCS_TRY(hbuf.ensure(kbytes + sizeof(float) * nout + 64));
        Delivery& D = pending;
        D.keys = hbuf.as<uint64_t>();
        D.vals = reinterpret_cast<float*>(hbuf.as<uint8_t>() + kbytes);
        D.stat = reinterpret_cast<const uint32_t*>(hs);
        D.rcnt = reinterpret_cast<const uint32_t*>(hs + o_chunk);
        D.nroi = nroi;
        D.cols.resize((size_t)nbl);
        for (int q = 0; q < nbl; q++) {
            const BeamletDev& d = J.beamlets[q];
            D.cols[(size_t)q] = {plans[sel[d.batch].plan].beam, d.fidx};
        }
        D.nparts = nparts;
        const uint64_t* sk = (nroi > 0 ? ctx->roi_keys : ctx->bl_keys).as<uint64_t>();
        const float* sv = (nroi > 0 ? ctx->roi_vals : ctx->bl_vals).as<float>();
        hipStream_t cs = ctx->cstream;
        for (int part = 0, b0 = 0; part < nparts; part++) {
            int b1 = nbl;
            if (part + 1 < nparts)
                b1 = (int)(std::lower_bound(out_off + b0, out_off + nbl, nout / nparts * (part + 1)) - out_off);
            hipEvent_t ev = ctx->col_ev[(njob & 1) * kColParts + part];
            if (part == 0) {
                CCCS_HIP(hipEventRecord(ev, ctx->stream));
                CCCS_HIP(hipStreamWaitEvent(cs, ev, 0));
                drain.queued = true;
            }
            const uint64_t e0 = out_off[b0], n = out_off[b1] - e0;
            if (n) {
                CCCS_HIP(hipMemcpyAsync(D.keys + e0, sk + e0, sizeof(uint64_t) * n, hipMemcpyDeviceToHost, cs));
                CCCS_HIP(hipMemcpyAsync(D.vals + e0, sv + e0, sizeof(float) * n, hipMemcpyDeviceToHost, cs));
            }
            CCCS_HIP(hipEventRecord(ev, cs));
            D.ev[part] = ev;
            D.end[part] = (size_t)b1;
            copy_done = ev;
            b0 = b1;
        }
        D.live = true;
        njob++;
    }
    CCCS_TRY(deliver());
    drain.queued = false;  // (the last part has arrived)
    return CCCS_OK;
}
