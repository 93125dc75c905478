// sample_replay.hip -- CPU replay of the beamlet sample stage.  TEST INFRASTRUCTURE.
//
// Builds the job tables of a workload on the host with the library's own planning code (this file includes
// endtoend_amd/csrc/beamlet.hip), lays out the REV store as the interval kernel and the sample kernel do, and
// replays the sample kernel's passes for groups of 64 lines, as a wave takes them, with the kernel's own
// functions (line_interval, line_pad, line_start, near_axis, in_foot_bounds, may_take_dose, bl_locate,
// fluence_cell).  Checked:
//   store:   offsets formed within blocks of kLineBlock lines and from the blocks' totals equal a running sum
//            over the lines, with and without zeros; every stored line lies with its zeros inside the store and
//            touches no other line's samples;
//   A.1:     the candidate list stays inside its array over the lines that share it, and its entries give back
//            line and sample; the cull keeps every footprint sample (each sample of every third line is
//            classified exactly);
//   A.2:     pillars and beamlet records inside their tables; the cell test equals the fluence test;
//   B.1:     a sample that is not listed takes no dose (its exact pillar
//            has no footprint sample on the line, or it is a wall);
//   B.2:     listed samples and store slots in bounds, no more requests than reserved; the trimmed interval lies
//            inside the stored one and every sample of it was written.
//   sample_replay <case dir> [group stride]
// The case directory is the one tests/shim_case.py writes.  Prints one JSON line of counts and exits 1 on any
// violation.
#include "../../endtoend_amd/csrc/beamlet.hip"

#include <cinttypes>
#include <cstdio>
#include <cstring>

#include "case.hpp"

namespace {

struct Counts {
    uint64_t groups = 0, shared_lists = 0, lines = 0, nonempty = 0, cand_lines = 0, foot_lines = 0, exact_lines = 0,
             samples = 0, cand = 0, foot = 0, exact = 0, requests = 0, shortfall = 0, cull_checked = 0, walls_checked = 0,
             untracked = 0, violations = 0;
    uint32_t max_len = 0, max_list = 0, max_pil_word = 0;
    std::string first;
    void fail(const char* what, uint64_t line) {
        violations++;
        if (first.empty()) first = std::string(what) + " (line " + std::to_string(line) + ")";
    }
    void merge(const Counts& o) {
        uint64_t* a = &groups;
        const uint64_t* b = &o.groups;
        for (; a <= &violations; a++, b++) *a += *b;
        max_len = std::max(max_len, o.max_len);
        max_list = std::max(max_list, o.max_list);
        max_pil_word = std::max(max_pil_word, o.max_pil_word);
        if (first.empty()) first = o.first;
    }
};

#define CHECK(cond, what, line)              \
    do {                                     \
        if (!(cond)) N.fail(what, line);     \
    } while (0)

// One direction's lines as the interval kernel leaves them and the sample kernel completes them: offsets within
// blocks, then the blocks before.
std::vector<LineMeta> lay_out(const BlArgs& a, Counts& N, uint64_t capacity) {
    const uint64_t nl = a.nlines;
    std::vector<LineMeta> meta(nl);
    const uint64_t nb = (nl + kLineBlock - 1) / kLineBlock;
    std::vector<uint32_t> total(nb, 0);
    for (uint64_t b = 0; b < nb; b++) {
        uint32_t before = 0;
        for (uint64_t line = b * kLineBlock; line < std::min(nl, (b + 1) * (uint64_t)kLineBlock); line++) {
            const int ci = find_cone(a.cones, a.nbatch, line);
            LineMeta m = line_interval(a, a.cones[ci], a.batches[ci], line);
            const uint32_t pad = line_pad(a.zeros, m.len);
            m.off = m.len > 0 ? before + pad : 0u;
            before += (uint32_t)m.len + pad;
            meta[line] = m;
        }
        total[b] = before;
    }
    uint32_t sum = 0;
    for (uint64_t b = 0; b < nb; b++) {
        for (uint64_t line = b * kLineBlock; line < std::min(nl, (b + 1) * (uint64_t)kLineBlock); line++)
            if (meta[line].len > 0) meta[line].off += sum;
        sum += total[b];
    }
    const uint64_t zeros = a.zeros ? 2 : 0;
    uint64_t end = 0;  // one past the last sample of the lines before
    for (uint64_t line = 0; line < nl; line++) {
        if (meta[line].len <= 0) {
            CHECK(meta[line].off == 0u, "an empty line with an offset", line);
            continue;
        }
        CHECK(meta[line].off == end + zeros, "block offsets differ from the running sum", line);
        end = (uint64_t)meta[line].off + (uint64_t)meta[line].len;
    }
    CHECK(end + zeros <= capacity + (a.zeros ? (uint64_t)kRevPad : 0), "store beyond its buffer", nl);
    CHECK(end <= capacity, "samples beyond the store", nl);
    return meta;
}

// The sample kernel's passes for the 64 lines base, base + G, ... of one wave.
void replay_group(const BlArgs& a, size_t nbeamlets, uint64_t base, uint64_t G, const std::vector<LineMeta>& meta,
                  uint64_t capacity, Counts& N) {
    N.groups++;
    struct Lane {
        LineMeta m{};
        int ci = 0, y = 0, z = 0, c0 = 0, c1 = 0;
        v3 p0 = mk3(0.f, 0.f, 0.f);
    } lane[64];
    uint64_t todo = 0;
    for (int k = 0; k < 64; k++) {
        const uint64_t line = base + (uint64_t)k * G;
        if (line >= a.nlines) break;
        Lane& l = lane[k];
        l.m = meta[line];
        l.ci = find_cone(a.cones, a.nbatch, line);
        const BlConeDev& c = a.cones[l.ci];
        const uint64_t q = line - c.line0;
        l.z = (int)(q / (uint64_t)c.ny);
        l.y = (int)(q - (uint64_t)l.z * (uint64_t)c.ny);
        l.p0 = line_start(a, c, l.y, l.z);
        N.lines++;
        if (l.m.len > 0) {
            todo |= 1ull << k;
            N.nonempty++;
            N.samples += (uint64_t)l.m.len;
            N.max_len = std::max(N.max_len, (uint32_t)l.m.len);
            CHECK(l.m.len <= kMaxLine && l.m.i0 >= 0 && l.m.i0 + l.m.len <= c.nx, "stored interval outside the line", line);
        }
    }
    uint16_t s_cand[kMaxLine], s_cpil[kMaxLine], s_list[kMaxLine];
    constexpr uint16_t kNoPil = 0xffff;
    while (todo) {
        const int ci = lane[__builtin_ctzll(todo)].ci;
        const BlConeDev& c = a.cones[ci];
        const BatchDev& B = a.batches[ci];
        const v3 ipd = mk3(B.ipd[0], B.ipd[1], B.ipd[2]);
        const v3 dl = line_step(c);
        const float pdx = (float)B.pd[0], pdz = (float)B.pd[2], ipdx = B.ipd[0], ipdz = B.ipd[2], cull = B.fw + 0.05f;
        const float dux = dl.x * ipdx, duz = dl.z * ipdz, cx = (cull + 0.05f) * ipdx, cz = (cull + 0.05f) * ipdz;
        const bool track = B.n <= (int)kPillarBits;
        uint64_t with_cand = 0;
        int ncand = 0, nlines = 0;
        // A.1
        while (todo) {
            const int k = __builtin_ctzll(todo), m = lane[k].m.len;
            if (lane[k].ci != ci || ncand + m > kMaxLine) break;
            todo &= todo - 1ull;
            nlines++;
            const uint64_t line = base + (uint64_t)k * G;
            const v3 p0 = lane[k].p0;
            const float t0 = (float)lane[k].m.i0;
            const float ux0 = fmaf(p0.x - B.fc[0], ipdx, 0.5f), uz0 = fmaf(p0.z - B.fc[1], ipdz, 0.5f);
            lane[k].c0 = ncand;
            for (int j = 0; j < m; j++) {
                const float t = t0 + (float)j;
                const bool near = near_axis(true, fmaf(t, dux, ux0), fmaf(t, duz, uz0), cx, cz);
                const bool cand = in_foot_bounds(near, B, p0.x + t * dl.x, p0.y + t * dl.y, p0.z + t * dl.z, pdx, pdz, ipdx,
                                                 ipdz, cull);
                if (line % 3 == 0 && !cand) {
                    int pe = -1;
                    v3 ie;
                    if (bl_locate(a, c, B, ipd, lane[k].m.i0 + j, lane[k].y, lane[k].z, pe, ie) &&
                        fabsf(ie.x - B.fc[0]) <= B.fw && fabsf(ie.z - B.fc[1]) <= B.fw) {
                        const PillarRec be = pillar_rec(a.beamlets[B.beamlet0 + pe]);
                        CHECK(fluence_cell(bl_terma_point(a, B, be, ie), B.beam) != be.fidx,
                              "the cull drops a footprint sample", line);
                    }
                    N.cull_checked++;
                }
                if (!cand) continue;
                CHECK(ncand < kMaxLine, "candidate list beyond its array", line);
                if (ncand >= kMaxLine) return;
                s_cand[ncand] = (uint16_t)(k << 10 | j);
                CHECK(s_cand[ncand] >> 10 == k && (s_cand[ncand] & 1023) == j, "candidate entry", line);
                ncand++;
            }
            if (ncand > lane[k].c0) {
                with_cand |= 1ull << k;
                lane[k].c1 = ncand;
                N.cand_lines++;
            }
        }
        if (nlines == 0) {
            N.fail("no line taken", base);
            return;
        }
        if (nlines > 1 && ncand > 0) N.shared_lists++;
        N.cand += (uint64_t)ncand;
        N.max_list = std::max(N.max_list, (uint32_t)ncand);
        // A.2
        for (int e = 0; e < ncand; e++) {
            const int k = s_cand[e] >> 10;
            const uint64_t line = base + (uint64_t)k * G;
            int pidx = -1;
            v3 inp;
            bool fp = false;
            if (bl_locate(a, c, B, ipd, lane[k].m.i0 + (s_cand[e] & 1023), lane[k].y, lane[k].z, pidx, inp) &&
                fabsf(inp.x - B.fc[0]) <= B.fw && fabsf(inp.z - B.fc[1]) <= B.fw) {
                CHECK(pidx >= 0 && pidx < B.n && (size_t)(B.beamlet0 + pidx) < nbeamlets, "pillar outside the batch", line);
                if (pidx < 0 || (size_t)(B.beamlet0 + pidx) >= nbeamlets) return;
                const PillarRec bl = pillar_rec(a.beamlets[B.beamlet0 + pidx]);
                const v3 tp = bl_terma_point(a, B, bl, inp);
                fp = fluence_cell(tp, B.beam) == bl.fidx;
                CHECK(fp == (point_fluence(tp, B.fmap, B.beam, bl.fidx) > 0.f), "cell test differs from the fluence test", line);
            }
            s_cpil[e] = !fp ? kNoPil : (uint16_t)(track ? pidx : 0);
        }
        while (with_cand) {
            const int k = __builtin_ctzll(with_cand);
            with_cand &= with_cand - 1ull;
            const Lane& l = lane[k];
            const uint64_t line = base + (uint64_t)k * G;
            const int i0 = l.m.i0, m = l.m.len;
            uint32_t nfoot = 0, s_foot[kMaxLine / 32] = {};
            std::vector<uint32_t> s_pil(kPillarBits / 32, 0u);
            for (int e = l.c0; e < l.c1; e++) {
                if (s_cpil[e] == kNoPil) continue;
                const uint32_t pil = s_cpil[e], j = s_cand[e] & 1023u;
                nfoot++;
                s_foot[j >> 5] |= 1u << (j & 31u);
                if (!track) continue;
                CHECK(pil >> 5 < kPillarBits / 32, "footprint pillar beyond the bit table", line);
                N.max_pil_word = std::max(N.max_pil_word, pil >> 5);
                s_pil[pil >> 5 & (kPillarBits / 32 - 1)] |= 1u << (pil & 31u);
            }
            if (nfoot == 0) continue;
            N.foot_lines++;
            N.foot += nfoot;
            if (!track) N.untracked++;
            auto has_foot = [&](int p) { return !track || (s_pil[p >> 5] >> (p & 31) & 1u) != 0u; };
            // B.1
            const float ux0 = l.p0.x * ipdx, uz0 = l.p0.z * ipdz, hx = 0.5f - 0.05f * ipdx, hz = 0.5f - 0.05f * ipdz;
            int nex = 0;
            bool listed[kMaxLine] = {};
            for (int j = 0; j < m; j++) {
                const float t = (float)(i0 + j), ux = fmaf(t, dux, ux0), uz = fmaf(t, duz, uz0);
                const bool exact = !track || may_take_dose(true, B, ux, uz, hx, hz, s_pil.data());
                if (!exact) {
                    int pe = -1;
                    v3 ie;
                    CHECK(!(bl_locate(a, c, B, ipd, i0 + j, l.y, l.z, pe, ie) && has_foot(pe)), "a wall that takes dose", line);
                    N.walls_checked++;
                    continue;
                }
                listed[j] = true;
                s_list[nex++] = (uint16_t)j;
            }
            if (nex == 0) {
                N.shortfall += nfoot;
                continue;
            }
            N.exact_lines++;
            N.exact += (uint64_t)nex;
            const int elo = s_list[0], ehi = s_list[nex - 1];
            // B.2
            uint32_t qdone = 0;
            int nlo = m, nhi = -1;
            for (int r = 0; r < nex; r++) {
                const int j = s_list[r];
                CHECK((uint64_t)l.m.off + (uint64_t)j < capacity, "slot beyond the store", line);
                int pidx = -1;
                v3 inp;
                if (!bl_locate(a, c, B, ipd, i0 + j, l.y, l.z, pidx, inp) || !has_foot(pidx)) continue;
                if (s_foot[j >> 5] >> (j & 31) & 1u) qdone++;
                nlo = std::min(nlo, j);
                nhi = std::max(nhi, j);
            }
            CHECK(qdone <= nfoot, "more requests than reserved", line);
            N.requests += qdone;
            N.shortfall += nfoot - std::min(qdone, nfoot);
            if (nhi < nlo) continue;
            CHECK(nlo >= 0 && nhi < m, "trimmed interval outside the stored one", line);
            for (int j = nlo; j <= nhi; j++) CHECK(listed[j] || (j > elo && j < ehi), "an unwritten sample", line);
        }
    }
}

}  // namespace

int main(int argc, char** argv) {
    if (argc < 2) {
        std::fprintf(stderr, "usage: %s <case dir> [group stride]\n", argv[0]);
        return 2;
    }
    const uint64_t stride = argc > 2 ? std::stoull(argv[2]) : 1;
    Case cs;
    load_case(argv[1], cs);
    std::vector<BeamPlan> plans;
    for (size_t i = 0; i < cs.beams.size(); i++) {
        BeamPlan P;
        if (plan_beam(&cs.ctx, cs.beams[i], cs.fmaps[i].data(), (int)i, P) != CCCS_OK) {
            std::fprintf(stderr, "plan: %s\n", cccs_last_error());
            return 2;
        }
        if (!P.bl.empty()) plans.push_back(std::move(P));
    }
    std::vector<const float*> fmaps;
    for (const BeamPlan& P : plans) fmaps.push_back(cs.fmaps[(size_t)P.beam].data());
    Job J;
    if (build_job(&cs.ctx, plans, all_batches(plans), fmaps, J) != CCCS_OK) {
        std::fprintf(stderr, "job: %s\n", cccs_last_error());
        return 2;
    }
    BlArgs a = base_args(&cs.ctx);
    a.batches = J.batches.data();
    a.beamlets = J.beamlets.data();
    const int nb = (int)J.batches.size();
    a.nbatch = nb;
    Counts total;
    for (int r = 0; r < cs.ctx.nrays; r++) {
        a.cones = J.cones.data() + (size_t)r * nb;
        a.nlines = J.ray_lines[r];
        a.zeros = false;
        lay_out(a, total, J.max_rev);
        a.zeros = line_zeros(J.max_rev, J.max_lines);
        const uint64_t capacity = store_samples(J.max_rev, J.max_lines);
        const std::vector<LineMeta> meta = lay_out(a, total, capacity);
        const uint64_t G = std::min<uint64_t>(a.nlines, (uint64_t)cs.ctx.sched.bl_sample_waves);
        const uint64_t rounds = (a.nlines + 64 * G - 1) / (64 * G);
#pragma omp parallel
        {
            Counts N;
#pragma omp for schedule(dynamic, 16)
            for (uint64_t g = 0; g < G * rounds; g += stride) {
                const uint64_t base = g / G * 64 * G + g % G;
                if (base < a.nlines) replay_group(a, J.beamlets.size(), base, G, meta, capacity, N);
            }
#pragma omp critical
            total.merge(N);
        }
    }
    std::printf("{\"beams\": %zu, \"batches\": %d, \"beamlets\": %zu, \"directions\": %d, \"zeros\": %d", plans.size(), nb,
                J.beamlets.size(), cs.ctx.nrays, (int)a.zeros);
    const char* names[] = {"groups", "shared_lists", "lines", "nonempty", "candidate_lines", "footprint_lines",
                           "exact_lines", "samples", "candidates", "footprint", "exact", "requests", "shortfall",
                           "cull_checked", "walls_checked", "untracked_lines", "violations"};
    const uint64_t* v = &total.groups;
    for (const char* n : names) std::printf(", \"%s\": %" PRIu64, n, *v++);
    std::printf(", \"max_len\": %u, \"max_list\": %u, \"max_pillar_word\": %u, \"first\": \"%s\"}\n", total.max_len,
                total.max_list, total.max_pil_word, total.first.c_str());
    return total.violations ? 1 : 0;
}
