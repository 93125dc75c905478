// footprint_check.hip -- CPU check of a beamlet call's stated device footprint.  TEST INFRASTRUCTURE.
//
// For every beam of a workload, the footprint that cccs_beamlet_footprint states against the buffers that the
// beam's job holds, formed here from the job's tables: packed grids, sparse-output bound, and one cone direction's
// REV store and half steps (two zero samples for every line beside the samples), line records and line grids.
//   footprint_check <case dir>
// Prints one JSON line and exits 1 on any difference.
#include "../../endtoend_amd/csrc/beamlet.hip"

#include <cinttypes>
#include <cstdio>

#include "case.hpp"

int main(int argc, char** argv) {
    if (argc < 2) return 2;
    Case c;
    load_case(argv[1], c);
    uint64_t differ = 0, stated = 0, held = 0;
    for (size_t i = 0; i < c.beams.size(); i++) {
        std::vector<BeamPlan> plans(1);
        Job J;
        const std::vector<const float*> fmaps{c.fmaps[i].data()};
        uint64_t bytes = 0;
        if (plan_beam(&c.ctx, c.beams[i], c.fmaps[i].data(), 0, plans[0]) != CCCS_OK ||
            build_job(&c.ctx, plans, all_batches(plans), fmaps, J) != CCCS_OK ||
            cccs_beamlet_footprint(&c.ctx, &c.beams[i], c.fmaps[i].data(), &bytes) != CCCS_OK) {
            std::fprintf(stderr, "%s\n", cccs_last_error());
            return 2;
        }
        const uint64_t samples = J.max_rev + 2 * J.max_lines;
        const uint64_t want = 4 * J.pdose + 12 * J.pvox + 2 * 4 * samples + 8 * J.max_lines + 4 * J.max_lines;
        if (samples >= (uint64_t(1) << 30) - 64 || bytes != want) differ++;
        stated += bytes;
        held += want;
    }
    std::printf("{\"beams\": %zu, \"stated\": %" PRIu64 ", \"held\": %" PRIu64 ", \"differences\": %" PRIu64 "}\n",
                c.beams.size(), stated, held, differ);
    return differ ? 1 : 0;
}
