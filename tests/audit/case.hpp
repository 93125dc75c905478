// case.hpp -- a workload directory (tests/shim_case.py writes it) as a host-only context, beams and maps, for
// the CPU checks that include the library's sources.  TEST INFRASTRUCTURE.
#pragma once

#include <fstream>
#include <map>
#include <sstream>
#include <stdexcept>
#include <string>
#include <vector>

struct Case {
    cccs_ctx ctx;
    std::vector<cccs_beam> beams;
    std::vector<std::vector<float>> fmaps;
};

inline std::vector<float> read_raw(const std::string& path, size_t n) {
    std::vector<float> v(n);
    std::ifstream f(path, std::ios::binary);
    if (!f.read(reinterpret_cast<char*>(v.data()), (std::streamsize)(n * sizeof(float))))
        throw std::runtime_error("cannot read " + path);
    return v;
}

inline void load_case(const std::string& dir, Case& c) {
    std::ifstream cf(dir + "/case.txt");
    std::map<std::string, std::vector<double>> kv;
    std::vector<std::vector<double>> rows;
    for (std::string ln; std::getline(cf, ln);) {
        std::istringstream is(ln);
        std::string key;
        if (!(is >> key)) continue;
        std::vector<double> vals;
        for (double x; is >> x;) vals.push_back(x);
        if (key == "beam") rows.push_back(vals);
        else kv[key] = vals;
    }
    cccs_problem& p = c.ctx.prob;
    for (int k = 0; k < 3; k++) {
        p.size[k] = (uint32_t)kv.at("size")[k];
        p.voxel[k] = (float)kv.at("voxel")[k];
        p.start[k] = (float)kv.at("start")[k];
        p.bbox_start[k] = (uint32_t)kv.at("bbox_start")[k];
        p.bbox_size[k] = (uint32_t)kv.at("bbox_size")[k];
        p.max_rev_size[k] = (uint32_t)kv.at("max_rev_size")[k];
    }
    p.rev_latspacing = (float)kv.at("rev_latspacing")[0];
    p.rev_longspacing = (float)kv.at("rev_longspacing")[0];
    p.kernel_extent = (float)kv.at("kernel_extent")[0];
    p.penumbra = (float)kv.at("penumbra")[0];
    p.ss_factor = (uint32_t)kv.at("ss_factor")[0];
    p.nphi = (uint32_t)kv.at("nphi")[0];
    p.ntheta = (uint32_t)kv.at("ntheta")[0];
    p.nradii = (uint32_t)kv.at("nradii")[0];
    c.ctx.nrays = (int)(p.nphi * (p.ntheta / 2));
    c.ctx.theta = read_raw(dir + "/theta", (size_t)c.ctx.nrays);
    c.ctx.phi = read_raw(dir + "/phi", (size_t)c.ctx.nrays);
    for (const std::vector<double>& b : rows) {
        cccs_beam o;
        o.azimuth = (float)b[1]; o.zenith = (float)b[2]; o.coll = (float)b[3];
        for (int k = 0; k < 3; k++) {
            o.source[k] = (float)b[4 + k];
            o.direction[k] = (float)b[7 + k];
            o.isocenter[k] = (float)b[10 + k];
        }
        o.sad = (float)b[13];
        o.fmap_size[0] = (uint32_t)b[14]; o.fmap_size[1] = (uint32_t)b[15];
        o.beamlet_size[0] = (float)b[16]; o.beamlet_size[1] = (float)b[17];
        c.fmaps.push_back(read_raw(dir + "/fmap_" + std::to_string(c.beams.size()),
                                   (size_t)o.fmap_size[0] * o.fmap_size[1]));
        c.beams.push_back(o);
    }
}
