// rot_check.hip -- CPU check of the short forms of the geometry.  TEST INFRASTRUCTURE.
//
// rot_fwd and rot_inv against rot2 for rotations from every host builder, over random angles and
// coordinates of all magnitudes that occur and zeros: equal (a zero may differ in sign).  div_by
// against the division: the same bits over random mantissas and exponents.  mad24 against the plain
// product.
//   rot_check [samples] [seed]
// Prints one JSON line of counts and exits 1 on any difference.
#include "../../endtoend_amd/csrc/cccs_internal.hpp"

#include <cinttypes>
#include <cstdio>
#include <cstdlib>
#include <cstring>
#include <random>

using namespace cccs;

int main(int argc, char** argv) {
    const int n = argc > 1 ? std::atoi(argv[1]) : 1000000;
    std::mt19937 rng(argc > 2 ? (unsigned)std::atoi(argv[2]) : 3u);
    std::uniform_real_distribution<float> U(-1.f, 1.f);
    auto bits = [&]() { return (uint32_t)rng(); };
    auto coord = [&]() {
        const uint32_t k = bits() % 16;
        return k == 0 ? 0.f : U(rng) * std::ldexp(1.f, (int)(bits() % 40) - 20);
    };
    uint64_t rots = 0, divs = 0, rot_bad = 0, div_bad = 0, mad_bad = 0;
    for (int i = 0; i < n; i++) {
        const float th = U(rng) * 6.3f, ph = U(rng) * 6.3f, co = bits() % 3 ? 0.f : U(rng) * 6.3f;
        const Rot2 f[2] = {rot2_beam_fwd(th, ph, co), rot2_kernel_fwd(th, ph)};
        const Rot2 b[2] = {rot2_beam_inv(th, ph, co), rot2_kernel_inv(th, ph)};
        const v3 p = mk3(coord(), coord(), coord());
        for (int k = 0; k < 2; k++) {
            const v3 x = rot_fwd(f[k], p), y = rot2(f[k], p), u = rot_inv(b[k], p), v = rot2(b[k], p);
            rots += 2;
            if (!(x.x == y.x && x.y == y.y && x.z == y.z)) rot_bad++;
            if (!(u.x == v.x && u.y == v.y && u.z == v.z)) rot_bad++;
        }
        // quotients between 2^-60 and 2^60, every mantissa
        const uint32_t mx = (bits() & 0x807fffffu) | ((97u + bits() % 60u) << 23);
        const uint32_t my = (bits() & 0x007fffffu) | ((97u + bits() % 60u) << 23);
        float x, y;
        std::memcpy(&x, &mx, 4);
        std::memcpy(&y, &my, 4);
        const float q = div_by(x, y, 1.f / y), r = x / y;
        divs++;
        if (std::memcmp(&q, &r, 4) != 0) div_bad++;
        if (div_by(0.f, y, 1.f / y) != 0.f) div_bad++;
        const uint32_t a = bits() >> 8, c = bits() >> 8, e = bits();
        if (mad24(a, c, e) != (uint32_t)((uint64_t)a * c + e)) mad_bad++;
    }
    std::printf("{\"rotations\": %" PRIu64 ", \"rotation_differences\": %" PRIu64 ", \"divisions\": %" PRIu64
                ", \"division_differences\": %" PRIu64 ", \"mad24_differences\": %" PRIu64 "}\n",
                rots, rot_bad, divs, div_bad, mad_bad);
    return rot_bad || div_bad || mad_bad;
}
