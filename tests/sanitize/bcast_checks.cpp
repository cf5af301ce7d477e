// The operators and azimuths of the broadcast FP64 M2L (build_bcast_m2l) for every
// order and part, built under the sanitizers: whole, finite, and the rotations'
// blocks orthogonal (stage 3 applies them transposed).
#include "../../simplefmm_amd/csrc/m2l_bcast.hpp"
#include "../../simplefmm_amd/csrc/tables.hpp"

#include <cmath>
#include <cstdio>
#include <string>
#include <vector>

namespace {

int failures = 0;
void check(bool ok, const std::string& what)
{
    if (ok) return;
    ++failures;
    std::printf("FAILED: %s\n", what.c_str());
}

bool finite(const std::vector<double>& v)
{
    for (double x : v)
        if (!std::isfinite(x)) return false;
    return !v.empty();
}

void order_case(const sfmm::Tables& t, int p, int mode)
{
    const std::string tag = "p=" + std::to_string(p) + " part " + std::to_string(mode);
    std::vector<double> rot, coax, fwd, back;
    sfmm::build_bcast_m2l(t, mode, rot, coax, fwd, back);
    const int nw = sfmm::bcast_waves(p);
    const sfmm::BcastUnits ur = sfmm::bcast_units(p, false, mode), ut = sfmm::bcast_units(p, true, mode);
    const size_t rr = sfmm::bcast_reg0(p, ur, false, nw), rt = sfmm::bcast_reg0(p, ut, true, nw);
    check(rot.size() == 70 * rr * 16 && coax.size() == 28 * rt * 16, tag + ": operator sizes");
    check(fwd.size() == 343 * 32 && back.size() == 343 * 32, tag + ": azimuth sizes");
    check(finite(rot) && finite(coax) && finite(fwd) && finite(back), tag + ": finite");
    double worst = 0.0;
    std::vector<bool> used(70, false);
    for (int c : t.off_class)
        if (c >= 0) used.at(c) = true;
    for (int cls = 0; cls < 70; ++cls)
        for (int w = 0; w < (used[cls] ? nw : 0); ++w)
            for (int q = 0; q < ur.count[w]; ++q) {
                const int S = sfmm::bcast_size(p, false, ur.idx[w][q], ur.part[w][q]);
                const double* b = rot.data() + (cls * rr + sfmm::bcast_reg0(p, ur, false, w)) * 16 +
                                  sfmm::bcast_block(p, ur, false, w, q);
                for (int i = 0; i < S; ++i)
                    for (int j = 0; j < S; ++j) {
                        double s = i == j ? -1.0 : 0.0;
                        for (int k = 0; k < S; ++k) s += b[i * S + k] * b[j * S + k];
                        worst = std::fmax(worst, std::fabs(s));
                    }
            }
    // the elements are rounded once, the check itself 17 times
    check(worst < 32 * 2.3e-16, tag + ": rotations orthogonal, off by " + std::to_string(worst * 1e16) + "e-16");
}

}  // namespace

int main()
{
    for (int p = 1; p <= sfmm::kBcastMaxP; ++p) {
        sfmm::Tables t;
        sfmm::build_tables(p, t);
        if (sfmm::bcast_parted(p)) {
            order_case(t, p, sfmm::kBcastCos);
            order_case(t, p, sfmm::kBcastSin);
        } else {
            order_case(t, p, sfmm::kBcastBoth);
        }
    }
    std::printf("%s (%d failed checks)\n", failures ? "FAILED" : "ok", failures);
    return failures ? 1 : 0;
}
