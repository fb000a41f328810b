// Wave schedules of the forward projector (fp_pair_schedule), without a GPU.
// Arguments: VolX, VolZ, band rows, staging.  Prints, per group of tilts, the sum
// over the bands of the busiest wave's load and what the best exchange of two
// pairs between waves would take off it.
#include <hip/hip_runtime.h>
static inline void __syncthreads() {}
#include <cmath>
#include <cstdio>
#include <cstdlib>

#include "atr_internal.h"
using namespace atr;

int main(int argc, char** argv)
{
    if (argc != 5) return 2;
    const int vol_x = atoi(argv[1]), vol_z = atoi(argv[2]), bz = atoi(argv[3]), pf = atoi(argv[4]);
    std::vector<float> tilts;
    for (int t = -60; t <= 60; t += 3) tilts.push_back((float)t);
    const int n = (int)tilts.size();
    Geometry g;
    cos_sin_table(tilts.data(), n, g.cos_sin);
    if (!build_fp_tables(g.cos_sin, n, vol_x, vol_z, vol_x, bz, g)) return 3;
    std::vector<int> list, tab;
    for (int t = 0; t < n; t += 5) list.push_back(t);
    const int group = fp_group(vol_x, (int)list.size(), fp_waves(pf));
    fp_pair_schedule(g, list.data(), (int)list.size(), vol_x, group, tab, pf);
    const int nb = g.fp_nbands, ntile = (vol_x + FP_WAVE - 1) / FP_WAVE;
    for (size_t base = 0; base < tab.size(); base += FP_WAVES * FP_MAXP) {
        std::vector<int> pair, owner;
        for (int i = 0; i < FP_WAVES * FP_MAXP; i++)
            if (tab[base + i] >= 0) {
                pair.push_back(tab[base + i] & 0xffffff);
                owner.push_back(i / FP_MAXP);
            }
        auto cost = [&](int p, int b) {
            const int4 d = g.fp_desc[(size_t)p * nb + b];
            const double wt = 1.0 + std::fabs((double)g.cos_sin[2 * (p / ntile) + 1]);
            return d.y > 0 ? d.y * wt * (d.w ? 1.0 : 1.4) + 8.0 : 0.0;
        };
        auto objective = [&] {
            std::vector<double> load((size_t)FP_WAVES * nb, 0.0);
            for (size_t i = 0; i < pair.size(); i++)
                for (int b = 0; b < nb; b++) load[owner[i] * nb + b] += cost(pair[i], b);
            double o = 0.0;
            for (int b = 0; b < nb; b++) {
                double m = 0.0;
                for (int w = 0; w < FP_WAVES; w++) m = std::max(m, load[w * nb + b]);
                o += m;
            }
            return o;
        };
        const double now = objective();
        double best = now;
        for (size_t i = 0; i < pair.size(); i++)
            for (size_t j = i + 1; j < pair.size(); j++) {
                std::swap(owner[i], owner[j]);
                best = std::min(best, objective());
                std::swap(owner[i], owner[j]);
            }
        std::printf("%.6f %.6f\n", now, now - best);
    }
    return 0;
}
