// Which shapes take the one-launch training passes (pixienn_amd/csrc/resident.h), on the host: every form that is chosen holds
// its slice, and the lines lie where they are said to.
#include "../../pixienn_amd/csrc/resident.h"

#include <cstdio>

using namespace pxh;

namespace {

int failed = 0, checks = 0;

void check(bool good, const char* what, int batch, int channels, int spatial)
{
    ++checks;
    if (!good && ++failed < 10) std::printf("%s: %d x %d x %d\n", what, batch, channels, spatial);
}

}  // namespace

int main()
{
    for (int channels: { 1, 5, 95, 96, 512, 513, 1024 })
        for (int spatial: { 1, 2, 3, 5, 7, 9, 49, 63, 169, 361, 1025, 2051 })
            for (int batch = 1; batch < 40000; batch += batch < 300 ? 1 : batch / 50) {
                const size_t values = static_cast<size_t>(batch) * spatial;
                if (values > 200000) break;
                for (bool backward: { false, true })
                    for (int activation: { PXH_LEAKY, PXH_MISH }) {
                        const ResidentForm form = resident_form(batch, channels, spatial, false, activation, backward);
                        check(!form.per_thread && !form.small, "vectors only where planes have them whole", batch, channels, spatial);
                        if (!form.odd) continue;
                        const ResidentGeom g = resident_geom(batch, channels, spatial);
                        const auto holds = [&]<int V, int R, int T>() {
                            const size_t items = V == 1 ? values : g.vectors;
                            check(static_cast<size_t>(R) * T >= items, "a form holds its slice", batch, channels, spatial);
                            check(V == 1 || spatial >= 4, "a vector fits a plane", batch, channels, spatial);
                            if (values <= 64) check(V == 1 && R == 1 && T == 64, "a value per lane", batch, channels, spatial);
                            else if (V == 4 && items <= 128) check(R == 1, "a vector per lane", batch, channels, spatial);
                            // vectors of up to 256 lanes: no lane has a step that none of the slice's is in
                            if (V == 4 && T <= 256 && (T < 256 || channels > kOddChannels))
                                check(static_cast<size_t>(R - (R == 6 ? 2 : 1)) * T < items, "no empty steps", batch, channels, spatial);
                        };
                        const auto one_step = [&](uint32_t most) {
                            return [&, most]<int V, int R, int T>() {
                                if (V == 4 && g.vectors <= most && channels <= kOddChannels) check(R == 1, "a vector per lane", batch, channels, spatial);
                                holds.template operator()<V, R, T>();
                            };
                        };
                        if (selects(activation)) dispatch_odd_form<kOddOneStep<PXH_LEAKY, true>>(form.odd, g, one_step(128));
                        else if (backward) dispatch_odd_form<kOddOneStep<PXH_MISH, true>>(form.odd, g, one_step(512));
                        else dispatch_odd_form<kOddOneStep<PXH_MISH, false>>(form.odd, g, one_step(256));
                    }
                const bool one = odd_slice(batch, channels, spatial, false, PXH_LEAKY, false) != 0;
                const size_t vectors = static_cast<size_t>(batch) * ((spatial + 3) / 4);
                for (bool backward: { false, true }) {
                    const size_t most = channels >= 96 ? 6144 : backward || spatial > 64 ? 3072 : 4096;
                    if (spatial >= 4) check((odd_slice(batch, channels, spatial, false, PXH_MISH, backward) != 0) == (vectors <= most), "a chain", batch, channels, spatial);
                    if (spatial >= 4) check((odd_slice(batch, channels, spatial, false, PXH_LOGISTIC, backward) != 0) == one, "no chain", batch, channels, spatial);
                }
                if (spatial >= 4) check(one == (vectors <= (channels < 96 ? 4096u : 6144u)), "light", batch, channels, spatial);
                if (spatial < 4) check(one == (values <= (channels < 96 ? 6144u : 24576u)), "planes below a vector", batch, channels, spatial);
                // a workspace too small is refused on both sides of lines that may move: this one does not
                check(asks_for_workspace(batch, channels, spatial, false) == (channels < 96 || values > 8192), "the workspace", batch, channels, spatial);
            }
    // sums in several launches: a value a step where a lane has one (two before an exponential), and never more steps than there are
    for (int spatial = 1; spatial < 5000; ++spatial)
        for (int activation: { PXH_LINEAR, PXH_LEAKY, PXH_MISH, PXH_SWISH }) {
            const bool vectors = sums_in_vectors(spatial, activation);
            check(vectors == (spatial > (activation == PXH_LINEAR || activation == PXH_LEAKY ? 64 : 128)), "sums", 0, 0, spatial);
            check(vectors ? spatial >= 4 : spatial <= kValueSteps * kWave, "steps of the sums", 0, 0, spatial);
        }
    std::printf("%d checks, %d failed\n", checks, failed);
    return failed != 0;
}
