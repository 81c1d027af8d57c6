// The first raycast pass names blocks inside a cube, and takes a ray whose ends
// lie ray_cube_margin blocks from its faces: no sample of the pass may come
// nearer to them than kTagReach, whatever the roundings of its steps. One axis
// of such marches, in the kernel's own float steps, at coordinates up to 2^24
// voxels, with step components chosen to round the same way every time.
//
// Prints "ok", or the march that leaves.
#include <algorithm>
#include <cmath>
#include <cstdio>

#include "../../semantic_icpslam_amd/csrc/sicp_kernels.hpp"

int main() {
    long marches = 0;
    for (int samples : {1, 15, 16, 48, 400, sicp::kRayTuneMaxSamples}) {
        const int margin = sicp::ray_cube_margin(samples), inside = margin - sicp::kTagReach;
        for (int e = 10; e < 24; ++e) {
            const float at = std::ldexp(1.0f, e) - 9000.0f * (e == 23), ulp = std::ldexp(1.0f, e - 23);
            for (float part : {0.01f, 0.26f, 0.49f, 0.51f, 0.74f, 0.99f})
                for (float k : {0.0f, 1.0f, 3.0f})
                    for (float step : {1.0f, 8.0f})
                        for (float sign : {1.0f, -1.0f}) {
                            const float d = sign * std::min(step, (k + part) * ulp);
                            const float start = sign > 0 ? at : 1.9f * at;
                            // the ends, a whole number of steps apart
                            const float end = start + (float)samples * d;
                            if (std::fabs(end) >= 0x1p24f || std::fabs(end) < 0.9f * at) continue;
                            const float lo = std::min(start, end), hi = std::max(start, end);
                            float p = start;
                            ++marches;
                            for (int i = 0; i < samples; ++i) {
                                const double out = std::max((double)lo - p, (double)p - hi);
                                if (out > 8.0 * inside) {
                                    std::printf("samples %d, 2^%d, step %g: %g voxels out\n",
                                                samples, e, d, out);
                                    return 1;
                                }
                                p = p + d;
                            }
                        }
        }
    }
    if (marches < 1000) {
        std::printf("only %ld marches\n", marches);
        return 1;
    }
    std::printf("ok\n");
    return 0;
}
