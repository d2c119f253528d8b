// Host check of the transfer's memory plan (slice_length, frame_group): the segment maps of a launch stay within MAPS_MAX,
// or within those of whole work items where one launch cannot be split, from one pixel to the largest launches, in both
// precisions and for every chunk length. Exit status 0 when every launch does.
#include <cstdio>
#include "../../kerrsplat_amd/csrc/ks_kernels.hpp"
using namespace ksd;
int main() {
    long bad = 0, n = 0, grouped = 0;
    const int64_t pixels[] = {1, 1850, 16384, 65536, 400921, 1048576, 4194304};
    for (int64_t npix : pixels)
        for (int N : {1, 7, 64, 301, 1024, 2048, 8000})
            for (int frames : {1, 2, 3, 48, 200, 800})
                for (int chunk : {8, 16, 32, 33, 128, 1024})
                    for (int real : {4, 8}) {
                        const int64_t map = SEG_FIELDS * real;
                        // a render: a group of frames
                        const int len = slice_length(chunk, npix * frames, N, npix, map);
                        const int g = frame_group(frames, npix, N, len, map);
                        const bool fits = maps_bytes(npix * g, N, len, map) <= MAPS_MAX;
                        if (len < 2 || len > chunk || g < 1 || g > frames || (!fits && (g > 1 || len != chunk))) {
                            if (++bad < 6) printf("render %lld x %d, %d frames, chunk %d: slices of %d, groups of %d\n", (long long)npix, N, frames, chunk, len, g);
                        }
                        grouped += g < frames;
                        // a dual sweep: every frame at once, w_in and T_out (64 bytes) beside each map
                        const int sl = slice_length(chunk, npix * frames, N, npix * frames, map + 64);
                        if (sl < 2 || sl > chunk || (maps_bytes(npix * frames, N, sl, map + 64) > MAPS_MAX && sl != chunk)) {
                            if (++bad < 6) printf("sweep %lld x %d, %d frames, chunk %d: slices of %d\n", (long long)npix, N, frames, chunk, sl);
                        }
                        ++n;
                    }
    // 400,921 points x 1024 samples x 48 frames in FP64: 394 GB of maps in one launch, two frames at a time here
    const int len = slice_length(32, (int64_t)400921 * 48, 1024, 400921, 160);
    printf("plans %ld, grouped %ld, outside the limit %ld; 400,921 x 1024 x 48 in FP64: slices of %d, groups of %d\n", n, grouped, bad, len,
           frame_group(48, 400921, 1024, len, 160));
    return bad != 0 || grouped == 0 || len != 8 || frame_group(48, 400921, 1024, len, 160) != 2;
}
