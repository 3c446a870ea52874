// Wave-tile gather (das_wave.h): k-order cubic, Akima and makima.
#include <type_traits>

#include "das_wave.h"

namespace pycbf {

int wave_launch_hermite(int gk, const DasArgs &a, const WaveArgs &w, int sum, int fc, int mode,
                        dim3 grid, int nw, size_t lds, hipStream_t s)
{
    if (gk == GK_KORDER) return wave_sum<GK_KORDER>(sum, fc, mode, a, w, grid, nw, lds, s);
    return wave_sum<GK_AKIMA>(sum, fc, mode, a, w, grid, nw, lds, s);
}

}  // namespace pycbf
