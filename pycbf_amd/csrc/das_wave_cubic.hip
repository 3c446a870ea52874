// Wave-tile gather (das_wave.h): natural cubic.
#include <type_traits>

#include "das_wave.h"

namespace pycbf {

int wave_launch_cubic(const DasArgs &a, const WaveArgs &w, int sum, int fc, int mode, dim3 grid,
                      int nw, size_t lds, hipStream_t s)
{
    return wave_sum<GK_CUBIC>(sum, fc, mode, a, w, grid, nw, lds, s);
}

}  // namespace pycbf
