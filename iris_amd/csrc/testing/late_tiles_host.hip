// Host builds of the words by which late tiles are shared out (late_tiles.hpp), for the CPU tests.
#include <hip/hip_runtime.h>

#include "../../../include/iris_amd_testing.h"
#include "../late_tiles.hpp"

extern "C" int32_t iris_late_join_host(int32_t word, int32_t most, int32_t tile) { return iris_amd::late_join(word, most, tile); }
extern "C" int32_t iris_late_next_host(int32_t word, int32_t link) { return iris_amd::late_next(word, link); }
