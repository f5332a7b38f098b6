// Translation unit of the second code object in libmaize_hip.so: the kernels of the launcher's own forms (forms.hpp).
#include "common.hpp"
#include "gemm_tile.hpp"
