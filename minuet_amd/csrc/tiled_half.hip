// tiled_forward_kernel (tiled_kernel.h) for half_t; a file per type because each is half a minute of compiling.
#include "tiled_kernel.h"

namespace mnt {

template void tiled_forward<half_t>(const half_t *, const half_t *, const int *, const int *, int64_t, int64_t, int64_t, int64_t,
                                 int64_t, const Epilogue &, half_t *, hipStream_t);

}  // namespace mnt
