// tiled_forward_kernel (tiled_kernel.h) for bf16_t; a file per type because each is half a minute of compiling.
#include "tiled_kernel.h"

namespace mnt {

template void tiled_forward<bf16_t>(const bf16_t *, const bf16_t *, const int *, const int *, int64_t, int64_t, int64_t, int64_t,
                                 int64_t, const Epilogue &, bf16_t *, hipStream_t);

}  // namespace mnt
