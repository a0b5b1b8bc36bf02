// streamed_forward_kernel (streamed_kernel.h) for bf16_t; a file per type because each is most of a minute of compiling.
#include "streamed_kernel.h"

namespace mnt {

template void streamed_forward<bf16_t>(const bf16_t *, const bf16_t *, const int *, const int *, int64_t, int64_t, int64_t,
                                    int64_t, int64_t, const Epilogue &, bf16_t *, hipStream_t);

}  // namespace mnt
