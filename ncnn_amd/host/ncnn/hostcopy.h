// memcpy spread over a few threads, for the host side of large uploads.
#ifndef NCNN_HOSTCOPY_H
#define NCNN_HOSTCOPY_H

#include <stddef.h>

namespace ncnn {

// Copies like memcpy.  From 1 MB up the bytes are shared out between the calling thread and a few helper threads of the
// process; a second caller that finds them busy copies alone, and so does a forked child.
void parallel_copy(void* dst, const void* src, size_t bytes);

} // namespace ncnn

#endif // NCNN_HOSTCOPY_H
