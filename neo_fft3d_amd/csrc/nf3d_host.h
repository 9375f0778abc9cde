// One frame of one plane from and to host memory in two halves, so that the
// front end queues every plane of a frame before it waits for the first
// (nf3d_engine.cpp; not part of the public C ABI).
#pragma once
#include <cstddef>

#include "../../include/nf3d.h"

// Queues the uploads, the filtering and the download.  On success the engine
// stays locked by the calling thread until its nf3d_engine_frame_end, which
// the caller owes it on every path.  Neither half throws.  Several engines are
// begun in one order by every caller (the front end: plane order, of engines
// that only it holds) and ended in the same order, so that a second caller's
// frame begins on the first engine while this one's ends on the others.
int nf3d_engine_frame_begin(nf3d_engine* e, int n, const nf3d_frame_ref* frames, int nframes, void* dst,
                            int dst_stride, char* err, size_t errlen);
// Waits for the frame and hands it to the dst given at the beginning.
int nf3d_engine_frame_end(nf3d_engine* e, char* err, size_t errlen);
