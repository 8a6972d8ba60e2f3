// ss_pack.h -- what the driver needs of the device: a buffer of the handle,
// copies on its stream, and the packing kernels.  No HIP headers here, so
// that host-only translation units can use it; an int result is a hipError_t.
#pragma once

#include <cstddef>
#include <cstdint>

#include "steadyscan.h"

namespace ss {

// n block matrices (nbm elements of esz bytes each) from raw frames of rawPix
// elements, through the table `at` (the pixel of every element, counted from
// `frames`, kNoPixel where the block is shorter: 0).  toFloat: the elements
// are doubles, and floats in the block matrices.
constexpr uint32_t kNoPixel = ~0u;
int pack_frames(void *stream, const uint32_t *at, int nbm, int esz, bool toFloat, const void *frames, size_t rawPix, int n,
                void *out);
// used[c] = 1 when column c (fh bytes) of mask has a nonzero byte.
int used_blocks(void *stream, const uint8_t *mask, int fh, int cols, uint8_t *used);

// The driver's device memory of at least `bytes`, in use until
// handle_stack_done; nullptr on failure (st set).  Kept by the handle across
// calls (grown on demand, freed by ss_destroy) as the batches' memory is, but
// either is given back for the other where the device does not hold both.
void *handle_stack(ss_handle *h, size_t bytes, ss_status *st);
void handle_stack_done(ss_handle *h);
// The handle's stream, as pack_frames takes it.
void *handle_raw_stream(const ss_handle *h);
// Host memory to the device through the handle's page-locked staging, which
// up to 16 host threads fill piece by piece; complete on return.
ss_status handle_upload(ss_handle *h, void *dst, const void *src, size_t bytes);
// Device memory to host, complete on return.
ss_status handle_download(ss_handle *h, void *dst, const void *src, size_t bytes);

}  // namespace ss
