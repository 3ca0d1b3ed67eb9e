// Downloads of large results into the caller's (pageable) arrays.
#pragma once
#include <hip/hip_runtime.h>
#include <cstddef>
#include <memory>
#include <vector>

namespace sfg {

// Pinned staging buffers of the process (at most four sets of 16 MB, one for each download
// under way), held by the objects that download through them and freed with the last of
// these.
struct Staging;
std::shared_ptr<Staging> staging();

// dst row map[i] (map null: i), `width` bytes long and tightly packed, = source row
// i, `pitch` bytes apart on the device, for i < rows; queued behind the work of
// stream st, complete on return.
//
// A fresh host array costs a page fault per 4 KB when it is first written, more than
// its transfer: 140 MB in four arrays took 42 ms as copies into staging vectors and from there
// into the arrays (32-45 ms copied there directly), and take 12 ms here, where 8 threads
// each copy what the DMA engine has put into their pinned buffers (1000 predictions of
// 32000 samples, all told: 16.5 ms then, 5.7 ms now).  Small results take fewer threads or
// none (kDirect, kOne).  Without pinned memory the copy is direct; rows to be copied apart
// then pass through scratch, which a caller of many downloads keeps.
hipError_t download(const std::shared_ptr<Staging> &staging, void *dst, const void *src, size_t pitch, size_t width,
                    size_t rows, const int *map, hipStream_t st, std::vector<char> *scratch = nullptr);

} // namespace sfg
