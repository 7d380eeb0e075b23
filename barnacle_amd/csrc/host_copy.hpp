// host_copy.hpp -- results from device memory into the caller's arrays.
#pragma once
#include <hip/hip_runtime.h>

#include <cstdint>
#include <vector>

namespace bnx {

// A copy to pageable memory goes through a page-locked buffer anyway; the
// runtime copies a megabyte in, waits, copies it out, and only then starts the
// next (17.7 GB/s for large films, 0.1 ms for the smallest).  Here one kernel
// writes the whole result into the context's page-locked buffer, piece after
// piece, and raises a flag behind each; the host copies the pieces out as they
// arrive (33 GB/s, what one core copies; 20 us for 0.2 MB).  Asynchronous
// copies with an event behind each 1 or 2 MB chunk reached 29 and 31 GB/s: the
// gaps between the copies bound them.  The wait holds a core, as the runtime's
// own does (a frame of 70.9 ms takes 70.9 ms of the calling thread, one that
// waited in the runtime took 114.9 of 114.9).  The buffer holds at most kBuffer
// bytes and lives as long as the context.
class HostCopy {
public:
    struct Part { void* dst; size_t bytes; };        // dst null: not wanted; bytes a multiple of 4
    HostCopy() = default;
    HostCopy(const HostCopy&) = delete;
    ~HostCopy();
    // The parts, which lie one after the other from `src` (16-byte aligned) on
    // in device memory, after everything enqueued on `s` so far.  Returns when
    // they have arrived.
    void download(const void* src, const std::vector<Part>& parts, hipStream_t s);

private:
    static constexpr size_t kPiece = (size_t)16 << 10, kBuffer = (size_t)16 << 20;
    static constexpr size_t kMaxPieces = kBuffer / kPiece;
    void grow(size_t bytes);
    void batch(const char* src, size_t at, size_t bytes, const std::vector<Part>& parts, hipStream_t s);

    char* buf_ = nullptr;
    uint32_t* flags_ = nullptr;                      // page-locked: the job that last wrote each piece
    size_t buf_bytes_ = 0;
    uint32_t job_ = 0;
};

}  // namespace bnx
