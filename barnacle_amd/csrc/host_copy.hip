// host_copy.hip -- results from device memory into the caller's arrays.
#include "host_copy.hpp"

#include <algorithm>
#include <cstring>

#include "abi_internal.hpp"

namespace bnx {

// Pieces of `per` 16-byte words, in order: few blocks, so that the first pieces
// arrive early (9.4 MB: 0.28 ms with 16 blocks of 16 KB pieces, 0.31 with 64,
// 0.39 with 64 of 64 KB).
constexpr int kCopyBlocks = 16;
static __global__ __launch_bounds__(256) void k_host_copy(const uint4* src, uint4* dst, uint32_t* flags, uint32_t job,
                                                          uint32_t words, uint32_t per) {
    const uint32_t n16 = words / 4, pieces = (n16 + per) / per;      // the last one holds the odd words too
    for (uint32_t p = blockIdx.x; p < pieces; p += gridDim.x) {
        const uint32_t end = min(n16, (p + 1) * per);
        for (uint32_t i = p * per + threadIdx.x; i < end; i += blockDim.x) dst[i] = src[i];
        if (p == pieces - 1 && threadIdx.x < words % 4) {
            const uint32_t i = 4 * n16 + threadIdx.x;
            reinterpret_cast<uint32_t*>(dst)[i] = reinterpret_cast<const uint32_t*>(src)[i];
        }
        __threadfence_system();
        __syncthreads();
        if (threadIdx.x == 0)
            __hip_atomic_store(&flags[p], job, __ATOMIC_RELEASE, __HIP_MEMORY_SCOPE_SYSTEM);
    }
}

HostCopy::~HostCopy() {
    if (buf_) (void)hipHostFree(buf_);
    if (flags_) (void)hipHostFree(flags_);
}

void HostCopy::grow(size_t bytes) {
    if (!flags_) {
        hip_check(hipHostMalloc((void**)&flags_, (kMaxPieces + 1) * sizeof(uint32_t), hipHostMallocDefault),
                  "hipHostMalloc");
        std::fill(flags_, flags_ + kMaxPieces + 1, 0u);
    }
    if (bytes <= buf_bytes_) return;
    if (buf_) (void)hipHostFree(buf_);
    buf_ = nullptr;
    buf_bytes_ = 0;
    bytes = std::min(kBuffer, (bytes + (1 << 20)) >> 20 << 20);
    hip_check(hipHostMalloc((void**)&buf_, bytes, hipHostMallocDefault), "hipHostMalloc");
    buf_bytes_ = bytes;
}

// Bytes [at, at + bytes) of the parts.
void HostCopy::batch(const char* src, size_t at, size_t bytes, const std::vector<Part>& parts, hipStream_t s) {
    grow(bytes);
    if (++job_ == 0) {                               // a flag never holds the job that is to come
        std::fill(flags_, flags_ + kMaxPieces + 1, 0u);
        job_ = 1;
    }
    const uint32_t words = (uint32_t)(bytes / 4), per = (uint32_t)(kPiece / 16);
    const size_t pieces = words / 4 / per + 1;
    hipLaunchKernelGGL(k_host_copy, dim3((unsigned)std::min<size_t>(pieces, kCopyBlocks)), dim3(256), 0, s,
                       (const uint4*)(src + at), (uint4*)buf_, flags_, job_, words, per);
    hip_check(hipGetLastError(), "kernel launch");
    size_t part = 0, begin = 0;                      // the part at hand and where it begins
    while (part < parts.size() && begin + parts[part].bytes <= at) begin += parts[part++].bytes;
    for (size_t p = 0; p < pieces; ++p) {
        for (uint32_t spins = 0; __atomic_load_n(&flags_[p], __ATOMIC_ACQUIRE) != job_; ++spins) {
            if (spins % 4096 != 4095) {
                __builtin_ia32_pause();
                continue;
            }
            const hipError_t e = hipStreamQuery(s);  // the stream is done, or has failed: the flag is there or never will be
            if (e == hipErrorNotReady) continue;
            hip_check(e, "result copy");
            if (__atomic_load_n(&flags_[p], __ATOMIC_ACQUIRE) != job_) throw bnh::Error(BN_E_DEVICE, "result copy incomplete");
            break;
        }
        const size_t a = at + p * kPiece, b = at + (p + 1 == pieces ? bytes : (p + 1) * kPiece);
        while (part < parts.size() && begin < b) {
            const size_t lo = std::max(a, begin), hi = std::min(b, begin + parts[part].bytes);
            if (lo < hi && parts[part].dst)
                std::memcpy((char*)parts[part].dst + (lo - begin), buf_ + (lo - at), hi - lo);
            if (begin + parts[part].bytes > b) break;
            begin += parts[part++].bytes;
        }
    }
}

void HostCopy::download(const void* src, const std::vector<Part>& parts, hipStream_t s) {
    size_t total = 0;
    for (const Part& p : parts) total += p.bytes;
    for (size_t at = 0; at < total; at += kBuffer)
        batch((const char*)src, at, std::min(kBuffer, total - at), parts, s);
}

}  // namespace bnx
