// Results to host memory (fetch.h).
//
// The device holds results compactly (u8 to u32 fields, one array each); the
// C ABI's arrays are 64-bit words.  A kernel packs the words straight into
// pinned host memory, a chunk of 2 MiB at a time, and host threads copy each
// chunk to the caller's arrays while the next ones are packed.  The kernel is
// bound by the link: 52 to 55 GB/s written, from 64 workgroups up, as fast as
// a plain copy of the finished words and without their pass through HBM.  One
// host thread copies about 30 GB/s out of pinned memory (and touches about 5
// GB/s of fresh pages), so long fetches use four.  Fetching the fields one by
// one through pageable copies and widening them on one host thread took 10.0
// ms for the vertices and faces of 101^3 vertices and 20 functions (134 MB);
// this takes 3.1 ms.
#include "fetch.h"

#include <algorithm>
#include <cstring>
#include <exception>
#include <thread>

#include "../devmem.h"

namespace rin {

namespace {

constexpr uint64_t kChunk = 262144;  // words: 2 MiB, about 40 us of the link

struct PackArgs {
    PackCol col[kPackCols];
    uint64_t first[kPackCols + 1];  // first word of each column in the whole stream
    int n;
};

template <class T>
__device__ inline uint64_t ld(const PackCol& C, int q, uint64_t i) {
    return (uint64_t) static_cast<const T*>(C.p[q])[i];
}

__device__ inline uint64_t pack_word(const PackCol& C, uint64_t i) {
    switch (C.kind) {
        case PACK_U32: return ld<uint32_t>(C, 0, i);
        case PACK_U8: return ld<uint8_t>(C, 0, i);
        case PACK_U8_NONE: {
            const uint64_t x = ld<uint8_t>(C, 0, i);
            return x == 0xFFu ? ~0ull : x;
        }
        case PACK_F64: return ld<uint64_t>(C, 0, i);
        case PACK_VERT: {
            const uint64_t v = i / 11;
            const uint32_t c = (uint32_t)(i - 11 * v);
            if (c == 0) return ld<uint32_t>(C, 0, v);
            if (c == 1) return ld<uint16_t>(C, 1, v);
            if (c == 2) return ld<uint8_t>(C, 2, v);
            if (c < 7) {
                const uint64_t x = ld<uint32_t>(C, 3, 4 * v + (c - 3));
                return x == 0xFFFFFFFFu ? ~0ull : x;
            }
            const uint64_t x = ld<uint8_t>(C, 4, 4 * v + (c - 7));
            return x == 0xFFu ? ~0ull : x;
        }
        case PACK_TET_FACE: return (i & 1) ? ld<uint16_t>(C, 1, i >> 1) : ld<uint32_t>(C, 0, i >> 1);
        case PACK_EDGE_OCC: {
            const uint64_t x = ld<uint32_t>(C, 0, i >> 1), f = ld<uint32_t>(C, 1, x);
            return (i & 1) ? x - ld<uint32_t>(C, 2, f) : f;
        }
        default: {  // PACK_ROWMAJOR
            const uint64_t v = i / C.rows, f = i - v * C.rows;
            return ld<uint64_t>(C, 0, f * C.stride + v);
        }
    }
}

// words [begin, end) of the stream to out[0..)
__global__ void __launch_bounds__(256) k_pack(PackArgs A, uint64_t begin, uint64_t end, uint64_t* __restrict__ out) {
    for (uint64_t w = begin + (uint64_t)blockIdx.x * 256 + threadIdx.x; w < end; w += (uint64_t)gridDim.x * 256) {
        int c = 0;
        while (c + 1 < A.n && w >= A.first[c + 1]) ++c;
        out[w - begin] = pack_word(A.col[c], w - A.first[c]);
    }
}

}  // namespace

void HostStage::need(int slots) {
    for (int i = 0; i < slots; ++i) {
        if (!host_[i]) {
            RIN_HIP(hipHostMalloc((void**)&host_[i], 8 * kChunk, hipHostMallocMapped | hipHostMallocCoherent));
            RIN_HIP(hipHostGetDevicePointer((void**)&dev_[i], host_[i], 0));
        }
        if (!done_[i]) RIN_HIP(hipEventCreateWithFlags(&done_[i], hipEventDisableTiming));
    }
}

void HostStage::release() {
    for (int i = 0; i < kSlots; ++i) {
        if (host_[i]) (void)hipHostFree(host_[i]);
        if (done_[i]) (void)hipEventDestroy(done_[i]);
        host_[i] = dev_[i] = nullptr;
        done_[i] = nullptr;
    }
}

void HostStage::fetch(int device, const std::vector<PackCol>& cols, hipStream_t s) {
    PackArgs A;
    A.n = 0;
    uint64_t words = 0;
    for (const PackCol& c : cols) {
        if (!c.words) continue;
        if (A.n == kPackCols) throw std::logic_error("too many columns");
        A.first[A.n] = words;
        A.col[A.n++] = c;
        words += c.words;
    }
    if (!words) {
        RIN_HIP(hipStreamSynchronize(s));
        return;
    }
    for (int c = A.n; c <= kPackCols; ++c) A.first[c] = words;
    const uint64_t chunks = (words + kChunk - 1) / kChunk;
    // a thread pays from a few chunks on (starting one costs about 15 us)
    const int threads = chunks >= 8 ? kThreads : (chunks >= 3 ? 2 : 1);
    need((int)std::min<uint64_t>(chunks, 2 * threads));
    // thread t takes chunks t, t + n, ... and two slots of its own, so that
    // one is packed while it copies the other
    auto work = [&](int t, int n) {
        auto launch = [&](uint64_t k) {
            const uint64_t b = k * kChunk, e = std::min(words, b + kChunk);
            const int slot = t + n * (int)((k / n) & 1);
            hipLaunchKernelGGL(k_pack, dim3((unsigned)((e - b + 255) / 256)), dim3(256), 0, s, A, b, e, dev_[slot]);
            RIN_HIP(hipGetLastError());
            RIN_HIP(hipEventRecord(done_[slot], s));
        };
        if ((uint64_t)t < chunks) launch((uint64_t)t);
        if ((uint64_t)(t + n) < chunks) launch((uint64_t)(t + n));
        for (uint64_t k = (uint64_t)t; k < chunks; k += n) {
            const int slot = t + n * (int)((k / n) & 1);
            RIN_HIP(hipEventSynchronize(done_[slot]));
            const uint64_t b = k * kChunk, e = std::min(words, b + kChunk);
            for (int c = 0; c < A.n; ++c) {
                const uint64_t lo = std::max(b, A.first[c]), hi = std::min(e, A.first[c + 1]);
                if (lo < hi)
                    std::memcpy(static_cast<uint64_t*>(A.col[c].dst) + (lo - A.first[c]), host_[slot] + (lo - b),
                                8 * (hi - lo));
            }
            if (k + 2 * (uint64_t)n < chunks) launch(k + 2 * (uint64_t)n);
        }
    };
    if (threads == 1) {
        work(0, 1);
        return;
    }
    std::vector<std::exception_ptr> err((size_t)threads);
    auto guarded = [&](int t) {
        try {
            RIN_HIP(hipSetDevice(device));
            work(t, threads);
        } catch (...) {
            err[(size_t)t] = std::current_exception();
        }
    };
    std::vector<std::thread> pool;
    pool.reserve((size_t)threads);
    int started = 1;
    try {
        for (; started < threads; ++started) pool.emplace_back(guarded, started);
    } catch (...) {
        // no thread to be had (or no memory for one; nothing may leave here
        // while others run): this one takes the rest's chunks after its own
    }
    guarded(0);
    for (int t = started; t < threads; ++t) guarded(t);
    for (auto& t : pool) t.join();
    // nothing of this fetch is left on the stream or in the slots
    const hipError_t sync = hipStreamSynchronize(s);
    for (auto& e : err)
        if (e) std::rethrow_exception(e);
    RIN_HIP(sync);
}

}  // namespace rin
