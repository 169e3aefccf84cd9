// Results to host memory: the arrays that the C ABI hands out, packed on the
// device into the caller's 64-bit layout.
#pragma once
#include <hip/hip_runtime.h>

#include <cstdint>
#include <vector>

namespace rin {

// One output array of 64-bit words and how its word i follows from device arrays.
enum PackKind : int {
    PACK_U32 = 0,   // p0: u32
    PACK_U8,        // p0: u8
    PACK_U8_NONE,   // p0: u8, 0xFF becomes all ones
    PACK_F64,       // p0: f64
    PACK_VERT,      // 11 words a vertex; p0..p4: tet u32, j u16, simplex size u8, simplex vertices 4 u32, functions 4 u8
    PACK_TET_FACE,  // 2 words an entry; p0: tet u32, p1: local face u16
    PACK_EDGE_OCC,  // 2 words an entry (face, corner); p0: face-corner position u32, p1: its face, p2: face starts
    PACK_ROWMAJOR   // p0: f64, `rows` columns of `stride` function-major values
};
struct PackCol {
    int kind = PACK_U32;
    uint32_t rows = 0;
    uint64_t stride = 0;
    const void* p[5] = {nullptr, nullptr, nullptr, nullptr, nullptr};
    uint64_t words = 0;
    void* dst = nullptr;  // host
};
constexpr int kPackCols = 6;

// Pinned staging that a context keeps for its fetches (nothing before the
// first; given back with the context).  Not for concurrent use.
class HostStage {
  public:
    HostStage() = default;
    HostStage(const HostStage&) = delete;
    HostStage& operator=(const HostStage&) = delete;
    ~HostStage() { release(); }
    // fills every column's host array; returns when they are complete
    void fetch(int device, const std::vector<PackCol>& cols, hipStream_t s);
    void release();

  private:
    static constexpr int kThreads = 4, kSlots = 2 * kThreads;
    uint64_t* host_[kSlots] = {};
    uint64_t* dev_[kSlots] = {};
    hipEvent_t done_[kSlots] = {};
    void need(int slots);
};

}  // namespace rin
