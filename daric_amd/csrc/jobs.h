// Device-side descriptors shared by the host launchers and the kernels.
#pragma once

#ifdef __HIPCC__
#include <hip/hip_runtime.h>
#endif

#include <cstdint>

#ifdef __HIPCC__
#define DARIC_HD __host__ __device__
#else
#define DARIC_HD
#endif

namespace daric {

// Fast 32-bit division by a run-time constant d (n, d < 2^31):
// q = (umulhi(n, m) + n) >> s with s = ceil(log2 d), m = floor(2^32 (2^s - d) / d) + 1.
struct FastDiv {
    uint32_t d = 1, m = 1, s = 0;
    FastDiv() = default;
    explicit FastDiv(uint32_t div) : d(div) {
        s = 0;
        while ((1ull << s) < div) ++s;
        m = static_cast<uint32_t>(((1ull << 32) * ((1ull << s) - div)) / div + 1);
    }
    inline DARIC_HD uint32_t div(uint32_t n) const {
        // (n * m) >> 32 lowers to v_mul_hi_u32 on the device.
        const uint32_t hi = static_cast<uint32_t>((static_cast<uint64_t>(n) * m) >> 32);
        return (hi + n) >> s;
    }
};

// Hand-over of a call's descriptors (jobs, segments, chunks, layer pointer
// tables) to its kernels. Descriptors of up to kInlineDescBytes travel inline
// in the kernel arguments (`ptr` null): no descriptor copy, no ring slot and
// no completion event, ~4 us per call on MI355X against ~9 us through the
// ring; such a launch also carries its descriptors by value, as a captured
// graph node needs. Larger sets go through the descriptor ring and `ptr`
// points at them (device memory, or the pinned host slot itself).
constexpr int kInlineDescBytes = 2816;
struct alignas(16) DescArg {
    const uint8_t* ptr;
    uint64_t reserved;
    alignas(16) uint8_t inl[kInlineDescBytes];
#ifdef __HIPCC__
    __host__ __device__
#endif
    const uint8_t* base() const { return ptr != nullptr ? ptr : inl; }
};

#ifdef __HIPCC__
// Descriptors are read-only and uniform across a workgroup: kernels address
// them in the constant address space, so they load through the scalar unit
// into SGPRs (a generic pointer would put them in VGPRs).
template <typename T>
using DescPtr = const __attribute__((address_space(4))) T*;
template <typename T>
__device__ __forceinline__ DescPtr<T> desc_at(const DescArg& d, int byte_off) {
    return (DescPtr<T>)(d.base() + byte_off);
}
typedef unsigned int DescWords __attribute__((ext_vector_type(4)));
// Copies one descriptor out of the constant address space. Its loads are all
// issued before the wait for any of them: left alone, the compiler sinks each
// load to its first use, and a workgroup's start becomes a chain of waits, each
// a round trip to the kernel arguments or to pinned memory (half a microsecond
// and more on MI355X).
template <typename T>
__device__ __forceinline__ T desc_load(DescPtr<T> p) {
    constexpr int N = sizeof(T) / 16;
    static_assert(sizeof(T) % 16 == 0 && (N == 2 || N == 5 || N == 7), "descriptors are whole 16-byte words");
    const __attribute__((address_space(4))) DescWords* src =
        reinterpret_cast<const __attribute__((address_space(4))) DescWords*>(p);
    DescWords w[N];
#pragma unroll
    for (int i = 0; i < N; ++i) w[i] = src[i];
    if constexpr (N == 2) asm volatile("" : "+s"(w[0]), "+s"(w[1]));
    else if constexpr (N == 5) asm volatile("" : "+s"(w[0]), "+s"(w[1]), "+s"(w[2]), "+s"(w[3]), "+s"(w[4]));
    else asm volatile("" : "+s"(w[0]), "+s"(w[1]), "+s"(w[2]), "+s"(w[3]), "+s"(w[4]), "+s"(w[5]), "+s"(w[6]));
    T v;
    __builtin_memcpy(&v, w, sizeof(T));
    return v;
}
// Has the listed kernel arguments (up to 8 words or pointers) in registers before
// what follows, so that their loads share one round trip.
#define DARIC_ARGS_TOGETHER4(a, b, c, d) asm volatile("" ::"s"(a), "s"(b), "s"(c), "s"(d))
#define DARIC_ARGS_TOGETHER6(a, b, c, d, e, f) asm volatile("" ::"s"(a), "s"(b), "s"(c), "s"(d), "s"(e), "s"(f))
// Reads one value of a list that every lane of the workgroup reads at the same
// place (a page id, a layer's address) through the scalar unit.
template <typename T>
__device__ __forceinline__ T uniform_load(const T* p) {
    return *(const __attribute__((address_space(4))) T*)p;
}
// The last descriptor whose tile_begin is at most `tile`, of n in ascending
// order that start at tile 0.
template <typename T>
__device__ __forceinline__ int find_by_tile(DescPtr<T> p, int n, int tile) {
    int lo = 0, hi = n - 1;
    while (lo < hi) {
        const int mid = (lo + hi + 1) >> 1;
        if (p[mid].tile_begin <= tile) lo = mid; else hi = mid - 1;
    }
    return lo;
}
#endif

// One page-copy job: one (layer, chunk) pair, the counterpart of the
// reference's PageCopyJobDesc (csrc/cache_ops/cache_ops.h:24-36). Byte units.
// Tile t of the job (t < prefix * n_sel) is prefix index p = t / n_sel and
// selected page s = t % n_sel; its staging bytes are
// stage[(p * n_sel + s) * span, +span) and its cache bytes are
// layer[p * prefix_stride + idx[s] * page_stride, +span).
struct alignas(16) CopyJob {
    uint8_t* layer;
    uint8_t* stage;
    const int32_t* idx;
    int64_t prefix_stride;
    int64_t page_stride;
    int32_t span;
    int32_t n_sel;
    int32_t prefix;
    int32_t num_pages;        // page ids outside [1, num_pages) are skipped
    int32_t n_tokens;         // fused rotate: tokens of the job to rotate
    float delta;              // fused rotate: fp32(new_pos - old_pos)
    int32_t part_units;       // page copies: accesses of a part of a tile
    FastDiv parts;            // page copies: parts a tile is cut into
};
static_assert(sizeof(CopyJob) == 80, "CopyJob layout");

// Row structure of a page span for the fused scatter + rotate kernel. The
// span is n_rows rows of W elements (rows dense, W contiguous). Rows
// [0, krows) of prefix index 0 hold K head rows: row r is token
// (r / tok_div) % PS and head h = tok_div == 1 ? (r / PS) % H : r % H.
// Elements [0, R) of a K row are rotated; everything else is copied.
struct RowGeom {
    int32_t W;         // row width in elements
    int32_t n_rows;    // rows per page span
    int32_t krows;     // K rows (prefix index 0 only)
    int32_t tok_div;   // 1 (head-major rows) or H (token-major rows)
    int32_t PS;        // tokens per page
    int32_t H;         // heads
    int32_t R;         // rotary dim
    int32_t n_rot;     // aligned: 16-byte units of a pair half (NeoX) or of the rotary dims (GPT-J)
    int32_t aligned;   // 1 when those are whole units
};

// In-place rotation geometry (elements): K element (b, s, h, d) of a layer is
// at base + b*sb + s*ss + h*sh + d, d < R (reference adapter.py:312-364).
struct InplaceGeom {
    int64_t sb;
    int64_t ss;
    int64_t sh;
    int32_t PS;
    int32_t H;
    int32_t R;
    int32_t num_blocks;
    int32_t n_rot;     // rotated items per head row (lane path: rotated units per pair half)
    int32_t tile_tokens;
    int32_t upr;       // lane and rows paths: 16-byte units per K row (lane: a power of two dividing 64)
    int32_t tok_div;   // lane and rows paths: rows per token step (H: token-major rows, 1: head-major)
    int32_t log2_parts;  // lane path: parts per page tile
    int32_t min_block;   // block ids below it are skipped: 0, or 1 to skip the null block too
    int32_t walk;        // rows path: units of a row that hold rotated values
    int32_t parts;       // rows path: parts per page, each but the last of part_rows rows
    int32_t part_rows;
    int32_t pad0;
};

struct RopeSeg {
    int64_t bt_offset;
    int32_t tok_start;
    int32_t n_tokens;
    float delta;
    int32_t tile_begin;   // first tile of this segment
    int32_t pad0;
    int32_t pad1;
};

// Paged K/V row geometry for the selection kernels (elements, D contiguous).
struct KVGeom {
    int64_t sb, ss, sh;     // block, slot, head strides
    int64_t v_off;          // element offset of V row relative to K row (-1: no V)
    int32_t PS, H, D, num_blocks;
};

struct SelChunk {
    int64_t bt_offset;
    int64_t row_offset;
    int32_t n_tokens;
    int32_t k;
    int32_t tile_begin;
    int32_t tok0;          // position of token 0 in the page at bt_offset (0 <= tok0 < PS)
};

}  // namespace daric
