// Recompute selection kernels (gfx950): per-token K deviation, per-chunk
// top-k by LDS radix select, and the merge of recomputed rows.
//
// Deviation order (the keys are bit-exact against the CPU oracle, which sums
// in exactly this order): a wavefront owns one token; the token's H*D
// elements, in (h, d) order, are cut into vectors of 8 elements; vector v is
// loaded by lane v % 64 in round v / 64; each lane accumulates
// acc = acc + diff * diff element by element (float32, no contraction),
// rounds ascending; the 64 lane sums are then combined by a butterfly over
// xor offsets 32, 16, 8, 4, 2, 1. Any NaN key is stored as 0x7FC00000.
//
// Top-k ranks keys by the IEEE total order of their float32 bits (NaN above
// +inf), ties to the lower token index, and writes the selected chunk-local
// indices in ascending order.
#include <hip/hip_runtime.h>

#include "common.h"
#include "elem.h"
#include "jobs.h"
#include "kernels.h"
#include "launch.h"

namespace daric {

namespace {

constexpr int kThreads = 256;
constexpr int kWaves = kThreads / 64;
// Tokens a lane group sums in the deviation kernel: 8 for 16-bit caches (16 loads
// of 16 bytes in flight per lane; 3-4% faster than 4 at config 3), 4 for fp8
// caches, where the 8-token form measured slower (config 5).
template <int CK> constexpr int dev_tok_per_group() { return CK == kE4M3 ? 4 : 8; }
constexpr int kMergeTok = 8;                       // selected tokens per merge workgroup
constexpr int kMaxGridYZ = 65535;                  // grid.y / grid.z limit; larger counts are sliced

// 8 elements: 16 bytes for 2-byte types, 8 bytes for fp8. Loaded raw (so a
// lane keeps few registers per load in flight) and converted when summed.
template <int KIND> struct Raw8 { u32x4 w; };
template <> struct Raw8<kE4M3> { u32x2 w; };

template <int KIND>
__device__ __forceinline__ Raw8<KIND> load_raw8(const uint8_t* p) {
    Raw8<KIND> r;
    if constexpr (KIND == kE4M3)
        r.w = __builtin_nontemporal_load(reinterpret_cast<const u32x2*>(p));
    else
        r.w = __builtin_nontemporal_load(reinterpret_cast<const u32x4*>(p));
    return r;
}

template <int KIND>
__device__ __forceinline__ void unpack8(const Raw8<KIND>& r, float* x, float scale) {
    if constexpr (KIND == kE4M3) {
#ifdef DARIC_FP8_SOFTWARE
#pragma unroll
        for (int b = 0; b < 4; ++b) { x[b] = e4m3_to_f32((r.w[0] >> (8 * b)) & 0xffu); x[4 + b] = e4m3_to_f32((r.w[1] >> (8 * b)) & 0xffu); }
#else
        e4m3x4_to_f32_hw(r.w[0], x);
        e4m3x4_to_f32_hw(r.w[1], x + 4);
#endif
#pragma unroll
        for (int i = 0; i < 8; ++i) x[i] = x[i] * scale;
    } else {
#pragma unroll
        for (int q = 0; q < 4; ++q) {
            if (KIND == kBF16) {
                x[2 * q] = u2f(r.w[q] << 16);
                x[2 * q + 1] = u2f(r.w[q] & 0xffff0000u);
            } else {
                const uint32_t word = r.w[q];
                x[2 * q] = f16_to_f32(word & 0xffffu);
                x[2 * q + 1] = f16_to_f32(word >> 16);
            }
        }
    }
}

// Keys of tokens of chunk c in layer l in the fixed order above. A group of G
// lanes sums TPG consecutive tokens, the first of them j0. G is 64, or the power
// of two that holds a token's vectors where they are fewer (heads split over
// GPUs, small models): the lanes of the fixed order that have no vector add
// +0 to sums that are not -0, so leaving them out gives the same bits, and a
// wavefront's loads serve 64 / G times the tokens. The butterfly leaves a key in
// every lane of its group. A token past the chunk's end, or whose block id lies
// outside [0, num_blocks), is not read and gets key 0; a NaN key is 0x7FC00000.
template <int CK, int NK, int TPG, int G>
__device__ __forceinline__ void group_keys(const SelChunk& c, int j0, int sub, const KVGeom& g,
                                           const uint8_t* __restrict__ base, const int32_t* __restrict__ bt,
                                           const uint8_t* __restrict__ k_new, int64_t T, int l,
                                           const float* __restrict__ ksc, float* key) {
#pragma clang fp contract(off)
    constexpr int CES = CK == kE4M3 ? 1 : 2;
    const int N = g.H * g.D;
    const int n_vec = N >> 3;
    const int rounds = G == 64 ? (n_vec + 63) >> 6 : 1;

    int64_t cache_row[TPG];
    const uint8_t* new_row[TPG];
    bool valid[TPG];
#pragma unroll
    for (int i = 0; i < TPG; ++i) {
        const int j = j0 + i;
        const int p = c.tok0 + j;                  // position in the chunk's block list
        int blk = -1;
        if (j < c.n_tokens) blk = bt[c.bt_offset + p / g.PS];
        valid[i] = j < c.n_tokens && blk >= 0 && blk < g.num_blocks;
        cache_row[i] = static_cast<int64_t>(blk) * g.sb + static_cast<int64_t>(p % g.PS) * g.ss;
        new_row[i] = k_new + ((static_cast<int64_t>(l) * T + c.row_offset + j) * N) * 2;
    }

    float acc[TPG];
#pragma unroll
    for (int i = 0; i < TPG; ++i) acc[i] = 0.0f;

    for (int r = 0; r < rounds; ++r) {
        const int v = r * 64 + sub;
        if (v >= n_vec) break;
        const int e0 = v << 3;
        const int h = e0 / g.D;
        const int d0 = e0 - h * g.D;
        const float scale = (CK == kE4M3 && ksc) ? ksc[h] : 1.0f;
        Raw8<NK> ra[TPG];
        Raw8<CK> rb[TPG];
#pragma unroll
        for (int i = 0; i < TPG; ++i) {
            if (!valid[i]) continue;
            ra[i] = load_raw8<NK>(new_row[i] + static_cast<int64_t>(e0) * 2);
            rb[i] = load_raw8<CK>(base + (cache_row[i] + static_cast<int64_t>(h) * g.sh + d0) * CES);
        }
#pragma unroll
        for (int i = 0; i < TPG; ++i) {
            if (!valid[i]) continue;
            float a[8], b[8];
            unpack8<NK>(ra[i], a, 1.0f);
            unpack8<CK>(rb[i], b, scale);
#pragma unroll
            for (int e = 0; e < 8; ++e) {
                const float df = a[e] - b[e];
                const float sq = df * df;
                acc[i] = acc[i] + sq;
            }
        }
    }
#pragma unroll
    for (int i = 0; i < TPG; ++i) {
        float s = acc[i];
#pragma unroll
        for (int off = G / 2; off >= 1; off >>= 1) s = s + __shfl_xor(s, off, 64);
        float k = valid[i] ? s : 0.0f;
        if (k != k) k = u2f(0x7fc00000u);
        key[i] = k;
    }
}

// Lanes per token: see group_keys.
inline int dev_group(int n_vec) { return n_vec > 32 ? 64 : n_vec > 16 ? 32 : n_vec > 8 ? 16 : 8; }

// Bound by HBM. G = 64 takes tokens of more than 256 values. A group of 16 lanes
// against it, MI355X: 8 chunks of 700 tokens of 80 values in one layer 8.7 -> 5.7
// us; with groups of 32 and 16 lanes the whole selection of 23 layers of 2 x 64
// (16 x 5 chunks) went from 268 to 116 us, of 59 layers of 1 x 256 from 390 to 233.
template <int CK, int NK, int G>
__global__ __launch_bounds__(kThreads) void deviation_kernel(
    DescArg d, int layer_off, KVGeom g, const int32_t* __restrict__ bt,
    const uint8_t* __restrict__ k_new, int64_t T, int n_chunks,
    const float* __restrict__ k_scales, float* __restrict__ keys, int l0) {
    const DescPtr<SelChunk> chunks = desc_at<SelChunk>(d, 0);
    const DescPtr<uint8_t*> layers = desc_at<uint8_t*>(d, layer_off);
    const int l = static_cast<int>(blockIdx.y) + l0;
    const int tile = static_cast<int>(blockIdx.x);
    const SelChunk c = desc_load(chunks + find_by_tile(chunks, n_chunks, tile));
    const int sub = static_cast<int>(threadIdx.x) & (G - 1);
    const int group = static_cast<int>(threadIdx.x) / G;
    constexpr int kTok = dev_tok_per_group<CK>();
    const int j0 = ((tile - c.tile_begin) * (kThreads / G) + group) * kTok;
    const float* ksc = k_scales ? k_scales + static_cast<int64_t>(l) * g.H : nullptr;
    float key[kTok];
    group_keys<CK, NK, kTok, G>(c, j0, sub, g, layers[l], bt, k_new, T, l, ksc, key);
#pragma unroll
    for (int i = 0; i < kTok; ++i) {
        const int j = j0 + i;
        if (sub == i % G && j < c.n_tokens) keys[static_cast<int64_t>(l) * T + c.row_offset + j] = key[i];
    }
}

__device__ __forceinline__ uint32_t order_key(float f) {
    uint32_t b = f2u(f);
    if ((b & 0x7fffffffu) > 0x7f800000u) b = 0x7fc00000u;
    return (b & 0x80000000u) ? ~b : (b | 0x80000000u);
}

// Per-chunk top-k by a workgroup of T lanes: the k largest of n order keys, ties
// to the lower index, written in ascending index order to orow[0 .. k-1] (when
// not null) and, when s_sel is not null, to the LDS array s_sel (visible to the
// other lanes after the caller's next barrier).
//
// Bound by latency: a chain of passes with barriers between them, so the passes
// are few and each pass is short. Wavefront w takes the consecutive keys of
// slots [w * slots, (w + 1) * slots) of 64, slot by slot, and holds them in
// registers (KPT slots; KPT = 0: it reads them again in each pass, for chunks
// longer than any register file). Radix passes find the k-th largest key: three
// of 11, 11 and 10 bits, or for a single wavefront, which would spend itself on
// 2048 bins, four of 8. A pass whose digit holds exactly the keys still wanted
// is the last. Lanes add to the LDS histogram one by one, except where all keys
// of a wavefront share the digit (ties, zeros), which one lane adds. The last
// step needs one barrier: the wavefronts' counts give each its place in the
// output.
// Against 256 lanes with four 8-bit passes over keys in LDS (from 8192 tokens,
// in memory), MI355X, 15% of the tokens selected: one chunk of 500 tokens 6.0 ->
// 4.6 us, 16 of 5000 29.2 -> 9.5 us, one of 12000 78 -> 18 us, 6 of 30000 194 ->
// 36 us, 6144 of 512 31.2 -> 23.6 us; all keys equal 6-440 -> 6-94 us.
constexpr int kTopkWave = 256, kTopkGroup = 2048;   // longest chunks of one and of four wavefronts
template <int T>
struct TopkLds {
    static constexpr int kBits = T == 64 ? 8 : 11;
    static constexpr int kBins = 1 << kBits;
    static constexpr int kPerLane = kBins / T;
    // Bin x lies at (x % kPerLane) * T + x / kPerLane, so that the lanes, which
    // sum kPerLane neighbouring bins each, read consecutive words.
    static __device__ __forceinline__ uint32_t at(uint32_t x) {
        return (x % kPerLane) * T + x / kPerLane;
    }
    uint32_t hist[kBins];
    uint32_t wave_a[T / 64], wave_b[T / 64];
    uint32_t digit, above, count;
};

template <int T, int KPT, typename KeyAt>
__device__ __forceinline__ void chunk_topk(KeyAt key_at, int n, int k, int32_t* __restrict__ orow, int32_t* s_sel,
                                           TopkLds<T>& sm) {
    constexpr int W = T / 64;
    using Lds = TopkLds<T>;
    constexpr int BPT = Lds::kPerLane;
    constexpr int R = KPT > 0 ? KPT : 1;
    const int tid = static_cast<int>(threadIdx.x);
    const int lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    // Places past 2^31 - 1 occur where KPT is 0 only; unsigned places ran the
    // register forms 2% slower.
    const int slots = KPT > 0 ? (n + T - 1) / T : topk_slots(n, T);
    const int i0 = wave * slots * 64 + lane;
    uint32_t key[R];
    if constexpr (KPT > 0) {
#pragma unroll
        for (int s = 0; s < KPT; ++s) {
            key[s] = 0;
            if (s < slots && i0 + s * 64 < n) key[s] = key_at(i0 + s * 64);
        }
    }
    // f(slot, key, whether there is one) for the wavefront's slots
    const auto each = [&](auto&& f) {
        if constexpr (KPT > 0) {
#pragma unroll
            for (int s = 0; s < KPT; ++s)
                if (s < slots) f(s, key[s], i0 + s * 64 < n);
        } else {
            for (int s = 0; s < slots; ++s) {
                const uint32_t i = static_cast<uint32_t>(i0) + static_cast<uint32_t>(s) * 64;
                const bool in = i < static_cast<uint32_t>(n);
                f(s, in ? key_at(static_cast<int>(i)) : 0u, in);
            }
        }
    };
#pragma unroll
    for (int b = 0; b < BPT; ++b) sm.hist[b * T + tid] = 0;
    __syncthreads();

    uint32_t prefix = 0, mask = 0, krem = static_cast<uint32_t>(k);
    bool whole = k >= n;      // every key from `prefix` up is taken
    int left_bits = 32;
    for (int pass = 0; left_bits > 0 && !whole; ++pass) {
        const int width = min(left_bits, Lds::kBits);
        const int shift = left_bits - width;
        left_bits = shift;
        const uint32_t dmask = (1u << width) - 1u;
        each([&](int, uint32_t v, bool in) {
            const bool act = in && (v & mask) == prefix;
            const uint32_t dig = (v >> shift) & dmask;
            const unsigned long long some = __ballot(act);
            if (some == 0) return;
            const int lead = __ffsll(static_cast<long long>(some)) - 1;
            const uint32_t d0 = static_cast<uint32_t>(__builtin_amdgcn_readlane(static_cast<int>(dig), lead));
            if (__ballot(act && dig != d0) == 0) {
                if (lane == lead) atomicAdd(&sm.hist[Lds::at(d0)], static_cast<uint32_t>(__popcll(some)));
            } else if (act) {
                atomicAdd(&sm.hist[Lds::at(dig)], 1u);
            }
        });
        __syncthreads();
        // Lane t sums bins [kBins - (t + 1) * BPT, kBins - t * BPT), highest first,
        // and leaves them empty for the next pass.
        uint32_t c[BPT], mine = 0;
#pragma unroll
        for (int b = 0; b < BPT; ++b) {
            const int at = (BPT - 1 - b) * T + (T - 1 - tid);
            c[b] = sm.hist[at];
            sm.hist[at] = 0;
            mine += c[b];
        }
        uint32_t incl = mine;
#pragma unroll
        for (int off = 1; off < 64; off <<= 1) {
            const uint32_t o = __shfl_up(incl, off, 64);
            if (lane >= off) incl += o;
        }
        if constexpr (W > 1) {
            if (lane == 63) sm.wave_a[wave] = incl;
            __syncthreads();
#pragma unroll
            for (int w = 0; w < W; ++w) incl += w < wave ? sm.wave_a[w] : 0u;
        }
        uint32_t above = incl - mine;          // keys with a larger digit
        if (above < krem && incl >= krem) {
#pragma unroll
            for (int b = 0; b < BPT; ++b) {
                if (above < krem && above + c[b] >= krem) {
                    sm.digit = static_cast<uint32_t>(Lds::kBins - 1 - tid * BPT - b);
                    sm.above = above;
                    sm.count = c[b];
                }
                above += c[b];
            }
        }
        __syncthreads();
        prefix |= sm.digit << shift;
        mask |= dmask << shift;
        krem -= sm.above;
        whole = sm.count == krem;
    }
    // Take every key with a larger prefix and, of those equal to it, all
    // (whole) or the first krem in index order.
    uint32_t n_gt = 0, n_eq = 0;
    const auto over = [&](uint32_t v, bool in) { return in && (whole ? v >= prefix : v > prefix); };
    each([&](int, uint32_t v, bool in) {
        n_gt += static_cast<uint32_t>(__popcll(__ballot(over(v, in))));
        n_eq += static_cast<uint32_t>(__popcll(__ballot(in && !whole && v == prefix)));
    });
    uint32_t gt = 0, eq = 0;                   // of the wavefronts before
    if constexpr (W > 1) {
        if (lane == 0) {
            sm.wave_a[wave] = n_gt;
            sm.wave_b[wave] = n_eq;
        }
        __syncthreads();
#pragma unroll
        for (int w = 0; w < W; ++w) {
            gt += w < wave ? sm.wave_a[w] : 0u;
            eq += w < wave ? sm.wave_b[w] : 0u;
        }
    }
    const unsigned long long below = (1ull << lane) - 1ull;
    each([&](int s, uint32_t v, bool in) {
        const bool g = over(v, in), e = in && !whole && v == prefix;
        const unsigned long long mg = __ballot(g), me = __ballot(e);
        const uint32_t eq_rank = eq + static_cast<uint32_t>(__popcll(me & below));
        const uint32_t pos = gt + static_cast<uint32_t>(__popcll(mg & below)) + min(eq_rank, krem);
        if ((g || (e && eq_rank < krem)) && pos < static_cast<uint32_t>(k)) {
            const int i = KPT > 0 ? i0 + s * 64 : static_cast<int>(static_cast<uint32_t>(i0) + static_cast<uint32_t>(s) * 64);
            if (orow != nullptr) orow[pos] = i;
            if (s_sel != nullptr) s_sel[pos] = i;
        }
        gt += static_cast<uint32_t>(__popcll(mg));
        eq += static_cast<uint32_t>(__popcll(me));
    });
}

// One workgroup per (layer, chunk), of T lanes and KPT slots for the call's longest
// chunk (launch_topk). A shorter chunk is done by the first lanes alone, with the
// fewest that hold it in registers, and the other wavefronts end at once (a
// barrier counts the live ones): the short chunks beside a long one would each
// pay for the barriers of 16 wavefronts. One chunk of 3000 tokens and 40 of 200 in
// 32 layers 28.5 -> 15.4 us, one of 9000 and 40 of 500 51.6 -> 24.9 us, calls of
// even chunks unchanged (MI355X).
template <int T, int KPT>
__global__ __launch_bounds__(T) void topk_kernel(const float* __restrict__ keys, int64_t stride, DescArg d,
                                                 int n_chunks, int32_t* __restrict__ out, int kmax, int l0) {
    const DescPtr<SelChunk> chunks = desc_at<SelChunk>(d, 0);
    static_assert(T <= 256 || sizeof(TopkLds<T>) >= sizeof(TopkLds<256>), "the short forms' LDS fits");
    __shared__ __align__(16) uint8_t s_mem[sizeof(TopkLds<T>)];
    const int l = static_cast<int>(blockIdx.y) + l0;
    const int ci = static_cast<int>(blockIdx.x);
    const SelChunk c = desc_load(chunks + ci);
    const int n = c.n_tokens;
    const int k = min(max(c.k, 0), n);
    int32_t* __restrict__ orow = out + (static_cast<int64_t>(l) * n_chunks + ci) * kmax;
    const int tid = static_cast<int>(threadIdx.x);
    const float* krow = keys + static_cast<int64_t>(l) * stride + c.row_offset;
    const auto key_at = [&](int i) -> uint32_t { return order_key(krow[i]); };
    const auto form = [&](auto lanes, auto slots) {
        constexpr int N = decltype(lanes)::value;
        if (tid >= N) return;
        for (int i = k + tid; i < kmax; i += N) orow[i] = -1;
        if (k == 0) return;
        chunk_topk<N, decltype(slots)::value>(key_at, n, k, orow, nullptr, *reinterpret_cast<TopkLds<N>*>(s_mem));
    };
    using std::integral_constant;
    if (T > 64 && n <= kTopkWave) form(integral_constant<int, 64>(), integral_constant<int, kTopkWave / 64>());
    else if (T > 256 && n <= kTopkGroup) form(integral_constant<int, 256>(), integral_constant<int, kTopkGroup / 256>());
    else form(integral_constant<int, T>(), integral_constant<int, KPT>());
}

template <int VW>
__global__ __launch_bounds__(kThreads) void merge_kernel(
    DescArg d, int layer_off, KVGeom g, int es, const int32_t* __restrict__ bt,
    const uint8_t* __restrict__ k_new, const uint8_t* __restrict__ v_new, int64_t T,
    int n_chunks, const int32_t* __restrict__ sel, int kmax, int c0, int l0) {
    const DescPtr<SelChunk> chunks = desc_at<SelChunk>(d, 0);
    const DescPtr<uint8_t*> layers = desc_at<uint8_t*>(d, layer_off);
    using V = typename std::conditional<VW == 16, u32x4, uint8_t>::type;
    const int l = static_cast<int>(blockIdx.z) + l0;
    const int ci = static_cast<int>(blockIdx.y) + c0;
    const SelChunk c = desc_load(chunks + ci);
    const int q0 = static_cast<int>(blockIdx.x) * kMergeTok;
    const int32_t* srow = sel + (static_cast<int64_t>(l) * n_chunks + ci) * kmax;
    uint8_t* __restrict__ base = layers[l];
    const int upr = g.D * es / VW;               // units per head row
    const int per_tok = 2 * g.H * upr;           // K and V rows
    const int items = kMergeTok * per_tok;
    const int64_t rowbytes = static_cast<int64_t>(g.H) * g.D * es;
    for (int it = threadIdx.x; it < items; it += kThreads) {
        const int t = it / per_tok;
        int rem = it - t * per_tok;
        const int kv = rem / (g.H * upr);
        rem -= kv * g.H * upr;
        const int h = rem / upr;
        const int u = rem - h * upr;
        const int q = q0 + t;
        if (q >= kmax || q >= c.k) continue;
        const int j = srow[q];
        if (j < 0 || j >= c.n_tokens) continue;
        if (kv == 1 && g.v_off < 0) continue;
        const int p = c.tok0 + j;
        const int blk = bt[c.bt_offset + p / g.PS];
        if (blk <= 0 || blk >= g.num_blocks) continue;
        const int64_t dst_el = static_cast<int64_t>(blk) * g.sb + static_cast<int64_t>(p % g.PS) * g.ss +
                               static_cast<int64_t>(h) * g.sh + (kv ? g.v_off : 0);
        const uint8_t* src = (kv ? v_new : k_new) +
                             (static_cast<int64_t>(l) * T + c.row_offset + j) * rowbytes +
                             static_cast<int64_t>(h) * g.D * es;
        *reinterpret_cast<V*>(base + dst_el * es + static_cast<int64_t>(u) * VW) =
            *reinterpret_cast<const V*>(src + static_cast<int64_t>(u) * VW);
    }
}

// Row merge for 16-byte-aligned rows. A workgroup writes `tpb` consecutive
// selected slots of one (layer, chunk): its first lanes resolve each slot's
// recomputed row and cache row (selection index, block table) into LDS; then
// its lanes walk the 16-byte source units of those K and V rows, up to
// kMergeUnits per lane, with every load issued before the first store. A lane
// holds only its loaded values and recomputes the addresses from LDS at store
// time (holding 16 destination pointers per lane took 112 VGPRs, capping the
// kernel at 4 waves per SIMD).
// MODE 0 copies bytes (rows and cache share their element type). MODE kBF16 /
// kF16 + 1 quantises bf16 / fp16 rows into an e4m3 cache as vLLM's fp8 cache
// write does: code = saturating RTNE of float32(x) / scale[l, h], the
// division correctly rounded (quant_quotient: one reciprocal per 16-byte unit
// and two FMAs per element instead of a division per element).
constexpr int kMergeUnits = 8;
// 256 lanes x 8 units in flight, nontemporal loads (and stores of copied
// rows): 2% faster for the copy and 4-5% for the quantising merge than plain
// accesses, in alternating processes. A same-process sweep at config 3 put 128
// or 512 lanes, 1 to 16 units, a precomputed slot table, two groups per
// workgroup and one-wavefront-per-token forms within +-2% of this. The
// layer-minor block order (LayerMinor) then took the config-3 merge from
// 704-749 to 622-689 us in same-process A/Bs, about the rate of a page
// scatter of the same bytes onto the same cache layers.
constexpr int kMergeThreads = 256;
constexpr int kMergeMaxTok = 64;
constexpr int kMergeCopy = 0;
constexpr int kMergeFromBF16 = kBF16 + 1;
constexpr int kMergeFromF16 = kF16 + 1;

// Where selected token j of chunk c in layer l is merged: *src, the byte
// offset of its recomputed rows (-1: skip the token: an index outside the
// chunk, or a block id of 0 or outside the cache), and *dst, the byte offset
// of its K row in the layer.
__device__ __forceinline__ void merge_slot(int j, const SelChunk& c, int l, const KVGeom& g, int64_t T,
                                           int64_t row_bytes, int ces, const int32_t* __restrict__ bt,
                                           int64_t* src, int64_t* dst) {
    *src = -1;
    *dst = 0;
    if (j < 0 || j >= c.n_tokens) return;
    const int p = c.tok0 + j;
    const int blk = bt[c.bt_offset + p / g.PS];
    if (blk <= 0 || blk >= g.num_blocks) return;
    *src = (static_cast<int64_t>(l) * T + c.row_offset + j) * row_bytes;
    *dst = (static_cast<int64_t>(blk) * g.sb + static_cast<int64_t>(p % g.PS) * g.ss) * ces;
}

// Copies (or quantises) the K and V rows of n_tok tokens whose slots
// s_src / s_dst (LDS) hold, walking their 16-byte source units in rounds of
// kMergeThreads x kMergeUnits: every load of a round is issued before its
// first store. Shared by merge_rows_kernel (one round per workgroup) and the
// fused selection kernel (all of a chunk's selected tokens).
template <int MODE, bool DENSE>
__device__ __forceinline__ void merge_units(
    int n_tok, const int64_t* s_src, const int64_t* s_dst, int l, uint8_t* __restrict__ base, const KVGeom& g,
    int ces, const uint8_t* __restrict__ k_new, const uint8_t* __restrict__ v_new, int units,
    FastDiv d_tok_units, FastDiv d_upr, const float* __restrict__ k_scales, const float* __restrict__ v_scales) {
    const int tid = static_cast<int>(threadIdx.x);
    const int tok_units = static_cast<int>(d_tok_units.d);   // units per token: K row, then V row
    const int total = n_tok * tok_units;
    const int upr = static_cast<int>(d_upr.d);
    for (int f0 = 0; f0 < total; f0 += kMergeThreads * kMergeUnits) {
        // Every slot loads (lanes past the end reload the last unit, skipped
        // rows read the first unit of k_new) so that the values stay plain
        // registers; only the stores are conditional.
        u32x4 v[kMergeUnits];
#pragma unroll
        for (int s = 0; s < kMergeUnits; ++s) {
            const int f = min(f0 + tid + s * kMergeThreads, total - 1);
            const int t = static_cast<int>(d_tok_units.div(static_cast<uint32_t>(f)));
            const int r = f - t * tok_units;
            const int kv = r >= units ? 1 : 0;
            const int64_t src = s_src[t];
            const uint8_t* p = src >= 0 ? (kv ? v_new : k_new) + src + static_cast<int64_t>(r - kv * units) * 16 : k_new;
            v[s] = __builtin_nontemporal_load(reinterpret_cast<const u32x4*>(p));
        }
        // An opaque copy of the thread index: the compiler would otherwise keep
        // every slot's decoded address alive across the loads (240 VGPRs).
        int tid_s = f0 + tid;
        asm volatile("" : "+v"(tid_s));
#pragma unroll
        for (int s = 0; s < kMergeUnits; ++s) {
            const int f = tid_s + s * kMergeThreads;
            if (f >= total) continue;
            const int t = static_cast<int>(d_tok_units.div(static_cast<uint32_t>(f)));
            const int r = f - t * tok_units;
            const int kv = r >= units ? 1 : 0;
            if (s_src[t] < 0) continue;
            const int u = r - kv * units;
            // DENSE: the head rows of a token are contiguous (sh == D), so unit u
            // of the token row lands at u * (cache bytes per unit)
            const int h = DENSE && MODE == kMergeCopy ? 0 : static_cast<int>(d_upr.div(static_cast<uint32_t>(u)));
            const int un = DENSE ? u : u - h * upr;
            uint8_t* dst = base + s_dst[t] + (static_cast<int64_t>(DENSE ? 0 : h) * g.sh + (kv ? g.v_off : 0)) * ces;
            if constexpr (MODE == kMergeCopy) {
                __builtin_nontemporal_store(v[s], reinterpret_cast<u32x4*>(dst + static_cast<int64_t>(un) * 16));
            } else {
                const QuantDiv qd = quant_div((kv ? v_scales : k_scales)[l * g.H + h]);
                float x[8];
#pragma unroll
                for (int w = 0; w < 4; ++w) Elem<MODE - 1>::unpack_word(v[s][w], x + 2 * w);
                if (qd.fast) {
#pragma unroll
                    for (int i = 0; i < 8; ++i) x[i] = quant_quotient_fast(qd, x[i]);
                } else {
#pragma unroll
                    for (int i = 0; i < 8; ++i) x[i] = x[i] / qd.s;
                }
                u32x2 o;
                o[0] = f32x4_to_e4m3_hw(x);
                o[1] = f32x4_to_e4m3_hw(x + 4);
                *reinterpret_cast<u32x2*>(dst + static_cast<int64_t>(un) * 8) = o;
            }
        }
    }
}

// A chunk's row batches begin at its tile_begin: the chunks' counts differ (the
// recompute policy gives a prompt's last document most of its budget), and a
// grid of the largest count times the chunks left most workgroups idle (MI355X,
// counts of 2% to 90% of 8 chunks of 3000 tokens, 22 layers of 4 x 96: 80 -> 60 us).
// Chunks of d_each.d batches each (0: uneven) are found by a division: the search's
// chain of loads cost 0.5 us in a short launch and 8 us in one of 400 chunks (32
// layers of 2 x 64, 10 rows each: 43.6 us, 36.0 by division).
template <int MODE, bool DENSE>
__global__ __launch_bounds__(kMergeThreads) void merge_rows_kernel(
    DescArg d, int chunk_off, int layer_off, KVGeom g, int ces, const int32_t* __restrict__ bt,
    const uint8_t* __restrict__ k_new, const uint8_t* __restrict__ v_new, int64_t T,
    int n_chunks, const int32_t* __restrict__ sel, int kmax, int tpb, int units,
    FastDiv d_tok_units, FastDiv d_upr, FastDiv d_each, const float* __restrict__ k_scales,
    const float* __restrict__ v_scales, LayerMinor lm) {
    __shared__ int64_t s_src[kMergeMaxTok];   // byte offset of the token's recomputed rows (-1: skip)
    __shared__ int64_t s_dst[kMergeMaxTok];   // byte offset of the token's K row in the layer
    const DescPtr<SelChunk> chunks = desc_at<SelChunk>(d, chunk_off);
    const DescPtr<uint8_t*> layers = desc_at<uint8_t*>(d, layer_off);
    // work item = (chunk, row batch), the batches of a chunk consecutive
    int l;
    int64_t item;
    lm.at(l, item);
    const int ci = d_each.d ? static_cast<int>(d_each.div(static_cast<uint32_t>(item)))
                            : find_by_tile(chunks, n_chunks, static_cast<int>(item));
    const SelChunk c = desc_load(chunks + ci);
    const int bx = static_cast<int>(item) - c.tile_begin;
    const int tid = static_cast<int>(threadIdx.x);
    const int ses = MODE == kMergeCopy ? ces : 2;                    // source element size
    const int64_t row_bytes = static_cast<int64_t>(g.H) * g.D * ses;
    if (tid < tpb) {
        const int q = bx * tpb + tid;
        const int j = q < min(kmax, c.k) ? sel[(static_cast<int64_t>(l) * n_chunks + ci) * kmax + q] : -1;
        merge_slot(j, c, l, g, T, row_bytes, ces, bt, &s_src[tid], &s_dst[tid]);
    }
    __syncthreads();
    merge_units<MODE, DENSE>(tpb, s_src, s_dst, l, layers[l], g, ces, k_new, v_new, units, d_tok_units, d_upr,
                             k_scales, v_scales);
}

// The whole selection of one (layer, chunk) in one workgroup: the chunk's
// deviation keys (group_keys, the fixed order of deviation_kernel; WITH_KEYS
// false: read from `keys` instead), its top-k (chunk_topk), then the slots of all
// its selected tokens (merge_slot) and the merge of their rows (merge_units).
// Keys and indices are written out as kv_deviation and topk_per_chunk write
// them. Dynamic LDS (select_merge_lds): n_max order keys (WITH_KEYS), kmax
// selected indices, kmax source and kmax destination offsets.
constexpr int kFusedSlots = 8;                          // key slots per wavefront
constexpr int kFusedMaxTokens = kThreads * kFusedSlots;
template <int CK, int NK, int MODE, bool DENSE, bool WITH_KEYS>
__global__ __launch_bounds__(kThreads) void select_merge_kernel(
    DescArg d, int layer_off, KVGeom g, int ces, const int32_t* __restrict__ bt,
    const uint8_t* __restrict__ k_new, const uint8_t* __restrict__ v_new, int64_t T, int n_chunks,
    const float* __restrict__ dev_scales, float* __restrict__ keys, int32_t* __restrict__ sel, int kmax,
    int n_max, int units, FastDiv d_tok_units, FastDiv d_upr, const float* __restrict__ k_scales,
    const float* __restrict__ v_scales, LayerMinor lm) {
    extern __shared__ __align__(16) uint32_t s_dyn[];   // keys, indices, then 8-byte offsets
    __shared__ TopkLds<kThreads> sm;
    uint32_t* s_keys = s_dyn;
    int32_t* s_sel = reinterpret_cast<int32_t*>(s_dyn + n_max);
    int64_t* s_src = reinterpret_cast<int64_t*>(s_dyn + ((n_max + kmax + 1) & ~1));
    int64_t* s_dst = s_src + kmax;
    const DescPtr<SelChunk> chunks = desc_at<SelChunk>(d, 0);
    const DescPtr<uint8_t*> layers = desc_at<uint8_t*>(d, layer_off);
    int l;
    int64_t item;
    lm.at(l, item);
    const int ci = static_cast<int>(item);
    const SelChunk c = desc_load(chunks + ci);
    const int tid = static_cast<int>(threadIdx.x);
    const int n = c.n_tokens;
    const int k = min(max(c.k, 0), n);
    uint8_t* __restrict__ base = layers[l];
    float* krow = keys + static_cast<int64_t>(l) * T + c.row_offset;
    if constexpr (WITH_KEYS) {
        constexpr int TPG = dev_tok_per_group<CK>();
        const int lane = tid & 63;
        const int wave = tid >> 6;
        const float* ksc = dev_scales ? dev_scales + static_cast<int64_t>(l) * g.H : nullptr;
        for (int j0 = wave * TPG; j0 < n; j0 += kWaves * TPG) {
            float key[TPG];
            group_keys<CK, NK, TPG, 64>(c, j0, lane, g, base, bt, k_new, T, l, ksc, key);
#pragma unroll
            for (int i = 0; i < TPG; ++i) {
                const int j = j0 + i;
                if (lane == i && j < n) {
                    krow[j] = key[i];
                    s_keys[j] = order_key(key[i]);
                }
            }
        }
        __syncthreads();
    }
    int32_t* __restrict__ orow = sel + (static_cast<int64_t>(l) * n_chunks + ci) * kmax;
    for (int i = k + tid; i < kmax; i += kThreads) orow[i] = -1;
    if (k == 0) return;
    chunk_topk<kThreads, kFusedSlots>(
        [&](int i) -> uint32_t { return WITH_KEYS ? s_keys[i] : order_key(krow[i]); }, n, k, orow, s_sel, sm);
    __syncthreads();
    const int ses = MODE == kMergeCopy ? ces : 2;
    const int64_t row_bytes = static_cast<int64_t>(g.H) * g.D * ses;
    for (int q = tid; q < k; q += kThreads) merge_slot(s_sel[q], c, l, g, T, row_bytes, ces, bt, &s_src[q], &s_dst[q]);
    __syncthreads();
    merge_units<MODE, DENSE>(k, s_src, s_dst, l, base, g, ces, k_new, v_new, units, d_tok_units, d_upr,
                             k_scales, v_scales);
}

}  // namespace

int deviation_tile_tokens(int cache_kind, const KVGeom& g) {
    const int group = dev_group(g.H * g.D / 8);
    return kThreads / group * (cache_kind == kE4M3 ? dev_tok_per_group<kE4M3>() : dev_tok_per_group<kBF16>());
}

void launch_deviation(const DescArg& d, int layer_off, int n_layers, const KVGeom& g, int cache_kind,
                      const int32_t* block_table, const uint8_t* k_new, int new_kind,
                      int64_t T, int n_chunks, int n_tiles,
                      const float* k_scales, float* keys, hipStream_t stream) {
    const int group = dev_group(g.H * g.D / 8);
    for (int l0 = 0; l0 < n_layers; l0 += kMaxGridYZ) {
        const dim3 grid(static_cast<unsigned>(n_tiles), static_cast<unsigned>(std::min(kMaxGridYZ, n_layers - l0)));
#define DARIC_DV(C, N, G) DARIC_LAUNCH((deviation_kernel<C, N, G>), grid, kThreads, 0, stream, d, layer_off, g, block_table, k_new, T, n_chunks, k_scales, keys, l0)
#define DARIC_DVG(C, N) do { if (group == 64) DARIC_DV(C, N, 64); else if (group == 32) DARIC_DV(C, N, 32); \
                             else if (group == 16) DARIC_DV(C, N, 16); else DARIC_DV(C, N, 8); } while (0)
        if (new_kind == kBF16) {
            if (cache_kind == kBF16) DARIC_DVG(kBF16, kBF16);
            else if (cache_kind == kF16) DARIC_DVG(kF16, kBF16);
            else DARIC_DVG(kE4M3, kBF16);
        } else {
            if (cache_kind == kBF16) DARIC_DVG(kBF16, kF16);
            else if (cache_kind == kF16) DARIC_DVG(kF16, kF16);
            else DARIC_DVG(kE4M3, kF16);
        }
#undef DARIC_DVG
#undef DARIC_DV
        check_launch("kv_deviation");
    }
}

// The fewest lanes whose registers hold the longest chunk's keys in a few slots:
// more wavefronts only add to the barriers. A CU holds one workgroup of 1024
// lanes, so beyond one per CU those of up to 8192 tokens take 512 lanes: 512
// chunks of 3000 tokens 17.4 -> 14.5 us, 3200 of 2100 tokens 84.9 -> 47.6 (256
// lanes over keys in LDS: 59.7), 3200 of 8000 168 -> 109; at 256 chunks of 8000
// they would take 19.4 instead of 14.9. Chunks read from memory again in each pass
// need fewer registers and fit twice; from 1024 of them on 512 lanes each: 1280 of
// 40000 tokens 475 -> 373 us, 3200 of 40000 1248 -> 940 (256 lanes and four passes:
// 1136), 4096 of 33000 1296 -> 927 (1099), where 1024 of 100000 would take 1079
// instead of 990 (MI355X).
void launch_topk(const float* keys, int n_layers, int64_t T, const DescArg& d,
                 int n_chunks, int max_tokens, int32_t* out_idx, int kmax, hipStream_t stream) {
    const int64_t groups = static_cast<int64_t>(n_chunks) * n_layers;
    for (int l0 = 0; l0 < n_layers; l0 += kMaxGridYZ) {
        const dim3 grid(static_cast<unsigned>(n_chunks), static_cast<unsigned>(std::min(kMaxGridYZ, n_layers - l0)));
#define DARIC_TK(TH, KPT) DARIC_LAUNCH((topk_kernel<TH, KPT>), grid, TH, 0, stream, keys, T, d, n_chunks, out_idx, kmax, l0)
        if (max_tokens <= kTopkWave) DARIC_TK(64, kTopkWave / 64);
        else if (max_tokens <= kTopkGroup) DARIC_TK(256, kTopkGroup / 256);
        else if (max_tokens <= 8192 && groups > 256) DARIC_TK(512, 16);
        else if (max_tokens <= 8192) DARIC_TK(1024, 8);
        else if (max_tokens <= 32768) DARIC_TK(1024, 32);
        else if (groups > 1024) DARIC_TK(512, 0);
        else DARIC_TK(1024, 0);
#undef DARIC_TK
        check_launch("topk_per_chunk");
    }
}

bool merge_fits_rows(const KVGeom& g, int elem_size, bool quant) {
    const int ses = quant ? 2 : elem_size;
    if ((g.D * ses) % 16 != 0) return false;
    const int64_t dst_unit = quant ? 8 : 16;     // cache bytes per 16-byte source unit
    if ((g.sb * elem_size) % dst_unit || (g.ss * elem_size) % dst_unit || (g.sh * elem_size) % dst_unit ||
        (g.v_off >= 0 && (g.v_off * elem_size) % dst_unit))
        return false;
    const int64_t tok_units = static_cast<int64_t>(g.v_off >= 0 ? 2 : 1) * g.H * (g.D * ses / 16);
    return tok_units <= static_cast<int64_t>(kMergeThreads) * kMergeUnits;
}

int64_t merge_max_row_bytes() { return static_cast<int64_t>(kMergeThreads) * kMergeUnits * 16; }

int merge_rows_per_block(const KVGeom& g, int elem_size, bool quant) {
    if (!merge_fits_rows(g, elem_size, quant)) return 0;
    const int tok_units = (g.v_off >= 0 ? 2 : 1) * g.H * (g.D * (quant ? 2 : elem_size) / 16);
    return std::min(kMergeMaxTok, std::max(1, kMergeThreads * kMergeUnits / tok_units));
}

void launch_merge(const DescArg& d, int chunk_off, int layer_off, int n_layers, const KVGeom& g, int elem_size,
                  const int32_t* block_table, const uint8_t* k_new, const uint8_t* v_new,
                  int64_t T, int n_chunks, const MergeBatches& batches, const int32_t* sel_idx, int kmax, int quant_from,
                  const float* k_scales, const float* v_scales, hipStream_t stream) {
    const bool quant = quant_from >= 0;
    if (merge_fits_rows(g, elem_size, quant)) {
        // one workgroup per (layer, chunk, batch of tpb selected rows), layer-minor
        const int ses = quant ? 2 : elem_size;
        const int upr = g.D * ses / 16;                              // source units per head row
        const int units = g.H * upr;                                 // per K (or V) token row
        const int tok_units = (g.v_off >= 0 ? 2 : 1) * units;
        const int tpb = merge_rows_per_block(g, elem_size, quant);
        const FastDiv dtu(static_cast<uint32_t>(tok_units)), dupr(static_cast<uint32_t>(upr));
        FastDiv deach(static_cast<uint32_t>(std::max<int64_t>(batches.each, 1)));
        if (batches.each == 0) deach.d = 0;
        const bool dense = g.sh == g.D;
        for_layer_minor(n_layers, batches.n, [&](const LayerMinor& lm, unsigned blocks) {
#define DARIC_MR(M, DN) DARIC_LAUNCH((merge_rows_kernel<M, DN>), blocks, kMergeThreads, 0, stream, d, chunk_off, \
                                     layer_off, g, elem_size, block_table, k_new, v_new, T, n_chunks, sel_idx, kmax, \
                                     tpb, units, dtu, dupr, deach, k_scales, v_scales, lm)
            if (!quant) { if (dense) DARIC_MR(kMergeCopy, true); else DARIC_MR(kMergeCopy, false); }
            else if (quant_from == kBF16) { if (dense) DARIC_MR(kMergeFromBF16, true); else DARIC_MR(kMergeFromBF16, false); }
            else { if (dense) DARIC_MR(kMergeFromF16, true); else DARIC_MR(kMergeFromF16, false); }
#undef DARIC_MR
            check_launch("merge_rows");
        });
        return;
    }
    // grid.y (chunks) and grid.z (layers) are cut into slices of at most 65535
    for (int l0 = 0; l0 < n_layers; l0 += kMaxGridYZ) {
        const int nl = std::min(kMaxGridYZ, n_layers - l0);
        for (int c0 = 0; c0 < n_chunks; c0 += kMaxGridYZ) {
            const int nc = std::min(kMaxGridYZ, n_chunks - c0);
            const dim3 grid(static_cast<unsigned>((kmax + kMergeTok - 1) / kMergeTok), static_cast<unsigned>(nc),
                            static_cast<unsigned>(nl));
            const bool vec = (g.D * elem_size) % 16 == 0 && (g.sb * elem_size) % 16 == 0 &&
                             (g.ss * elem_size) % 16 == 0 && (g.sh * elem_size) % 16 == 0 &&
                             (g.v_off < 0 || (g.v_off * elem_size) % 16 == 0);
            if (vec)
                DARIC_LAUNCH((merge_kernel<16>), grid, kThreads, 0, stream, d, layer_off, g, elem_size, block_table,
                             k_new, v_new, T, n_chunks, sel_idx, kmax, c0, l0);
            else
                DARIC_LAUNCH((merge_kernel<1>), grid, kThreads, 0, stream, d, layer_off, g, elem_size, block_table,
                             k_new, v_new, T, n_chunks, sel_idx, kmax, c0, l0);
            check_launch("merge_rows");
        }
    }
}

// Dynamic LDS of the fused kernel: keys (one pass only) and indices (4 bytes
// each), then the source and destination offsets of the selected tokens (8 bytes
// each).
size_t select_merge_lds(int64_t max_tokens, int64_t kmax, bool one_pass) {
    const int64_t n = one_pass ? std::max<int64_t>(max_tokens, 1) : 0, k = std::max<int64_t>(kmax, 1);
    return static_cast<size_t>(((n + k + 1) & ~int64_t(1)) * 4 + 2 * k * 8);
}

constexpr size_t kSelectMergeMaxLds = 40 * 1024;   // beside the 8 KiB of the top-k
// A fused workgroup merges its chunk's selected rows alone, in rounds of
// kMergeThreads x kMergeUnits 16-byte units. Up to this many rounds per chunk
// the fused top-k + merge is as fast as topk_kernel + merge_rows_kernel or faster;
// beyond it the merge kernel's spread over (chunk, row batch) wins. MI355X, whole
// selections, fused against three launches: 96 chunks of 512 tokens in 32 layers of
// 8 x 128 bf16 1318 and 1320 us at 10 rounds, 1412 and 1414 at 12, 1961 and 1942 at
// 26; 6 of 1500 220.3 and 219.0 at 10, 240 and 234 at 16; 64 of 1000 in 80 layers of
// 1 x 128 495 and 509 at 1, 1173 and 1192 at 11; 16 of 512 in 80 e4m3 layers 382 and
// 388 at 3, 517 and 504 at 12, 571 and 549 at 16.
constexpr int64_t kFusedMaxRounds = 12;

bool select_merge_fits(const KVGeom& g, int elem_size, bool quant, int64_t max_tokens, int64_t kmax,
                       bool one_pass) {
    if (!merge_fits_rows(g, elem_size, quant) || max_tokens > kFusedMaxTokens ||
        select_merge_lds(max_tokens, kmax, one_pass) > kSelectMergeMaxLds)
        return false;
    const int ses = quant ? 2 : elem_size;
    const int64_t tok_units = static_cast<int64_t>(g.v_off >= 0 ? 2 : 1) * g.H * (g.D * ses / 16);
    const int64_t rounds = (kmax * tok_units + kMergeThreads * kMergeUnits - 1) / (kMergeThreads * kMergeUnits);
    return one_pass || rounds <= kFusedMaxRounds;
}

void launch_select_merge(const DescArg& d, int layer_off, int n_layers, const KVGeom& g, int cache_kind,
                         int elem_size, const int32_t* block_table, const uint8_t* k_new, int new_kind,
                         const uint8_t* v_new, int64_t T, int n_chunks, int max_tokens, bool with_keys,
                         float* keys, int32_t* sel_idx, int kmax, bool quant, const float* k_scales,
                         const float* v_scales, hipStream_t stream) {
    static_assert(kThreads == kMergeThreads, "the fused kernel's merge batches use every lane");
    const int ses = quant ? 2 : elem_size;
    const int upr = g.D * ses / 16;
    const int units = g.H * upr;
    const int tok_units = (g.v_off >= 0 ? 2 : 1) * units;
    const FastDiv dtu(static_cast<uint32_t>(tok_units)), dupr(static_cast<uint32_t>(upr));
    const bool dense = g.sh == g.D;
    const int n_max = with_keys ? std::max(max_tokens, 1) : 0;
    const size_t lds = select_merge_lds(max_tokens, kmax, with_keys);
    // deviation scales: per-head K scales of an fp8 cache (the quantising
    // merge's K scales are the same ones)
    const float* dev_scales = cache_kind == kE4M3 ? k_scales : nullptr;
    // one workgroup per (layer, chunk), layer-minor
    for_layer_minor(n_layers, n_chunks, [&](const LayerMinor& lm, unsigned blocks) {
#define DARIC_SM(C, N, M, DN, WK) DARIC_LAUNCH((select_merge_kernel<C, N, M, DN, WK>), blocks, kThreads, lds, stream, \
                                           d, layer_off, g, elem_size, block_table, k_new, v_new, T, n_chunks, \
                                           dev_scales, keys, sel_idx, kmax, n_max, units, dtu, dupr, \
                                           k_scales, v_scales, lm)
#define DARIC_SM_K(C, N, M, DN) do { if (with_keys) DARIC_SM(C, N, M, DN, true); else DARIC_SM(C, N, M, DN, false); } while (0)
#define DARIC_SM_D(C, N, M) do { if (dense) DARIC_SM_K(C, N, M, true); else DARIC_SM_K(C, N, M, false); } while (0)
        if (cache_kind == kBF16) {
            if (new_kind == kBF16) DARIC_SM_D(kBF16, kBF16, kMergeCopy);
            else DARIC_SM_D(kBF16, kF16, kMergeCopy);
        } else if (cache_kind == kF16) {
            if (new_kind == kBF16) DARIC_SM_D(kF16, kBF16, kMergeCopy);
            else DARIC_SM_D(kF16, kF16, kMergeCopy);
        } else if (quant) {
            if (new_kind == kBF16) DARIC_SM_D(kE4M3, kBF16, kMergeFromBF16);
            else DARIC_SM_D(kE4M3, kF16, kMergeFromF16);
        } else {
            throw Error(DARIC_ERR_INVALID, "select_merge on an fp8 cache merges bf16/fp16 rows with scales");
        }
#undef DARIC_SM_D
#undef DARIC_SM_K
#undef DARIC_SM
        check_launch("select_merge");
    });
}

}  // namespace daric
