// Paged-KV gather / scatter and the fused scatter + K re-rotation (gfx950).
//
// Work decomposition: a job is one (layer, chunk) pair; a tile is one page
// span of one prefix index (the K or V half of a page for vLLM's
// [2, blocks, PS, H, D] layout: 32 KiB at Llama-3-8B shape). A 256-lane
// workgroup streams a tile, or a part of one, with 16-byte accesses, 8 in
// flight per lane, loads before stores. Staging-side loads and cache-side
// stores are nontemporal: every byte is touched once.
//
// Block order (measured on MI355X at the Llama-3-8B shape): both directions
// cut each tile into parts of 8 KiB (page_part_bytes). In large calls the scatter
// direction and the fused scatter + rotation deal runs of 128 KiB of each job to
// the XCDs (JobRuns); the gather direction runs job by job, tile by tile (JobRows),
// which sustained ~6.3 TB/s (256 jobs of 64 pages) and 5.8-6.0 TB/s (32 of 4096),
// against 5.5-5.6 TB/s for whole-tile workgroups and job-minor orders.
//
// Pages whose block id is 0 (vLLM's null block) are skipped, as the
// reference's kernels skip them (csrc/cache_ops/kernels.cu:26,39,69,79,104,117);
// ids outside [0, num_pages) are skipped as well instead of faulting.
#include <hip/hip_runtime.h>

#include <algorithm>

#include "elem.h"
#include "jobs.h"
#include "kernels.h"
#include "launch.h"
#include "rotate_rows.h"

namespace daric {

constexpr int kThreads = 256;
constexpr int kUnroll = 8;
constexpr int kMaxHalfRot = 256;  // rotary_dim / 2 limit of the LDS cos/sin table

template <int VW> struct VecOf;
template <> struct VecOf<16> { using T = u32x4; };
template <> struct VecOf<4> { using T = uint32_t; };
template <> struct VecOf<1> { using T = uint8_t; };

template <typename T>
__device__ __forceinline__ T ld_nt(const T* p) { return __builtin_nontemporal_load(p); }
template <typename T>
__device__ __forceinline__ void st_nt(T* p, T v) { __builtin_nontemporal_store(v, p); }

// Copies n_units units of VW bytes from src to dst (n_units < 2^31) by the LANES
// lanes of a workgroup.
template <int VW, int LANES = kThreads>
__device__ __forceinline__ void copy_units(const uint8_t* __restrict__ src,
                                           uint8_t* __restrict__ dst, int n_units) {
    using T = typename VecOf<VW>::T;
    const T* s = reinterpret_cast<const T*>(src);
    T* d = reinterpret_cast<T*>(dst);
    for (int base = 0; base < n_units; base += LANES * kUnroll) {
        T v[kUnroll];
#pragma unroll
        for (int u = 0; u < kUnroll; ++u) {
            const int i = base + u * LANES + static_cast<int>(threadIdx.x);
            if (i < n_units) v[u] = ld_nt(s + i);
        }
#pragma unroll
        for (int u = 0; u < kUnroll; ++u) {
            const int i = base + u * LANES + static_cast<int>(threadIdx.x);
            if (i < n_units) st_nt(d + i, v[u]);
        }
    }
}

// Resolves tile t of job j. Returns false when the tile is beyond the job or
// its page is skipped.
__device__ __forceinline__ bool resolve_tile(const CopyJob& j, int t, int& p, int& s,
                                             uint8_t*& cache, uint8_t*& stage) {
    const int n_sel = j.n_sel;
    if (t >= j.prefix * n_sel) return false;
    if (t < n_sel) p = 0;
    else if (t < 2 * n_sel) p = 1;      // the K/V pair of vLLM's caches: no division
    else p = t / n_sel;
    s = t - p * n_sel;
    const int page = uniform_load(j.idx + s);
    if (page <= 0 || page >= j.num_pages) return false;
    cache = j.layer + p * j.prefix_stride + static_cast<int64_t>(page) * j.page_stride;
    stage = j.stage + static_cast<int64_t>(t) * j.span;
    return true;
}

// A unit is a part of a tile: part_units accesses of VW bytes, the last part of a
// tile what is left. LANES: copy_lanes of the longest unit.
template <int VW, bool GATHER, class Grid, int LANES>
__global__ __launch_bounds__(LANES) void copy_pages_kernel(DescArg d, int job0, Grid grid) {
    DARIC_ARGS_TOGETHER4(d.ptr, job0, grid.begin[1], grid.cls[0].div.d);
    int jb, unit;
    grid.at_block(blockIdx.x, jb, unit);
    const CopyJob j = desc_load(desc_at<CopyJob>(d, 0) + job0 + jb);
    const int tile = static_cast<int>(j.parts.div(static_cast<uint32_t>(unit)));
    int p, s;
    uint8_t *cache, *stage;
    if (!resolve_tile(j, tile, p, s, cache, stage)) return;
    const int u0 = (unit - tile * static_cast<int>(j.parts.d)) * j.part_units;
    const int cnt = min(j.part_units, j.span / VW - u0);
    if (cnt <= 0) return;
    const int64_t b0 = static_cast<int64_t>(u0) * VW;
    if (GATHER)
        copy_units<VW, LANES>(cache + b0, stage + b0, cnt);
    else
        copy_units<VW, LANES>(stage + b0, cache + b0, cnt);
}

// Fused scatter + rotation for any row width (rotate_rows.h). A workgroup takes
// a part of a page span: whole rows, up to 16 KiB, in the order of JobRuns. The
// loads are issued before the workgroup computes the tile's cos/sin values into
// LDS, so the sincos latency overlaps the memory latency. Rows that are not
// rotated (V rows, tokens past the job's n_tokens) are copied bit-exactly. fp8
// codes are rotated as stored: a per-head scale cancels in a linear rotation.
// Bound by HBM. Against one workgroup per page span with a lane per pair of
// units, on MI355X: 48 layers x 78 pages of 64 x 576 bf16 122 -> 109 us (5.1
// TB/s), 60 layers x 855 pages of 16 x 576 e4m3 365 -> 216 us, 6 layers x 76
// K+V pages of 64 x 8 x 192 bf16 99 -> 69 us. Rotary halves inside a unit took a
// scatter and a pass per layer before: 18 layers, 8 heads of 80 with 40 rotated,
// 22000 tokens 686 -> 362 us in one launch instead of 19.
// Eight wavefronts per SIMD: the compiler took 66 to 68 registers of its own accord,
// seven wavefronts (fp16 pairs of 96 in K+V pages 30.1 -> 29.0 us, 80 layers of 1 x
// 192 bf16 82.7 -> 75.5).
template <int KIND, bool NEOX, bool ALIGNED>
__global__ __launch_bounds__(kThreads, 8) void scatter_rotate_rows_kernel(
    DescArg d, int job0, JobRuns jr, RowGeomDiv gd, const float* __restrict__ inv_freq) {
    static_assert(kThreads == kRowThreads && kRowPartUnits == kRowUnits, "one part per workgroup");
    using RR = RowRotation<KIND, NEOX, ALIGNED>;
    __shared__ u32x4 s_row[NEOX ? kRowUnits : 1];
    __shared__ float4 s_cs[kRowMaxHalf / 2];

    DARIC_ARGS_TOGETHER6(d.ptr, job0, jr.begin[1], jr.cls[0].div.d, gd.parts.d, gd.ps.d);
    int jb, unit;
    jr.at_block(blockIdx.x, jb, unit);
    const CopyJob j = desc_load(desc_at<CopyJob>(d, 0) + job0 + jb);
    const int tile = static_cast<int>(gd.parts.div(static_cast<uint32_t>(unit)));
    int p, s;
    uint8_t *cache, *stage;
    if (!resolve_tile(j, tile, p, s, cache, stage)) return;

    const RowGeom& g = gd.g;
    const int upr = static_cast<int>(gd.upr.d);
    const int r0 = (unit - tile * static_cast<int>(gd.parts.d)) * gd.part_rows;
    const int n = min(gd.part_rows, g.n_rows - r0) * upr;
    const u32x4* __restrict__ src = reinterpret_cast<const u32x4*>(stage) + static_cast<int64_t>(r0) * upr;
    u32x4* __restrict__ dst = reinterpret_cast<u32x4*>(cache) + static_cast<int64_t>(r0) * upr;
    const int n_valid = min(max(j.n_tokens - s * g.PS, 0), g.PS);
    if (p != 0 || n_valid == 0 || j.delta == 0.0f || r0 >= g.krows) {
        copy_units<16>(reinterpret_cast<const uint8_t*>(src), reinterpret_cast<uint8_t*>(dst), n);
        return;
    }

    // A row wider than the part: its rotated dims (at most 512) lie in the first
    // kRowUnits units.
    if (n > kRowUnits)
        copy_units<16>(reinterpret_cast<const uint8_t*>(src + kRowUnits), reinterpret_cast<uint8_t*>(dst + kRowUnits),
                       n - kRowUnits);
    const int tid = static_cast<int>(threadIdx.x);
    u32x4 v[kRowUnroll];
#pragma unroll
    for (int u = 0; u < kRowUnroll; ++u) {
        const int i = u * kThreads + tid;
        v[u] = u32x4{0u, 0u, 0u, 0u};
        if (i < n) v[u] = ld_nt(src + i);
    }
    RR::fill(s_cs, g.R / 2, j.delta, inv_freq);
    if constexpr (NEOX) {
#pragma unroll
        for (int u = 0; u < kRowUnroll; ++u) s_row[u * kThreads + tid] = v[u];
    }
    __syncthreads();
    const int rot_units = RR::rotated_units(g.R);
#pragma unroll
    for (int u = 0; u < kRowUnroll; ++u) {
        const int i = u * kThreads + tid;
        if (i >= n) continue;
        const int row = static_cast<int>(gd.upr.div(static_cast<uint32_t>(i)));
        const int k = i - row * upr;
        const uint32_t q = gd.tok_div.div(static_cast<uint32_t>(r0 + row));
        const int token = static_cast<int>(q - gd.ps.div(q) * static_cast<uint32_t>(g.PS));
        const bool rot = k < rot_units && r0 + row < g.krows && token < n_valid;
        st_nt(dst + i, rot ? RR::turn(v[u], s_row + (NEOX ? i - k : 0), k, s_cs, g.R / 2) : v[u]);
    }
}

// Lane-exchange variant of the fused kernel, used when the 16-byte units of a
// row (upr = W / VE) divide the 64-lane wavefront. Lanes keep the plain
// copy's access pattern -- unit i of the tile is lane i % 256 of round
// i / 256, fully coalesced -- so a lane's position k = i % upr inside its row
// is fixed, and so are its rotary pair indices: its cos/sin values are read
// from LDS into registers once per tile. NeoX pair halves (units k and
// k +- n_rot of the same row, always in the same wavefront) are exchanged with
// ds_bpermute. GPT-J pairs are adjacent elements of one unit and need no
// exchange. Values are converted, rotated and repacked one 32-bit word at a
// time. Rows that are not rotated are stored as loaded.
//
// fp8 (e4m3) with per-head scales: dequantise -> rotate -> requantise is
// sat_rtne(rot(q * s) / s) with one scale s for both members of a pair (they
// lie in the same head row), and a rotation is linear, so that equals
// sat_rtne(rot(q)) up to float32 rounding (relative 2^-24, far below the
// e4m3 quantum). The kernel therefore rotates the code values directly and
// saturates on requantisation; the registered scales are needed only where
// cached values meet other data (kv_deviation).
// Units in flight per lane in the lane kernel.
constexpr int kRotLaneUnroll = 4;

template <int KIND, bool NEOX>
__global__ __launch_bounds__(kThreads) void scatter_rotate_lane_kernel(
    DescArg d, int job0, JobRuns jr, RowGeomDiv gd, const float* __restrict__ inv_freq, int log2_parts) {
    using E = Elem<KIND>;
    constexpr int VE = E::VE;
    constexpr int EPW = E::EPW;
    // A lane's cos/sin values (one per pair it touches) stay in registers for
    // 16-bit types. For e4m3 a 16-byte unit spans 16 pairs, and 32 registers
    // of them held the kernel at 114 VGPRs (4 waves/SIMD); it reads them from
    // LDS instead, interleaved (cos, sin) so one float4 serves two pairs: 66
    // VGPRs, 7 waves/SIMD, 1.6% faster at config 5 in a same-process A/B. For
    // bf16 the register form measured 1% faster. Both give identical bits.
    constexpr bool CSL = KIND == kE4M3;
    constexpr int NC = CSL ? 1 : (NEOX ? VE : VE / 2);  // cos/sin values per lane
    constexpr int UNR = kRotLaneUnroll;
    __shared__ float s_cos[kMaxHalfRot];
    __shared__ float s_sin[kMaxHalfRot];
    __shared__ float4 s_cs[kMaxHalfRot / 2];   // CSL: (cos, sin) of pairs 2i and 2i+1

    DARIC_ARGS_TOGETHER6(d.ptr, job0, jr.begin[1], jr.cls[0].div.d, gd.ps.d, log2_parts);
    int jb, unit;
    jr.at_block(blockIdx.x, jb, unit);
    const CopyJob j = desc_load(desc_at<CopyJob>(d, 0) + job0 + jb);
    int p, s;
    uint8_t *cache, *stage;
    if (!resolve_tile(j, unit >> log2_parts, p, s, cache, stage)) return;
    const int n_units = j.span / 16;
    const int per = n_units >> log2_parts;
    const int u0 = (unit & ((1 << log2_parts) - 1)) * per;
    const int u1 = u0 + per;

    const RowGeom& g = gd.g;
    const int n_valid = min(max(j.n_tokens - s * g.PS, 0), g.PS);
    if (p != 0 || n_valid == 0 || j.delta == 0.0f || g.krows == 0) {
        copy_units<16>(stage + static_cast<int64_t>(u0) * 16, cache + static_cast<int64_t>(u0) * 16, per);
        return;
    }

    const int tid = static_cast<int>(threadIdx.x);
    const int lane = tid & 63;
    const int upr = g.W / VE;                       // a power of two <= 64
    const int log2_upr = __builtin_ctz(static_cast<unsigned>(upr));
    const int k = tid & (upr - 1);
    const int nr = g.n_rot;
    const bool rot_lane = NEOX ? k < 2 * nr : k < nr;
    const bool first = k < nr;
    const int src_lane = (NEOX && rot_lane) ? (first ? lane + nr : lane - nr) : lane;
    const int pi0 = NEOX ? (first ? k : k - nr) * VE : k * (VE / 2);
    const int half = g.R / 2;
    const u32x4* __restrict__ src = reinterpret_cast<const u32x4*>(stage);
    u32x4* __restrict__ dst = reinterpret_cast<u32x4*>(cache);

    float cs[NC], ss[NC];
    for (int base = u0; base < u1; base += kThreads * UNR) {
        u32x4 v[UNR];
#pragma unroll
        for (int u = 0; u < UNR; ++u) {
            const int i = base + u * kThreads + tid;
            v[u] = u32x4{0u, 0u, 0u, 0u};
            if (i < u1) v[u] = ld_nt(src + i);
        }
        if (base == u0) {
            // 16-bit types: lane k takes pairs kk*NC .. kk*NC + NC-1 into
            // registers. The table is stored transposed, pair i at
            // (i % NC) * (half / NC) + i / NC, so the lanes of a wavefront
            // read consecutive words for each e (the row-major, stride-NC
            // reads took 5.5 M bank-conflict cycles per launch at config 2).
            // e4m3 (CSL): the (cos, sin) entries are transposed the same way
            // -- NeoX float4 j (pairs 2j, 2j+1 of a unit) of unit kk at
            // j * (half / VE) + kk, GPT-J float2 pair pi at pi * (half /
            // (VE / 2)) + kk -- so each LDS read instruction takes consecutive
            // entries across the lanes (interleaved in pair order, they took
            // 30% of the kernel's LDS cycles in bank conflicts at config 5).
            const int cols = half / NC;
            for (int i = tid; i < half; i += kThreads) {
                float sn, c;
                sincosf(j.delta * inv_freq[i], &sn, &c);
                if (CSL) {
                    float* q;
                    if (NEOX) {
                        const int f = i >> 1;
                        q = reinterpret_cast<float*>(s_cs + (f % (VE / 2)) * (half / VE) + f / (VE / 2)) + 2 * (i & 1);
                    } else {
                        q = reinterpret_cast<float*>(s_cs) + 2 * ((i % (VE / 2)) * (half / (VE / 2)) + i / (VE / 2));
                    }
                    q[0] = c;
                    q[1] = sn;
                } else {
                    const int at = (i % NC) * cols + i / NC;
                    s_cos[at] = c;
                    s_sin[at] = sn;
                }
            }
            __syncthreads();
            if (!CSL) {
                const int kk = pi0 / NC;
#pragma unroll
                for (int e = 0; e < NC; ++e) {
                    const int at = rot_lane ? e * cols + kk : 0;
                    cs[e] = s_cos[at];
                    ss[e] = (NEOX && first) ? -s_sin[at] : s_sin[at];
                }
            }
        }
#pragma unroll
        for (int u = 0; u < UNR; ++u) {
            const int i = base + u * kThreads + tid;
            u32x4 pv = v[u];
            if (NEOX) {
#pragma unroll
                for (int w = 0; w < 4; ++w)
                    pv[w] = static_cast<uint32_t>(__shfl(static_cast<int>(v[u][w]), src_lane, 64));
            }
            if (i >= u1) continue;
            const uint32_t r = static_cast<uint32_t>(i >> log2_upr);
            const uint32_t q = gd.tok_div.div(r);
            const int token = static_cast<int>(q - gd.ps.div(q) * g.PS);
            const bool rot = rot_lane && static_cast<int>(r) < g.krows && token < n_valid;
            if (!rot) {
                st_nt(dst + i, v[u]);
                continue;
            }
            u32x4 out;
#pragma unroll
            for (int w = 0; w < 4; ++w) {
                float x[EPW];
                E::unpack_word(v[u][w], x);
                if (NEOX) {
                    float y[EPW];
                    E::unpack_word(pv[w], y);
                    if (CSL) {
                        // pairs pi0 + w*EPW .. +EPW-1: EPW/2 float4 reads
                        const int kk = pi0 / VE;
#pragma unroll
                        for (int h2 = 0; h2 < EPW / 2; ++h2) {
                            const float4 t = s_cs[(w * (EPW / 2) + h2) * (half / VE) + kk];
                            const float s0 = first ? -t.y : t.y, s1 = first ? -t.w : t.w;
                            x[2 * h2] = x[2 * h2] * t.x + y[2 * h2] * s0;
                            x[2 * h2 + 1] = x[2 * h2 + 1] * t.z + y[2 * h2 + 1] * s1;
                        }
                    } else {
#pragma unroll
                        for (int e = 0; e < EPW; ++e)
                            x[e] = x[e] * cs[w * EPW + e] + y[e] * ss[w * EPW + e];
                    }
                } else {
#pragma unroll
                    for (int m = 0; m < EPW / 2; ++m) {
                        const int pi = w * (EPW / 2) + m;
                        float c, sn;
                        if (CSL) {
                            const float* csq = reinterpret_cast<const float*>(s_cs) +
                                               2 * (pi * (half / (VE / 2)) + pi0 / (VE / 2));
                            c = csq[0];
                            sn = csq[1];
                        } else {
                            c = cs[pi];
                            sn = ss[pi];
                        }
                        const float x1 = x[2 * m], x2 = x[2 * m + 1];
                        x[2 * m] = x1 * c - x2 * sn;
                        x[2 * m + 1] = x2 * c + x1 * sn;
                    }
                }
                out[w] = E::pack_word(x);
            }
            st_nt(dst + i, out);
        }
    }
}

// Descriptor upload: one 16-byte unit per lane, read from host memory.
__global__ __launch_bounds__(kThreads) void upload_kernel(const u32x4* __restrict__ src,
                                                         u32x4* __restrict__ dst, uint32_t n16) {
    const uint32_t i = blockIdx.x * kThreads + threadIdx.x;
    if (i < n16) dst[i] = src[i];
}

void launch_copy_pages(const DescArg& d, const JobClasses& classes, int64_t part, int vw,
                       bool gather, hipStream_t stream) {
    if (classes.empty()) return;
    const int lanes = copy_lanes(part, vw);
#define DARIC_CP(VW, G, GRID, T) DARIC_LAUNCH((copy_pages_kernel<VW, G, GRID, T>), blocks, T, 0, stream, d, j0, g)
#define DARIC_CPV(G, GRID)                                                                               \
    do {                                                                                                 \
        if (vw == 16 && lanes == 64) DARIC_CP(16, G, GRID, 64);                                          \
        else if (vw == 16 && lanes == 128) DARIC_CP(16, G, GRID, 128);                                   \
        else if (vw == 16) DARIC_CP(16, G, GRID, 256);                                                   \
        else if (vw == 4) DARIC_CP(4, G, GRID, 256);                                                     \
        else DARIC_CP(1, G, GRID, 256);                                                                  \
    } while (0)
    if (gather) {
        for_job_rows(classes, 1, part, [&](int j0, const JobRows& g, unsigned blocks) {
            DARIC_CPV(true, JobRows);
            check_launch("gather_pages");
        });
        return;
    }
    for_job_runs(classes, 1, part, kScatterRunsFrom, [&](int j0, const JobRuns& g, unsigned blocks) {
        DARIC_CPV(false, JobRuns);
        check_launch("scatter_pages");
    });
#undef DARIC_CPV
#undef DARIC_CP
}

void launch_upload(const void* src, void* dst, size_t n16, hipStream_t stream) {
    if (n16 == 0) return;
    const dim3 grid(static_cast<unsigned>((n16 + kThreads - 1) / kThreads));
    upload_kernel<<<grid, kThreads, 0, stream>>>(static_cast<const u32x4*>(src), static_cast<u32x4*>(dst),
                                                 static_cast<uint32_t>(n16));
    check_launch("descriptor upload");
}

void launch_scatter_rotate(const DescArg& d, const JobClasses& classes, const RowGeom& g, int kind,
                           bool neox, const float* inv_freq, hipStream_t stream) {
    RowGeomDiv gd;
    gd.g = g;
    gd.tok_div = FastDiv(static_cast<uint32_t>(g.tok_div));
    gd.ps = FastDiv(static_cast<uint32_t>(g.PS));
    const int unit_elems = kind == kE4M3 ? 16 : 8;
    gd.upr = FastDiv(static_cast<uint32_t>(g.W / unit_elems));
    const FusedCut cut(g, unit_elems);
    const int lp = cut.log2_parts;
    if (cut.lane) {
        for_job_runs(classes, cut.parts, cut.unit_bytes, fused_runs_from(cut.unit_bytes),
                     [&](int j0, const JobRuns& jr, unsigned blocks) {
#define DARIC_SR(K, N) DARIC_LAUNCH((scatter_rotate_lane_kernel<K, N>), blocks, kThreads, 0, stream, d, j0, jr, gd, inv_freq, lp)
            if (kind == kBF16) { if (neox) DARIC_SR(kBF16, true); else DARIC_SR(kBF16, false); }
            else if (kind == kF16) { if (neox) DARIC_SR(kF16, true); else DARIC_SR(kF16, false); }
            else { if (neox) DARIC_SR(kE4M3, true); else DARIC_SR(kE4M3, false); }
#undef DARIC_SR
            check_launch("scatter_pages_rerotate");
        });
        return;
    }
    gd.parts = FastDiv(static_cast<uint32_t>(cut.parts));
    gd.part_rows = static_cast<int32_t>(cut.part_rows);
    for_job_runs(classes, cut.parts, cut.unit_bytes, fused_runs_from(cut.unit_bytes),
                 [&](int j0, const JobRuns& jr, unsigned blocks) {
#define DARIC_SR(K, N, A) DARIC_LAUNCH((scatter_rotate_rows_kernel<K, N, A>), blocks, kThreads, 0, stream, d, j0, jr, gd, inv_freq)
#define DARIC_SRA(K, N) do { if (g.aligned) DARIC_SR(K, N, true); else DARIC_SR(K, N, false); } while (0)
        if (kind == kBF16) { if (neox) DARIC_SRA(kBF16, true); else DARIC_SRA(kBF16, false); }
        else if (kind == kF16) { if (neox) DARIC_SRA(kF16, true); else DARIC_SRA(kF16, false); }
        else { if (neox) DARIC_SRA(kE4M3, true); else DARIC_SRA(kE4M3, false); }
#undef DARIC_SRA
#undef DARIC_SR
        check_launch("scatter_pages_rerotate");
    });
}

}  // namespace daric
