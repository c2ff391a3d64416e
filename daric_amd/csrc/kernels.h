// Launchers of the gfx950 kernels (defined in the .hip files).
#pragma once

#include <algorithm>
#include <mutex>
#include <vector>

#include <hip/hip_runtime_api.h>

#include <cstdint>

#include "jobs.h"

namespace daric {

struct RowGeomDiv {
    RowGeom g;
    FastDiv tok_div, ps;
    FastDiv upr;     // 16-byte units per row
    FastDiv parts;   // parts a page span is cut into, each but the last of part_rows rows (rows kernel)
    int32_t part_rows = 0;
};

// Page spans of rows of `upr` 16-byte units, cut into parts of whole rows for
// a kernel whose workgroups hold up to kRowPartUnits units: the fewest parts,
// of nearly equal size.
constexpr int64_t kRowPartUnits = 1024;
struct RowParts {
    int32_t parts = 1, part_rows = 1;
    RowParts(int64_t n_rows, int64_t upr) {
        const int64_t most = std::max<int64_t>(1, kRowPartUnits / std::max<int64_t>(upr, 1));
        const int64_t n = (n_rows + most - 1) / most;
        part_rows = static_cast<int32_t>((n_rows + n - 1) / n);
        parts = static_cast<int32_t>((n_rows + part_rows - 1) / part_rows);
    }
};

// Stores the first n bytes (even; all 16 from 16 up) of a 16-byte unit, w its four
// words, and leaves the rest of dst alone: in place, the bytes past a row's rotary
// dims may be V, or a tail that another stream writes meanwhile.
template <class Words>
inline DARIC_HD void store_unit_head(uint8_t* dst, const Words& w, int n) {
#ifdef __HIP_DEVICE_COMPILE__
#pragma unroll
#endif
    for (int i = 0; i < 4; ++i) {
        if (4 * i + 4 <= n) *reinterpret_cast<uint32_t*>(dst + 4 * i) = w[i];
        else if (4 * i + 2 <= n) *reinterpret_cast<uint16_t*>(dst + 4 * i) = static_cast<uint16_t>(w[i]);
    }
}

// Layer-minor block order for kernels over (layer, work item) pairs: block b
// of a launch takes layer l0 + b % nl and work item w0 + b / nl. Workgroups
// are dispatched to the 8 XCDs in turn, so with nl a multiple of 8 each XCD
// works on a fixed eighth of the layers, and its address translations and L2
// see an eighth of the layers' memory. On MI355X that made the row merge 8-12%
// faster, the fused top-k + merge 5-7% and the in-place re-rotation 4-10%
// than work-item-major grids (in same-process A/Bs at configs 2, 3 and 5);
// the deviation kernel, which streams each layer's rows in order, ran 4-5%
// slower that way and keeps its tile-major grid.
struct LayerMinor {
    int32_t l0 = 0;     // first layer of the launch
    int32_t nl = 1;     // layers of the launch
    int64_t w0 = 0;     // first work item of the launch
    // (layer, work item) of block b of the launch
    inline DARIC_HD void at_block(uint32_t b, int& l, int64_t& w) const {
        const uint32_t n = static_cast<uint32_t>(nl);
        l = l0 + static_cast<int>(b % n);
        w = w0 + static_cast<int64_t>(b / n);
    }
#ifdef __HIPCC__
    __device__ inline void at(int& l, int64_t& w) const { at_block(blockIdx.x, l, w); }
#endif
};

// Largest grid.x of a 256-lane launch (grid.x * 256 lanes < 2^32).
constexpr int64_t kMaxGridBlocks = (1ll << 24) - 1;

// Calls launch(LayerMinor, blocks) for launches that together cover
// n_layers x n_items, each of at most kMaxGridBlocks blocks.
template <class F>
void for_layer_minor(int n_layers, int64_t n_items, F&& launch) {
    if (n_layers <= 0 || n_items <= 0) return;
    const int64_t nl = std::min<int64_t>(n_layers, kMaxGridBlocks);
    const int64_t per = std::max<int64_t>(1, kMaxGridBlocks / nl);
    for (int64_t l0 = 0; l0 < n_layers; l0 += nl) {
        LayerMinor lm;
        lm.l0 = static_cast<int32_t>(l0);
        lm.nl = static_cast<int32_t>(std::min<int64_t>(nl, n_layers - l0));
        for (int64_t w0 = 0; w0 < n_items; w0 += per) {
            lm.w0 = w0;
            const int64_t ni = std::min<int64_t>(per, n_items - w0);
            launch(lm, static_cast<unsigned>(lm.nl * ni));
        }
    }
}

// The jobs of a page copy by length: classes of consecutive jobs of `tiles`
// tiles each (the longest of the class), longest first (order_jobs). A grid made
// from them has workgroups for the tiles that are there; one sized by the
// longest job gave every job as many, and a workgroup that finds nothing to do
// still costs its place in the queue (about 0.7 ns on the whole chip). Same
// process, MI355X, against the grid of the longest job, in 8 KiB parts: gather
// into rows of 24 KiB pages 168 -> 157 us (three chunks of 1111 to 3000 tokens),
// 48 KiB 411 -> 392 us (five of 1462 to 2629), 72 KiB 172 -> 161 us (six of 64
// to 4000).
struct JobClass {
    int64_t jobs, tiles;
};
constexpr int kJobClasses = 8;
struct JobClasses {
    int n = 0;
    JobClass c[kJobClasses];
    bool empty() const { return n == 0; }
    const JobClass& operator[](int k) const { return c[k]; }
    int64_t jobs() const {
        int64_t s = 0;
        for (int k = 0; k < n; ++k) s += c[k].jobs;
        return s;
    }
    // One class of `jobs` jobs (none of jobs without tiles).
    static JobClasses even(int64_t jobs, int64_t tiles) {
        JobClasses r;
        if (tiles > 0 && jobs > 0) r.c[r.n++] = {jobs, tiles};
        return r;
    }
};

// Joins neighbours of a descending list of lengths until at most kJobClasses
// are left, each time those where that adds the fewest idle workgroups.
// joined[i] is the class that entry i ends up in. Returns their number.
inline int join_classes(JobClass* d, int n, int* joined) {
    int at[64], live = n;
    for (int i = 0; i < n; ++i) at[i] = i;     // the entry that starts live class k
    while (live > kJobClasses) {
        int best = 0;
        int64_t least = -1;
        for (int k = 0; k + 1 < live; ++k) {
            const int64_t idle = (d[at[k]].tiles - d[at[k + 1]].tiles) * d[at[k + 1]].jobs;
            if (least < 0 || idle < least) { least = idle; best = k; }
        }
        d[at[best]].jobs += d[at[best + 1]].jobs;
        for (int k = best + 1; k + 1 < live; ++k) at[k] = at[k + 1];
        --live;
    }
    for (int i = 0, k = -1; i < n; ++i) {
        if (k + 1 < live && at[k + 1] == i) ++k;
        joined[i] = k;
    }
    for (int k = 0; k < live; ++k) d[k] = d[at[k]];
    return live;
}

// Sorts `jobs` by descending class of count(job), keeping the order within a
// class, and returns the classes (jobs without tiles come last, in none).
template <class Job, class Count>
JobClasses order_jobs(std::vector<Job>& jobs, Count&& count) {
    JobClasses out;
    const size_t n = jobs.size();
    if (n == 0) return out;
    constexpr int kLengths = 64;
    JobClass d[kLengths];
    int nd = 0, last = 0;
    int64_t longest = count(jobs[0]);
    bool even = true;
    for (size_t i = 1; i < n; ++i) {
        const int64_t t = count(jobs[i]);
        even = even && t == longest;
        longest = std::max(longest, t);
    }
    if (even) return JobClasses::even(static_cast<int64_t>(n), longest);
    std::vector<uint32_t> to(n);      // a job's length, then its place
    // lengths in at most 63 steps of the longest (exact up to 63 tiles, or where
    // no more than 64 lengths occur), rounded up
    int64_t step = 1;
    for (size_t i = 0; i < n; ++i) {
        const int64_t tiles = count(jobs[i]);
        const int64_t t = step == 1 ? tiles : (tiles + step - 1) / step * step;
        if (nd == 0 || d[last].tiles != t) {
            for (last = 0; last < nd && d[last].tiles != t;) ++last;
            if (last == nd) {
                if (nd == kLengths) {     // too many lengths: start again in coarser steps
                    step = (longest + 62) / 63;
                    nd = 0;
                    i = static_cast<size_t>(-1);
                    continue;
                }
                d[nd++] = {0, t};
            }
        }
        ++d[last].jobs;
        to[i] = static_cast<uint32_t>(last);
    }
    if (nd == 1) return JobClasses::even(static_cast<int64_t>(n), longest);
    int rank[kLengths], joined[kLengths];
    JobClass s[kLengths];
    int ns = 0;
    for (int i = 0; i < nd; ++i) {
        rank[i] = 0;
        for (int k = 0; k < nd; ++k) rank[i] += d[k].tiles > d[i].tiles ? 1 : 0;
        if (d[i].tiles > 0) ++ns;
    }
    for (int i = 0; i < nd; ++i)
        if (d[i].tiles > 0) s[rank[i]] = d[i];
    out.n = join_classes(s, ns, joined);
    size_t at[kJobClasses + 1] = {0};
    for (int k = 0; k < out.n; ++k) {
        out.c[k] = {s[k].jobs, std::min(s[k].tiles, longest)};
        at[k + 1] = at[k] + static_cast<size_t>(s[k].jobs);
    }
    uint32_t cls[kLengths];
    for (int i = 0; i < nd; ++i) cls[i] = d[i].tiles > 0 ? joined[rank[i]] : out.n;
    for (size_t i = 0; i < n; ++i) to[i] = static_cast<uint32_t>(at[cls[to[i]]]++);
    // In place: with a second, zeroed array of jobs and a division per job 432 uneven
    // jobs of 112 bytes took 9.8 us instead of 4.5, 1280 took 72 instead of 16 (one
    // host core).
    for (size_t i = 0; i < n; ++i) {
        if (to[i] == i) continue;
        Job held = jobs[i];
        for (uint32_t k = static_cast<uint32_t>(i); to[k] != k;) {
            const uint32_t next = to[k];
            to[k] = k;
            std::swap(held, jobs[next]);
            k = next;
        }
    }
    return out;
}

// Bytes of the parts that a page copy cuts its tiles into, the last part of a
// tile what is left, for a job of `tiles` tiles of `span` bytes: one up to 11 KiB,
// two equal ones up to 16 KiB, then 8 KiB (two accesses of 16 bytes per lane), and
// more where a job's parts would not fit in one launch. A part as long as the tile ends the doubling: a job of up to
// kMaxGridBlocks tiles then has a workgroup per tile. Each job is cut by its own
// span: by the call's largest, 60 layers of 8 KiB pages beside 4 of 128 KiB had
// 16 workgroups to each of their pages, 15 of them idle (gather of 584 MiB 645 ->
// 195 us).
// Exact 8 KiB parts left pages of 8.5 to 15 KiB a small second part: gathers of
// 300 MiB in pages of 8.5, 9, 10 and 12 KiB ran at 0.79, 0.81, 0.88 and 0.97 of
// the rate of one part per page, scatters at 0.87, 0.91, 0.95 and 1.01, and by
// this rule at 1.02, 0.99, 0.99 and 1.00, and 1.00, 0.98, 1.00 and 1.03. From
// 16 KiB up exact parts are 0.99-1.05 of parts of 8 to 16 KiB, and equal parts
// 0.97-1.03 of exact ones; above 64 KiB they are 1.1-1.25 of eight parts each, and
// parts of 4 KiB 0.88-1.05 of these rates (MI355X).
inline int64_t page_part_bytes(int64_t span, int64_t tiles) {
    int64_t part = span <= 11 * 1024 ? std::max<int64_t>(span, 8192)
                 : span <= 16 * 1024 ? ((span + 1) / 2 + 255) / 256 * 256 : 8192;
    while (part < span && (span + part - 1) / part * tiles > kMaxGridBlocks) part *= 2;
    return part;
}

// Parts of a page span in the fused scatter, whose jobs share a row geometry; lane:
// the lane-exchange kernel (whole rows inside a wavefront, pair halves of whole
// units), log2_parts of its pages. The rows kernel takes the other rows. unit_elems:
// values in 16 bytes.
struct FusedCut {
    bool lane;
    int log2_parts = 0;
    int64_t parts, unit_bytes, part_rows = 0;
    FusedCut(const RowGeom& g, int unit_elems) {
        const int upr = g.W / unit_elems;
        const int64_t units = static_cast<int64_t>(g.n_rows) * upr;   // 16-byte units per page span
        lane = g.aligned && 64 % upr == 0;
        if (lane) {
            // Pages cut into parts of at least 16 KiB, whole rows each. Two 16 KiB
            // halves of the 32 KiB bf16 pages measured ~1% faster than whole pages
            // at config 2, kernel and whole call alike (347.2 against 350.2 us per
            // kernel, 347.5 against 350.7 us per call; bit-identical output);
            // 8 KiB parts were 4% slower.
            while ((units >> (log2_parts + 1)) * 16 >= 16384 && units % (2ll << log2_parts) == 0 &&
                   (units >> (log2_parts + 1)) % upr == 0)
                ++log2_parts;
            parts = 1ll << log2_parts;
            unit_bytes = (units * 16) >> log2_parts;
        } else {
            const RowParts rp(g.n_rows, upr);
            parts = rp.parts;
            part_rows = rp.part_rows;
            unit_bytes = part_rows * upr * 16;
        }
    }
};

// Jobs of the fused scatter whose parts would not fit one launch (2^24 - 1 pages of
// two parts and more) go as several: of consecutive pages, of K and of V apart. V's
// are copied, which a delta of 0 asks for; PS: tokens of a page.
inline void split_long_jobs(std::vector<CopyJob>& jobs, int64_t parts, int64_t PS) {
    const int64_t most = std::max<int64_t>(1, kMaxGridBlocks / parts);
    std::vector<CopyJob> out;
    for (size_t i = 0; i < jobs.size(); ++i) {
        const CopyJob& j = jobs[i];
        const bool fits = static_cast<int64_t>(j.prefix) * j.n_sel <= most;
        if (fits && out.empty()) continue;
        if (out.empty()) out.assign(jobs.begin(), jobs.begin() + static_cast<std::ptrdiff_t>(i));
        if (fits) {
            out.push_back(j);
            continue;
        }
        for (int64_t p = 0; p < j.prefix; ++p) {
            for (int64_t s = 0; s < j.n_sel; s += most) {
                CopyJob piece = j;
                piece.layer += p * j.prefix_stride;
                piece.stage += (p * j.n_sel + s) * j.span;
                piece.idx += s;
                piece.prefix = 1;
                piece.n_sel = static_cast<int32_t>(std::min<int64_t>(most, j.n_sel - s));
                piece.n_tokens = static_cast<int32_t>(std::max<int64_t>(0, j.n_tokens - s * PS));
                if (p > 0) piece.delta = 0.0f;
                out.push_back(piece);
            }
        }
    }
    if (!out.empty()) jobs.swap(out);
}

// Cuts the jobs' tiles into parts for accesses of vw bytes and orders the jobs by
// their parts. *part gets the longest part's bytes, of pages shorter than a part the
// page's.
inline JobClasses cut_pages(std::vector<CopyJob>& jobs, int vw, int64_t* part) {
    *part = 0;
    const CopyJob* like = nullptr;     // job whose tiles the last one had: no divisions again
    bool even = true;                  // no second pass over the jobs of the usual call
    for (CopyJob& j : jobs) {
        const int64_t tiles = static_cast<int64_t>(j.prefix) * j.n_sel;
        if (like != nullptr && like->span == j.span && like->n_sel == j.n_sel && like->prefix == j.prefix) {
            j.part_units = like->part_units;
            j.parts = like->parts;
        } else {
            const int64_t bytes = page_part_bytes(j.span, tiles);
            j.part_units = static_cast<int32_t>((bytes + vw - 1) / vw);
            j.parts = FastDiv(static_cast<uint32_t>(std::max<int64_t>(1, (j.span + bytes - 1) / bytes)));
            if (tiles > 0) *part = std::max(*part, std::min<int64_t>(bytes, j.span));
            even = like == nullptr;
            like = &j;
        }
    }
    if (even && like != nullptr)
        return JobClasses::even(static_cast<int64_t>(jobs.size()), static_cast<int64_t>(like->prefix) * like->n_sel * like->parts.d);
    return order_jobs(jobs, [](const CopyJob& j) {
        return static_cast<int64_t>(j.prefix) * j.n_sel * j.parts.d;
    });
}

// Lanes of a copy's workgroups of up to unit_bytes: 256, or as many as have two
// accesses of 16 bytes each where units are small. Such workgroups are bound by
// their start, a chain of loads from the grid's class over the job and the page id
// to the data, times those a CU holds, 8 of 256 lanes: 640 MiB in pages of 2 KiB (80
// layers of 1 x 64 bf16) were gathered in 418 us by 256 lanes each, in 222 by 128 and
// in 216 by 64, scattered in 405, 253 and 246, token by token in 529, 269 and 221; in
// pages of 4 KiB (1 x 128) in 222, 216 and 229, scattered in 252, 244 and 248, token
// by token in 273, 221 and 227 (MI355X).
inline int copy_lanes(int64_t unit_bytes, int vw) {
    return vw != 16 || unit_bytes > 4096 ? 256 : unit_bytes > 2048 ? 128 : 64;
}

// Most bytes of job descriptors that a copy's kernels read from the pinned slot
// itself, without an upload kernel (4-5 us with its gap) before the copy;
// unit_bytes: its largest workgroup's bytes. Every pair of CUs reads every job over
// the host link once, or again and again beyond the 16 KiB of its scalar cache.
// Gathers, whose neighbouring workgroups wait for the same job, feel that first,
// and all do where copies fill the link (the store's gather beside the last batch's
// way to the host). MI355X, uploaded against read in place, idle and beside
// host-to-device copies: gathers of 40 jobs (3.1 KiB) 44.2 and 45.6 -> 41.5 and 45.7
// us, 40 (4.4) 45.4 and 47.3 -> 44.0 and 50.0, 96 (10.5) 73.0 and 75.1 -> 75.1 and
// 85.2, 160 of 4 KiB pages (12.5; 256 lanes) 57.1 and 59.8 -> 65.8 and 81.6; scatters of 48
// (5.3) 28.4 and 29.7 -> 23.2 and 24.8, 128 (14) 104.9 and 108.9 -> 100.2 and 103.9,
// 160 of 4 KiB pages 64.2 and 66.4 -> 65.6 and 74.2.
inline size_t direct_desc_bytes(bool gather, int64_t unit_bytes) {
    return gather ? 4096 : unit_bytes < 8192 ? 12 * 1024 : 16 * 1024;
}

// Where the blocks of each class begin, and what they divide by. A block compares
// its place with all the begins, without a branch before the last: returning
// early for the first class ran the gathers of even jobs 2-4% slower and the
// scatters up to 1% (MI355X).
struct JobGrid {
    struct Class {
        uint32_t first = 0;
        FastDiv div;
    };
    uint32_t begin[kJobClasses];
    Class cls[kJobClasses];
    uint32_t log2_run = 0;
    JobGrid() {
        for (uint32_t& b : begin) b = 0xffffffffu;
        begin[0] = 0;
    }
    inline DARIC_HD Class find(uint32_t r, uint32_t& base) const {
        uint32_t k = 0;
        base = 0;
#ifdef __HIP_DEVICE_COMPILE__
#pragma unroll
#endif
        for (int i = 1; i < kJobClasses; ++i)
            if (r >= begin[i]) { k = static_cast<uint32_t>(i); base = begin[i]; }
#ifdef __HIP_DEVICE_COMPILE__
        const DescPtr<uint32_t> p = (DescPtr<uint32_t>)(const uint32_t*)cls + 4 * k;
        Class c;
        c.first = p[0]; c.div.d = p[1]; c.div.m = p[2]; c.div.s = p[3];
        return c;
#else
        return cls[k];
#endif
    }
};
static_assert(sizeof(JobGrid::Class) == 16, "JobGrid::Class layout");

// Block order of the kernels that scatter from staging into the pages of many
// jobs (one job per layer and chunk). Workgroups are dispatched to the 8 XCDs
// in turn; block b is place b / 8 % run of the (b / 8 / run)-th run of XCD
// b % 8, and the runs of `run` consecutive units are dealt to the XCDs job by
// job: round q takes unit block q of each of the n jobs that reach it, job
// (i + q) % n being the i-th. So an XCD reads and writes a job's consecutive
// parts while all jobs advance together, and the shift by q moves a job on to
// the next XCD with each run, so that a call of few jobs still loads the XCDs
// alike. A class's `first` is its first round, its divisor the jobs that reach
// those rounds.
// The scatters wait on HBM writes to random pages, whose rate depends on how
// the concurrent writes fall on the memory channels. Runs of 128 KiB against
// the plain job-minor order (run = 1), on MI355X, same process: fused scatter
// of 256 jobs (32 layers x 8 chunks of 1024 tokens, bf16) 408 -> 391 us on
// layers 256 MiB apart and 346 -> 341 us on layers 4 GiB apart, plain scatter
// 404 -> 381 and 345 -> 332 us; fused fp8 scatter of 1280 jobs 2135 -> 2016 us.
// Runs of 64 KiB gained half as much and runs of 512 KiB nothing on the
// fused scatter. Below `runs_from` bytes, where a call's traffic stays mostly in
// the 256 MB Infinity Cache, runs gained nothing and cost up to 5% (kScatterRunsFrom,
// fused_runs_from; token-major scatter 0.92-1.04x at 384 MiB, 0.93-1.05x at 512,
// 0.96-1.05x at 768). Fewer than 16 runs per XCD leave some XCDs idle at the end, so such
// calls take shorter runs. Runs of one unit are not shifted: units of 72 KiB ran
// 2.5% slower so.
struct JobRuns : JobGrid {
    static constexpr uint32_t kXcds = 8;
    static constexpr int64_t kRunBytes = 128 * 1024;
    static constexpr int64_t kMinRuns = 16 * kXcds;
    inline DARIC_HD void at_block(uint32_t b, int& job, int& unit) const {
        const uint32_t i = b >> 3;
        const uint32_t r = ((i >> log2_run) << 3) + (b & (kXcds - 1));
        uint32_t base;
        const Class c = find(r, base);
        const uint32_t q0 = c.div.div(r - base);
        const uint32_t q = c.first + q0;
        uint32_t j = r - base - q0 * c.div.d;
        if (log2_run != 0) {
            j += q - c.div.div(q) * c.div.d;
            if (j >= c.div.d) j -= c.div.d;
        }
        job = static_cast<int>(j);
        unit = static_cast<int>((q << log2_run) + (i & ((1u << log2_run) - 1)));
    }
};

// Block order of the gathers: job by job, unit by unit, since consecutive units
// write consecutive staging bytes. Workgroups are dispatched to the 8 XCDs in
// turn, so neighbouring parts of the staging side would be written from
// different XCDs: in rows of a multiple of 8 units (every job's row is padded to
// one, except rows of fewer than 64) the units are permuted so that XCD x's i-th
// unit becomes unit (i / run * 8 + x) * run + i % run: each XCD writes runs of
// `run` consecutive units. Runs of ~256 KiB measured fastest on MI355X (gathers
// 1-3% faster than the plain order); runs of 32-64 KiB were slower than the plain
// order. Units past the last whole group keep their place. A class's `first` is
// its first job, its divisor the units of a job's row.
struct JobRows : JobGrid {
    static constexpr uint32_t kXcds = 8;
    static constexpr int64_t kRunBytes = 256 * 1024;
    inline DARIC_HD void at_block(uint32_t b, int& job, int& unit) const {
        uint32_t base;
        const Class c = find(b, base);
        const uint32_t j = c.div.div(b - base);
        const uint32_t u = b - base - j * c.div.d;
        job = static_cast<int>(c.first + j);
        const uint32_t full = c.div.d % kXcds ? 0 : c.div.d >> (3 + log2_run) << (3 + log2_run);
        const uint32_t i = u >> 3, x = u & (kXcds - 1);
        unit = static_cast<int>(u >= full ? u : ((((i >> log2_run) << 3) + x) << log2_run) + (i & ((1u << log2_run) - 1)));
    }
};

// Calls launch(first job, grid, blocks) for launches that together cover the
// jobs' units, parts per tile, each launch of at most kMaxGridBlocks blocks:
// slices of jobs where one launch cannot hold them all.
template <class Grid, class Build, class F>
void for_job_slices(const JobClasses& classes, int64_t parts, Build&& build, F&& launch) {
    if (classes.empty() || parts <= 0) return;
    const int64_t n = classes.jobs();
    const int64_t row = classes[0].tiles * parts + 8;
    const int64_t slice = std::max<int64_t>(1, std::min<int64_t>(n, kMaxGridBlocks / row));
    for (int64_t j0 = 0; j0 < n; j0 += slice) {
        JobClasses part;
        int64_t at = 0;
        for (int k = 0; k < classes.n; ++k) {
            const int64_t lo = std::max(at, j0), hi = std::min(at + classes[k].jobs, j0 + slice);
            if (hi > lo) part.c[part.n++] = {hi - lo, classes[k].tiles * parts};
            at += classes[k].jobs;
        }
        Grid g;
        const int64_t blocks = build(part, g);
        launch(static_cast<int>(j0), g, static_cast<unsigned>(blocks));
    }
}

// JobRuns launches. Runs longer than one unit are used where the units make at
// least runs_from bytes.
template <class F>
void for_job_runs(const JobClasses& classes, int64_t parts, int64_t unit_bytes, int64_t runs_from, F&& launch) {
    int64_t total = 0;
    for (int k = 0; k < classes.n; ++k) total += classes[k].jobs * classes[k].tiles * parts;
    for_job_slices<JobRuns>(classes, parts, [&](const JobClasses& cl, JobRuns& g) {
        const auto runs = [&](uint32_t log2) {
            int64_t r = 0;
            for (int k = 0; k < cl.n; ++k) r += cl[k].jobs * ((cl[k].tiles + (1ll << log2) - 1) >> log2);
            return r;
        };
        const auto blocks = [&](uint32_t log2) {
            return log2 == 0 ? runs(0) : ((runs(log2) + JobRuns::kXcds - 1) / JobRuns::kXcds * JobRuns::kXcds) << log2;
        };
        if (total * unit_bytes >= runs_from)
            while (g.log2_run < 10 && (unit_bytes << (g.log2_run + 1)) <= JobRuns::kRunBytes) ++g.log2_run;
        while (g.log2_run > 0 && (runs(g.log2_run) < JobRuns::kMinRuns || blocks(g.log2_run) > kMaxGridBlocks))
            --g.log2_run;
        // rounds [0, shortest class's runs) hold every job, the next ones the
        // longer classes' jobs, and so on
        int64_t n = cl.jobs(), at = 0, round = 0;
        int k = 0;
        for (int i = cl.n - 1; i >= 0; --i) {
            const int64_t end = (cl[i].tiles + (1ll << g.log2_run) - 1) >> g.log2_run;
            if (end > round) {
                g.begin[k] = static_cast<uint32_t>(at);
                g.cls[k].first = static_cast<uint32_t>(round);
                g.cls[k].div = FastDiv(static_cast<uint32_t>(n));
                ++k;
                at += n * (end - round);
                round = end;
            }
            n -= cl[i].jobs;
        }
        return blocks(g.log2_run);
    }, launch);
}

// Fewest bytes of a call from which its scatters run in runs (JobRuns). Plain order
// against runs, MI355X, layers of 8 x 64 fp16, 8 x 96 and 8 x 128 bf16, 8 x 128
// e4m3, one chunk and four: plain scatter 0.95-1.05x at 64 MiB, 0.97-1.02x at 128,
// 1.01-1.07x at 160, 0.99-1.05x at 256, 1.00-1.07x from 384.
constexpr int64_t kScatterRunsFrom = 144ll << 20;
// Fused scatter with units of 8 KiB and more, and 2 x 128 bf16, 8 x 192 and MLA rows
// beside those: 0.95-0.99x at 64 MiB, 0.95-1.02x at 128, 0.96-1.03x at 160 (mean
// 0.99), 0.97-1.03x at 192 (1.00), 0.99-1.06x at 224 (1.01), 0.98-1.04x at 256
// (1.01), 0.99-1.06x at 320 (1.01), 0.98-1.05x at 352 (1.01). Smaller units never: those of 4 KiB
// ran 0.75-0.91x from 64 to 256 MiB (96 MiB in four chunks of 80 layers 49 -> 64 us,
// 56 in the plain order of earlier grids) and 0.90-0.99x at 768, of 2 KiB
// 0.69-0.95x, since each reads its job over the host link.
inline int64_t fused_runs_from(int64_t unit_bytes) {
    return unit_bytes < 8192 ? INT64_MAX : 208ll << 20;
}

// JobRows launches.
template <class F>
void for_job_rows(const JobClasses& classes, int64_t parts, int64_t unit_bytes, F&& launch) {
    for_job_slices<JobRows>(classes, parts, [&](const JobClasses& cl, JobRows& g) {
        while (g.log2_run < 10 && (unit_bytes << (g.log2_run + 1)) <= JobRows::kRunBytes) ++g.log2_run;
        int64_t at = 0, job = 0;
        for (int k = 0; k < cl.n; ++k) {
            const int64_t padded = (cl[k].tiles + 7) / 8 * 8;
            const int64_t row = cl[k].tiles < 64 || padded > kMaxGridBlocks ? cl[k].tiles : padded;
            g.begin[k] = static_cast<uint32_t>(at);
            g.cls[k].first = static_cast<uint32_t>(job);
            g.cls[k].div = FastDiv(static_cast<uint32_t>(row));
            at += row * cl[k].jobs;
            job += cl[k].jobs;
        }
        return at;
    }, launch);
}

// One token-major copy job: the pages idx[0 .. n_sel) of one layer to or from
// staging laid out as [n_kv][n_sel * PS][H][row_bytes] (K rows, then V rows).
// A workgroup moves one part: part_tokens consecutive tokens (all heads) of
// one page and one of K or V. Byte units.
struct alignas(16) TokenJob {
    uint8_t* layer;          // K element [0, ..., 0] of the layer
    uint8_t* stage;          // first byte of the job's staging range
    const int32_t* idx;      // page ids; ids outside [1, num_blocks) are skipped
    int64_t sb, ss, sh;      // page, token and head strides
    int64_t v_off;           // V plane relative to K (n_kv == 2)
    int32_t n_sel;
    int32_t num_blocks;
    int32_t PS;
    int32_t H;
    int32_t row_bytes;       // D * element size
    int32_t n_kv;            // 2, or 1 for a cache without V (MLA)
    int32_t part_tokens;
    int32_t parts_per_page;  // ceil(PS / part_tokens)
    FastDiv d_upr;           // row_bytes / access width
    FastDiv d_h;             // H
};
static_assert(sizeof(TokenJob) == 112, "TokenJob layout");

// Tokens of a part of a page (one of K or V) of PS tokens of tok_bytes each, for
// the row kernel with accesses of vw bytes: 8 KiB, two accesses per lane, where whole
// tokens make them up, else up to a quarter more where that saves a part, and parts
// of a page equal in size; pages of up to 28 KiB in one part or two, of up to 14
// KiB. Against 16 KiB (MI355X): 1.00-1.13x on gathers, 0.95-1.13x on scatters; 4 KiB
// 0.7-1.05x. Gathers of 400 MiB in pages of 11, 12, 13, 14 and 28 KiB, against 16
// KiB: 1.05, 1.04, 1.04, 1.03 and 1.02x, where parts of up to 10 KiB left them two
// parts or four and 0.88, 0.91, 0.91, 0.97 and 0.96x; 24 KiB 1.15x for 1.10x, 16 KiB
// 1.07x in two parts and 1.02x in one, 32 KiB 1.07x in four and 1.02x in two. Pages
// of 64, 96, 128 and 512 KiB of 512- and 2048-byte tokens, gathers and scatters of
// 300 MiB: 1.02-1.03, 1.06, 1.01 and 1.06x, 1.06, 1.06, 1.07 and 1.02x, in parts of
// 10 KiB 0.98-1.00, 1.04, 1.00 and 1.05x, 1.03, 1.04, 1.03 and 1.02x; tokens of
// 576 to 3072 bytes ran up to 1.13x faster in parts of up to 10 KiB than of 8.
// A job of `pages` pages whose parts would not fit one launch takes parts of 16 KiB.
inline int64_t token_row_part(int64_t PS, int64_t tok_bytes, int vw, int64_t pages) {
    constexpr int64_t kPart = 10 * 1024, kEven = 8 * 1024, kMost = 14 * 1024, kLongest = 16 * 1024;
    const int64_t bytes = vw != 16 ? 4096 : PS * tok_bytes <= 2 * kMost ? kMost : kEven % tok_bytes == 0 ? kEven : kPart;
    const int64_t most = std::min<int64_t>(PS, std::max<int64_t>(1, bytes / tok_bytes));
    const int64_t parts = (PS + most - 1) / most;
    if (vw == 16 && parts * pages > kMaxGridBlocks) return std::min<int64_t>(PS, std::max<int64_t>(1, kLongest / tok_bytes));
    return (PS + parts - 1) / parts;
}

// Token-major gather (staging <- cache) or scatter; lds selects the
// LDS-staged transpose for head-major pages ([H, PS, D] dense); vw is 16 or 1.
// part_bytes: the largest part's staging bytes (sets the XCD run length). The
// jobs are ordered by their parts (order_jobs).
void launch_token_copy(const DescArg& d, const JobClasses& classes, int64_t part_bytes, int vw,
                       bool lds, bool gather, hipStream_t stream);

// Plain page copies of the CopyJobs in `d`, cut and ordered by cut_pages for
// accesses of vw bytes (16, 4 or 1); part is its longest part.
void launch_copy_pages(const DescArg& d, const JobClasses& classes, int64_t part, int vw,
                       bool gather, hipStream_t stream);

// Fused scatter + K re-rotation of the CopyJobs in `d`, ordered by their tiles
// (order_jobs); kind is an ElemKind. All jobs share `geom`.
void launch_scatter_rotate(const DescArg& d, const JobClasses& classes, const RowGeom& geom, int kind,
                           bool neox, const float* inv_freq, hipStream_t stream);

// In-place K re-rotation over segments of tokens. `d` holds the n_segs
// RopeSegs, then (at byte layer_off) the n_layers K base pointers. `path`:
// kRotElem (per-element access), kRotVec (16-byte items, tiles of
// g.tile_tokens tokens), kRotLane or kRotRows (tiles of pages of dense K rows, see
// rerotate_lane_kernel and rerotate_rows_kernel). fp8 codes are rotated as stored (a per-head scale
// cancels in a linear rotation).
enum RotPath { kRotElem = 0, kRotVec = 1, kRotLane = 2, kRotRows = 3 };
void launch_rerotate_inplace(const DescArg& d, int layer_off, int n_layers, const InplaceGeom& g,
                             int n_segs, int n_tiles, const int32_t* block_table,
                             const float* inv_freq, int kind, bool neox, int path, hipStream_t stream);

// Slots of 64 keys a wavefront of the top-k takes of a chunk of n tokens, with T
// lanes in the workgroup: T * topk_slots(n, T) may pass 2^31 - 1, but not 2^32.
inline DARIC_HD int topk_slots(int n, int T) {
    return static_cast<int>((static_cast<uint32_t>(n) + static_cast<uint32_t>(T) - 1) / static_cast<uint32_t>(T));
}

// Selection kernels. deviation_tile_tokens: tokens per deviation workgroup
// (the tiling launch_deviation expects in SelChunk::tile_begin).
int deviation_tile_tokens(int cache_kind, const KVGeom& g);
// Selection launchers: `d` holds the n_chunks SelChunks, then (deviation and
// merge, at byte layer_off) the n_layers layer base pointers.
void launch_deviation(const DescArg& d, int layer_off, int n_layers, const KVGeom& g, int cache_kind,
                      const int32_t* block_table, const uint8_t* k_new, int new_kind,
                      int64_t T, int n_chunks, int n_tiles,
                      const float* k_scales, float* keys, hipStream_t stream);
void launch_topk(const float* keys, int n_layers, int64_t T, const DescArg& d,
                 int n_chunks, int max_tokens, int32_t* out_idx, int kmax, hipStream_t stream);
// Sets each chunk's first batch of `rows` index slots in tile_begin: n batches in
// all, `each` per chunk (0 where the chunks differ); none where rows is 0 (the
// element kernel has a grid of its own). top_k: the indices are the top-k's own,
// whose slots past the chunk's tokens are empty. A caller's may stand in any of a
// chunk's first min(k, kmax) slots.
struct MergeBatches {
    int64_t n = 0, each = 0;
};
inline MergeBatches merge_batches(std::vector<SelChunk>& chunks, int64_t kmax, int rows, bool top_k) {
    MergeBatches b;
    if (rows == 0) return b;
    for (size_t i = 0; i < chunks.size(); ++i) {
        SelChunk& c = chunks[i];
        c.tile_begin = static_cast<int32_t>(b.n);
        const int64_t slots = std::min<int64_t>(c.k, kmax);
        const int64_t own = ((top_k ? std::min<int64_t>(slots, c.n_tokens) : slots) + rows - 1) / rows;
        b.each = i == 0 || b.each == own ? own : 0;
        b.n += own;
        if (b.n > 0x7fffffff) break;      // refused by the caller
    }
    return b;
}
// merge: the SelChunks at byte chunk_off have their batches of merge_rows_per_block
// index slots (merge_batches; 0 rows and batches where the row kernel does not
// take the geometry). quant_from is -1
// (rows are copied as bytes) or the ElemKind of bf16 / fp16 rows quantised into
// an e4m3 cache with the [n_layers, H] fp32 k_scales / v_scales.
// merge_fits_rows: whether the row kernel takes the geometry (required for
// quantising); merge_max_row_bytes: the most bytes of recomputed K+V values per
// token it takes.
bool merge_fits_rows(const KVGeom& g, int elem_size, bool quant);
int64_t merge_max_row_bytes();
int merge_rows_per_block(const KVGeom& g, int elem_size, bool quant);
void launch_merge(const DescArg& d, int chunk_off, int layer_off, int n_layers, const KVGeom& g, int elem_size,
                  const int32_t* block_table, const uint8_t* k_new, const uint8_t* v_new,
                  int64_t T, int n_chunks, const MergeBatches& batches, const int32_t* sel_idx, int kmax, int quant_from,
                  const float* k_scales, const float* v_scales, hipStream_t stream);
// Fused selection, one workgroup per (layer, chunk): top-k on the chunk's
// keys held in LDS and the merge of its selected rows, with (with_keys) or
// without (keys already hold them) the chunk's deviation keys computed first
// in the same workgroup. select_merge_fits: whether it takes the geometry and
// chunk sizes, and (unless one_pass) whether a chunk's selected rows are few
// enough for one workgroup to merge faster than the merge kernel (else the
// three launches above do the same work).
bool select_merge_fits(const KVGeom& g, int elem_size, bool quant, int64_t max_tokens, int64_t kmax,
                       bool one_pass);
void launch_select_merge(const DescArg& d, int layer_off, int n_layers, const KVGeom& g, int cache_kind,
                         int elem_size, const int32_t* block_table, const uint8_t* k_new, int new_kind,
                         const uint8_t* v_new, int64_t T, int n_chunks, int max_tokens, bool with_keys,
                         float* keys, int32_t* sel_idx, int kmax, bool quant, const float* k_scales,
                         const float* v_scales, hipStream_t stream);

// Copies n16 16-byte units from host-pinned `src` to device `dst` on `stream`
// (descriptor upload; both 16-byte aligned).
void launch_upload(const void* src, void* dst, size_t n16, hipStream_t stream);

// Allocation-free descriptor staging (noalloc.hip). Each GPU holds a static
// device array of kNoAllocScratchBytes; noalloc_scratch returns its address on
// `device` (looked up once per device). stash_descriptors enqueues kernels on
// `stream` that write `bytes` (a multiple of 16) from host memory `src` to
// `dst` in that array, carrying them in their kernel arguments.
constexpr size_t kNoAllocScratchBytes = 256 * 1024;
uint8_t* noalloc_scratch(int device);
void stash_descriptors(const void* src, size_t bytes, uint8_t* dst, hipStream_t stream);

// One call's use of a GPU's scratch array. The constructor takes the device's
// call lock and, when the previous eager call used another stream, makes
// `stream` wait for that call's last kernel; finish() is called after the
// call's last launch that reads the array and records the device's event on
// `stream`. Under stream capture neither the wait nor the record is made.
struct ScratchState;
class ScratchUse {
public:
    ScratchUse(int device, hipStream_t stream);
    // A call that stops before finish() (an error after some of its kernels
    // were enqueued) still records the event, so that later calls order
    // after whatever it enqueued.
    ~ScratchUse();
    ScratchUse(const ScratchUse&) = delete;
    ScratchUse& operator=(const ScratchUse&) = delete;
    uint8_t* ptr() const;
    void finish();

private:
    ScratchState* state_;
    hipStream_t stream_;
    std::unique_lock<std::mutex> lock_;
    bool capture_ = false;
    bool finished_ = false;
};
// Cross-stream waits ScratchUse has enqueued since the library was loaded.
int64_t scratch_stream_waits();

// Launch-configuration error check after a <<<>>> launch.
void check_launch(const char* what);

}  // namespace daric
