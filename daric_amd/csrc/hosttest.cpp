// Host-only hooks for the CPU test suite: the scalar element conversions and
// the fast divider that the kernels use, compiled for the host from the same
// headers. Not part of the product ABI (include/daric_cache_ops.h).
#include <cstdint>
#include <vector>

#include "elem.h"
#include "kernels.h"

extern "C" {

uint32_t daric_hosttest_f32_to_bf16(float f) { return daric::f32_to_bf16(f); }
uint32_t daric_hosttest_f32_to_f16(float f) { return daric::f32_to_f16(f); }
uint32_t daric_hosttest_f32_to_e4m3(float f) { return daric::f32_to_e4m3(f); }
float daric_hosttest_e4m3_to_f32(uint32_t c) { return daric::e4m3_to_f32(c); }

// Encodes n floats into out (uint8 codes).
void daric_hosttest_encode_e4m3(const float* in, uint8_t* out, int64_t n) {
    for (int64_t i = 0; i < n; ++i) out[i] = static_cast<uint8_t>(daric::f32_to_e4m3(in[i]));
}
void daric_hosttest_encode_bf16(const float* in, uint16_t* out, int64_t n) {
    for (int64_t i = 0; i < n; ++i) out[i] = static_cast<uint16_t>(daric::f32_to_bf16(in[i]));
}

// out[i * n_x + j] = the quantising writes' quotient of x[j] by scales[i].
void daric_hosttest_quant_quotients(const float* x, int64_t n_x, const float* scales, int64_t n_s,
                                    float* out) {
    for (int64_t i = 0; i < n_s; ++i) {
        const daric::QuantDiv d = daric::quant_div(scales[i]);
        for (int64_t j = 0; j < n_x; ++j) out[i * n_x + j] = daric::quant_quotient(d, x[j]);
    }
}

// Returns the number of n in [n0, n1) for which FastDiv(d).div(n) != n / d.
int64_t daric_hosttest_fastdiv_errors(uint32_t d, uint32_t n0, uint32_t n1) {
    const daric::FastDiv f(d);
    int64_t bad = 0;
    for (uint64_t n = n0; n < n1; ++n)
        if (f.div(static_cast<uint32_t>(n)) != static_cast<uint32_t>(n) / d) ++bad;
    return bad;
}


// Walks the launches for_layer_minor makes for n_layers x n_items and
// decodes every block with LayerMinor::at_block. Returns the number of
// launches when every (layer, item) pair is covered exactly once and no
// launch exceeds kMaxGridBlocks, else -1 (a pair missed, repeated or out of
// range) or -2 (an oversized launch).
int64_t daric_hosttest_layer_minor(int n_layers, int64_t n_items) {
    std::vector<uint8_t> seen(static_cast<size_t>(n_layers) * static_cast<size_t>(n_items), 0);
    int64_t launches = 0;
    bool bad = false, big = false;
    daric::for_layer_minor(n_layers, n_items, [&](const daric::LayerMinor& lm, unsigned blocks) {
        ++launches;
        if (static_cast<int64_t>(blocks) > daric::kMaxGridBlocks || blocks == 0) big = true;
        for (uint32_t b = 0; b < blocks; ++b) {
            int l;
            int64_t w;
            lm.at_block(b, l, w);
            if (l < 0 || l >= n_layers || w < 0 || w >= n_items) { bad = true; continue; }
            uint8_t& s = seen[static_cast<size_t>(l) * static_cast<size_t>(n_items) + static_cast<size_t>(w)];
            if (s) bad = true;
            s = 1;
        }
    });
    for (uint8_t s : seen)
        if (!s) bad = true;
    if (big) return -2;
    return bad ? -1 : launches;
}

// Walks the launches for_job_runs (gather 0) or for_job_rows (gather 1) makes for
// jobs of tiles[i] tiles of `parts` units, ordered by order_jobs, and decodes
// every block. Returns the number of launches when every unit of every job is
// taken by exactly one block, every job lies in its launch and no launch exceeds
// kMaxGridBlocks, else -1 or -2 (an oversized launch). *log2_run gets the last
// launch's run length, *idle the blocks that no unit of a job answers to.
int64_t daric_hosttest_job_grid(int gather, const int64_t* tiles, int64_t n, int64_t parts, int64_t unit_bytes,
                                int64_t runs_from, int32_t* log2_run, int64_t* idle) {
    struct Job { int64_t id, tiles; };
    std::vector<Job> jobs;
    for (int64_t i = 0; i < n; ++i) jobs.push_back({i, tiles[i]});
    const daric::JobClasses classes = daric::order_jobs(jobs, [](const Job& j) { return j.tiles; });
    std::vector<std::vector<uint8_t>> seen(static_cast<size_t>(n));
    for (int64_t i = 0; i < n; ++i) seen[static_cast<size_t>(i)].assign(static_cast<size_t>(tiles[i] * parts), 0);
    int64_t launches = 0;
    bool bad = false, big = false;
    *idle = 0;
    int64_t at = 0;
    for (int k = 0; k < classes.n; ++k) {    // longest class first, the jobs of a class in their order
        for (int64_t i = at; i < at + classes[k].jobs; ++i) {
            const int64_t t = jobs[static_cast<size_t>(i)].tiles;
            if (t > classes[k].tiles || t <= 0 || (i > at && jobs[static_cast<size_t>(i)].id < jobs[static_cast<size_t>(i - 1)].id)) bad = true;
        }
        at += classes[k].jobs;
        if (k > 0 && classes[k].tiles >= classes[k - 1].tiles) bad = true;
    }
    for (int64_t i = at; i < n; ++i) bad = bad || jobs[static_cast<size_t>(i)].tiles != 0;
    const auto walk = [&](int j0, const auto& g, unsigned blocks) {
        ++launches;
        *log2_run = static_cast<int32_t>(g.log2_run);
        if (static_cast<int64_t>(blocks) > daric::kMaxGridBlocks || blocks == 0) big = true;
        for (uint32_t b = 0; b < blocks; ++b) {
            int job, unit;
            g.at_block(b, job, unit);
            if (job < 0 || j0 + job >= n || unit < 0) { bad = true; continue; }
            const Job& j = jobs[static_cast<size_t>(j0 + job)];
            if (unit >= j.tiles * parts) { ++*idle; continue; }   // the kernels' tile check drops it
            uint8_t& s = seen[static_cast<size_t>(j.id)][static_cast<size_t>(unit)];
            if (s) bad = true;
            s = 1;
        }
    };
    if (gather) daric::for_job_rows(classes, parts, unit_bytes, walk);
    else daric::for_job_runs(classes, parts, unit_bytes, runs_from, walk);
    for (const auto& v : seen)
        for (uint8_t s : v)
            if (!s) bad = true;
    if (big) return -2;
    return bad ? -1 : launches;
}

void daric_hosttest_store_unit_head(uint8_t* dst, const uint32_t* words, int n) {
    daric::store_unit_head(dst, words, n);
}

int64_t daric_hosttest_token_row_part(int64_t page_tokens, int64_t tok_bytes, int vw, int64_t pages) {
    return daric::token_row_part(page_tokens, tok_bytes, vw, pages);
}

int daric_hosttest_topk_slots(int n, int lanes) { return daric::topk_slots(n, lanes); }

// Units (parts of tiles) that a page copy of one call has for jobs of tiles[i]
// tiles of span[i] bytes: units[i], in the order of the arguments.
// Returns the longest unit's bytes.
int64_t daric_hosttest_page_units(const int64_t* tiles, const int64_t* span, int64_t n, int vw, int64_t* units) {
    std::vector<daric::CopyJob> jobs(static_cast<size_t>(n));
    for (int64_t i = 0; i < n; ++i) {
        daric::CopyJob& j = jobs[static_cast<size_t>(i)];
        j.prefix = 1;
        j.n_sel = static_cast<int32_t>(tiles[i]);
        j.span = static_cast<int32_t>(span[i]);
        j.n_tokens = static_cast<int32_t>(i);
    }
    int64_t part;
    daric::cut_pages(jobs, vw, &part);
    for (const daric::CopyJob& j : jobs) units[j.n_tokens] = static_cast<int64_t>(j.n_sel) * j.parts.d;
    return part;
}

int daric_hosttest_copy_lanes(int64_t unit_bytes, int vw) { return daric::copy_lanes(unit_bytes, vw); }

int64_t daric_hosttest_page_part_bytes(int64_t max_span, int64_t tiles) {
    return daric::page_part_bytes(max_span, tiles);
}

// The batches that the row merge makes of chunks of n_tokens[i] tokens and k[i]
// slots: begin[i] and, as return value, their number; *each as MergeBatches has it.
int64_t daric_hosttest_merge_batches(const int32_t* n_tokens, const int32_t* k, int64_t n, int64_t kmax, int rows,
                                     int top_k, int32_t* begin, int64_t* each) {
    std::vector<daric::SelChunk> chunks(static_cast<size_t>(n));
    for (size_t i = 0; i < chunks.size(); ++i) {
        chunks[i].n_tokens = n_tokens[i];
        chunks[i].k = k[i];
    }
    const daric::MergeBatches b = daric::merge_batches(chunks, kmax, rows, top_k != 0);
    for (size_t i = 0; i < chunks.size(); ++i) begin[i] = chunks[i].tile_begin;
    *each = b.each;
    return b.n;
}

int64_t daric_hosttest_direct_desc_bytes(int gather, int64_t unit_bytes) {
    return static_cast<int64_t>(daric::direct_desc_bytes(gather != 0, unit_bytes));
}

int64_t daric_hosttest_fused_runs_from(int64_t unit_bytes) { return daric::fused_runs_from(unit_bytes); }

// Splits one job (split_long_jobs) and lists, for every tile of the pieces in
// order, the page span it takes: place in the layer before the page id, place in
// staging, place in the id list and tokens it rotates (-1: copied). Returns the
// tiles, or -1 where a piece has more units than a launch holds.
int64_t daric_hosttest_split_job(int prefix, int n_sel, int64_t prefix_stride, int span, int n_tokens, int64_t parts,
                                 int64_t page_tokens, int64_t* out, int64_t cap) {
    uint8_t base[1];
    const int32_t ids[1] = {0};
    daric::CopyJob j{};
    j.layer = base;
    j.stage = base;
    j.idx = ids;
    j.prefix = prefix;
    j.n_sel = n_sel;
    j.prefix_stride = prefix_stride;
    j.span = span;
    j.n_tokens = n_tokens;
    j.delta = 3.0f;
    std::vector<daric::CopyJob> jobs(3, j);
    jobs[0].n_sel = jobs[2].n_sel = 1;
    jobs[0].prefix = jobs[2].prefix = 1;
    daric::split_long_jobs(jobs, parts, page_tokens);
    if (jobs.front().n_sel != 1 || jobs.back().n_sel != 1) return -2;
    int64_t n = 0;
    for (size_t i = 1; i + 1 < jobs.size(); ++i) {
        const daric::CopyJob& q = jobs[i];
        if (static_cast<int64_t>(q.prefix) * q.n_sel * parts > daric::kMaxGridBlocks) return -1;
        for (int64_t t = 0; t < static_cast<int64_t>(q.prefix) * q.n_sel && n < cap; ++t, ++n) {
            const int64_t p = t / q.n_sel, s = t % q.n_sel;
            out[4 * n] = reinterpret_cast<intptr_t>(q.layer) - reinterpret_cast<intptr_t>(base) + p * q.prefix_stride;
            out[4 * n + 1] = reinterpret_cast<intptr_t>(q.stage) - reinterpret_cast<intptr_t>(base) + t * q.span;
            out[4 * n + 2] = (reinterpret_cast<intptr_t>(q.idx) - reinterpret_cast<intptr_t>(ids)) / 4 + s;
            const int64_t left = q.n_tokens - s * page_tokens;
            out[4 * n + 3] = p == 0 && q.delta != 0.0f && left > 0 ? (left < page_tokens ? left : page_tokens) : -1;
        }
    }
    return n;
}

}
