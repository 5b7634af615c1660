// How the fused prefill kernels (m3_ssd_wide.hip, m3_ssd_f32.hip) cut sequences into segments, and
// what of a call a workspace holds at a time. Host arithmetic, but for seg_start.
#pragma once

#include <algorithm>
#include <cstddef>
#include <cstdint>

#include <hip/hip_runtime.h>

namespace m3 {

// First token of segment i: four segments each of seg0, 2 seg0 and 4 seg0 tokens, then 16 seg0.
__host__ __device__ inline int64_t seg_start(int i, int seg0) {
    const int u = i <= 4 ? i : i <= 8 ? 4 + 2 * (i - 4) : i <= 12 ? 12 + 4 * (i - 8) : 28 + 16 * (i - 12);
    return (int64_t)u * seg0;
}

// Segments of a sequence. The first cut is free, as the state at it is the walk's own: up to two
// segments a sequence is walked in one piece, with the same bits.
inline int seg_count(int64_t seqlen, int seg0) {
    if (seqlen <= 2 * seg0) return 1;
    int n = 1;
    while (seg_start(n, seg0) < seqlen) ++n;
    return n;
}

inline size_t al256(size_t n) { return (n + 255) & ~(size_t)255; }

// Bytes of one sequence: its B^ (and C^) rows, one segment's state, log-decay, angle increments.
struct SegSizes {
    size_t rows, state, decay, angle;
};

// Workspace: B^ and C^ rows, then the segments' states, log-decays and angle increments.
struct SegPlan {
    int segs;
    int batch;         // sequences per slice
    int slots, group;  // states kept, segments per group of launches
    size_t rows, hseg, lseg, aseg, total;  // bytes of B^ (and of C^); offsets; bytes in all
};

inline void seg_layout(SegPlan& p, const SegSizes& z) {
    const size_t n = p.segs - 1, b = p.batch;
    p.rows = al256(b * z.rows);
    p.hseg = 2 * p.rows;
    p.lseg = p.hseg + (n ? al256(p.slots * b * z.state) : 0);
    p.aseg = p.lseg + al256(n * b * z.decay);
    p.total = p.aseg + al256(n * b * z.angle);
}

// The plan of a call in `limit` bytes. A workspace that does not hold every segment's state takes
// the batch in slices (where the caller can: `slice`), and one that does not hold those of one
// slice takes its segments in groups, from two states on: the same arithmetic in more launches.
// Below that the sequences are walked in one piece, which moves their results by rounding.
inline SegPlan plan_segments(int batch, int segs, const SegSizes& z, size_t limit, bool slice) {
    SegPlan p;
    p.segs = p.group = segs;
    p.batch = batch;
    p.slots = std::max(segs - 1, 1);
    seg_layout(p, z);
    if (segs == 1 || p.total <= limit) return p;
    if (slice) {
        // the sequences of a slice, give or take alignment
        p.batch = std::min(batch, 1 + (int)((double)limit / p.total * batch));
        seg_layout(p, z);
        while (p.batch > 1 && p.total > limit) {
            --p.batch;
            seg_layout(p, z);
        }
    }
    while (p.slots > 2 && p.total > limit) {
        --p.slots;
        p.group = p.slots - 1;
        seg_layout(p, z);
    }
    if (p.total > limit) {
        p.segs = p.slots = p.group = 1;
        p.batch = batch;
        seg_layout(p, z);
    }
    return p;
}

}  // namespace m3
