// Host tables of the field histogram: what is copied to the start of the
// caller's workspace, what the kernels add behind it, and which form counts.
// Plain C++, so that it can be checked without a device.
#ifndef MXB_FIELD_PLAN_H
#define MXB_FIELD_PLAN_H

#include <algorithm>
#include <cmath>
#include <cstdint>
#include <vector>

namespace mxb {

// Bytes of a field histogram's workspace beside 4 per voxel coordinate of each axis.
constexpr int64_t kFieldHistWorkspace = 2 * 65536 * 4;
inline int64_t field_workspace_bytes(int64_t nZ, int64_t nY, int64_t nX) {
    return kFieldHistWorkspace + (nZ + nY + nX) * 4 + 256;
}

constexpr int64_t kGroupCells = 32768;   // 32-bit counters of a block's table (128 KB)
constexpr int64_t kMaxGroups = 2048;
constexpr int64_t kMaxBricks = 49152;    // 192 KB of ranges in the workspace
constexpr int64_t kMaxBox = 512;         // voxels per field value

// `words` holds the field coordinate of every voxel coordinate (z, y, x axis
// after axis) and, for the grouped form, then the first voxel coordinate of
// every segment, and the extent.  A segment is a run of voxel coordinates with
// one field coordinate.  The grouped form goes on with ng + 1 bounds, ng + 2
// starts and the bricks' ranges.
struct FieldPlan {
    std::vector<int32_t> words;
    int64_t ns[3] = {0, 0, 0}, width[3] = {0, 0, 0};  // segments, the widest
    bool grouped = false;
    int64_t G = 0, ng = 0;                    // field bins per group, groups
    int64_t nb[3] = {0, 0, 0}, bricks = 0;    // bricks along each axis, and in all
    int lb[3] = {3, 3, 4};                    // log2 of brick edges (x at least 16)

    // Words of the workspace in use, once the plan is made.
    int64_t table_words() const {
        return (int64_t)words.size() + (grouped ? 2 * ng + 3 + bricks : 0);
    }
};

// The plan of n voxels (z, y, x) against a field of nf, fb x vb bins.
// `monotone`: the field's bins rise with its values, and both maps take the
// fast division.
inline void make_field_plan(const int64_t n[3], const int64_t nf[3], int64_t fb, int64_t vb, bool monotone,
                            FieldPlan &p) {
    std::vector<int32_t> &words = p.words;
    const int64_t nmaps = n[0] + n[1] + n[2];
    words.clear();
    for (int k = 0; k < 3; ++k) {
        const double d = (double)nf[k] / (double)n[k];  // histograms.cc:246-249, :284-287
        for (int64_t i = 0; i < n[k]; ++i)
            words.push_back((int32_t)std::min<int64_t>(nf[k] - 1, (int64_t)std::floor((double)i * d)));
    }
    // runs of equal field coordinates
    auto segments = [&](int k, int64_t at, auto &&begins) {
        for (int64_t i = 0; i < n[k]; ++i)
            if (i == 0 || words[at + i] != words[at + i - 1]) begins(i);
    };
    const int64_t first[3] = {0, n[0], n[0] + n[1]};
    for (int k = 0; k < 3; ++k) {
        int64_t from = 0;
        segments(k, first[k], [&](int64_t i) {
            p.width[k] = std::max(p.width[k], i - from);
            from = i;
            ++p.ns[k];
        });
        p.width[k] = std::max(p.width[k], n[k] - from);
    }
    // The grouped form: every field coordinate is sampled (the segments are the
    // field's coordinates), the tables fit the workspace, a group holds at least one row
    // of bins, and bins are monotone in the value.
    p.G = std::min<int64_t>(2047, std::min(fb, kGroupCells / vb));
    p.grouped = p.G >= 1 && (fb + p.G - 1) / p.G <= kMaxGroups && p.width[0] * p.width[1] * p.width[2] <= kMaxBox &&
                monotone && nmaps <= 40000;
    for (int k = 0; k < 3; ++k) p.grouped = p.grouped && p.ns[k] == nf[k] && nf[k] <= 8192;  // brick numbers of 11, 10 and 11 bits
    // bricks: 16 x 8 x 8 field values, doubled along the shortest edge (in
    // voxels) until the table of ranges fits
    while (p.grouped) {
        p.bricks = 1;
        for (int k = 0; k < 3; ++k) {
            p.nb[k] = (nf[k] + (int64_t(1) << p.lb[k]) - 1) >> p.lb[k];
            p.bricks *= p.nb[k];
        }
        if (p.bricks <= kMaxBricks) break;
        int best = 0;
        for (int k = 1; k < 3; ++k)
            if ((p.width[k] << p.lb[k]) < (p.width[best] << p.lb[best])) best = k;
        if (++p.lb[best] > 7) p.grouped = false;
    }
    if (!p.grouped) return;
    p.ng = (fb + p.G - 1) / p.G;
    // the segments' starts, which only this form reads: for long axes they would
    // not fit the workspace beside the maps
    for (int k = 0; k < 3; ++k) {
        segments(k, first[k], [&](int64_t i) { words.push_back((int32_t)i); });
        words.push_back((int32_t)n[k]);
    }
}

}  // namespace mxb

#endif  // MXB_FIELD_PLAN_H
