// How the grid form's workgroups cut the column ranges of their row blocks into segments.  Plain integer
// arithmetic, the same on the device and on the host.
#pragma once

namespace km {

#define KM_GROUP 4                /* row blocks, and wavefronts, of a workgroup */
#define KM_GROUP_CORE_SHARED 256  /* columns of the core beyond which all wavefronts take a piece */
// Lanes of the plan: the segments whose sums the row blocks add (the first cell in halves, two cells, the core,
// whole or in halves, two cells, the last cell in halves), the wavefronts' pieces of a shared core, the row blocks.
#define KM_GROUP_SEGMENTS 10
#define KM_GROUP_CORE 4
#define KM_GROUP_PIECE 10
#define KM_GROUP_ROW 14

struct GroupCut {
    int segment[KM_GROUP_SEGMENTS + 1];  // segment i: the columns [segment[i], segment[i + 1])
    int piece[KM_GROUP + 1];             // the same of a shared core's pieces
    bool shared;
};

// Half of the columns [from, to), in whole steps of 32 where there are as many.
constexpr int group_half(int from, int to) { return ((to - from + 1) / 2 + 31) & ~31; }

// The segments between the ends of the ranges, at[] in ascending order.  Every bound lies within its cell: a quarter
// of the core in whole steps, three times, is more than the core where that has 260 to 287 columns.
constexpr GroupCut group_cut(const int (&at)[2 * KM_GROUP]) {
    static_assert(KM_GROUP == 4, "eight ends of ranges");
    const int core = at[4] - at[3];
    const bool shared = core > KM_GROUP_CORE_SHARED;
    const int from_first = at[1] - group_half(at[0], at[1]);
    const int in_core = at[3] + group_half(at[3], at[4]);
    const int from_last = at[6] + group_half(at[6], at[7]);
    GroupCut c = {{at[0], from_first > at[0] ? from_first : at[0], at[1], at[2], at[3], shared || in_core > at[4] ? at[4] : in_core,
                   at[4], at[5], at[6], from_last < at[7] ? from_last : at[7], at[7]},
                  {at[3], at[4], at[4], at[4], at[4]},
                  shared};
    const int quarter = (core / KM_GROUP + 31) & ~31;
    for (int i = 1; i < KM_GROUP; i++) {
        c.piece[i] = core > i * quarter ? at[3] + i * quarter : at[4];
    }
    return c;
}

// The row blocks whose range holds the columns [start, end), as bits; ends[]: the starts of the ranges, then
// their ends.  No columns: none.
constexpr int group_rows(const int (&ends)[2 * KM_GROUP], int start, int end) {
    int rows = 0;
    for (int r = 0; r < KM_GROUP; r++) {
        rows |= ends[r] <= start && end <= ends[KM_GROUP + r] && start < end ? 1 << r : 0;
    }
    return rows;
}

}  // namespace km
