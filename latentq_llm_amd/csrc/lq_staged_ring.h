// Which groups of 128 k a workgroup of the staged forward kernel (lq_gemm_staged.hip) works on, stage by stage, and the LDS ring
// that holds their scales and zeros. Arithmetic only: the host test walks it through every slice of a row.
#pragma once

constexpr int kStagedStages = 3;  // LDS stages: stage u + 2 is requested during stage u

// Groups first .. end - 1 of a row, a stage being a pair of them or (pairs = false) one
struct StagedSlice {
    int first, end;
    bool pairs;

    constexpr int groups() const { return end - first; }
    // pairs of groups; the last of an odd number begins a group earlier, and only its second group is new
    constexpr int pair_start(int j) const {
        const int g = first + 2 * j < end - 2 ? first + 2 * j : end - 2;
        return g > 0 ? g : 0;
    }
    constexpr int units() const { return pairs ? (groups() + 1) / 2 : groups(); }  // stages of the workgroup,
    constexpr int units_of(int kg) const { return pairs && kg == 0 ? groups() / 2 : units(); }  // and of the waves that take the kg-th group of a pair
    constexpr int group_of(int u, int kg) const { return pairs ? pair_start(u) + kg : first + u; }
    constexpr int last_group(int u) const { return pairs ? (first + 2 * u + 1 < end ? first + 2 * u + 1 : end - 1) : first + u; }
};

// Pieces of 2^q_log groups' values. In the interval between two barriers in which stage u's values are read, group
// first + 2 u on, the pieces up to stage u + 2's are requested, group first + 2 u + 5 with pairs: six groups, which are parts of up to
// three pieces of four, two of eight, or six of one. The slots hold that many: with two slots for pieces of four the third piece
// would take the place of one that a slower wave has yet to read. (One group per stage: three groups, two pieces of four.)
struct ScaleRing {
    int q_log;
    bool pairs;

    constexpr int piece(int g) const { return g >> q_log; }
    constexpr unsigned slot(int piece) const { return (unsigned)piece & (q_log ? (pairs ? 3u : 1u) : 7u); }
    static constexpr int bytes(bool pairs) { return pairs ? 4 * 4096 : 2 * 4096; }  // slots of 4 KB, or of 1 KB for single groups
};
