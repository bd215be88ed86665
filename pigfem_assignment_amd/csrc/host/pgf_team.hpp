// Shares of a system's rows for the blocks of a PCG team (kernels/pgf_team.hpp).
#pragma once

#include <cstdint>
#include <vector>

namespace pgft {

struct GroupRec {  // up to dim consecutive free rows with one column list
    int32_t row, begin, len_k, stride;  // first row, its first entry, columns << 2 | rows, entries per row
};

// Team blocks have TEAM_THREADS threads; team_lanes(dim) of them serve a group
// together, each taking up to team_cols(dim) of its columns in one step: a
// regular node's row group (18 columns in 2D, 45 in 3D) is one step.
constexpr int TEAM_THREADS = 512;
constexpr int team_lanes(int dim) { return dim == 3 ? 16 : 4; }
constexpr int team_cols(int dim) { return dim == 3 ? 3 : 5; }

// One step of a lane group: up to lanes * columns of a row group.
// Longer groups take consecutive steps of the same lane group, which carries
// its sums from the first to the last.
struct StepRec {
    int32_t begin, row, stride;  // first entry (in the group's first row), row in the share, entries per row
    int32_t what;                // columns | rows << 8 | STEP_CONT | STEP_LAST; 0: nothing to do
};
constexpr int32_t STEP_CONT = 1 << 10, STEP_LAST = 1 << 11;

struct TeamPlan {
    int blocks = 0;                      // per team
    std::vector<int32_t> part;           // [systems][blocks + 1] first group of each block's share
    std::vector<int32_t> row_ptr;        // [systems][blocks + 1] first row of each block's share
    std::vector<int64_t> step_ptr;       // [systems * blocks + 1] first pass of each share (lane groups per block wide)
    std::vector<StepRec> steps;
    std::vector<int64_t> halo_ptr;       // [systems * blocks + 1]
    std::vector<int32_t> halo;           // ascending columns outside a share's rows
    std::vector<int32_t> sys_window;     // largest window of each system's shares
    int max_rows = 0, max_passes = 0, max_window = 0;
};

// A system's groups [lo, hi) of a batch (or all groups); its columns are its
// own rows.
struct SysGroups {
    int64_t lo, hi;
};

// Shares with about equal numbers of steps (the passes of a block follow from
// them); grp has one record past the last group (its row is the row count).
// The steps and halos are found in parallel over the shares.  False, and no
// plan but its sys_window, where a share has a window of more than fit_window
// columns.
bool make_team_plan(int dim, const std::vector<GroupRec>& grp, const std::vector<SysGroups>& sys, const int32_t* colidx,
                    int blocks, int64_t fit_window, TeamPlan& plan);

}  // namespace pgft
