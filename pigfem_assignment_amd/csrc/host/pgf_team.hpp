// Shares of a system's rows for the blocks of a PCG team (kernels/pgf_team.hpp).
#pragma once

#include <cstdint>
#include <vector>

namespace pgft {

struct GroupRec {  // up to dim consecutive free rows with one column list
    int32_t row, begin, len_k, stride;  // first row, its first entry, columns << 2 | rows, entries per row
};

// Team blocks have TEAM_THREADS threads; TEAM_LANES(dim) of them serve a group
// together, each taking up to TEAM_COLS of its columns in one step.
constexpr int TEAM_THREADS = 512, TEAM_COLS = 3;
constexpr int team_lanes(int dim) { return dim == 3 ? 16 : 8; }

// One step of a lane group: up to TEAM_COLS * lanes columns of a row group.
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
    int max_rows = 0, max_passes = 0, max_window = 0;
};

// Shares with about equal numbers of steps (the passes of a block follow from
// them); grp has one record past the last group (its row is the row count);
// system s owns the groups [sys_grp[s], sys_grp[s+1]).  The steps and halos are
// found in parallel over the shares.
void make_team_plan(int dim, const std::vector<GroupRec>& grp, const std::vector<int64_t>& sys_grp, const int32_t* colidx,
                    int blocks, TeamPlan& plan);

}  // namespace pgft
