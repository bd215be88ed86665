// Shares, steps and halos of the PCG teams.
#include "pgf_team.hpp"

#include <algorithm>
#include <exception>
#include <omp.h>

namespace pgft {

bool make_team_plan(int dim, const std::vector<GroupRec>& grp, const std::vector<SysGroups>& sys, const int32_t* colidx,
                    int blocks, int64_t fit_window, TeamPlan& plan) {
    const int n_sys = (int)sys.size();
    plan = TeamPlan();
    plan.blocks = blocks;
    plan.part.reserve((size_t)n_sys * (blocks + 1));
    const int lg = TEAM_THREADS / team_lanes(dim), cols = team_cols(dim) * team_lanes(dim);
    auto cost = [&](int64_t g) { return (int64_t)std::max(1, ((grp[g].len_k >> 2) + cols - 1) / cols); };
    for (int s = 0; s < n_sys; ++s) {
        const int64_t hi = sys[s].hi;
        int64_t g = sys[s].lo, total = 0, run = 0;
        for (int64_t i = g; i < hi; ++i) total += cost(i);
        for (int k = 0; k <= blocks; ++k) {
            const int64_t upto = 2 * (total / blocks * k + total % blocks * k / blocks);
            while (g < hi && (k == blocks || 2 * run + cost(g) <= upto)) run += cost(g++);
            plan.part.push_back((int32_t)g);
        }
    }
    const int n_shares = n_sys * blocks;
    plan.row_ptr.resize(plan.part.size());
    for (size_t i = 0; i < plan.part.size(); ++i) plan.row_ptr[i] = grp[plan.part[i]].row;
    int64_t sys_rows = 0;
    for (const SysGroups& s : sys) sys_rows = std::max<int64_t>(sys_rows, grp[s.hi].row - grp[s.lo].row);
    // a share's window is no smaller than its rows
    plan.sys_window.assign(n_sys, 0);
    bool fits = true;
    for (size_t i = 1; i < plan.row_ptr.size(); ++i)
        if (i % (blocks + 1) != 0) {
            int32_t& w = plan.sys_window[i / (blocks + 1)];
            w = std::max(w, plan.row_ptr[i] - plan.row_ptr[i - 1]);
            fits = fits && w <= fit_window;
        }
    if (!fits) return false;
    std::vector<int32_t> share_window(n_shares);
    std::vector<std::vector<int32_t>> found(n_shares);
    std::vector<std::vector<StepRec>> steps(n_shares);
    int rows = 0, passes = 0, window = 0;
    // an exception must not leave a parallel region: the first is thrown on behind it
    std::exception_ptr failed;
#pragma omp parallel num_threads(std::min(omp_get_max_threads(), 16)) reduction(max : rows, passes, window)
    {
        // the share that last met each column of its system, per thread
        std::vector<int32_t> seen;
#pragma omp for schedule(dynamic, 4)
        for (int k = 0; k < n_shares; ++k) try {
            if (seen.empty()) seen.assign((size_t)sys_rows, -1);
            const int32_t* pt = &plan.part[(size_t)(k / blocks) * (blocks + 1) + k % blocks];
            const int32_t r0 = grp[pt[0]].row, r1 = grp[pt[1]].row, first = grp[sys[k / blocks].lo].row;
            rows = std::max(rows, r1 - r0);
            // longest groups first, each to the lane group with the fewest
            // steps, the next one in order among equals: few passes, and
            // neighbours stay side by side
            std::vector<StepRec>& st = steps[k];
            std::vector<int> used(lg, 0);
            int at = 0, most = 1;
            for (int32_t g = pt[0]; g < pt[1]; ++g) most = std::max(most, (int)cost(g));
            for (int n = most; n >= 1; --n)
                for (int32_t g = pt[0]; g < pt[1]; ++g) {
                    if (cost(g) != n) continue;
                    int best = at;
                    for (int i = 1; i < lg; ++i) {
                        const int s = (at + i) % lg;
                        if (used[s] < used[best]) best = s;
                    }
                    at = (best + 1) % lg;
                    const int len = grp[g].len_k >> 2;
                    if ((size_t)(used[best] + n) * lg > st.size()) st.resize((size_t)(used[best] + n) * lg, StepRec{0, 0, 0, 0});
                    for (int s = 0; s < n; ++s)
                        st[(size_t)(used[best] + s) * lg + best] =
                            StepRec{grp[g].begin + s * cols, grp[g].row - r0, grp[g].stride,
                                    std::min(cols, len - s * cols) | (grp[g].len_k & 3) << 8 | (s ? STEP_CONT : 0) |
                                        (s + 1 == n ? STEP_LAST : 0)};
                    used[best] += n;
                }
            passes = std::max(passes, (int)(st.size() / lg));
            std::vector<int32_t>& h = found[k];
            for (int32_t g = pt[0]; g < pt[1]; ++g)
                for (const int32_t *c = colidx + grp[g].begin, *e = c + (grp[g].len_k >> 2); c < e; ++c)
                    if ((*c < r0 || *c >= r1) && seen[*c - first] != k) {
                        seen[*c - first] = k;
                        h.push_back(*c);
                    }
            std::sort(h.begin(), h.end());
            share_window[k] = r1 - r0 + (int32_t)h.size();
            window = std::max(window, share_window[k]);
        } catch (...) {
#pragma omp critical(pgf_team_plan)
            if (!failed) failed = std::current_exception();
        }
    }
    if (failed) std::rethrow_exception(failed);
    plan.max_rows = rows;
    plan.max_passes = passes;
    plan.max_window = window;
    for (int k = 0; k < n_shares; ++k)
        plan.sys_window[k / blocks] = std::max(plan.sys_window[k / blocks], share_window[k]);
    if (window > fit_window) return false;
    plan.halo_ptr.assign(n_shares + 1, 0);
    for (int k = 0; k < n_shares; ++k) plan.halo_ptr[k + 1] = plan.halo_ptr[k] + (int64_t)found[k].size();
    plan.step_ptr.assign(n_shares + 1, 0);
    for (int k = 0; k < n_shares; ++k) plan.step_ptr[k + 1] = plan.step_ptr[k] + (int64_t)steps[k].size() / lg;
    plan.halo.resize((size_t)plan.halo_ptr[n_shares]);
    plan.steps.resize((size_t)plan.step_ptr[n_shares] * lg);
#pragma omp parallel for schedule(static)
    for (int k = 0; k < n_shares; ++k) {
        std::copy(found[k].begin(), found[k].end(), plan.halo.begin() + plan.halo_ptr[k]);
        std::copy(steps[k].begin(), steps[k].end(), plan.steps.begin() + plan.step_ptr[k] * lg);
    }
    return true;
}

}  // namespace pgft
