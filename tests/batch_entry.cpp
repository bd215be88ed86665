// Calls pgf_batch_pcg where no GPU is visible, on a context made by hand: what
// the C entry does when memory of the host or the device runs out, and what it
// does again on a repeated call.
//   batch_entry workspace        teams laid out already, the solve's device memory fails
//   batch_entry plan BYTES       one system of 400 x 400 rows, host blocks of BYTES or more fail
//   batch_entry unfit            a system of 800 x 800 rows, four right-hand sides: fits no team; twice
// Prints the status and the host bytes that each call allocated, or dies of an
// exception that leaves the entry.
#include <atomic>
#include <cstdio>
#include <cstdlib>
#include <cstring>
#include <new>

#include "../include/pgfem.h"
#include "../pigfem_assignment_amd/csrc/kernels/pgf_device.hpp"

static size_t g_limit = ~(size_t)0;
static std::atomic<size_t> g_bytes{0};
void* operator new(size_t n) {
    g_bytes += n;
    void* p = n >= g_limit ? nullptr : std::malloc(n);
    if (!p) throw std::bad_alloc();
    return p;
}
void operator delete(void* p) noexcept { std::free(p); }
void operator delete(void* p, size_t) noexcept { std::free(p); }

struct pgf_ctx : public pgfd::Ctx {};

// n x n rows in groups of one, each with its neighbours in the grid
static void grid_pattern(pgf_ctx& c, int n) {
    c.dim = 2;
    c.n_free = c.n_rows = (int64_t)n * n;
    c.n_cu = 256;
    c.h_rowptr.push_back(0);
    for (int r = 0; r < n * n; ++r) {
        const int b = (int)c.h_colidx.size(), y = r / n, x = r % n;
        for (int j = std::max(y - 1, 0); j <= std::min(y + 1, n - 1); ++j)
            for (int i = std::max(x - 1, 0); i <= std::min(x + 1, n - 1); ++i) c.h_colidx.push_back(j * n + i);
        const int len = (int)c.h_colidx.size() - b;
        c.h_rowsplit.push_back(len);
        c.h_rowptr.push_back((int64_t)c.h_colidx.size());
        c.h_grp.push_back(pgft::GroupRec{r, b, len << 2 | 1, len});
    }
    c.n_grp = (int64_t)c.h_grp.size();
    c.h_grp.push_back(pgft::GroupRec{n * n, 0, 0, 0});
    c.nnz = (int64_t)c.h_colidx.size();
}

int main(int argc, char** argv) {
    pgf_ctx* c = new pgf_ctx();
    const char* mode = argc > 1 ? argv[1] : "";
    const bool unfit = !std::strcmp(mode, "unfit");
    const int n = !std::strcmp(mode, "workspace") ? 4 : unfit ? 800 : 400, nrhs = unfit ? 4 : 1;
    grid_pattern(*c, n);
    const int64_t sys[2] = {0, c->n_free};
    double* b = (double*)std::calloc((size_t)n * n * nrhs, sizeof(double));
    double* x = (double*)std::calloc((size_t)n * n * nrhs, sizeof(double));
    if (!std::strcmp(mode, "workspace")) {
        c->batch_teams.emplace_back();
        c->batch_sys = {0, c->n_free};
        c->batch_nrhs = 1;
    }
    for (int call = 0; call < (unfit ? 2 : 1); ++call) {
        if (argc > 2) g_limit = (size_t)std::atoll(argv[2]);
        g_bytes = 0;
        const int rc = pgf_batch_pcg(c, 1, sys, nrhs, b, x, 1e-8, 10, nullptr, nullptr, nullptr, nullptr);
        g_limit = ~(size_t)0;
        std::printf("status %d, %zu bytes: %s\n", rc, (size_t)g_bytes, pgf_last_error(c));
    }
    std::fflush(stdout);
    std::_Exit(0);  // (the context holds nothing of the device)
}
