// Every load of the flexible kernels' ordered sums (list_sum, row_sum in
// scan_flex.hip) lies inside the LDS a block asks for: the loads are repeated
// here, loop by loop, on lists of every shape of small systems.
#include <cstdio>
#include <cstring>
#include <vector>

#include "../mechafm_amd/csrc/flex.hpp"

using namespace mafm;

// largest place (in doubles from v) that list_sum<S>(v, n) loads
static size_t list_last(int S, int n) {
    auto batch = [&](int q) { return (size_t)S * (q / 2 + FLEX_BATCH / 2 - 1) + 1; };
    size_t last = batch(0);
    for (int q = 0; q < n; q += 2 * FLEX_BATCH) {
        last = batch(q + FLEX_BATCH);
        if (q + FLEX_BATCH >= n) break;
        last = batch(q + 2 * FLEX_BATCH);
    }
    return last;
}

// largest place that row_sum<DIV>(v, row, nq, p) loads; past: it read the table past its n_rows
static size_t row_last(int DIV, const std::vector<int32_t>& row, int nq, int p, bool& past) {
    size_t last = 0;
    auto four = [&](int q) {
        for (int j = 0; j < 4; ++j) {
            if (q + j >= (int)row.size()) { past = true; return; }
            last = std::max(last, (size_t)(row[q + j] / DIV + p + 1));
        }
    };
    const int n2 = (nq + 1) / 2;
    four(0);
    int q = 0;
    for (; q + 4 <= n2; q += 4) four(q + 4);
    if (q + 8 > (int)row.size()) past = true;   // the places loaded ahead
    return last;
}

int main() {
    long checked = 0, outside = 0;
    for (int n = 2; n <= 6; ++n)
        for (int n_tip = 0; n_tip <= 70; ++n_tip)
            for (int shape = 0; shape < 6; ++shape) {
                // slots of the other atoms by rank: none, one on one atom, some, even, falling, many
                std::vector<int> cnt(n - 1);
                for (int k = 0; k < n - 1; ++k)
                    cnt[k] = shape == 0 ? 0 : shape == 1 ? (k == 0) : shape == 2 ? std::max(0, 3 - k) : shape == 3 ? 2
                             : shape == 4 ? std::max(0, 9 - 4 * k) : 40 - k;
                const int n_rows = (cnt[0] + 1) / 2;
                std::vector<int32_t> row((n_rows + 12 + 3) / 4 * 4, 0);
                const int others = 4 * flex_padded(n_tip);
                int width = n - 1, n_res = others;
                for (int q = 0; q < n_rows; ++q) {
                    while (width > 0 && cnt[width - 1] <= 2 * q) --width;
                    row[q] = n_res - others;
                    n_res += 6 * width;
                }
                auto check = [&](size_t bytes, size_t all) {
                    const size_t results = flex_padded(n) + 4;
                    bool past = false;
                    size_t last = list_last(2, n);                                       // the powers
                    last = std::max(last, results + 6 + list_last(8, n_tip));            // the tip, its energy's lane
                    for (int k = 0; k < n - 1; ++k) {
                        last = std::max(last, results + others + row_last(1, row, cnt[k], 6 * k + 4, past));
                        if (all) last = std::max(last, results + n_res + 8 + row_last(3, row, cnt[k], 2 * k, past));
                    }
                    ++checked;
                    if (past || (last + 1) * sizeof(double) > bytes) {
                        if (outside++ < 5)
                            printf("%d atoms, %d tip slots, shape %d: byte %zu of %zu%s\n", n, n_tip, shape,
                                   (last + 1) * sizeof(double), bytes, past ? ", table" : "");
                    }
                };
                for (int rk4 = 0; rk4 < 2; ++rk4) {
                    FlexArgs a;
                    memset(&a, 0, sizeof a);
                    a.n_atoms = n; a.n_res = n_res; a.n_tip = n_tip; a.n_rows = (int)row.size();
                    a.minimiser = MAFM_MIN_FIRE; a.integrator = rk4 ? MAFM_INT_RK4 : MAFM_INT_MIDPOINT;
                    check(flex_block_lds(a), 0);
                    for (int op : {SYS_EVAL, SYS_STEP, SYS_MINIMISE}) {
                        SysArgs s;
                        memset(&s, 0, sizeof s);
                        s.n_atoms = n; s.n_res = n_res; s.n_tip = n_tip; s.n_rows = (int)row.size();
                        s.op = op; s.minimiser = MAFM_MIN_FIRE; s.integrator = a.integrator;
                        check(sys_block_bytes(s), sys_all_energies(s));
                    }
                }
            }
    printf("checked %ld outside %ld\n", checked, outside);
    return outside ? 1 : 0;
}
