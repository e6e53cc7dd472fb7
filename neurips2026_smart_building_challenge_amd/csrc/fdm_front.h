// Host plan of the default field solve (see sbf::FrontTab): which columns form
// a front, the fronts' boundaries, heights, assembly lists and tasks. Plain
// C++, no device calls.
#pragma once
#include <utility>
#include <vector>

#include "fdm.h"

namespace sbf {

typedef std::vector<std::vector<std::pair<int, double>>> RowTerms;

struct FrontPlan {
    std::vector<Front> fronts;          // by height, leaves first
    std::vector<int> pos;               // [n] row of the permuted system -> row in front order
    std::vector<int> front_of, local;   // [n] row of the permuted system -> its front, its place there
    std::vector<int> bperm;             // the B rows as rows of the permuted system (ascending), laid out as brow
    std::vector<int> brow;              // the B rows as positions
    std::vector<AsmRow> arow;
    std::vector<int> xsrc;
    std::vector<FrontTask> tasks;
    std::vector<FrontLevel> levels;
    int n_leaf = 0, n_c = 0;
    size_t ops = 0;                     // doubles of the operators, padding included
};

// lower[i]: row i's off-diagonal terms of L; upper[i]: row i's of U.
void plan_fronts(const RowTerms& lower, const RowTerms& upper, FrontPlan* out);

}  // namespace sbf
