// ekm_mg5.h -- the MUDPACK replica's form for grids without cross terms
// (ekm_mg5.hip), used by ekm_mg.hip.
#pragma once
#include <vector>

#include "ekm_host.h"
#include "ekm_internal.h"

// every level's rows are 5-point rows (the corner coefficients are zero)
bool mg5_applies(const std::vector<HostMgLevel>& hl, int ngrid);
// ops: the cycle programs of mg ((op << 8) | level; the full multigrid start,
// then one W cycle)
int mg5_plan_build(Mg5Plan& mp, const MgPlan& mg, const Dims& d, const std::vector<HostMgLevel>& hl,
                   const std::vector<int>& ops, size_t lds_budget_doubles);
int mg5_solve(const MgPlan& mg, const Dims& d, int nsolve, int iguess, hipStream_t st);
