// sor_plan_driver.cpp -- prints the plans of hydro_amd/csrc/sor_plan.h for grids
// and iteration limits (built by tests/test_sor_plan.py with g++
// -fsanitize=undefined): for each "nx ny limit w" on the input, w the
// doubles of workspace (0: any number), one line
//   ok_one Q rounds doubles_one | use_chain Q G span le doubles_many a b end
//   first workspace
#include <cstdio>

#include "../hydro_amd/csrc/sor_plan.h"

int main() {
  int nx, ny, limit;
  long w;
  while (std::scanf("%d %d %d %ld", &nx, &ny, &limit, &w) == 4) {
    const long all = w ? w : 1L << 60;
    const hg::SorPlan p = hg::PlanSor(nx, ny, limit, all), c = hg::PlanChain(nx, ny, limit, all);
    const bool many = hg::UseChain(p, c);
    const int P = 2 * c.Q;
    const long end = many ? hg::ChainDoneStep(limit, P, c.G * P, c.span, c.a, c.b) : 0;
    std::printf("%d %d %d %ld %d %d %d %d %d %ld %d %d %ld %d %ld\n", int(p.ok), p.Q, p.rounds,
                p.ok ? p.doubles : 0, int(many), c.Q, c.G, c.span, c.le, c.ok ? c.doubles : 0, c.a,
                c.b, end, int(many ? c.first : p.first), hg::SorWorkspaceDoubles(nx, ny, limit));
  }
  return 0;
}
