// The Adams-Bashforth sums of crm_round.hpp on the host: for every shape, engine and velocity
// component, one line of the shape and the bits of the sum for each set of operands read.
#include <cstdio>
#include <initializer_list>

#include "crm_round.hpp"

using namespace crm;

static double sum(AbAlone x, const double* v) {
  switch (x) {
    case AbAlone::A: return ab_sum<AbAlone::A>(v[0], v[1], v[2], v[3], v[4], v[5]);
    case AbAlone::B: return ab_sum<AbAlone::B>(v[0], v[1], v[2], v[3], v[4], v[5]);
    default: return ab_sum<AbAlone::C>(v[0], v[1], v[2], v[3], v[4], v[5]);
  }
}

int main() {
  double v[6];
  while (std::scanf("%la %la %la %la %la %la", v, v + 1, v + 2, v + 3, v + 4, v + 5) == 6)
    for (int columns : {8, 16, 32, 64, 128})
      for (int y3 = 0; y3 < (columns == 16 || columns == 64 ? 2 : 1); y3++)
        for (int fp64 = 0; fp64 < 2; fp64++)
          for (char f : {'u', 'v', 'w'}) {
            if (f == 'v' && !y3) continue;
            const AbField field = f == 'u' ? AbField::U : f == 'v' ? AbField::V : AbField::W;
            std::printf("%d %d %d %c %a\n", columns, y3, fp64, f, sum(ab_alone(field, columns, y3, fp64), v));
          }
}
