/* Accuracy of mdt_exp_t (md_tian2_amd/csrc/mdt_math.h) against libm's exp of the
 * same argument: prints the largest error as a multiple of the bound
 * (2 + 2 |x|) 2^-53 relative -- 2 for table, polynomial and product, 1 each per unit
 * of x for the rounding of the constant and of the scaled argument -- over
 * [-690, 690] and, finely, over the EMT pair range [-120, 70]. */
#include <math.h>
#include <stdio.h>
#include "../../md_tian2_amd/csrc/mdt_math.h"

int main(void) {
    static const double tab[MDT_EXP_TAB_N] = MDT_EXP_TAB_INIT;
    double worst = 0.0, wx = 0.0;
    for (int pass = 0; pass < 2; ++pass)
        for (long i = 0; i <= 4000000; ++i) {
            const double x = pass ? -120.0 + 190.0 * (double)i / 4000000.0 : -690.0 + 1380.0 * (double)i / 4000000.0;
            const double y = exp(x), e = fabs(mdt_exp_t(x * MDT_EXP_K, tab) - y) / y;
            const double m = e / ((2.0 + 2.0 * fabs(x)) * 1.1102230246251565e-16);
            if (!(m <= worst)) worst = m, wx = x;
        }
    printf("%.6f %.17g\n", worst, wx);
    return 0;
}
