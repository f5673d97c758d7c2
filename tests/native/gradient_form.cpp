// Host evaluation of the bracket D of dW/dq of the gradient sweep and the force pass (kernED,
// common.hpp), for the CPU tests: for each q on stdin prints D, and D as the gradient sweep has it (kernVGD).
#include "../../cosmosphere_amd/csrc/common.hpp"

#include <cstdio>

int main()
{
    double q;
    while (std::scanf("%lf", &q) == 1)
    {
        double E, D, V, G, D2;
        csph::kernED<double>(q, E, D);
        csph::kernVGD<double>(q, V, G, D2);
        std::printf("%.17g %.17g\n", D, D2);
    }
    return 0;
}
