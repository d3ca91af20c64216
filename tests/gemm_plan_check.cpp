// The route of FP8 GEMM launches, by the launcher's own rule
// (hy-nomas_amd/csrc/gemm_plan.h): one line per "MODE M N K CUS" read from the
// standard input (MODE 0 row/column, 1 blockwise), made of
//   64x64, 128x192, ...   one launch of gemm_small_kernel in such tiles
//   256x256 [edge]        the persistent or the 8-wave blockwise kernel [with edge tiles]
//   tail 4x1              gemm_tail_kernel, K split over 4 waves, 1 row block
//   light                 the tail stripe on the persistent launch's light workgroups
#include <cstdio>

#include "../hy-nomas_amd/csrc/gemm_plan.h"

using namespace hn::gemm;

int main() {
    int mode, cus;
    long long M, N, K;
    while (scanf("%d %lld %lld %lld %d", &mode, &M, &N, &K, &cus) == 5) {
        const Route r = gemm_route(mode, M, N, K, cus);
        if (r.small >= 0) {
            const TileCost& t = (mode == ROWCOL ? kSmallRowcol : kSmallBlockwise)[r.small];
            printf("%dx%d\n", t.tm, t.tn);
            continue;
        }
        const char* sep = "";
        if (r.Mt > 0) printf("256x256%s", r.tiles.tiles_part ? " edge" : ""), sep = " ";
        if (r.Mt < M && r.tail_cols > 0) printf("%slight", sep);
        else if (r.Mt < M) printf("%stail %dx%d", sep, r.tail_waves, r.tail_blocks);
        printf("\n");
    }
    return 0;
}
