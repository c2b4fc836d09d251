// Host check of tftq_one_piece, by which a workgroup of a list of one tensor finds its block: the
// same workgroup ids lead to the same blocks as through the table of the planner (which
// tests/plan_mapping.cpp walks), and every block is visited exactly once.  Prints "ok" on success.

#include <stdio.h>

#include <vector>

#include "../include/tftq.h"
#include "../torchft_amd/csrc/tftq_internal.h"

int main()
{
    for (int natural = 0; natural < 2; natural++) {
        for (int32_t nwg : {1, 2, 7, 8, 9, 15, 16, 17, 63, 255, 256, 1023, 100001}) {
            std::vector<uint8_t> seen((size_t)nwg, 0);
            for (uint32_t b = 0; b < 8u * (uint32_t)((nwg + 7) / 8); b++) {
                const int32_t at = tftq_one_piece(nwg, natural, b);
                if (at == -1) continue;
                if (at < 0 || at >= nwg || seen[(size_t)at]++) return printf("%d workgroups: id %u leads to %d\n", nwg, b, at), 1;
            }
            for (uint8_t s : seen)
                if (!s) return printf("%d workgroups: one is missing\n", nwg), 1;
        }
        if (tftq_one_piece(INT32_MAX - 4096, natural, 0) != 0) return printf("large launch\n"), 1;
    }
    const int64_t shapes[][2] = {{1, 1}, {4096, 1}, {33, 130}, {5000, 17}, {777, 4096}, {1000, 5000}, {3, 70000}, {4096, 1024}};
    for (const auto &shape : shapes) {
        for (int ws : {1, 3, 8, 64}) {
            for (int by_columns = 0; by_columns < 2; by_columns++) {
                const int64_t strides[2] = {by_columns ? 1 : shape[1], by_columns ? shape[0] : 1};
                tftq_plan *p = nullptr;
                if (tftq_plan_create(TFTQ_BF16, 1, shape, strides, ws, &p)) return printf("plan\n"), 1;
                for (int st = 0; st < N_LAUNCHES; st++) {
                    if (p->nwg[st] == 0) continue;
                    const Dealt &d = p->dealt[st];
                    for (uint32_t b = 0; b < 8u * (uint32_t)p->dealt_per_xcd[st]; b++) {
                        const int x = (int)(b & 7), i = p->natural[st] ? (int)b : (int)(b >> 3);
                        const int32_t want = i < d.cum_end[x][0] ? d.base[x][0] + i : -1;
                        const int32_t at = tftq_one_piece(p->nwg[st], p->natural[st], b);
                        if (at != want) return printf("%lld x %lld, stage %d, id %u: %d, not %d\n", (long long)shape[0], (long long)shape[1], st, b, at, want), 1;
                    }
                }
                tftq_plan_destroy(p);
            }
        }
    }
    printf("ok\n");
    return 0;
}
