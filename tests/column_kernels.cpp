// What quantize's second launch runs for lists of matrices stored column by column.
//
// Reads lists from the standard input, one per line: dtype, slots, and rows and columns of every tensor.
// Prints, for every list, one word for each variant of a kernel that its blocks take: the kernel
// (QcKernel), the groups of rows and the steps that the variant holds (16: a row of more than 12).

#include <stdio.h>

#include <iostream>
#include <set>
#include <sstream>
#include <string>
#include <vector>

#include "../include/tftq.h"
#include "../torchft_amd/csrc/tftq_internal.h"

int main()
{
    static const char *const names[] = {"any4", "any12", "two4", "two8", "two12"};
    std::string line;
    while (std::getline(std::cin, line)) {
        std::istringstream in(line);
        int dtype, ws;
        int64_t m, n;
        std::vector<int64_t> shapes, strides;
        in >> dtype >> ws;
        while (in >> m >> n) {
            shapes.insert(shapes.end(), {m, n});
            strides.insert(strides.end(), {1, m});
        }
        tftq_plan *p = nullptr;
        if (tftq_plan_create(dtype, (int)shapes.size() / 2, shapes.data(), strides.data(), ws, &p)) return 1;
        std::set<std::string> words;
        for (const Seg &s : p->segs) {
            if (s.kind[ST_Q] != K_COLS) continue;
            const int steps = tftq_qc_steps(s.n, s.lg_groups);
            if (!tftq_qc_has(s.lg_groups, steps)) return 1;
            const int held = steps <= 2 ? steps : steps <= 4 ? 4 : steps <= 8 ? 8 : steps <= 12 ? 12 : 16;
            words.insert(std::string(names[tftq_qc_kernel(*p)]) + "/" + std::to_string(1 << s.lg_groups) + "/" + std::to_string(held));
        }
        for (const std::string &w : words) printf("%s ", w.c_str());
        printf("\n");
        tftq_plan_destroy(p);
    }
    return 0;
}
