// The launchers' host rules, from the library's own headers: each line of
// standard input is a question, each line of output its answer.
//   rows CUS N...   -> rows per workgroup, workgroups of the launch
//   small N K M     -> 1 if the GEMM entry's call goes to the small-batch kernel
//   dequant B       -> super-blocks and threads of each launch for B super-blocks
#include <iostream>
#include <sstream>
#include <string>
#include <vector>

#include "dequant_plan.h"
#include "small_batch_plan.h"

int main() {
    std::string line, what;
    while (std::getline(std::cin, line)) {
        std::istringstream in(line);
        in >> what;
        std::vector<int64_t> v;
        for (int64_t x; in >> x;) v.push_back(x);
        if (what == "rows") {
            const int count = (int)v.size() - 1;
            const int64_t rows = iq4xs::gm_rows(count, v.data() + 1, v[0]);
            int64_t wgs = 0;
            for (int i = 1; i <= count; ++i) wgs += (v[i] + rows - 1) / rows;
            std::cout << rows << " " << wgs << "\n";
        } else if (what == "small") {
            std::cout << (iq4xs::use_small_batch(v[0], v[1], v[2]) ? 1 : 0) << "\n";
        } else if (what == "dequant") {
            for (int64_t left = v[0]; left > 0;) {
                const int64_t n = iq4xs::dequant_chunk(left);
                const int64_t wgs = (n * iq4xs::DEQUANT_THREADS + iq4xs::DEQUANT_WG - 1) / iq4xs::DEQUANT_WG;
                std::cout << n << " " << wgs * iq4xs::DEQUANT_WG << " ";
                left -= n;
            }
            std::cout << "\n";
        } else {
            return 1;
        }
    }
    return 0;
}
