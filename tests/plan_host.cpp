// Sizes the library's host code plans with, printed for the tests: no GPU is
// touched.  Lines of standard input:
//   pagerank V log2S H edges  -> words of the edges, room of them with their groups' rows, bins, parts
//   sort n                    -> scratch words of a batch sort
#include <cstdio>
#include <cstring>

#include "kernels.hpp"

int main() {
    char what[32];
    unsigned long long a, b, c, e;
    while (scanf("%31s", what) == 1) {
        if (!strcmp(what, "pagerank") && scanf("%llu %llu %llu %llu", &a, &b, &c, &e) == 4) {
            pma::DevState d{};
            d.V = (pma::u32)a;
            d.log2S = (pma::u32)b;
            d.H = (pma::u32)c;
            const pma::PrBins p = pma::pr_bins_plan(d, e);
            printf("%llu %llu %u %u\n", (unsigned long long)p.words, (unsigned long long)pma::pr_bins_edge_words(p),
                   p.bins, p.parts);
        } else if (!strcmp(what, "sort") && scanf("%llu", &a) == 1) {
            printf("%llu\n", (unsigned long long)pma::sort_scratch_words(a));
        } else {
            return 1;
        }
    }
    return 0;
}
