// Prints prefill_page_span for the argument lines "tk window rw group log2_page" on stdin.
#include <cstdio>
#include <cinttypes>
#include "prefill_span.h"
int main() {
    int64_t tk, window, rw, group, lp;
    while (std::scanf("%" SCNd64 " %" SCNd64 " %" SCNd64 " %" SCNd64 " %" SCNd64, &tk, &window, &rw, &group, &lp) == 5)
        std::printf("%" PRId64 "\n", sandy_hip::prefill_page_span(tk, window, rw, group, static_cast<int>(lp)));
}
