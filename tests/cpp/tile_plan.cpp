// Prints the tiled GEMM's plan (tile, K slices) for each "rows cols n bytes" line of the input, on 256
// CUs: x0ne_gemm_tile_plan of the built library.
#include <cstdio>

#include <hip/hip_runtime.h>

#include "launch.h"

int main() {
    unsigned rows, cols, n;
    unsigned long long bytes;
    while (std::scanf("%u %u %u %llu", &rows, &cols, &n, &bytes) == 4) {
        const X0neTilePlan p = x0ne_gemm_tile_plan(rows, cols, n, 256, bytes);
        std::printf("%d %u\n", p.tile, p.slices);
    }
}
