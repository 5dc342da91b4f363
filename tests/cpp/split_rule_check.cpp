// Prints what the library's rules pick on 256 CUs for the launches given as arguments (width batch heads length radius, causal, all
// loads 128-bit): workgroup shapes of the split-product forward, dQ and dK/dV kernels, and which of forward, default and
// deterministic backward run them. No GPU.
#include <cstdio>
#include <cstdlib>

#include "attention_launch.hpp"

int main(int argc, char **argv) {
    for (int i = 1; i + 4 < argc; i += 5) {
        const int D = std::atoi(argv[i]), batch = std::atoi(argv[i + 1]), heads = std::atoi(argv[i + 2]), length = std::atoi(argv[i + 3]),
                  radius = std::atoi(argv[i + 4]);
        constexpr int kCus = 256;
        rk::ForwardArgs f{};
        rk::BackwardArgs b{};
        f.batch = b.batch = batch;
        f.heads = b.heads = heads;
        f.queries = b.queries = f.keys = b.keys = length;
        f.radius = b.radius = radius;
        f.causal = b.causal = 1;
        const rk::SplitWorkgroup forward = rk::forward_split_workgroup(D, f, kCus), dq = rk::dq_split_workgroup(D, b, kCus),
                                 dkdv = rk::dkdv_split_workgroup(D, b, kCus);
        std::printf("%d %d %d %d %d %d %d %d %d\n", forward.tiles, forward.streams, dq.tiles, dq.streams, dkdv.tiles, dkdv.streams,
                rk::forward_split_pays(D, f, kCus), rk::backward_split_pays(D, b, kCus, true, false),
                rk::backward_split_pays(D, b, kCus, true, true));
    }
    return 0;
}
