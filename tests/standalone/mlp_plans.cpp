// Reads sizes (tokens d_model hidden, one a line) and prints which of the block's kernels each of them runs on 256 compute units:
// the product, the tile's number, and "parts" where k is split; for every set of gradients that a backward pass can be asked for.
#include <cstdio>

#include "../../mgrrmsnorm_amd/csrc/mlp_plan.hpp"

int main() {
    constexpr int kCus = 256;
    long long t, d, h;
    const auto show = [](const char* what, mg::MlpPlan p) {
        if (p.shape >= 0) printf(" %s-%d%s", what, p.shape, p.splits > 1 ? "-parts" : "");
    };
    while (scanf("%lld %lld %lld", &t, &d, &h) == 3) {
        const mg::MlpForward f(t, d, h, kCus);
        show("gate_up", f.gate_up);
        show("down", f.down);
        for (int want = 1; want < 8; ++want) {
            const mg::MlpBackward b(t, d, h, want & 1, want & 2, want & 4, kCus);
            show("weight_grad", b.w3);
            show("weight_grad", b.w12);
            show("activation_bwd", b.act);
            show("input_grad", b.x);
            if (b.w12.splits > 1 && b.x.splits > 1) printf(" both-parts");
        }
        printf("\n");
    }
}
