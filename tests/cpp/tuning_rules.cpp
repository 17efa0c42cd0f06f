// Prints what a rule of gi_tuning.h gives: "walk <sims> <n>" (lanes per
// particle of the contact walk of equal simulations) or "piece <n> <L0>" (j per
// piece in the batched engine).
#include <cstdlib>

#include "gi_tuning.h"

int main(int argc, char** argv) {
    if (argc == 4 && !std::strcmp(argv[1], "walk")) {
        const double k = std::atof(argv[2]), n = std::atof(argv[3]);
        std::printf("%d\n", gi::contact_walk_by_rows(k * n, k * n * n) ? 9 : 1);
        return 0;
    }
    if (argc == 4 && !std::strcmp(argv[1], "piece")) {
        std::printf("%lld\n", gi::batched_piece_len(std::atoll(argv[2]), std::atoll(argv[3])));
        return 0;
    }
    return 2;
}
