// Prints the LDS class of every mesh of a plan: arguments "nsub,entries" per mesh.
#include <cstdio>
#include <vector>

#include "md_analysis.h"

int main(int argc, char **argv) {
    std::vector<md::SubSize> meshes;
    for (int k = 1; k < argc; ++k) {
        md::SubSize s{};
        if (std::sscanf(argv[k], "%d,%d", &s.nsub, &s.entries) != 2) return 2;
        meshes.push_back(s);
    }
    std::vector<int> cls;
    md::subtree_classes(meshes, cls);
    for (int c : cls) std::printf("%d ", c);
    std::printf("\n");
    return 0;
}
