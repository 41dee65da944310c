// Two host threads bring their own trees' coefficients out of HBM at the same
// time through the C++ API (evalf and saveTree, FunctionTree.cpp:375-435,524-546
// of MRCPP's src/trees): each has to see its own values.  Trees of more than
// 16 MiB, several pieces of the download.  Exit status 0 when every check holds, 2
// without a GPU.
#include <array>
#include <cstdio>
#include <string>
#include <thread>
#include <vector>

#include "MRCPP/Gaussians"
#include "MRCPP/MWFunctions"

using Tree = mrcpp::FunctionTree<3>;

int run(const std::string &dir) {
    mrcpp::BoundingBox<3> world(-4, std::array<int, 3>{-1, -1, -1}, std::array<int, 3>{2, 2, 2});
    mrcpp::LegendreBasis basis(7);
    mrcpp::MultiResolutionAnalysis<3> mra(world, basis, 25);
    const std::vector<mrcpp::Coord<3>> points{{0.1, 0.2, 0.3}, {1.01, 1.0, 0.98}, {-1.02, 0.99, 1.0}, {5.0, -7.0, 3.0}};
    const auto make = [&](Tree &f, int which) {
        mrcpp::GaussExp<3> g;
        for (int i = 0; i < 4; i++)
            g.append(mrcpp::GaussFunc<3>(60.0 + 20.0 * i, 1.0 + which + i, mrcpp::Coord<3>{which ? -1.0 : 1.0, 1.0, 1.0 - 0.7 * i}, std::array<int, 3>{0, 0, 0}));
        mrcpp::build_grid(f, g);
        mrcpp::project(1e-6, f, g);
    };
    const auto values = [&](Tree &f) {
        std::vector<double> v;
        for (const auto &r : points) v.push_back(f.evalf(r));
        return v;
    };
    std::vector<double> want[2];
    for (int w = 0; w < 2; w++) {
        Tree f(mra);
        make(f, w);
        std::printf("tree %d: %d nodes\n", w, f.getNNodes());
        if ((size_t)f.getNNodes() * 8 * 512 * sizeof(double) <= (16u << 20)) return 1;
        want[w] = values(f);
    }
    int wrong = 0;
    for (int round = 0; round < 6; round++) {
        Tree a(mra), b(mra);
        make(a, 0);
        make(b, 1);
        std::vector<double> got[2];
        // the second tree goes through a file in every other round
        std::thread ta([&] { got[0] = values(a); });
        std::thread tb([&] {
            if (round % 2 == 0) {
                got[1] = values(b);
                return;
            }
            b.saveTree(dir + "/b");
            Tree c(mra);
            c.loadTree(dir + "/b");
            got[1] = values(c);
        });
        ta.join();
        tb.join();
        for (int w = 0; w < 2; w++)
            if (got[w] != want[w]) {
                std::printf("round %d: tree %d has other values\n", round, w);
                wrong++;
            }
        std::printf("round %d done\n", round);
        std::fflush(stdout);
    }
    std::printf("%s: %d wrong\n", wrong ? "FAILED" : "PASSED", wrong);
    return wrong ? 1 : 0;
}

int main(int argc, char **argv) {
    try {
        return run(argc > 1 ? argv[1] : ".");
    } catch (const std::exception &e) {
        std::printf("ERROR: %s\n", e.what());
        return 2;
    }
}
