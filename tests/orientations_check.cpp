// Checks the orientation file reader and the seed table (exaca_amd/csrc/init.cpp): the shipped file and
// small files with every form of number that takes the reader's slow path, against getline and atof
// as the reference reads them (src/CAinitialize.cpp:1408-1442), bit for bit; and the table's rows, built on
// threads, against one orientation at a time. Prints the number of mismatches and exits nonzero on any.
#include <cstdio>
#include <cstring>
#include <fstream>
#include <sstream>

#include "ca_common.hpp"
#include "init.hpp"

static std::vector<float> by_lines(const std::string &path) {
    std::vector<float> guv(9 * 10000, 0.0f);
    std::ifstream in(path);
    std::string line;
    std::getline(in, line);
    for (int i = 0; i < 10000; i++) {
        if (!std::getline(in, line)) break;
        std::istringstream ss(line);
        std::string tok;
        int slot = 0;
        while (slot < 9 && std::getline(ss, tok, ',')) guv[9 * i + slot++] = static_cast<float>(std::atof(tok.c_str()));
    }
    return guv;
}

int main(int, char **argv) {
    int bad = 0;
    auto same = [&](const std::string &path) {
        const std::vector<float> a = exaca::read_orientations(path), b = by_lines(path);
        if (std::memcmp(a.data(), b.data(), 4 * b.size())) bad++, printf("differs: %s\n", path.c_str());
    };
    same(argv[1]);
    const std::string tmp = argv[2];
    for (const char *text : {"3\n1,2,3,4,5,6,7,8,9\r\n.5,-.25, 1e-3,,+2,abc,1.5x,123456789012345678,9,10\n\n-0,1", "", "2\n", "4",
                             "1\n1.0000000000000000001,0.1234567890123456,5e400,-,.,7.,-.5,0x10,inf\n1,2\n,,3,,,,,,,4\n",
                             "2\n1,2,3,4,5,6,7,8,9,10,11\n-1.5,999999999999999,0.000000000000001,1,1,1,1,1,1"}) {
        std::ofstream(tmp) << text;
        same(tmp);
    }
    const std::vector<float> guv = exaca::read_orientations(argv[1]);
    for (int rows : {1, 7, 1000, 2003, 10000}) {
        const std::vector<float> t = exaca::seed_table(guv, rows);
        for (int o = 0; o < rows; o++) {
            float one[exaca::kCdlStride] = {};
            exaca::seed_critical_lengths(&guv[9 * o], one);
            bad += std::memcmp(one, &t[static_cast<size_t>(o) * exaca::kCdlStride], sizeof one) != 0;
        }
    }
    printf("mismatches %d\n", bad);
    return bad != 0;
}
