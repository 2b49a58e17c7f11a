// Reads the orientation file of the first argument and the same contents from standard input (a pipe, which has
// no size and no positions), and exits nonzero where the two differ or hold nothing.
#include <cstdio>

#include "init.hpp"

int main(int, char **argv) {
    const std::vector<float> a = exaca::read_orientations(argv[1]), b = exaca::read_orientations("/dev/stdin");
    int given = 0;
    for (float x : a) given += x != 0.0f;
    printf("%d components, %s\n", given, a == b ? "the same" : "different");
    return a != b || !given;
}
