// Prints the launch shape (1-based) that each size on the command line takes by default.
#include "sl_ordered_rule.hpp"

#include <cstdio>
#include <cstdlib>

int main(int argc, char** argv)
{
    for (int k = 1; k < argc; k++) std::printf("%d\n", sl::ordered_default_shape(std::atoi(argv[k])) + 1);
    return 0;
}
