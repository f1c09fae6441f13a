// Prints the generated HIP source of a lowered program read from stdin, for
// tests/test_codegen_acos.py.
#include <iostream>
#include "codegen.hpp"

int main() {
    std::cout << ivarp::codegen::generate(ivarp::flat::Program::read(std::cin), "t");
    return 0;
}
