// eig_rule BATCH N: prints 1 if the eigenvalues of BATCH N x N matrices run a wavefront per matrix
#include <cstdio>

#include "../../pyrpa_amd/csrc/linalg.h"

int main(int, char** argv) { printf("%d\n", gmod::eig_by_wave(atol(argv[1]), atoi(argv[2])) ? 1 : 0); }
