// fft_rule PREC NX NY NZ M MASK N: the box passes of N transforms on 256 CUs,
// a letter each: w whole boxes, s small ones, a capital where untiled boxes
// run one per CU
#include <cstdio>

#include "../../pyrpa_amd/csrc/fftbox.h"

using namespace gmod;

template <typename R>
static void print(char** v) {
  const size_t lds = 160 * 1024;
  long budget = 1;
  while ((budget * 2) * (long)sizeof(cpx<R>) * 33 / 32 <= (long)lds) budget *= 2;
  BoxPlan<R> p, q;
  const int nx = atoi(v[2]), ny = atoi(v[3]), nz = atoi(v[4]), m = atoi(v[5]), mask = atoi(v[6]);
  p.build(nx, ny, nz, m, mask, budget, lds);
  q.build(nx, ny, nz, m, mask, budget, lds, budget / 4);
  const bool two = q.ok && q.fwd.size() == p.fwd.size();
  const long n = atol(v[7]), ncu = 256;
  for (size_t i = 0; i < p.fwd.size(); ++i) {
    const bool small = two && box_take_small(p.fwd[i], q.fwd[i], n, ncu, budget);
    const BoxArgs& a = small ? q.fwd[i] : p.fwd[i];
    const size_t shm = (size_t)(a.lds_elems + a.ntwl) * sizeof(cpx<R>);
    const bool one = box_kind(a, a.blocks() * n, shm, lds, small, ncu) == BOX_ONE;
    putchar(small ? (one ? 'S' : 's') : (one ? 'W' : 'w'));
  }
  putchar('\n');
}

int main(int, char** v) { *v[1] == '0' ? print<double>(v) : print<float>(v); }
