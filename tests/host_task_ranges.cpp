// Host unit test of csrc/hpx_task_ranges.h (compiled and run by tests/test_task_ranges.py).
#include "hpx_task_ranges.h"

#include <cstdio>
#include <cstdlib>
#include <random>

#define CHECK(c)                                                            \
  do {                                                                      \
    if (!(c)) {                                                             \
      std::printf("%s:%d: %s\n", __FILE__, __LINE__, #c);                   \
      std::exit(1);                                                         \
    }                                                                       \
  } while (0)

namespace {
float* tensor_at(uintptr_t x) { return reinterpret_cast<float*>(x); }
uint8_t* bytes_at(uintptr_t x) { return reinterpret_cast<uint8_t*>(x); }

hpx_task_t task(uintptr_t tensor, int64_t numel, uintptr_t B, uintptr_t C, int64_t bytes) {
  hpx_task_t t{};
  t.tensor = tensor_at(tensor); t.tensor_numel = numel;
  t.B = bytes_at(B); t.B_bytes = bytes;
  t.C = bytes_at(C); t.C_bytes = bytes;
  return t;
}
bool share(const hpx_task_t& a, const hpx_task_t& b) {  // in one batch, and in two
  hpx::Ranges both, x, y;
  both.add(a); both.add(b);
  x.add(a); y.add(b);
  CHECK(!x.close() && !y.close());
  const bool s = both.close();
  CHECK(x.meets(y) == s && y.meets(x) == s);
  return s;
}
}  // namespace

int main() {
  const hpx_task_t a = task(0x10000, 1000, 0x40000, 0x80000, 250);
  CHECK(share(a, a));
  CHECK(!share(a, task(0x10000 + 4000, 1000, 0x40100, 0x80100, 250)));       // neighbours in one bucket
  CHECK(share(a, task(0x10000 + 3996, 1000, 0x40100, 0x80100, 250)));        // the last element
  CHECK(share(a, task(0x10000 + 400, 10, 0x40100, 0x80100, 3)));             // a slice, at another address
  CHECK(share(task(0x10000 + 400, 10, 0x40100, 0x80100, 3), a));
  CHECK(share(a, task(0x20000, 1000, 0x40000 + 249, 0x80100, 250)));         // B
  CHECK(share(a, task(0x20000, 1000, 0x40100, 0x80000 - 249, 250)));         // C
  CHECK(!share(a, task(0x20000, 1000, 0x40100, 0x80000 - 250, 250)));
  hpx_task_t gathered = task(0x20000, 1000, 0x50000, 0x80000 - 500, 250);    // slot 2 of it is a's C
  gathered.C_bytes = 750;
  CHECK(share(a, gathered));
  gathered.C_bytes = 500;
  CHECK(!share(a, gathered));
  hpx_task_t r = a;                                                          // a residual of unstated length
  r.residual = tensor_at(0x18000);
  CHECK(share(r, task(0x18000 + 3996, 1, 0x50000, 0x90000, 1)));
  CHECK(!share(r, task(0x18000 + 4000, 1, 0x50000, 0x90000, 1)));
  hpx_task_t p{};                                                            // the factors of a matrix
  p.tensor = tensor_at(0x100000); p.residual = tensor_at(0x200000); p.tensor_numel = p.residual_numel = 60;
  p.M = tensor_at(0x300000); p.P = tensor_at(0x400000); p.Q = tensor_at(0x500000);
  p.n = 10; p.m = 6; p.r = 2;
  CHECK(share(p, task(0x300000 + 59 * 4, 1, 0x50000, 0x90000, 1)) && !share(p, task(0x300000 + 60 * 4, 1, 0x50000, 0x90000, 1)));
  CHECK(share(p, task(0x400000 + 19 * 4, 1, 0x50000, 0x90000, 1)) && !share(p, task(0x400000 + 20 * 4, 1, 0x50000, 0x90000, 1)));
  CHECK(share(p, task(0x500000 + 11 * 4, 1, 0x50000, 0x90000, 1)) && !share(p, task(0x500000 + 12 * 4, 1, 0x50000, 0x90000, 1)));

  hpx::Ranges none, some;
  CHECK(!none.close() && !none.meets(none));
  some.add(nullptr, 8);
  some.add(tensor_at(16), 0);
  CHECK(!some.close() && !some.meets(some));

  // against every pair of bytes
  std::mt19937 gen(1);
  for (int trial = 0; trial < 20000; trial++) {
    bool byte[2][64] = {}, twice[2] = {};
    hpx::Ranges s[2];
    for (int k = 0; k < 2; k++) {
      for (int c = int(gen() % 4); c > 0; c--) {
        const int lo = 1 + int(gen() % 60), n = int(gen() % 4);
        s[k].add(bytes_at(uintptr_t(lo)), n);
        for (int i = lo; i < lo + n; i++) {
          twice[k] = twice[k] || byte[k][i];
          byte[k][i] = true;
        }
      }
      CHECK(s[k].close() == twice[k]);
    }
    bool any = false;
    for (int i = 0; i < 64; i++) any = any || (byte[0][i] && byte[1][i]);
    CHECK(s[0].meets(s[1]) == any && s[1].meets(s[0]) == any);
  }
  std::puts("OK");
  return 0;
}
