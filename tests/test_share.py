"""How contexts share a device's compute units in the resident PCG (csrc/share.h), on the CPU."""
import os
import subprocess

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))

SOURCE = r"""
#include "share.h"
#include <cstdio>
#include <cstdlib>
using namespace hobak;
#define CHECK(c) do { if (!(c)) { std::printf("line %d: %s\n", __LINE__, #c); std::exit(1); } } while (0)
struct Use { int u[kShareDies]; };
Use all(int n) { Use x; for (int& v : x.u) v = n; return x; }
Use one(int d, int n) { Use x = all(0); x.u[d] = n; return x; }
void hold(Claim& c, Use x, double ms) { std::copy(x.u, x.u + kShareDies, c.use); c.ms = ms; c.live = true; }
Use held(const Share& s, const Claim* mine) { Use x; s.held(mine, x.u); return x; }
bool fits(const Share& s, const Claim* mine, Use use) { return Share::fits(held(s, mine).u, use.u, 32); }
int first_die(const Share& s, const Claim* mine, const int* w, int n) { return Share::first_die(held(s, mine).u, w, n, 32); }
int main() {
  Share s;
  Claim a, b, c;
  s.claims = {&a, &b, &c};
  // nobody here: room for everything, no turns
  CHECK(fits(s, &a, all(32)) && !fits(s, &a, all(33)));
  CHECK(s.turn_ms(&a, 10.0) == 0.0);
  int w[2] = {28, 8};
  CHECK(first_die(s, &a, w, 2) == 0);
  // b holds 26 compute units of each die: 6 are left
  hold(b, all(26), 4.7);
  CHECK(fits(s, &a, all(6)) && !fits(s, &a, one(3, 7)));
  CHECK(first_die(s, &a, w, 2) == -1);
  // its own claim is not in a context's way
  CHECK(fits(s, &b, all(32)));
  // contexts that met take turns of the other's length, for a while
  CHECK(s.turn_ms(&a, 10.0) == 0.0);
  a.ms = 14.0;
  s.meets(&a, 10.0);
  CHECK(s.turn_ms(&a, 10.0) == 4.7 && s.turn_ms(&b, 10.01) == 14.0 && s.turn_ms(&c, 10.0) == 0.0);
  CHECK(s.turn_ms(&a, 11.0) == 0.0 && s.turn_ms(&b, 11.0) == 0.0);
  // of 2 ms at least
  hold(c, one(0, 8), 0.5);
  s.meets(&a, 12.0);
  CHECK(s.turn_ms(&a, 12.0) == kShareTurnMs && s.turn_ms(&b, 12.0) == kShareTurnMs && s.turn_ms(&c, 12.0) == 4.7);
  // a claim given back leaves room at once; contexts used in turn do not meet
  b.live = c.live = false;
  CHECK(fits(s, &a, all(32)));
  s.meets(&a, 20.0);
  CHECK(s.turn_ms(&a, 20.0) == 0.0 && s.turn_ms(&b, 20.0) == 0.0);
  // groups of the two-kernel form: seen while they are queued and for a while after
  CHECK(!Share::large(all(8).u, 32) && Share::large(all(9).u, 32) && !Share::large(one(0, 32).u, 32));
  // calls of short kernels: likewise
  CHECK(Share::fills(all(32).u, 32) && !Share::fills(one(0, 32).u, 32) && !s.calls_lately(&a, 20.0));
  b.calls = 1;
  CHECK(s.calls_lately(&a, 20.0) && !s.calls_lately(&b, 20.0));
  b.calls = 0;
  CHECK(s.calls_lately(&a, 20.01) && !s.calls_lately(&a, 21.0));
  int event = 0;
  CHECK(!s.groups_lately(&a, 20.0));
  b.groups.push_back(&event);
  CHECK(s.groups_lately(&a, 20.0) && !s.groups_lately(&b, 20.0));
  b.groups.clear();
  CHECK(s.groups_lately(&a, 20.01) && !s.groups_lately(&a, 21.0));
  b.groups.push_back(&event);  // (groups that came and went between launches: contexts used in turn)
  b.groups.clear();
  CHECK(!s.groups_lately(&a, 21.0));
  // the emptiest dies
  hold(b, one(0, 28), 1.0);
  CHECK(first_die(s, &a, w, 1) == 1);
  hold(c, one(1, 28), 1.0);
  CHECK(first_die(s, &a, w, 2) == 2);
  int v[8] = {4, 4, 4, 4, 4, 4, 4, 4}, x[8] = {5, 5, 5, 5, 5, 5, 5, 5};
  CHECK(first_die(s, &a, v, 8) == 0 && first_die(s, &a, x, 8) == -1);
  return 0;
}
"""


def test_claims(tmp_path):
    src, exe = tmp_path / "share.cpp", tmp_path / "share"
    src.write_text(SOURCE)
    subprocess.run(["g++", "-std=c++17", "-Wall", "-Werror", "-I", os.path.join(ROOT, "hobakv1_amd", "csrc"), str(src),
                    "-o", str(exe), "-pthread"], check=True)
    out = subprocess.run([str(exe)], capture_output=True, text=True)
    assert out.returncode == 0, out.stdout
