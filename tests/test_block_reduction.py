"""The reduction of the contraction's blocks by the interaction's symmetries
(taurus_vap_amd/csrc/tg_blocks.h) against the whole blocks, on the CPU.

A host program fills the blocks of both channels with small integers that have a chosen set
of symmetries (time reversal with hermiticity, charge reflection, their product alone, both,
none, one with a single element changed), with the phases of half-integer spin and with
phases that make elements their own image with a minus, in full and with most elements zero
(signs found per connected part).  It checks that
  * products with the reduced blocks, through the orbit sums and back, equal those with
    the whole block (exactly: integers and their quarters),
  * a block splits by every symmetry that it has, down to its largest orbit, and by none that
    it lacks."""
import os
import subprocess

import pytest

CSRC = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "taurus_vap_amd", "csrc")
PROGRAM = r"""
#include <cstdio>
#include <cstdlib>
#include <cstring>
#include <random>
#include "tg_blocks.h"
int main(int, char** argv) {
  const bool pp = !std::strcmp(argv[1], "pp");
  const int kind = std::atoi(argv[2]);      // bits: time reversal, reflection, their product
  const bool odd = std::atoi(argv[3]), sparse = std::atoi(argv[4]), broken = std::atoi(argv[5]);
  std::mt19937 rng(7);
  auto pick = [&](int lo, int hi) { return lo + (int)(rng() % (unsigned)(hi - lo + 1)); };
  // shells (l, 2j), protons then neutrons, by (2m, parity) inside each half
  const int shells[6][2] = {{0, 1}, {1, 3}, {1, 1}, {2, 5}, {0, 1}, {2, 3}};
  struct St { int t, m, l, sh; };
  std::vector<St> st;
  for (int t = -1; t <= 1; t += 2)
    for (int q = 0; q < 6; ++q)
      for (int m = -shells[q][1]; m <= shells[q][1]; m += 2) st.push_back({t, m, shells[q][0], q});
  std::stable_sort(st.begin(), st.end(), [](const St& a, const St& b) {
    return std::make_tuple(a.t, a.m, a.l & 1) < std::make_tuple(b.t, b.m, b.l & 1);
  });
  const int n = (int)st.size(), h = n / 2;
  std::vector<int> m(n), t(n), l(n), tr(n), ph(n);
  for (int i = 0; i < n; ++i) {
    m[i] = st[i].m; t[i] = st[i].t; l[i] = st[i].l;
    for (int k = 0; k < n; ++k)
      if (st[k].t == st[i].t && st[k].sh == st[i].sh && st[k].m == -st[i].m) tr[i] = k;
  }
  for (int i = 0; i < h; ++i)
    if (m[i] > 0) {
      ph[i] = pick(0, 1) ? 1 : -1;
      ph[tr[i]] = odd ? ph[i] : -ph[i];
    }
  for (int i = 0; i < h; ++i) ph[i + h] = ph[i];
  const SpBasis basis{n, m, t, l, tr};
  long long reduced = 0, whole = 0, splits = 0;
  for (auto& kv : channel_classes(basis, pp)) {
    const std::vector<int>& el = kv.second;
    const int s = (int)el.size();
    std::vector<int> at(n * n, -1);
    for (int k = 0; k < s; ++k) at[el[k]] = k;
    // the chosen symmetries that map this class to itself
    struct P { std::vector<int> to, sg; };
    std::vector<P> gen;
    for (int q = 0; q < 3; ++q) {
      if (!(kind >> q & 1)) continue;
      const bool T = q != 1, C = q != 0;
      P g;
      bool ok = true;
      for (int k = 0; k < s && ok; ++k) {
        int x = el[k] % n, y = el[k] / n, sg = 1;
        if (T) {
          sg = ph[x] * ph[y];
          const int tx = tr[x], ty = tr[y];
          x = pp ? tx : ty;
          y = pp ? ty : tx;
        }
        if (C) { x = (x + h) % n; y = (y + h) % n; }
        if (pp && x < y) { std::swap(x, y); sg = -sg; }
        const int e = at[x + y * n];
        ok = e >= 0;
        g.to.push_back(e);
        g.sg.push_back(sg);
      }
      if (ok) gen.push_back(g);
    }
    // B(p, q), symmetric, summed over the group: 4 rounds reach every product
    std::vector<double> B((size_t)s * s, 0.0);
    for (int p = 0; p < s; ++p)
      for (int q = 0; q <= p; ++q)
        if (!sparse || pick(0, 2 * s) == 0 || p == q) B[p + (size_t)q * s] = B[q + (size_t)p * s] = pick(-9, 9);
    for (const P& g : gen) {
      std::vector<double> D = B;
      for (int p = 0; p < s; ++p)
        for (int q = 0; q < s; ++q) D[g.to[q] + (size_t)g.to[p] * s] += g.sg[p] * g.sg[q] * B[q + (size_t)p * s];
      B = D;
    }
    // the largest orbit of the symmetries it has now
    size_t largest = 1;
    for (int k = 0; k < s; ++k) {
      std::vector<int> orbit(1, k);
      for (size_t i = 0; i < orbit.size(); ++i)
        for (const P& g : gen)
          if (std::find(orbit.begin(), orbit.end(), g.to[orbit[i]]) == orbit.end()) orbit.push_back(g.to[orbit[i]]);
      largest = std::max(largest, orbit.size());
    }
    if (broken && s > 2) {
      B[0] += 1000.0;                     // no longer like any image
      bool moved = false;
      for (const P& g : gen) moved = moved || g.to[0] != 0;
      if (moved) largest = 0;             // (which symmetries are left is not followed)
    }
    const std::vector<double> B0 = B;      // (B is reduced in place)
    std::vector<double> tmp;
    B.resize(block_len(s));
    const Reduced R = reduce_class(basis, pp, el, B.data(), [&](int e) { return at[e]; }, tmp);
    int got = 1, elements = 0, sums = 0;
    for (const Orbit& o : R.orb) { got = std::max(got, o.m); elements += o.m; }
    for (int z : R.size) sums += z;
    if (elements != s || sums != s) { std::printf("class of %d: %d elements, %d sums\n", s, elements, sums); return 1; }
    if (largest && got != (int)largest && (!sparse || got < (int)largest) && s > 2) {
      std::printf("class of %d: orbits of %d, expected %d\n", s, got, (int)largest);
      return 1;
    }
    // x -> sums -> blocks -> elements against B x
    std::vector<double> x(s), X(s, 0.0), C(s, 0.0), y(s, 0.0);
    for (double& v : x) v = pick(-20, 20);
    auto sign = [](const Orbit& o, int j, int i) { return (o.mask >> (4 * j + i) & 1u) ? -1.0 : 1.0; };
    std::vector<int> used(s, 0);
    for (const Orbit& o : R.orb)
      for (int j = 0; j < o.m; ++j) {
        if (o.pos[j] < 0 || o.pos[j] >= s || used[o.pos[j]]++) { std::printf("position %d\n", o.pos[j]); return 1; }
        for (int i = 0; i < o.m; ++i) X[o.pos[j]] += sign(o, j, i) * x[at[o.lin[i]]];
      }
    size_t w0 = 0;
    int off = 0;
    for (int z : R.size) {
      for (int k = 0; k < z; ++k)
        for (int j = 0; j < z; ++j) C[off + j] += B[w0 + (size_t)k * z + j] * X[off + k];
      off += z;
      w0 += block_len(z);
      if (s > 2) {                        // (two elements can agree by chance)
        reduced += (long long)z * z;
        splits += z && z < s;
      }
    }
    for (const Orbit& o : R.orb)
      for (int i = 0; i < o.m; ++i)
        for (int j = 0; j < o.m; ++j) y[at[o.lin[i]]] += sign(o, j, i) * C[o.pos[j]];
    for (int p = 0; p < s; ++p) {
      double v = 0.0;
      for (int q = 0; q < s; ++q) v += B0[q + (size_t)p * s] * x[q];
      if (v != y[p]) { std::printf("class of %d, element %d: %g instead of %g\n", s, p, y[p], v); return 1; }
    }
    if (s > 2) whole += (long long)s * s;
  }
  std::printf("%lld %lld %lld\n", whole, reduced, splits);
  return 0;
}
"""


@pytest.fixture(scope="module")
def program(tmp_path_factory):
    d = tmp_path_factory.mktemp("blocks")
    src, exe = d / "b.cpp", d / "b"
    src.write_text(PROGRAM)
    flags = ["-std=c++17", "-O1", "-g", "-fsanitize=undefined", "-fno-sanitize-recover",
             "-D_GLIBCXX_ASSERTIONS", "-I", CSRC]
    subprocess.run(["g++", *flags, str(src), "-o", str(exe)], check=True)
    return str(exe)


@pytest.mark.parametrize("broken", [0, 1])
@pytest.mark.parametrize("sparse", [0, 1])
@pytest.mark.parametrize("odd", [0, 1])
@pytest.mark.parametrize("kind", [0, 1, 2, 4, 3])
@pytest.mark.parametrize("channel", ["ph", "pp"])
def test_reduced_blocks_equal_whole_ones(program, channel, kind, odd, sparse, broken):
    r = subprocess.run([program, channel, str(kind), str(odd), str(sparse), str(broken)],
                       capture_output=True, text=True, timeout=60)
    assert r.returncode == 0, r.stdout + r.stderr
    whole, reduced, splits = map(int, r.stdout.split())
    if kind == 0 and not sparse:
        assert reduced == whole and splits == 0
    if kind and not broken:
        assert reduced < whole and splits > 0
