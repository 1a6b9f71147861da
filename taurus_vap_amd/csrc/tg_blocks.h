// The interaction's blocks and their reduction by symmetry (host).
//
// A channel's blocks hold the elements (x, y) of one class: (2m_x - 2m_y, 2t_x - 2t_y, parity)
// in ph, the sums of them for x > y in pp.
//
// The interaction's symmetries are signed permutations of a block's elements:
//   ph: time reversal with hermiticity, (a,c) -> (c~,a~);  pp: time reversal,
//       (x,y) -> (x~,y~); the signs follow from the elements;
//   charge reflection, proton <-> neutron of every state (+1 in ph; a stored pp pair
//       changes its order, -1), and the product of the two.
// One that maps a block to itself and leaves its matrix the same BIT BY BIT (checked at
// tg_init on the values as stored, so no element is changed; a charge-dependent
// interaction, or one whose elements carry different rounding, simply does not pass)
// commutes with the block: the elements fall into orbits, and the sums
// a_chi(O) = sum_p c_chi(p) x_p over an orbit, c = +-1, mix only within a character
// chi.  A block of s elements becomes 2 (or 4) of about s/2 (s/4): half (a quarter) of
// the multiply-adds.  Their elements are sums of 2 (4) stored ones over the power of two
// |O|, rounded to FP64 once (exact for FP32 elements within 29 binary places of each other),
// and take the bytes of the FP32 block.  A block with no symmetry keeps its elements as
// stored (FP32 when the TBMEs are FP32).
#pragma once
#include <algorithm>
#include <map>
#include <tuple>
#include <utility>
#include <vector>

// Single-particle states in the order the matrices are kept in
struct SpBasis {
  int n;
  const std::vector<int>&sp_2mj, &sp_2mt, &sp_l, &sp_tr;   // sp_tr from 0
};

// An orbit of matrix elements under the symmetries of its block and the sums the
// contraction takes over it (kernels of tg_fields.hip); m elements and m sums.
struct Orbit {
  int lin[4];                   // linear indices x + y*n of the elements
  int pos[4];                   // positions of the sums
  unsigned mask;                // bit 4 j + i: element i enters sum j with a minus
  int m;
};

typedef std::tuple<int, int, int> ClassKey;

// Elements of a block channel by class, in patches of 8 x 8 (linear indices x + y n)
inline std::map<ClassKey, std::vector<int>> channel_classes(const SpBasis& c, bool pp) {
  const int n = c.n;
  const std::vector<int>&m = c.sp_2mj, &t = c.sp_2mt, &l = c.sp_l;
  // runs of states with the same m, t and parity; the elements of two runs are of one class
  std::vector<int> run(1, 0);
  for (int i = 1; i < n; ++i)
    if (m[i] != m[i - 1] || t[i] != t[i - 1] || (l[i] & 1) != (l[i - 1] & 1)) run.push_back(i);
  run.push_back(n);
  std::map<ClassKey, std::vector<int>> cls;
  for (size_t rx = 0; rx + 1 < run.size(); ++rx)
    for (size_t ry = 0; ry + 1 < run.size(); ++ry) {
      const int x0 = run[rx], x1 = run[rx + 1], y0 = run[ry], y1 = run[ry + 1];
      if (pp && x1 - 1 <= y0) continue;              // (every x > y)
      std::vector<int>& el = cls[pp ? ClassKey(m[x0] + m[y0], t[x0] + t[y0], (l[x0] + l[y0]) & 1)
                                    : ClassKey(m[x0] - m[y0], t[x0] - t[y0], (l[x0] + l[y0]) & 1)];
      for (int yb = y0; yb < y1; yb += 8)
        for (int xb = x0; xb < x1; xb += 8)
          for (int y = yb; y < std::min(yb + 8, y1); ++y)
            for (int x = xb; x < std::min(xb + 8, x1); ++x)
              if (!pp || x > y) el.push_back(x + y * n);
    }
  return cls;
}

// A signed permutation of a class: element k -> to[k] with sign sg[k]
struct Sym {
  std::vector<int> to, sg;
};

// Whether B(to p, to q) = sg_p sg_q B(p, q) for all p, q, bit by bit (B symmetric in
// meaning, stored at B[q + p s], p the input).  With `find` the signs are found first: +-1 spread
// over the elements that B connects, an element and its images (imgs) alike.
inline bool sym_holds(const double* B, int s, Sym& g, bool find,
                      const std::vector<const std::vector<int>*>& imgs) {
  if (find) {
    g.sg.assign(s, 0);
    std::vector<int> todo;
    auto visit = [&](int k, int sg) {
      std::vector<int> st(1, k);
      while (!st.empty()) {
        const int e = st.back();
        st.pop_back();
        if (g.sg[e] != 0) continue;
        g.sg[e] = sg;
        todo.push_back(e);
        for (const std::vector<int>* im : imgs) st.push_back((*im)[e]);
      }
    };
    for (int r = 0; r < s; ++r) {
      if (g.sg[r] != 0) continue;
      visit(r, 1);
      while (!todo.empty()) {
        const int p = todo.back();
        todo.pop_back();
        const double* bp = B + (size_t)p * s;
        const double* bt = B + (size_t)g.to[p] * s;
        for (int q = 0; q < s; ++q)
          if (g.sg[q] == 0 && bp[q] != 0.0) visit(q, (bp[q] == bt[g.to[q]]) ? g.sg[p] : -g.sg[p]);
      }
    }
  }
  for (int p = 0; p < s; ++p) {
    const double* bp = B + (size_t)p * s;
    const double* bt = B + (size_t)g.to[p] * s;
    const double sp = g.sg[p];
    for (int q = 0; q < s; ++q)
      if (!(bt[g.to[q]] == sp * g.sg[q] * bp[q])) return false;
  }
  return true;
}

// One class of a channel reduced by its symmetries: its orbits (positions relative to
// the class) and the orders of the character blocks.
struct Reduced {
  std::vector<Orbit> orb;
  std::vector<int> size;
  bool split = false;
};

// Elements a block of order s takes: a whole number of 16 bytes
inline size_t block_len(size_t s) { return (s * s + 1) / 2 * 2; }

// Reduces a class in place: the blocks (matrix [in * size + out], block_len(size) apart)
// replace B, which has room for block_len(s).  place(e): index of element e in the
// class, or -1; tmp: scratch.

template <typename Place>
Reduced reduce_class(const SpBasis& c, bool pp, const std::vector<int>& el, double* B, const Place& place,
                     std::vector<double>& tmp) {
  const int n = c.n, h = n / 2, s = (int)el.size();
  // the proton and the neutron half hold the same states, in the same order
  bool halves = true;
  for (int i = 0; i < h && halves; ++i)
    halves = c.sp_2mj[i] == c.sp_2mj[i + h] && c.sp_l[i] == c.sp_l[i + h] &&
             c.sp_tr[i] < h && c.sp_tr[i + h] == c.sp_tr[i] + h;
  bool tr_ok = true;
  for (int i = 0; i < n && tr_ok; ++i) tr_ok = c.sp_tr[c.sp_tr[i]] == i && c.sp_tr[i] != i;
  // image of element (x, y): time reversal (and transposition in ph), reflection; the
  // sign where a pp pair changes its order
  auto image = [&](int e, bool tr, bool ch, int& sg) {
    int x = e % n, y = e / n;
    sg = 1;
    if (tr) {
      const int tx = c.sp_tr[x], ty = c.sp_tr[y];
      x = pp ? tx : ty;
      y = pp ? ty : tx;
    }
    if (ch) {
      x = (x + h) % n;
      y = (y + h) % n;
    }
    if (pp && x < y) {
      std::swap(x, y);
      sg = -1;
    }
    return x + y * n;
  };
  Sym g[3];               // time reversal, reflection, their product
  bool ok[3];
  for (int q = 0; q < 3; ++q) {
    const bool tr = q != 1, ch = q != 0;
    ok[q] = (!tr || tr_ok) && (!ch || halves) && s > 1;
    g[q].to.assign(s, 0);
    g[q].sg.assign(s, 1);
    for (int k = 0; k < s && ok[q]; ++k) {
      g[q].to[k] = place(image(el[k], tr, ch, g[q].sg[k]));
      ok[q] = g[q].to[k] >= 0;
    }
    for (int k = 0; k < s && ok[q]; ++k) ok[q] = g[q].to[g[q].to[k]] == k;
  }
  std::vector<const std::vector<int>*> imgs;
  for (int q = 0; q < 3; ++q)
    if (ok[q]) imgs.push_back(&g[q].to);
  // the reflection's signs are known; those with time reversal are found
  if (ok[1]) ok[1] = sym_holds(B, s, g[1], false, imgs);
  if (ok[0]) ok[0] = sym_holds(B, s, g[0], true, imgs);
  if (ok[2] && !(ok[0] && ok[1])) ok[2] = sym_holds(B, s, g[2], true, imgs);
  // signs of an involution agree on an element and its image
  for (int q = 0; q < 3; ++q)
    for (int k = 0; k < s && ok[q]; ++k) ok[q] = g[q].sg[k] == g[q].sg[g[q].to[k]];
  std::vector<const Sym*> gen;
  if (ok[0] && ok[1]) {
    bool commute = true;
    for (int k = 0; k < s && commute; ++k)
      commute = g[0].to[g[1].to[k]] == g[1].to[g[0].to[k]] &&
                g[0].sg[g[1].to[k]] * g[1].sg[k] == g[1].sg[g[0].to[k]] * g[0].sg[k];
    gen.push_back(&g[0]);
    if (commute) gen.push_back(&g[1]);
  } else {
    for (int q = 0; q < 3; ++q)
      if (ok[q]) {
        gen.push_back(&g[q]);
        break;
      }
  }
  Reduced R;
  R.split = !gen.empty();
  if (!R.split) {
    R.size.assign(1, s);
    R.orb.resize(s);
    for (int k = 0; k < s; ++k) {
      R.orb[k] = Orbit{};
      R.orb[k].lin[0] = el[k];
      R.orb[k].pos[0] = k;
      R.orb[k].m = 1;
    }
    return R;
  }
  const int ng = (int)gen.size(), order = 1 << ng;
  // orbits: element e_b = (product of the generators in b) of the first one, its sign
  std::vector<char> seen(s, 0);
  R.size.assign(order, 0);
  std::vector<std::vector<int>> members;          // elements of each orbit (class index)
  std::vector<unsigned> masks;                    // bit 4 j + i: minus of element i in sum j
  std::vector<std::vector<int>> chars;            // character of each of the orbit's sums
  for (int k = 0; k < s; ++k) {
    if (seen[k]) continue;
    int im[4], sg[4];
    for (int b = 0; b < order; ++b) {
      int e = k, sgn = 1;
      for (int q = 0; q < ng; ++q)
        if (b >> q & 1) {
          sgn *= gen[q]->sg[e];
          e = gen[q]->to[e];
        }
      im[b] = e;
      sg[b] = sgn;
    }
    std::vector<int> mem, first;
    for (int b = 0; b < order; ++b)
      if (std::find(mem.begin(), mem.end(), im[b]) == mem.end()) {
        mem.push_back(im[b]);
        first.push_back(b);
        seen[im[b]] = 1;
      }
    std::vector<int> ch;
    unsigned mask = 0;
    for (int x = 0; x < order; ++x) {
      // character x: sign (-1)^(bits of b & x) of the group element b
      auto cs = [&](int b) { return (__builtin_popcount(b & x) & 1 ? -1 : 1) * sg[b]; };
      bool fits = true;
      for (int b = 0; b < order && fits; ++b)
        for (int b2 = 0; b2 < b && fits; ++b2)
          if (im[b] == im[b2]) fits = cs(b) == cs(b2);
      if (!fits) continue;
      const int j = (int)ch.size();
      for (size_t i = 0; i < mem.size(); ++i)
        if (cs(first[i]) < 0) mask |= 1u << (4 * j + (int)i);
      ch.push_back(x);
    }
    members.push_back(mem);
    masks.push_back(mask);
    chars.push_back(ch);
    for (int x : ch) ++R.size[x];
  }
  // positions: character blocks one after another, orbits in order inside each
  std::vector<int> base(order, 0), fill(order, 0);
  std::vector<size_t> wbase(order, 0);
  size_t wsz = 0;
  for (int x = 0, o = 0; x < order; ++x) {
    base[x] = o;
    o += R.size[x];
    wbase[x] = wsz;
    wsz += block_len(R.size[x]);
  }
  tmp.assign(wsz, 0.0);
  const size_t no = members.size();
  std::vector<std::vector<int>> idx(no);          // index of each of its sums in its block
  for (size_t o = 0; o < no; ++o) {
    Orbit ob{};
    ob.m = (int)members[o].size();
    ob.mask = masks[o];
    for (int i = 0; i < ob.m; ++i) {
      ob.lin[i] = el[members[o][i]];
      const int x = chars[o][i];
      idx[o].push_back(fill[x]);
      ob.pos[i] = base[x] + fill[x]++;
    }
    R.orb.push_back(ob);
  }
  // the first elements of the orbits of each block, in its order: the outputs of a row
  std::vector<std::vector<int>> head(order);
  for (size_t o = 0; o < no; ++o)
    for (int x : chars[o]) head[x].push_back(members[o][0]);
  for (size_t o = 0; o < no; ++o)
    for (size_t j = 0; j < chars[o].size(); ++j) {
      const int x = chars[o][j], size = R.size[x], m = (int)members[o].size();
      const int* out = head[x].data();
      double* w = tmp.data() + wbase[x] + (size_t)idx[o][j] * size;
      const double* row[4];
      double sg[4];
      for (int i = 0; i < m; ++i) {
        row[i] = B + (size_t)members[o][i] * s;
        sg[i] = (masks[o] >> (4 * j + i) & 1u) ? -1.0 : 1.0;
      }
      const double over = 1.0 / m;             // a power of two
      // (0.0 +: no element is a negative zero)
      if (m == 1)
        for (int k = 0; k < size; ++k) w[k] = 0.0 + sg[0] * row[0][out[k]];
      else if (m == 2)
        for (int k = 0; k < size; ++k) w[k] = ((0.0 + sg[0] * row[0][out[k]]) + sg[1] * row[1][out[k]]) * over;
      else
        for (int k = 0; k < size; ++k)
          w[k] = ((((0.0 + sg[0] * row[0][out[k]]) + sg[1] * row[1][out[k]]) + sg[2] * row[2][out[k]]) +
                  sg[3] * row[3][out[k]]) * over;
    }
  std::copy(tmp.begin(), tmp.end(), B);
  return R;
}
