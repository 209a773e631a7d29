// Walks the dealing of decode attention's keys (csrc/q36_deal.h) on the host: what the split kernel's workgroups
// write and what the combine kernel reads, over many batches.  Prints each batch that fails and exits 1.
//   deal_check SEED BATCHES
#include <algorithm>
#include <cmath>
#include <cstdio>
#include <cstdlib>
#include <random>
#include <vector>

#define __host__
#define __device__
#define __forceinline__ inline
#include "q36_deal.h"

using namespace q36;

// One KV head (h), one batch: the split kernel's steps per request and partial slots, then the combine's reads.
static const char* walk(const std::vector<int>& len, int RT, int width, int cus, int h) {
  // (the split count of the equal splits, as the host passes it on)
  const int so = std::max(1, std::min(64, cus / (2 * (int)len.size())));
  const int splits = so <= (RT == 1 ? 4 : 2) && (int)len.size() * 2 * so <= (RT == 1 ? 2 : 1) * cus ? so : 0;
  const int B = (int)len.size(), max_steps = table_steps(width), nocut = table_uncut(max_steps);
  const int G = deal_groups(B, max_steps, (RT == 1 ? 2 : 1) * cus / 2);
  std::vector<int> st(B), first(B, -1), last(B, -1), whole(B, 0), firsts(B, 0), lasts(B, 0);
  std::vector<std::vector<int>> done(B);
  int steps = 0, longest = 0;
  for (int b = 0; b < B; ++b) {
    st[b] = std::min(req_steps(len[b]), max_steps);
    steps += st[b], longest = std::max(longest, st[b]);
    done[b].assign(req_steps(len[b]), 0);
  }
  const int total = steps + B * ovh(RT), Gp = piece_places(RT, B, G, steps), c0 = piece_least(steps, Gp);
  const int even = even_pieces(RT, B, G, G / B, splits, steps, longest);
  std::vector<int> pieces(B, even);  // of each request, where the call is dealt in pieces
  int np = even * B;
  if (!np && B <= std::min(Gp, 256)) {
    for (int k = 0; k < kSizes; ++k) {
      int n = 0;
      for (int b = 0; b < B; ++b) n += pieces[b] = req_pieces(st[b], piece_size(c0, k));
      if (n > Gp) continue;
      if (piece_size(c0, k) <= piece_most(RT, total, Gp)) np = n;
      // (the kernel does not search where this many requests are too long)
      if (np && B + std::count_if(st.begin(), st.end(), [&](int v) { return v > piece_most(RT, total, Gp); }) > Gp)
        return "pieces that fit are not searched for";
      break;
    }
  }
  const int nsh = line_shares(total, G);
  const int slots = 4 * (RT == 1 ? cus : cus / 2);  // of 16 RT rows
  std::vector<int> owner(slots, -1);                // request that wrote the slot in this call
  const char* err = nullptr;
  auto run = [&](int b, const DealRun& r, int w) {
    if (r.st0 < 0 || r.st0 + r.nst > (int)done[b].size()) err = "a run outside its request";
    for (int s = r.st0; !err && s < r.st0 + r.nst; ++s) ++done[b][s];
    if (r.part == 0 || (r.part & kFirst)) first[b] = r.part ? w : 0, ++firsts[b];
    if (r.part == 0 || (r.part & kLast)) last[b] = r.part ? w : 0, ++lasts[b];
    if (r.part == 0) {
      ++whole[b];
      return;
    }
    const int slot = part_slot(w, h, r.part);
    if (w >= G) err = "a piece past the workgroups";
    else if (slot < 0 || slot >= slots) err = "a slot outside the workspace";
    else if (owner[slot] >= 0) err = "a slot written twice";
    else owner[slot] = b;
  };
  if (np) {
    for (int b = 0, w = 0; b < B; ++b)
      for (int p = 0; p < pieces[b]; ++p, ++w) run(b, piece_run(req_steps(len[b]), pieces[b], p), w);
  } else {
    for (int w = 0; w < nsh; ++w) {
      const int x0 = share_begin(total, nsh, w), x1 = share_begin(total, nsh, w + 1);
      for (int b = 0, off = 0; b < B; ++b) {
        const int wt = st[b] + ovh(RT), off0 = off, n_all = req_steps(len[b]);
        off += wt;
        if (off <= x0 || off0 >= x1) continue;
        const DealRun r = line_run(n_all, off0, ovh(RT) / 2, n_all <= kWhole || n_all > max_steps, x0, x1);
        if (r.nst >= 0) run(b, r, w);
      }
    }
  }
  if (err) return err;
  int used = 0;
  for (int b = 0; b < B; ++b) {
    for (int d : done[b])
      if (d != 1) return "a step not in exactly one run";
    if (firsts[b] != 1 || lasts[b] != 1) return "a request whose pieces are not told to the combine once";
    const int n = last[b] - first[b] + 1;
    if ((n <= 1) != (whole[b] == 1) || whole[b] > 1) return "a request neither whole nor in pieces";
    if (n <= 1) continue;
    if (nocut) return "a cut request without a combine";
    for (int p = 0; p < n; ++p) {
      const int slot = part_slot(first[b] + p, h, p == 0 ? kFirst : 0);
      if (slot >= slots || owner[slot] != b) return "the combine reads a slot that this call did not write";
      ++used;
    }
  }
  if (used != (int)std::count_if(owner.begin(), owner.end(), [](int o) { return o >= 0; })) return "a partial not read";
  return nullptr;
}

int main(int argc, char** argv) {
  std::mt19937 g(argc > 1 ? atoi(argv[1]) : 0);
  const int batches = argc > 2 ? atoi(argv[2]) : 1000;
  auto uni = [&](int lo, int hi) { return (int)(lo + g() % (unsigned)(hi - lo + 1)); };
  auto logu = [&](int lo, int hi) {  // spread over the logarithm
    const double u = (double)g() / 4294967296.0;
    return std::max(lo, std::min(hi, (int)(lo * std::pow((hi + 1.0) / lo, u))));
  };
  int bad = 0;
  auto check = [&](const std::vector<int>& len, int RT, int width, int cus) {
    const char* e = walk(len, RT, width, cus, uni(0, 1));
    if (!e) return;
    if (++bad <= 10)
      printf("B=%zu row tiles %d width %d CUs %d lengths %d .. %d: %s\n", len.size(), RT, width, cus,
             *std::min_element(len.begin(), len.end()), *std::max_element(len.begin(), len.end()), e);
  };
  // equal lengths in tables as wide as they are and much wider
  for (int RT = 1; RT <= 2; ++RT)
    for (int B = 1; B <= 300; B = B < 20 ? B + 1 : B + B / 7)
      for (int width : {128, 384, 1280, 4096, 32768, 262144})
        for (int len = 0; len <= std::min(width, 40000); len = len < 40 ? len + 13 : len + len / 5)
          check(std::vector<int>(B, len), RT, width, 256);
  // ragged batches: widths from the longest request's up to 262144, some requests empty, a few longer than the table
  for (int i = 0; i < batches; ++i) {
    const int B = uni(0, 3) ? logu(1, 300) : logu(1, 3000), hi = logu(1, B > 300 ? 2000 : 40000), lo = uni(0, 1) ? hi : logu(1, hi);
    std::vector<int> len(B);
    for (int& n : len) n = uni(0, 15) ? logu(lo, hi) : 0;
    if (uni(0, 3) == 0) len[uni(0, B - 1)] = logu(1, 100000);
    const int longest = std::max(1, *std::max_element(len.begin(), len.end()));
    const int width = uni(0, 9) == 0 ? std::max(1, longest - uni(0, 100)) : std::min(262144, longest + (uni(0, 1) ? uni(0, 3) : logu(1, 262144)));
    check(len, 1 + uni(0, 1), width, uni(0, 7) ? 256 : uni(2, 304) & ~1);
  }
  printf("%d of the batches fail\n", bad);
  return bad != 0;
}
