// How decode attention deals one call's keys to the workgroups of a KV head: the integer arithmetic, for the
// kernels, the host and a program that checks it over many batches on the CPU.
#pragma once
#include <stdint.h>

namespace q36 {

constexpr int kST = 32;              // keys per wave step
constexpr int kMinPiece = 4, kWhole = 8;
constexpr int kAlone = 12, kEven = 40;  // even dealing: steps
constexpr int even_over(int RT) { return RT == 1 ? 18 : 12; }
constexpr int ovh(int RT) { return RT == 1 ? 8 : 16; }

__host__ __device__ __forceinline__ int req_steps(int nk) { return nk > 0 ? (nk + kST - 1) / kST : 0; }

// The host's part, from the page table's width: the steps a request can have, whether every request is dealt whole, and
// the workgroups a KV head gets of the `places` that fit on the chip (no more than pieces of a table of this width).
inline int table_steps(int width) { return (width - 1) / kST + 1; }
inline int table_uncut(int max_steps) { return max_steps <= kAlone; }
inline int deal_groups(int B, int max_steps, int places) {
  const int64_t pieces = (int64_t)B * ((max_steps - 1) / kMinPiece + 1);
  return pieces < places ? (int)pieces : places > 1 ? places : 1;
}

// ---- pieces: Gp workgroups take part; the sizes tried are c0 and 15 more up to about 2 c0
__host__ __device__ __forceinline__ int piece_places(int RT, int B, int G, int steps) {
  return RT == 1 && B <= G / 2 && steps >= kMinPiece * (G / 2) ? G / 2 : G;
}
__host__ __device__ __forceinline__ int piece_least(int steps, int Gp) {
  const int c = (steps + Gp - 1) / Gp;
  return c > kMinPiece ? c : kMinPiece;
}
constexpr int kSizes = 16;
__host__ __device__ __forceinline__ int piece_size(int c0, int k) { return c0 + (c0 * k + kSizes - 1) / kSizes; }
__host__ __device__ __forceinline__ int req_pieces(int steps, int c) { return steps > c ? (steps + c - 1) / c : 1; }
constexpr int piece_slack(int RT) { return RT == 1 ? 8 : 4; }
// The largest piece taken, of a call whose line is `total` long: the least, or not much more than an equal share
__host__ __device__ __forceinline__ int piece_most(int RT, int total, int Gp) {
  const int c = total / Gp + total / (piece_slack(RT) * Gp) + 2;
  return c > kMinPiece ? c : kMinPiece;
}

// ---- even: every request in the same number of pieces, piece p of request b at workgroup b n + p
// From the page table's width alone (0: not): whole requests up to kAlone steps, and `splits` (0: none) of at most
// kEven steps, in the two-row-tile form of kEven steps together.
inline int even_table(int RT, int splits, int max_steps) {
  if (max_steps <= kAlone) return 1;
  return max_steps <= kEven * (RT == 1 ? splits : splits > 0) ? splits : 0;
}
// From the lengths: whole requests up to kAlone steps; `splits` while a piece of the longest is no more than even_over
// steps above a workgroup's share of all steps (what dealing the steps out more evenly costs); as many as fit where all
// lengths are alike.  per: the requests' share of the G workgroups, G / B.
// Measured, us a call (steps above the share: even, other): one row tile 101 x 2 rows over 250 .. 877 keys (15) 22.5, 24.2;
// 240 x 1 over 300 .. 900 (12) 39.6, 42.8; 40 x 1 over 100 .. 3000 (23) 25.2, 17.9; 70 x 2 over 20 .. 1280 (35) 23.0,
// 16.7; two row tiles 128 x 4 over 200 .. 700 (8) 27.3, 29.8; 64 x 4 over 20 .. 1280 (15) 28.0, 23.5.
__host__ __device__ __forceinline__ int even_pieces(int RT, int B, int G, int per, int splits, int steps, int longest) {
  if (longest <= kAlone) return 1;
  const int Gp = piece_places(RT, B, G, steps);
  if (splits > 0 && (int64_t)longest * Gp <= (int64_t)splits * (steps + even_over(RT) * Gp)) return splits;
  if (B > G || steps != B * longest) return 0;
  const int most = Gp < G ? per / 2 : per, fit = (longest + kMinPiece - 1) / kMinPiece;
  const int k = most < fit ? most : fit, slack = piece_slack(RT), total = steps + B * ovh(RT);
  // longest / k steps a piece, against piece_most
  return k == fit || (int64_t)longest * (slack * Gp) <= k * ((int64_t)total * (slack + 1) + 2 * slack * Gp) ? k : 0;
}

// ---- the line
// Shares of the line.  No more than positions: G comes from the page table's width and total from the lengths, and the
// combine reads a partial of every share between a request's first and last, so none of these may be empty (a
// workgroup past the last share leaves).
__host__ __device__ __forceinline__ int line_shares(int total, int G) { return total < G ? total : G; }
// share w of nsh begins at total * w / nsh (in 32 bits: the remainder's part is below nsh * nsh)
__host__ __device__ __forceinline__ int share_begin(int total, int nsh, int w) {
  const int q = total / nsh, r = total - q * nsh;
  return q * w + r * w / nsh;
}

// A run of a request's steps [st0, st0 + nst) and what becomes of it: 0 the whole request (written out), else a partial
// (kPart), a request's first and last so marked.  nst < 0: the share holds no step of the request.
constexpr int kPart = 1, kFirst = 2, kLast = 4;
struct DealRun {
  int st0, nst, part;
};
// Piece p of n of a request of `steps`.
__host__ __device__ __forceinline__ DealRun piece_run(int steps, int n, int p) {
  if (n == 1) return DealRun{0, steps, 0};
  const int per = steps / n, rem = steps - per * n;
  return DealRun{p * per + (p < rem ? p : rem), per + (p < rem ? 1 : 0), kPart | (p == 0 ? kFirst : 0) | (p == n - 1 ? kLast : 0)};
}
// The share [x0, x1) of the line against a request of `steps` whose weight begins at off0.  whole: it is not cut.
__host__ __device__ __forceinline__ DealRun line_run(int steps, int off0, int half, bool whole, int x0, int x1) {
  if (whole) return DealRun{0, off0 < x0 ? -1 : steps, 0};
  const int off = off0 + half;  // of its first step
  const int e = x1 - off < steps ? x1 - off : steps, st0 = x0 > off ? x0 - off : 0, nst = e - st0;
  return DealRun{st0, nst > 0 ? nst : -1, nst == steps ? 0 : kPart | (st0 == 0 ? kFirst : 0) | (e == steps ? kLast : 0)};
}
// The partial of workgroup w (of KV head h); a workgroup can hold one request's last piece and the next one's first.
// The pieces of a request lie in consecutive workgroups.
__host__ __device__ __forceinline__ int part_slot(int w, int h, int part) { return 2 * (2 * w + h) + (part & kFirst ? 1 : 0); }

}  // namespace q36
