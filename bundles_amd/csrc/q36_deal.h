// How decode attention deals one call's keys to the workgroups of a KV head: the integer arithmetic, for the
// kernels, the host and a program that checks it over many batches on the CPU.
#pragma once
#include <stdint.h>

namespace q36 {

constexpr int kST = 32;              // keys per wave step
constexpr int kMinPiece = 4, kWhole = 8;
constexpr int ovh(int RT) { return RT == 1 ? 8 : 16; }

__host__ __device__ __forceinline__ int req_steps(int nk) { return nk > 0 ? (nk + kST - 1) / kST : 0; }

// The host's part, from the page table's width: the steps a request can have, whether no request is cut, and the
// workgroups a KV head gets of the `places` that fit on the chip (no more than pieces of a table of this width).
inline int table_steps(int width) { return (width - 1) / kST + 1; }
inline int table_uncut(int max_steps) { return max_steps <= kMinPiece; }
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
// n pieces of at most c steps, of a call whose line is `total` long: whether they are taken (they fit, and c is the
// least or not much more than an equal share)
__host__ __device__ __forceinline__ bool pieces_taken(int RT, int n, int c, int total, int Gp) {
  const int slack = RT == 1 ? 8 : 4, most = total / Gp + total / (slack * Gp) + 2;
  return n <= Gp && (c <= kMinPiece || c <= most);
}

// ---- the line
// Shares of the line.  No more than positions: G comes from the page table's width and total from the lengths, and the
// combine reads a partial of every share between a request's first and last, so none of these may be empty (a
// workgroup past the last share leaves).
__host__ __device__ __forceinline__ int line_shares(int total, int G) { return total < G ? total : G; }
// share w of nsh begins at total * w / nsh; the share that holds position x
__host__ __device__ __forceinline__ int share_begin(int total, int nsh, int w) { return (int)((int64_t)total * w / nsh); }
__host__ __device__ __forceinline__ int share_of(int total, int nsh, int x) {
  return (int)((((int64_t)x + 1) * nsh - 1) / total);
}

// A run of a request's steps [st0, st0 + nst) and what becomes of it: 0 the whole request (written out), 1 a partial, 2
// a request's first partial.  nst < 0: the share holds no step of the request.
struct DealRun {
  int st0, nst, part;
};
// Piece p of n of a request of `steps`.
__host__ __device__ __forceinline__ DealRun piece_run(int steps, int n, int p) {
  const int per = steps / n, rem = steps % n;
  return DealRun{p * per + (p < rem ? p : rem), per + (p < rem ? 1 : 0), n > 1 ? 1 + (p == 0) : 0};
}
// The share [x0, x1) of the line against a request of `steps` whose weight begins at off0.  whole: it is not cut.
__host__ __device__ __forceinline__ DealRun line_run(int steps, int off0, int half, bool whole, int x0, int x1) {
  if (whole) return DealRun{0, off0 < x0 ? -1 : steps, 0};
  const int off = off0 + half;  // of its first step
  const int e = x1 - off < steps ? x1 - off : steps, st0 = x0 > off ? x0 - off : 0, nst = e - st0;
  return DealRun{st0, nst > 0 ? nst : -1, nst == steps ? 0 : 1 + (st0 == 0)};
}
// Where a request's pieces lie: the partial of workgroup w (of its KV head) at slot 4 w + 2 h + part - 1, the pieces
// of one request in the workgroups first .. last.
__host__ __device__ __forceinline__ int part_slot(int w, int h, int part) { return 2 * (2 * w + h) + (part == 2); }

}  // namespace q36
