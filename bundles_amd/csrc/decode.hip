// Decode / verify attention for gfx950 over an e4m3 KV cache: 16 query heads grouped onto 2 KV
// heads of 256 dims, up to 4 query tokens per request (the verify draft; 1 for plain decode) with
// the causal rule among them, one-token pages through a page table, split over the keys.
//
// Reference behaviour (R = qwen36_nodes_kb34, L = R/qwen36_layer): L/qk_attn_verify.cu:354-760
// (attn_verify_kernel: q -> e4m3, scores of e4m3 q and k, base-2 online softmax, P rounded to
// f16 for P V with V widened to f16, the split partials and their combine), L/attn_fused.py:110-124
// (split count min(64, CUs / (requests * KV heads))).  The new tokens' K/V go into the cache at
// their slots first (the reference writes them there as well).  The output is the normalised
// attention bf16(o / l); the o_proj applies the sigmoid gate.
//
// Kernels:
//   kv_scatter      the new tokens' e4m3 K and V rows into the cache slots out_loc[t].
//   decode_split    workgroup = an equal share of all requests' keys (or one of a fixed number of splits
//                   of a request, when the caller asks for that), for one KV head; 4 independent waves,
//                   each streaming its own contiguous run of 32-key steps for the group's 8 query heads x NT tokens
//                   (16 or 32 query rows) with its own running max / weight sum / output, and the
//                   four are merged once at the end.  Scores S^T = K Q^T: e4m3 16x16x128 MFMA with
//                   the keys as operand A straight from the cache (registers) and the e4m3 query
//                   fragments as operand B, so a lane holds one query row: the row max needs two
//                   cross-lane steps and the output rescale is one factor per lane.  O^T += V^T P^T:
//                   f16 16x16x32 MFMA, V^T read from LDS with the transpose read (V rows staged by
//                   buffer DMA in the key order the lane's weights are in), P^T the lane's own
//                   weights rounded to f16.  Keys, values and page-table entries stream through a
//                   per-wave pipeline (2 stages at two waves a SIMD for one row tile, 4 at one wave
//                   a SIMD for two) with no workgroup barrier; the output is rescaled only
//                   when a row max grows by more than 2^8 (weights up to 2^8 are exact in f16).
//   decode_combine  a cut request's partials weighted by exp2(m_p - M) / L (a request that one
//                   workgroup holds whole is written by the split kernel itself).
#include <math.h>

#include <atomic>
#include <type_traits>

#include "q36_device.h"
#include "q36_host.h"
#include "q36_deal.h"

namespace q36 {
namespace {

constexpr int kQH = 16, kKVH = 2, kDD = 256, kGQ = kQH / kKVH, kDNT = 4, kDRows = kGQ * kDNT;
// NS (kernel template): key / value stages per wave (steps in flight + 1); the page-table entries run
// 2 NS steps ahead, so an entry's DMA is older than every key and value load a wait leaves in flight
// The two forms' shapes (alternating builds on one box, three rounds): the one-row-tile form (decode,
// NT <= 2) with 2 stages fits 224 registers and 77 KB of LDS, so two workgroups share a CU (two waves
// a SIMD): decode 189.9 -> 182.7 us against 3 stages at one wave a SIMD; the two-row-tile form
// (verify) keeps one wave a SIMD and runs 4 stages (456 registers, 145 KB): 62.0 -> 60.6 us.
constexpr int kDecNS1 = 2, kDecWPE1 = 2, kDecNS2 = 4;
constexpr int kVG = 4 * kDD + 64;    // a group of 4 value rows in LDS (64 bytes of padding)
constexpr int kVW = 8 * kVG;         // one wave's 32 value rows
constexpr int kVS = 4 * kVW;         // one stage of the four waves' value rows
constexpr float kLazy = 8.f;
// Key and value reads carry the non-temporal cache policy (nt): each row is read once per call, and
// inside the hybrid node (after a GDN verify has left ~0.5 GB of snapshot writes dirty in the
// caches) the plain reads ran at half speed, evicting that data; measured 111 -> 63 us per call.
constexpr int kKVAux = 2;         // rescale when a row max grows past the reference by 2^8
static_assert(kVS >= 2 * 16 * kDD * 4, "a stage holds two waves' fp32 output of one row tile at the merge");

typedef _Float16 v8h __attribute__((ext_vector_type(8)));
typedef _Float16 v2h __attribute__((ext_vector_type(2)));

struct DecodeDev {
  int B, NT, pt_stride;
  int splits;               // > 0: every request in this many equal splits; 0: balanced (see decode_split)
  int groups, per;          // balanced: workgroups of a KV head the keys are dealt to, and these over B
  int even;                 // balanced: the pieces of every request where the lengths allow it (0: none)
  int max_steps;            // steps the page table's width holds: the most a request weighs
  const uint16_t* q;        // bf16 [B*NT, 16, 256]
  const uint8_t* kc;        // e4m3 [slots, 2, 256]
  const uint8_t* vc;
  int64_t kv_bytes;         // bytes of each cache
  const int32_t* pt;        // [B, pt_stride]
  const int32_t* seqlens;   // [B], new tokens included
  float scale_log2;
  float* ws_o;              // [slots][16 RT][256] unnormalised partial outputs
  float* ws_ml;             // [slots][2][16 RT]: running max (base 2) and weight sum per row
  int2* meta;               // balanced: [B] first and last share of each request
  uint16_t* out;            // bf16 [B*NT, 16, 256]
  const uint16_t* gate;     // bf16 [B*NT, 16 * 256] or null: with oq, the o_proj's quantized input
  uint8_t* oq;              // e4m3 [B*NT, 16 * 256] of bf16(out * sigmoid(gate)) per 128-group
  float* oqs;               // [B*NT, 32] group scales
};

// The gate's 4 values at dims 4c .. 4c + 3 of row (token tok, head); zeros without a gate.  Read through a descriptor, so
// that no branch holds the load back.
__device__ __forceinline__ v2i gate_row(const DecodeDev& d, int tok, int head, int c) {
  const __amdgpu_buffer_rsrc_t rs = __builtin_amdgcn_make_buffer_rsrc(
      (void*)(d.gate + (size_t)tok * (kQH * kDD)), (short)0, d.oq ? kQH * kDD * 2 : 0, 0x00020000);
  return __builtin_bit_cast(v2i, __builtin_amdgcn_raw_buffer_load_b64(rs, (head * kDD + 4 * c) * 2, 0, 0));
}
// Max over each half of the wave (32 lanes), without LDS.
__device__ __forceinline__ float half_max(float v) {
  v = fmaxf(v, __uint_as_float(dpp_u32<0xB1>(__float_as_uint(v))));
  v = fmaxf(v, __uint_as_float(dpp_u32<0x4E>(__float_as_uint(v))));
  v = fmaxf(v, __uint_as_float(dpp_u32<0x141>(__float_as_uint(v))));
  v = fmaxf(v, __uint_as_float(dpp_u32<0x140>(__float_as_uint(v))));
  const auto p16 = __builtin_amdgcn_permlane16_swap(__float_as_uint(v), __float_as_uint(v), false, false);
  return fmaxf(__uint_as_float(p16[0]), __uint_as_float(p16[1]));
}
// The output's 4 values at dims 4c .. 4c + 3 of row (token tok, head) after the bf16 store: the o_proj
// input bf16(o * sigmoid(gate)) in e4m3 per 128-channel group (32 neighbouring lanes of one wave hold
// a group), the same arithmetic as the o_proj's own quantization of the bf16 output.
__device__ __forceinline__ void gated_e4m3(const DecodeDev& d, int tok, int head, int c, uint32_t o01, uint32_t o23, v2i gv) {
  const size_t at = (size_t)tok * (kQH * kDD) + head * kDD + 4 * c;
  const uint32_t g01 = (uint32_t)gv.x, g23 = (uint32_t)gv.y;
  float f[4] = {rbf_hw(bf_lo(o01) * sigmoid_q(bf_lo(g01))), rbf_hw(bf_hi(o01) * sigmoid_q(bf_hi(g01))),
                rbf_hw(bf_lo(o23) * sigmoid_q(bf_lo(g23))), rbf_hw(bf_hi(o23) * sigmoid_q(bf_hi(g23)))};
  const float m = half_max(fmaxf(fmaxf(fabsf(f[0]), fabsf(f[1])), fmaxf(fabsf(f[2]), fabsf(f[3]))));
  const float inv = m > 0.f ? 448.f / m : 0.f;
  *reinterpret_cast<uint32_t*>(d.oq + at) = f2e4m3x2_hw(f[0] * inv, f[1] * inv) | (f2e4m3x2_hw(f[2] * inv, f[3] * inv) << 16);
  if ((c & 31) == 0) d.oqs[(size_t)tok * (kQH * kDD / 128) + head * 2 + c / 32] = m / 448.f;
}

__device__ __forceinline__ v4f mfma_e4m3(v8i a, v8i b, v4f c) {
  return __builtin_amdgcn_mfma_scale_f32_16x16x128_f8f6f4(a, b, c, 0, 0, 0, 127, 0, 127);
}
__device__ __forceinline__ v8i cat8d(v4i a, v4i b) {
  v8i r = {a.x, a.y, a.z, a.w, b.x, b.y, b.z, b.w};
  return r;
}
// 8 e4m3 codes (two words) -> 8 f16 (every e4m3 value is an f16 value: exact at scale 1)
__device__ __forceinline__ v8h widen8(int w0, int w1) {
  const v2h a = __builtin_amdgcn_cvt_scalef32_pk_f16_fp8(w0, 1.f, false);
  const v2h b = __builtin_amdgcn_cvt_scalef32_pk_f16_fp8(w0, 1.f, true);
  const v2h c = __builtin_amdgcn_cvt_scalef32_pk_f16_fp8(w1, 1.f, false);
  const v2h e = __builtin_amdgcn_cvt_scalef32_pk_f16_fp8(w1, 1.f, true);
  return v8h{a.x, a.y, b.x, b.y, c.x, c.y, e.x, e.y};
}
__device__ __forceinline__ uint32_t lds_addr(const void* p) {
  return (uint32_t)(uintptr_t)((const __attribute__((address_space(3))) uint8_t*)p);
}
// LDS read by asm: the compiler counts the buffer DMA into the same array as a pending write and
// would wait for every load in flight; the caller waits (lgkmcnt) before using the value.
__device__ __forceinline__ int lds_ld32_asm(const void* p) {
  int v;
  asm volatile("ds_read_b32 %0, %1" : "=v"(v) : "v"(lds_addr(p)) : "memory");
  return v;
}

__global__ __launch_bounds__(256) void kv_scatter_kernel(const uint8_t* k8, const uint8_t* v8, const int64_t* loc, int T,
                                                        int64_t num_slots, uint8_t* kc, uint8_t* vc) {
  // thread: 16 bytes of one token's K or V row pair (2 heads x 256 bytes = 32 pieces per row);
  // a slot outside the cache is skipped
  const int i = blockIdx.x * 256 + threadIdx.x;
  if (i >= T * 64) return;
  const int t = i / 64, piece = i % 64, isv = piece >= 32, p = piece & 31;
  if (loc[t] < 0 || loc[t] >= num_slots) return;
  const size_t src = (size_t)t * (kKVH * kDD) + 16 * p, dst = (size_t)loc[t] * (kKVH * kDD) + 16 * p;
  *reinterpret_cast<v4i*>((isv ? vc : kc) + dst) = *reinterpret_cast<const v4i*>((isv ? v8 : k8) + src);
}

// How one call's keys are dealt to the workgroups of a KV head (G of them fit on the chip at once), in
// steps of kST keys (the arithmetic is q36_deal.h's):
//   even    batches of short or equal requests: every request whole, or in the same few pieces, one a workgroup;
//   pieces  each request in ceil(steps / c) equal pieces, one piece a workgroup, with the smallest c (from
//           kMinPiece up) that needs no more than G pieces.  The one-row-tile form, of which two workgroups
//           fit a CU, takes no more than G / 2: one a CU reads as fast, and longer runs leave fewer
//           partials (us, G against G / 2 pieces: 125 x 2 rows over 2580 .. 2995 keys 79.3 -> 73.4,
//           52 x 1 over 2325 37.6 -> 35.1, 3 x 1 over 20000 .. 32000 30.1 -> 26.8, 12 x 1 over 2984 ..
//           3471 22.2 -> 19.3);
//   line    where there are more requests than G, or a few long ones among many would make that c much
//           more than an equal share: a request weighs its steps plus ovh (what starting and merging a
//           run costs beside its steps), half before and half after them, and the line of all
//           weights is cut into G equal shares (as many as positions if these are fewer).  A share
//           holds the end of one request, whole requests and the start of another; requests of at most kWhole
//           steps are not cut but belong to the share that holds their start.
// Every workgroup works the dealing out for itself from seqlens before its first key, so a captured launch follows the
// lengths it finds.  That takes 0.5 us more than one load where it is even, 2 to 3 us else, and the combine launch
// 1.5 to 2.5 us where it finds nothing cut; a call whose page table holds no long request is spared both (see
// q36_attn_decode).  Measured, us a call (a fixed number of splits per request -> dealt): 64 x 4 rows over 128 .. 8192
// keys 85.4 -> 45.4, 256 x 1 over 20 .. 4000 96 -> 51, 150 x 4 over 300 .. 6000 130 -> 87, 12 x 2 over 3000 ..
// 30000 53.7 -> 36.6, 1 x 1 over 1000 42.9 -> 11.0.  Equal lengths have only that to lose: 64 x 4 over 4096 60.1 ->
// 62.3, 256 x 1 over 4096 181.6 -> 184.1; so have short ones in a table of 32768 entries: 84 x 1 over 191 8.9 -> 11.1,
// 56 x 1 over 646 14.8 -> 16.0, 117 x 3 over 131 .. 187 16.1 -> 16.4, 300 x 1 over 100 .. 300 20.9 -> 23.3, 1000 x 1 over 50 .. 300
// 48.6 -> 54.9 (by pieces and line as the others: 18.0, 18.5, 19.0, 32.0 and 60.0).
// ovh: 4 / 12 / 20 / 28 steps gave 58.5 / 52.2 / 49.3 / 50.3 us on the first of these (two row tiles) and
// 56.5 / 57.2 / 63.7 / 70.7 on the second (one).  kMinPiece: 2 / 4 / 8 steps 25.0 / 22.5 / 22.9 us for one
// request of 4 rows over 8000 keys, 14.0 / 14.6 / 16.0 us for one of 1 row over 1000.
// Integer sum over the wave, and inclusive scan, without LDS (the plan runs before the first load of a key).
__device__ __forceinline__ int wave_sum_i(int v) {
  v += (int)dpp_u32<0xB1>((uint32_t)v);
  v += (int)dpp_u32<0x4E>((uint32_t)v);
  v += (int)dpp_u32<0x141>((uint32_t)v);
  v += (int)dpp_u32<0x140>((uint32_t)v);
  const auto p16 = __builtin_amdgcn_permlane16_swap((uint32_t)v, (uint32_t)v, false, false);
  v = (int)(p16[0] + p16[1]);
  const auto p32 = __builtin_amdgcn_permlane32_swap((uint32_t)v, (uint32_t)v, false, false);
  return (int)(p32[0] + p32[1]);
}
__device__ __forceinline__ int wave_rows_sum_i(int v) {  // over the wave's four rows of 16 lanes
  const auto p16 = __builtin_amdgcn_permlane16_swap((uint32_t)v, (uint32_t)v, false, false);
  v = (int)(p16[0] + p16[1]);
  const auto p32 = __builtin_amdgcn_permlane32_swap((uint32_t)v, (uint32_t)v, false, false);
  return (int)(p32[0] + p32[1]);
}
__device__ __forceinline__ int wave_imax(int v) {
  v = max(v, (int)dpp_u32<0xB1>((uint32_t)v));
  v = max(v, (int)dpp_u32<0x4E>((uint32_t)v));
  v = max(v, (int)dpp_u32<0x141>((uint32_t)v));
  v = max(v, (int)dpp_u32<0x140>((uint32_t)v));
  const auto p16 = __builtin_amdgcn_permlane16_swap((uint32_t)v, (uint32_t)v, false, false);
  v = max((int)p16[0], (int)p16[1]);
  const auto p32 = __builtin_amdgcn_permlane32_swap((uint32_t)v, (uint32_t)v, false, false);
  return max((int)p32[0], (int)p32[1]);
}
__device__ __forceinline__ int wave_scan_i(int v) {
  v += __builtin_amdgcn_update_dpp(0, v, 0x111, 0xf, 0xf, false);  // row_shr 1, 2, 4, 8: within rows of 16
  v += __builtin_amdgcn_update_dpp(0, v, 0x112, 0xf, 0xf, false);
  v += __builtin_amdgcn_update_dpp(0, v, 0x114, 0xf, 0xf, false);
  v += __builtin_amdgcn_update_dpp(0, v, 0x118, 0xf, 0xf, false);
  const int r0 = __builtin_amdgcn_readlane(v, 15), r1 = __builtin_amdgcn_readlane(v, 31),
            r2 = __builtin_amdgcn_readlane(v, 47), row = (threadIdx.x & 63) >> 4;
  return v + (row > 0 ? r0 : 0) + (row > 1 ? r1 : 0) + (row > 2 ? r2 : 0);
}
// threadIdx.x through an empty asm: values derived from it are formed afresh for each run of steps
// instead of being kept, or spilled, across the step loop of the run before
__device__ __forceinline__ int run_tid() {
  int t = (int)threadIdx.x;
  asm volatile("" : "+v"(t));
  return t;
}

template <int RT, int NS, int WPE>
__global__ __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(WPE, WPE))) void decode_split_kernel(DecodeDev d) {
  constexpr int PTD = 2 * NS, kPTR = PTD <= 4 ? 4 : 8;  // page-table entries ahead, ring entries (one step each)
  constexpr int kRows = 16 * RT;
  static_assert(NS >= 2 && NS <= 4, "the prologue and the step loop are written out for 2 to 4 stages");
  static_assert(kPTR >= PTD, "the ring holds the entries of every step in flight");
  // one object per stage: the compiler then sees that a stage's DMA does not write what another
  // stage's reads read (in one array it waits for every DMA in flight before each read)
  __shared__ __align__(16) uint8_t vs0[kVS];
  __shared__ __align__(16) uint8_t vs1[kVS];
  __shared__ __align__(16) uint8_t vs2[NS >= 3 ? kVS : 16];
  __shared__ __align__(16) uint8_t vs3[NS >= 4 ? kVS : 16];
  __shared__ __align__(16) int32_t ptl[4][kPTR][64];
  __shared__ float mw[4][kRows], lwv[4][kRows], rowM[kRows], rowL[kRows];
  // balanced: offset and key count of each of 256 requests, the waves' sums, and the loop's state (in LDS,
  // so that no register holds it across a run): the share, the next request, the chunk of requests
  __shared__ int roff[256], rkeys[256], rsum[4], rmax[4], npiece[64];
  __shared__ int lx0, lx1, li, lhi, lc0, lbase;
  const int h = blockIdx.x & 1;
  // The run's request and key count; of a call dealt in pieces also the request's pieces and which of them (pn 0: not)
  int b = 0, nk = 0, pn = 0, pp = 0;
  if (d.splits == 0) {
    const int t = run_tid(), lane = t & 63, wv = __builtin_amdgcn_readfirstlane(t >> 6), wg = blockIdx.x >> 1, G = d.groups;
    // Up to 256 requests every wave reads all lengths (request 64 j + lane), so that a call dealt evenly is dealt with no
    // exchange between waves.
    int len[4] = {0, 0, 0, 0}, steps = 0, longest = 0;
    const bool few = d.B <= 256;
    if (few) {
#pragma unroll
      for (int j = 0; j < 4; ++j) len[j] = d.seqlens[min(64 * j + lane, d.B - 1)];
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        if (64 * j + lane >= d.B) len[j] = 0;
        const int v = min(req_steps(len[j]), d.max_steps);
        steps += v, longest = max(longest, v);
      }
    } else {
#pragma unroll 4
      for (int q = t; q < d.B; q += 256) {
        const int v = min(req_steps(d.seqlens[q]), d.max_steps);
        steps += v, longest = max(longest, v);
      }
    }
    steps = wave_sum_i(steps), longest = wave_imax(longest);
    if (!few) {
      if (lane == 0) rsum[wv] = steps, rmax[wv] = longest;
      __syncthreads();
      steps = rsum[0] + rsum[1] + rsum[2] + rsum[3], longest = max(max(rmax[0], rmax[1]), max(rmax[2], rmax[3]));
    }
    steps = __builtin_amdgcn_readfirstlane(steps), longest = __builtin_amdgcn_readfirstlane(longest);
    pn = even_pieces(RT, d.B, G, d.per, d.even, steps, longest);
    if (pn) {
      if (wg >= d.B * pn) return;
      b = pn == 1 ? wg : wg / pn, pp = wg - b * pn;
      nk = few ? __builtin_amdgcn_readlane(b < 64 ? len[0] : b < 128 ? len[1] : b < 192 ? len[2] : len[3], b & 63)
               : d.seqlens[b];
    } else {
      // (rolled loops: the plan's code is fetched cold on every launch, and longer code took longer)
      const int total = steps + d.B * ovh(RT), Gp = piece_places(RT, d.B, G, steps);
      if (few) {
        const int rk = wv == 0 ? len[0] : wv == 1 ? len[1] : wv == 2 ? len[2] : len[3];
        rkeys[t] = rk;
        roff[t] = min(req_steps(rk), d.max_steps);
      }
      __syncthreads();
      // (no search where the requests longer than the largest piece taken are too many already)
      const int most = piece_most(RT, total, Gp);
      int longs = 0;
#pragma unroll
      for (int j = 0; j < 4; ++j)
        longs += __builtin_popcountll(__builtin_amdgcn_ballot_w64(min(req_steps(len[j]), d.max_steps) > most));
      if (few && d.B + longs <= Gp) {
        // the kSizes piece sizes at once: thread t adds up size t % 16's pieces of every 16th request
        const int c0 = piece_least(steps, Gp), ct = piece_size(c0, t & (kSizes - 1));
        int n = 0;
#pragma unroll 2
        for (int q = t / kSizes; q < d.B; q += 256 / kSizes) n += req_pieces(roff[q], ct);
        n = wave_rows_sum_i(n);
        if (lane < kSizes) npiece[wv * kSizes + lane] = n;
        __syncthreads();
        n = npiece[t & 15] + npiece[16 + (t & 15)] + npiece[32 + (t & 15)] + npiece[48 + (t & 15)];
        const uint64_t fits = __builtin_amdgcn_ballot_w64(n <= Gp) & 0xffffu;
        const int k = fits ? __builtin_ctzll(fits) : 0, c = piece_size(c0, k), np = __builtin_amdgcn_readlane(n, k);
        if (np <= Gp && c <= most) {
          if (wg >= np) return;
          // the request that piece wg belongs to
          int end = 0;
#pragma unroll 1
          for (int q = 0; end <= wg; q += 64) {
            const int w = q + lane < d.B ? req_pieces(roff[q + lane], c) : 0;
            const int e = end + wave_scan_i(w);
            const uint64_t at = __builtin_amdgcn_ballot_w64(wg < e);
            end = __builtin_amdgcn_readlane(e, 63);
            if (at == 0) continue;
            const int l = __builtin_ctzll(at);
            b = q + l, pn = __builtin_amdgcn_readlane(w, l), nk = rkeys[b];
            pp = wg - __builtin_amdgcn_readlane(e, l) + pn;
          }
        }
      }
      if (!pn) {
        const int nsh = line_shares(total, G);
        if (wg >= nsh) return;
        const int x0 = share_begin(total, nsh, wg), x1 = share_begin(total, nsh, wg + 1);
        if (t == 0) lx0 = x0, lx1 = x1, li = 0, lhi = 0, lc0 = -256, lbase = 0;
        __syncthreads();
      }
    }
  }
  for (bool again = false;; again = true) {
  // the run of steps [st0, st0 + nst) of request b, and the slot of its partial result (-1: the whole request, written
  // out here)
  int st0, nst, slot, part;
  const int wg = (int)blockIdx.x >> 1;
  if (pn) {
    if (again) {  // only whole requests can be more than workgroups
      b += gridDim.x >> 1;
      if (pn > 1 || b >= d.B) return;
      nk = d.seqlens[b];
    }
    const DealRun r = piece_run(req_steps(nk), pn, pp);
    st0 = r.st0, nst = r.nst;
    part = r.part;
  } else if (d.splits == 0) {
    const int t = run_tid(), x0 = __builtin_amdgcn_readfirstlane(lx0), x1 = __builtin_amdgcn_readfirstlane(lx1);
    int i = __builtin_amdgcn_readfirstlane(li);
    if (i >= __builtin_amdgcn_readfirstlane(lhi)) {  // the next 256 requests
      const int c0 = __builtin_amdgcn_readfirstlane(lc0) + 256, base = __builtin_amdgcn_readfirstlane(lbase);
      if (c0 >= d.B || base >= x1) return;
      const bool in = c0 + t < d.B;
      const int rk = d.B <= 256 ? rkeys[t] : in ? d.seqlens[c0 + t] : 0;
      const int w = in ? min(req_steps(rk), d.max_steps) + ovh(RT) : 0, inc = wave_scan_i(w), v = t >> 6;
      __syncthreads();  // the state above has been read
      if ((t & 63) == 63) rsum[v] = inc;
      __syncthreads();
      const int off = base + inc - w + (v > 0 ? rsum[0] : 0) + (v > 1 ? rsum[1] : 0) + (v > 2 ? rsum[2] : 0);
      roff[t] = off;
      rkeys[t] = rk;
      // the requests of the chunk that touch the share
      const int lo = __builtin_popcountll(__builtin_amdgcn_ballot_w64(in && off + w <= x0));
      const int hi = __builtin_popcountll(__builtin_amdgcn_ballot_w64(in && off < x1));
      if ((t & 63) == 0) npiece[v] = lo, npiece[4 + v] = hi;
      __syncthreads();
      if (t == 0) {
        li = npiece[0] + npiece[1] + npiece[2] + npiece[3], lhi = npiece[4] + npiece[5] + npiece[6] + npiece[7];
        lc0 = c0, lbase = base + rsum[0] + rsum[1] + rsum[2] + rsum[3];
      }
      __syncthreads();
      continue;
    }
    b = __builtin_amdgcn_readfirstlane(lc0) + i;
    nk = __builtin_amdgcn_readfirstlane(rkeys[i]);
    const int off0 = __builtin_amdgcn_readfirstlane(roff[i]);
    const int steps = req_steps(nk);
    __syncthreads();
    if (t == 0) li = i + 1;
    __syncthreads();
    // (a key count past the page table's width is not cut either: its weight is the table's)
    const DealRun r = line_run(steps, off0, ovh(RT) / 2, steps <= kWhole || steps > d.max_steps, x0, x1);
    if (r.nst < 0) continue;
    st0 = r.st0, nst = r.nst;
    part = r.part;
  } else {
    if (again) return;
    const int S = d.splits;
    b = S == 1 ? wg : wg / S;
    const int s = wg - b * S;
    nk = d.seqlens[b];
    const DealRun r = piece_run(req_steps(nk), S, s);
    st0 = r.st0, nst = r.nst, part = 0;
    slot = S > 1 ? (b * kKVH + h) * S + s : -1;
  }
  // scalars: the descriptors made from them stay in SGPRs
  b = __builtin_amdgcn_readfirstlane(b), nk = __builtin_amdgcn_readfirstlane(nk);
  st0 = __builtin_amdgcn_readfirstlane(st0), nst = __builtin_amdgcn_readfirstlane(nst);
  if (d.splits == 0) {
    slot = part ? part_slot(wg, h, part) : -1;
    if (threadIdx.x == 0 && h == 0) {  // the workgroups that hold the request's first and last piece
      if (part == 0 || (part & kFirst)) d.meta[b].x = part ? wg : 0;
      if (part == 0 || (part & kLast)) d.meta[b].y = part ? wg : 0;
    }
  }
  const int tid = run_tid(), lane = tid & 63, l16 = lane & 15, lg = lane >> 4, NT = d.NT;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);  // uniform: LDS bases stay scalar
  const int npre = nk - NT;
  // the wave's share of the run, contiguous
  const int ws0 = st0 + (wave * nst) / 4, ws1 = st0 + ((wave + 1) * nst) / 4;
  const int kbeg = ws0 * kST, kend = min(ws1 * kST, nk);  // the wave's keys [kbeg, kend)
  const int kfull = min(kend - 1, npre);  // keys up to here are visible to every query row
  const __amdgpu_buffer_rsrc_t krs = __builtin_amdgcn_make_buffer_rsrc((void*)d.kc, (short)0, (int)d.kv_bytes, 0x00020000);
  const __amdgpu_buffer_rsrc_t vrs = __builtin_amdgcn_make_buffer_rsrc((void*)d.vc, (short)0, (int)d.kv_bytes, 0x00020000);
  // the request's page-table row through a bounded buffer (an entry past the row reads as slot 0)
  const __amdgpu_buffer_rsrc_t prs = __builtin_amdgcn_make_buffer_rsrc(
      (void*)(d.pt + (size_t)b * d.pt_stride), (short)0, 4 * d.pt_stride, 0x00020000);
  int32_t* ring = &ptl[wave][0][0];
  // Page-table entries of step j into ring entry j % kPTR (lanes 32..63 repeat lanes 0..31).  Keys past
  // the wave's range take the slot of its last key: their loads are repeats that stay in L2, their
  // scores are masked and their values are real cache rows (finite), so 0 * V stays 0.
  auto pt_dma = [&](int j) {
    const int key = max(min(kbeg + kST * j + (lane & 31), kend - 1), 0);
    __builtin_amdgcn_raw_ptr_buffer_load_lds(prs, ring + (j & (kPTR - 1)) * 64, 4, 4 * key, 0, 0, 0);
  };
  // the entries of the prologue's steps first: the query rows below come with them in one round trip
  for (int j = 0; j <= PTD - NS; ++j) pt_dma(j);
  // query fragments (score operand B): column 16 rt + l16 = query row (token row / 8, head
  // h * 8 + row % 8), dims 128 kb + 32 lg .. +31 rounded to e4m3; rows of tokens past NT are zero
  v8i qb[RT][2];
  int lim[RT];  // the row's last visible key (-1: none): causal among the new tokens, wave range
#pragma unroll
  for (int rt = 0; rt < RT; ++rt) {
    const int row = 16 * rt + l16, t = row >> 3;
    lim[rt] = t < NT ? min(kend - 1, npre + t) : -1;
#pragma unroll
    for (int kb = 0; kb < 2; ++kb) {
      int w[8] = {0, 0, 0, 0, 0, 0, 0, 0};
      if (t < NT) {
        const uint16_t* src = d.q + (((size_t)b * NT + t) * kQH + h * kGQ + (row & 7)) * kDD + 128 * kb + 32 * lg;
#pragma unroll
        for (int c = 0; c < 4; ++c) {
          const v4i raw = *reinterpret_cast<const v4i*>(src + 8 * c);
#pragma unroll
          for (int j = 0; j < 2; ++j)
            w[2 * c + j] = (int)(f2e4m3x2_hw(bf_lo((uint32_t)raw[2 * j]), bf_hi((uint32_t)raw[2 * j])) |
                                 (f2e4m3x2_hw(bf_lo((uint32_t)raw[2 * j + 1]), bf_hi((uint32_t)raw[2 * j + 1])) << 16));
        }
      }
      qb[rt][kb] = v8i{w[0], w[1], w[2], w[3], w[4], w[5], w[6], w[7]};
    }
  }
  // Step j into stage Q: the 32 keys' rows as score operand A (kf[Q][kt]: key 16 kt + l16, dims
  // 128 half + 32 lg ..), and the 32 value rows into the wave's LDS rows: DMA call m writes rows
  // 4 m .. 4 m + 3 with key 16 (m & 1) + 4 (m >> 1) + (row % 4), so rows 8 g .. 8 g + 7 hold keys
  // 4 g .. 4 g + 3 and 16 + 4 g .. 16 + 4 g + 3 (the order of lane group g's weights).  Row group m
  // (one DMA call, 1 KB) starts at m * (1 KB + 64 B) and 16-byte piece p of its row i sits at position
  // p ^ i: the eight rows a lane group reads for one dim tile fall on eight distinct 16-byte bank
  // slots, and only the low two bits of a piece's position depend on the lane.
  v4i kf[NS][2][4];
  auto stage = [&](auto qc) -> uint8_t* {
    constexpr int Q = decltype(qc)::value;
    return (Q == 0 ? vs0 : Q == 1 ? vs1 : Q == 2 ? vs2 : vs3) + wave * kVW;
  };
  auto fetch = [&](int j, auto qc) {
    constexpr int Q = decltype(qc)::value;
    const int32_t* e = ring + (j & (kPTR - 1)) * 64;
    int ks0 = lds_ld32_asm(e + l16), ks1 = lds_ld32_asm(e + 16 + l16);
    int vsl0 = lds_ld32_asm(e + lg), vsl1 = lds_ld32_asm(e + 16 + lg), vsl2 = lds_ld32_asm(e + 4 + lg),
        vsl3 = lds_ld32_asm(e + 20 + lg), vsl4 = lds_ld32_asm(e + 8 + lg), vsl5 = lds_ld32_asm(e + 24 + lg),
        vsl6 = lds_ld32_asm(e + 12 + lg), vsl7 = lds_ld32_asm(e + 28 + lg);
    asm volatile("s_waitcnt lgkmcnt(0)"
                 : "+v"(ks0), "+v"(ks1), "+v"(vsl0), "+v"(vsl1), "+v"(vsl2), "+v"(vsl3), "+v"(vsl4), "+v"(vsl5),
                   "+v"(vsl6), "+v"(vsl7)::"memory");
    const int kb0 = (ks0 * kKVH + h) * kDD + 32 * lg, kb1 = (ks1 * kKVH + h) * kDD + 32 * lg;
    kf[Q][0][0] = __builtin_amdgcn_raw_buffer_load_b128(krs, kb0, 0, kKVAux);
    kf[Q][0][1] = __builtin_amdgcn_raw_buffer_load_b128(krs, kb0 + 16, 0, kKVAux);
    kf[Q][0][2] = __builtin_amdgcn_raw_buffer_load_b128(krs, kb0 + 128, 0, kKVAux);
    kf[Q][0][3] = __builtin_amdgcn_raw_buffer_load_b128(krs, kb0 + 144, 0, kKVAux);
    kf[Q][1][0] = __builtin_amdgcn_raw_buffer_load_b128(krs, kb1, 0, kKVAux);
    kf[Q][1][1] = __builtin_amdgcn_raw_buffer_load_b128(krs, kb1 + 16, 0, kKVAux);
    kf[Q][1][2] = __builtin_amdgcn_raw_buffer_load_b128(krs, kb1 + 128, 0, kKVAux);
    kf[Q][1][3] = __builtin_amdgcn_raw_buffer_load_b128(krs, kb1 + 144, 0, kKVAux);
    uint8_t* vb = stage(qc);
    const int vsl[8] = {vsl0, vsl1, vsl2, vsl3, vsl4, vsl5, vsl6, vsl7};
#pragma unroll
    for (int m = 0; m < 8; ++m)
      __builtin_amdgcn_raw_ptr_buffer_load_lds(vrs, vb + m * kVG, 16, (vsl[m] * kKVH + h) * kDD + 16 * (l16 ^ lg), 0, 0,
                                               kKVAux);
  };
  // per-lane state: running max (base 2) of query row 16 rt + l16, the lane's share of its weight
  // sum, and O^T (lane: row 16 rt + l16, dims 16 dt + 4 lg + r)
  float m[RT], l[RT];
  v4f o[RT][16];
#pragma unroll
  for (int rt = 0; rt < RT; ++rt) {
    m[rt] = -1e30f;
    l[rt] = 0.f;
#pragma unroll
    for (int dt = 0; dt < 16; ++dt) o[rt][dt] = v4f{0.f, 0.f, 0.f, 0.f};
  }
  // lane's value-read address: row 8 lg + l16 / 2 = group 2 lg + l16 / 8, row (l16 / 2) % 4 in it,
  // half l16 % 2; dim tile dt adds 64 (dt / 4) + 16 ((dt % 4) ^ row)
  const int vri = (l16 >> 1) & 3, vbase = (2 * lg + (l16 >> 3)) * kVG + vri * kDD + 8 * (l16 & 1);
  auto compute = [&](int j, auto qc) {
    constexpr int Q = decltype(qc)::value;
    // this stage's values have landed (newer: NS page-table DMAs and NS - 1 steps' requests); all
    // sixteen transposed reads are issued now and complete under the scores and the softmax
    asm volatile("s_waitcnt vmcnt(%0)" ::"n"(NS + (NS - 1) * 16) : "memory");
    const uint8_t* vb = stage(qc) + vbase;
    v2i vraw[16];
#pragma unroll
    for (int dt = 0; dt < 16; ++dt)
      vraw[dt] = __builtin_amdgcn_ds_read_tr8_b64_v2i32(
          (__attribute__((address_space(3))) v2i*)(vb + 64 * (dt >> 2) + 16 * ((dt & 3) ^ vri)));
    v4f sc[RT][2];
#pragma unroll
    for (int rt = 0; rt < RT; ++rt)
#pragma unroll
      for (int kt = 0; kt < 2; ++kt) {
        sc[rt][kt] = mfma_e4m3(cat8d(kf[Q][kt][0], kf[Q][kt][1]), qb[rt][0], v4f{0.f, 0.f, 0.f, 0.f});
        sc[rt][kt] = mfma_e4m3(cat8d(kf[Q][kt][2], kf[Q][kt][3]), qb[rt][1], sc[rt][kt]);
      }
    // Softmax weights.  Only a step with keys some query row must not see (the causal edge, the end
    // of the wave's range) masks them to -inf; rows of tokens past NT have zero queries, stay finite
    // and are never written.  The running max starts at a finite -1e30, so exp2 of a masked score
    // is 0 with no special case.  Scores are raw MFMA sums, scaled inside the exponent's fma.
    const float sl2 = d.scale_log2;
    float sv[RT][8];
#pragma unroll
    for (int rt = 0; rt < RT; ++rt)
#pragma unroll
      for (int i = 0; i < 8; ++i) sv[rt][i] = sc[rt][i >> 2][i & 3];
    if (kbeg + kST * j + kST - 1 > kfull) {  // uniform over the wave
      const int key0 = kbeg + kST * j + 4 * lg;  // lane's keys: key0 + 16 kt + r
#pragma unroll
      for (int rt = 0; rt < RT; ++rt)
#pragma unroll
        for (int i = 0; i < 8; ++i)
          if (key0 + 16 * (i >> 2) + (i & 3) > lim[rt]) sv[rt][i] = -INFINITY;
    }
    float tmax[RT];
    bool need = false;
#pragma unroll
    for (int rt = 0; rt < RT; ++rt) {
      float mx = fmaxf(fmaxf(fmaxf(sv[rt][0], sv[rt][1]), fmaxf(sv[rt][2], sv[rt][3])),
                       fmaxf(fmaxf(sv[rt][4], sv[rt][5]), fmaxf(sv[rt][6], sv[rt][7])));
      // across the four lane groups (rows of 16 lanes) that hold the same query row
      const auto p16 = __builtin_amdgcn_permlane16_swap(__float_as_uint(mx), __float_as_uint(mx), false, false);
      mx = fmaxf(__uint_as_float(p16[0]), __uint_as_float(p16[1]));
      const auto p32 = __builtin_amdgcn_permlane32_swap(__float_as_uint(mx), __float_as_uint(mx), false, false);
      tmax[rt] = fmaxf(__uint_as_float(p32[0]), __uint_as_float(p32[1])) * sl2;
      need |= tmax[rt] > m[rt] + kLazy;
    }
    // Rare (a row max grew past its reference by 2^8), and marked so: with the branch at its default
    // weight the compiler placed the output accumulators' AGPR -> VGPR copies for it above the branch,
    // some 120 copies every step.
    if (__builtin_expect(__builtin_amdgcn_ballot_w64(need) != 0, 0)) {
#pragma unroll
      for (int rt = 0; rt < RT; ++rt) {
        const float mn = fmaxf(m[rt], tmax[rt]);
        const float al = __builtin_amdgcn_exp2f(m[rt] - mn);
        m[rt] = mn;
        l[rt] *= al;
        // four dim tiles at a time: the accumulators live in AGPRs and go through VGPRs to scale
#pragma unroll
        for (int dg = 0; dg < 16; dg += 4) {
#pragma unroll
          for (int i = 0; i < 4; ++i) {
            // taken from the AGPRs here (an opaque redefinition: a VGPR copy made before the branch
            // would be stale), scaled, and put back (no VGPR copy across the join)
            asm volatile("" : "+a"(o[rt][dg + i]));
            o[rt][dg + i] *= al;
            asm volatile("" : "+a"(o[rt][dg + i]));
          }
          __builtin_amdgcn_sched_barrier(0);
        }
      }
    }
    v8h pb[RT];
#pragma unroll
    for (int rt = 0; rt < RT; ++rt) {
      float ps = 0.f;
#pragma unroll
      for (int i = 0; i < 8; ++i) {
        const float p = __builtin_amdgcn_exp2f(__builtin_fmaf(sv[rt][i], sl2, -m[rt]));
        ps += p;
        pb[rt][i] = (_Float16)p;
      }
      l[rt] += ps;
    }
#pragma unroll
    for (int dt = 0; dt < 16; ++dt) {
      const v8h vv = widen8(vraw[dt].x, vraw[dt].y);
#pragma unroll
      for (int rt = 0; rt < RT; ++rt) o[rt][dt] = __builtin_amdgcn_mfma_f32_16x16x32_f16(vv, pb[rt], o[rt][dt], 0, 0, 0);
    }
  };
  // prologue: the entries of steps 0 .. PTD - NS have landed; the first NS - 1 steps' requests, each
  // followed by the page-table DMA PTD steps ahead (the order every step keeps)
  asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
  fetch(0, std::integral_constant<int, 0>{});
  pt_dma(PTD - NS + 1);
  if constexpr (NS >= 3) {
    fetch(1, std::integral_constant<int, 1>{});
    pt_dma(PTD - NS + 2);
  }
  if constexpr (NS == 4) {
    fetch(2, std::integral_constant<int, 2>{});
    pt_dma(PTD - NS + 3);
  }
  auto step = [&](int j, auto qc) {
    constexpr int Q = decltype(qc)::value;
    fetch(j + NS - 1, std::integral_constant<int, (Q + NS - 1) % NS>{});
    pt_dma(j + PTD);
    __builtin_amdgcn_sched_barrier(0);  // requests first: the compute below waits for step j's data
    compute(j, qc);
    __builtin_amdgcn_sched_barrier(0);  // and the next step's requests stay after it
  };
  const int nj = ws1 - ws0;
  for (int j = 0; j < nj; j += NS) {
    step(j, std::integral_constant<int, 0>{});
    if (j + 1 >= nj) break;
    step(j + 1, std::integral_constant<int, 1>{});
    if constexpr (NS >= 3) {
      if (j + 2 >= nj) break;
      step(j + 2, std::integral_constant<int, 2>{});
    }
    if constexpr (NS == 4) {
      if (j + 3 >= nj) break;
      step(j + 3, std::integral_constant<int, 3>{});
    }
  }
  asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
  // merge the four waves: M = max of the waves' maxima, L = sum of exp2(m_w - M) l_w; per row
  // tile, each wave's output scaled by exp2(m - M) into its own 16 KB (fp32 [16 rows][256], 16-byte
  // piece c of row r at c ^ r), then summed in wave order into this split's partial (or, with one
  // split, normalised by L into the bf16 output)
#pragma unroll
  for (int rt = 0; rt < RT; ++rt) {
    float lt = l[rt] + __shfl_xor(l[rt], 16);
    lt = lt + __shfl_xor(lt, 32);
    if (lg == 0) {
      mw[wave][16 * rt + l16] = m[rt];
      lwv[wave][16 * rt + l16] = lt;
    }
  }
  __syncthreads();
  if (tid < kRows) {
    const int row = tid;
    const float M = fmaxf(fmaxf(mw[0][row], mw[1][row]), fmaxf(mw[2][row], mw[3][row]));
    float L = 0.f;
#pragma unroll
    for (int w = 0; w < 4; ++w) L += __builtin_amdgcn_exp2f(mw[w][row] - M) * lwv[w][row];
    rowM[row] = M;
    rowL[row] = L;
    if (slot >= 0) {
      d.ws_ml[(size_t)slot * 2 * kRows + row] = M;
      d.ws_ml[(size_t)slot * 2 * kRows + kRows + row] = L;
    }
  }
  __syncthreads();
  float* ob = reinterpret_cast<float*>((wave < 2 ? vs0 : vs1) + (wave & 1) * (kVS / 2));
  const float* o0 = reinterpret_cast<const float*>(vs0);
  const float* o1 = reinterpret_cast<const float*>(vs0 + kVS / 2);
  const float* o2 = reinterpret_cast<const float*>(vs1);
  const float* o3 = reinterpret_cast<const float*>(vs1 + kVS / 2);
  float* wo = d.ws_o + (size_t)(slot >= 0 ? slot : 0) * kRows * kDD;
#pragma unroll
  for (int rt = 0; rt < RT; ++rt) {
    if (rt > 0) __syncthreads();  // the previous tile's sums have read the buffers
    const float M = rowM[16 * rt + l16];
    const float f = __builtin_amdgcn_exp2f(m[rt] - M);
#pragma unroll
    for (int dt = 0; dt < 16; ++dt)
      *reinterpret_cast<v4f*>(ob + l16 * kDD + 4 * ((4 * dt + lg) ^ l16)) = o[rt][dt] * f;
    __syncthreads();
    const int rows = min(16, NT * kGQ - 16 * rt);
    for (int e = tid; e < rows * (kDD / 4); e += 256) {
      const int r = e / (kDD / 4), c = e % (kDD / 4), at = r * kDD + 4 * (c ^ r), row = 16 * rt + r;
      const v4f a = (*reinterpret_cast<const v4f*>(o0 + at) + *reinterpret_cast<const v4f*>(o1 + at)) +
                    (*reinterpret_cast<const v4f*>(o2 + at) + *reinterpret_cast<const v4f*>(o3 + at));
      if (slot >= 0) {
        *reinterpret_cast<v4f*>(wo + row * kDD + 4 * c) = a;
      } else {
        const float L = rowL[row], il = L > 0.f ? 1.f / L : 0.f;
        uint16_t* dst = d.out + (((size_t)b * NT + (row >> 3)) * kQH + h * kGQ + (row & 7)) * kDD + 4 * c;
        const uint32_t o01 = pack_bf2_hw(a[0] * il, a[1] * il), o23 = pack_bf2_hw(a[2] * il, a[3] * il);
        *reinterpret_cast<uint2*>(dst) = make_uint2(o01, o23);
        // a wave holds one row (rows * 64 threads, whole waves): its two 128-groups are its lane halves
        if (d.oq) {
          const int tok = b * NT + (row >> 3), head = h * kGQ + (row & 7);
          gated_e4m3(d, tok, head, c, o01, o23, gate_row(d, __builtin_amdgcn_readfirstlane(tok), head, c));
        }
      }
    }
  }
  __syncthreads();  // every wave has read the buffers before the next run's requests write them
  }
}

// out = bf16(sum_p exp2(m_p - M) o_p / L), L = sum_p exp2(m_p - M) l_p over the pieces of a request, for each query row
// (b, t, head).  Latency-bound (the request's pieces, then their maxima, sums and outputs at once): a request of a few
// pieces takes one pass by one wave (decode_combine_few); 4 or 16 waves a row where a call of few requests has
// them in tens (3 requests of 42 splits: 23.3 us for one thread per 4 dims walking the splits, 5.5 us for 16
// waves).  kRows: rows of a slot.
struct Pieces {
  int n, g0, gstep, first;  // piece p of the request is at slot g0 + p * gstep, the first at g0 + first
  __device__ __forceinline__ int at(int p) const { return p * gstep + (p == 0 ? first : 0); }
};
__device__ __forceinline__ Pieces req_parts(const DecodeDev& d, int b, int h) {
  if (d.splits > 0) return Pieces{d.splits, (b * kKVH + h) * d.splits, 1, 0};
  const int2 w = d.meta[b];
  return Pieces{w.y - w.x + 1, part_slot(w.x, h, 0), part_slot(1, 0, 0), part_slot(0, 0, kFirst)};
}
__device__ __forceinline__ void put_row(const DecodeDev& d, int bt, int head, int c, v4f a, float L, v2i gate) {
  const float il = L > 0.f ? 1.f / L : 0.f;
  const uint32_t o01 = pack_bf2_hw(a[0] * il, a[1] * il), o23 = pack_bf2_hw(a[2] * il, a[3] * il);
  *reinterpret_cast<uint2*>(d.out + ((size_t)bt * kQH + head) * kDD + 4 * c) = make_uint2(o01, o23);
  // the wave holds the row: lanes 0-31 / 32-63 its two 128-groups
  if (d.oq) gated_e4m3(d, bt, head, c, o01, o23, gate);
}

// A workgroup a token, each of its 4 waves 4 query rows, each lane 4 dims of them.  Up to kNF pieces are in flight at
// once, read through descriptors of the request's slots (a piece past the last reads zeros and costs no traffic);
// more go in rounds, the sums rescaled to the new maximum.  Where nothing was cut the launch is pure overhead, so
// it is kept small: a wave a row took 0.3 us more for 84 tokens and 1.5 us more for 1000.
constexpr int kNF = 4;
__global__ __launch_bounds__(256) void decode_combine_few_kernel(DecodeDev d, int kRows) {
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), c = threadIdx.x & 63;
  const int bt = blockIdx.x, t = bt % d.NT, b = bt / d.NT, head = 4 * wave, h = head / kGQ, gr = t * kGQ + head % kGQ;
  const Pieces P = req_parts(d, b, h);
  if (d.splits == 0 && P.n <= 1) return;  // written by the split kernel
  const int span = (P.at(P.n - 1) + P.first + 1) * kRows;
  const __amdgpu_buffer_rsrc_t ors = __builtin_amdgcn_make_buffer_rsrc(
      (void*)(d.ws_o + (size_t)P.g0 * kRows * kDD), (short)0, span * (kDD * 4), 0x00020000);
  const __amdgpu_buffer_rsrc_t mrs = __builtin_amdgcn_make_buffer_rsrc(
      (void*)(d.ws_ml + (size_t)P.g0 * 2 * kRows), (short)0, span * (2 * 4), 0x00020000);
  v2i gate[4];
#pragma unroll
  for (int i = 0; i < 4; ++i) gate[i] = gate_row(d, bt, head + i, c);
  v4f a[4] = {}, M = {-1e30f, -1e30f, -1e30f, -1e30f}, L = {};  // the pieces' maxima are finite (-1e30: no visible key)
  for (int p0 = 0; p0 < P.n; p0 += kNF) {
    v4f m[kNF], l[kNF], o[kNF][4];
#pragma unroll
    for (int k = 0; k < kNF; ++k) {
      const bool in = p0 + k < P.n;
      const int row = P.at(p0 + k) * kRows, past = 0x7fffff00;
      const int mo = in ? (2 * row + gr) * 4 : past, oo = in ? (row + gr) * (kDD * 4) + 16 * c : past;
      m[k] = __builtin_bit_cast(v4f, __builtin_amdgcn_raw_buffer_load_b128(mrs, mo, 0, 0));
      l[k] = __builtin_bit_cast(v4f, __builtin_amdgcn_raw_buffer_load_b128(mrs, mo, kRows * 4, 0));
#pragma unroll
      for (int i = 0; i < 4; ++i)
        o[k][i] = __builtin_bit_cast(v4f, __builtin_amdgcn_raw_buffer_load_b128(ors, oo, i * kDD * 4, 0));
    }
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      float mk[kNF], mx = M[i];
#pragma unroll
      for (int k = 0; k < kNF; ++k) {
        mk[k] = p0 + k < P.n ? m[k][i] : -1e30f;
        mx = fmaxf(mx, mk[k]);
      }
      if (p0) {
        const float s = __builtin_amdgcn_exp2f(M[i] - mx);
        L[i] *= s;
        a[i] *= s;
      }
      M[i] = mx;
#pragma unroll
      for (int k = 0; k < kNF; ++k) {
        const float w = __builtin_amdgcn_exp2f(mk[k] - mx);
        L[i] += w * l[k][i];
        a[i] += w * o[k][i];
      }
    }
  }
#pragma unroll
  for (int i = 0; i < 4; ++i) put_row(d, bt, head + i, c, a[i], L[i], gate[i]);
}

// A workgroup a row: wave v adds pieces v, v + WPR, ..., each lane 4 dims, four in flight, and the waves' sums meet in LDS
// in wave order.
template <int WPR>
__global__ __launch_bounds__(64 * WPR) void decode_combine_kernel(DecodeDev d, int kRows) {
  __shared__ v4f sums[WPR][64];
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), lane = threadIdx.x & 63, c = lane;
  const int head = blockIdx.x % kQH, bt = blockIdx.x / kQH, t = bt % d.NT, b = bt / d.NT;
  const int h = head / kGQ, gr = t * kGQ + head % kGQ;
  const Pieces P = req_parts(d, b, h);
  const int n = P.n;
  if (d.splits == 0 && n <= 1) return;  // written by the split kernel
  auto slot = [&](int p) { return (size_t)(P.g0 + P.at(p)); };
  v4f o[4];
  auto fetch = [&](int p0, int q0, int m) {  // pieces p0 + q0, p0 + q0 + WPR, .. (past the m-th: the last again)
#pragma unroll
    for (int k = 0; k < 4; ++k)
      o[k] = *reinterpret_cast<const v4f*>(d.ws_o + (slot(p0 + min(q0 + k * WPR, m - 1)) * kRows + gr) * kDD + 4 * c);
  };
  auto ml = [&](int p, int what) { return d.ws_ml[(slot(p) * 2 + what) * kRows + gr]; };
  const v2i gate = gate_row(d, bt, head, c);
  float mp = ml(min(lane, n - 1), 0), lp = ml(min(lane, n - 1), 1);
  fetch(0, wave, min(64, n));
  float M = mp;
  for (int p = lane + 64; p < n; p += 64) M = fmaxf(M, ml(p, 0));
  M = wave_max(M);
  float L = 0.f;
  v4f a = {0.f, 0.f, 0.f, 0.f};
  for (int p0 = 0; p0 < n; p0 += 64) {
    if (p0) mp = ml(min(p0 + lane, n - 1), 0), lp = ml(min(p0 + lane, n - 1), 1);
    const float w = p0 + lane < n ? exp2f(mp - M) : 0.f;
    L += w * lp;
    const int m = min(64, n - p0);
    for (int q0 = wave; q0 < m; q0 += 4 * WPR) {
      if (p0 + q0 != wave) fetch(p0, q0, m);
#pragma unroll
      for (int k = 0; k < 4; ++k) {
        const int q = q0 + k * WPR, qc = min(q, m - 1);
        const float r = __int_as_float(__builtin_amdgcn_readlane(__float_as_int(w), qc));
        a += (q < m ? r : 0.f) * o[k];
      }
    }
  }
  L = wave_sum_bfly(L);
  sums[wave][lane] = a;
  __syncthreads();
  if (wave != 0) return;
#pragma unroll
  for (int v = 1; v < WPR; ++v) a += sums[v][lane];
  put_row(d, bt, head, c, a, L, gate);
}

int decode_cus() {
  static std::atomic<int> known[64];  // per device, 0: not asked yet
  int cus = 256, dev = 0;
  if (hipGetDevice(&dev) != hipSuccess) return cus;
  const bool slot = dev >= 0 && dev < 64;
  if (slot && known[dev].load(std::memory_order_relaxed)) return known[dev].load(std::memory_order_relaxed);
  if (hipDeviceGetAttribute(&cus, hipDeviceAttributeMultiprocessorCount, dev) == hipSuccess && slot)
    known[dev].store(cus, std::memory_order_relaxed);
  return cus;
}
// Equal splits per request: as asked for, or (a workspace too small for the balanced form) enough to
// give every CU a workgroup.
int decode_splits(int B, int splits) {
  if (splits > 0) return min(splits, 64);
  return max(1, min(64, decode_cus() / (B * kKVH)));
}
size_t decode_slots_bytes(size_t slots) {  // slots of kDRows rows (or twice as many of half the rows)
  return align_up(sizeof(float) * slots * kDRows * kDD, 256) + align_up(sizeof(float) * slots * 2 * kDRows, 256);
}
size_t decode_ws_bytes(int B, int S) { return decode_slots_bytes((size_t)B * kKVH * S); }
// Balanced: two slots a workgroup, one workgroup a CU of kDRows rows or two a CU of half the rows
size_t decode_bal_bytes(int B) { return decode_slots_bytes(2 * (size_t)decode_cus()) + align_up(sizeof(int2) * (size_t)B, 256); }

}  // namespace
}  // namespace q36

using namespace q36;

extern "C" size_t q36_attn_decode_workspace_bytes(int32_t B, int32_t splits) {
  return splits > 0 ? decode_ws_bytes(B, decode_splits(B, splits))
                    : std::max(decode_bal_bytes(B), decode_ws_bytes(B, decode_splits(B, 0)));
}

extern "C" int q36_attn_decode(const q36_decode_args* a, q36_stream_t stream) {
  Q36_REQUIRE(a != nullptr, "q36_attn_decode: null args");
  Q36_REQUIRE(a->HQ == kQH && a->HKV == kKVH && a->D == kDD,
              "q36_attn_decode: HQ=%d HKV=%d D=%d unsupported (this build: 16 / 2 / 256)", a->HQ, a->HKV, a->D);
  Q36_REQUIRE(a->B >= 1 && a->B <= 65535 && a->NT >= 1 && a->NT <= kDNT, "q36_attn_decode: B=%d NT=%d out of range",
              a->B, a->NT);
  Q36_REQUIRE(a->q && a->k_cache && a->v_cache && a->page_table && a->seqlens && a->out && a->workspace,
              "q36_attn_decode: a required pointer is null");
  Q36_REQUIRE(aligned16(a->q) && aligned16(a->k_cache) && aligned16(a->v_cache) &&
                  (reinterpret_cast<uintptr_t>(a->workspace) & 255u) == 0,
              "q36_attn_decode: q, k_cache, v_cache must be 16-byte and workspace 256-byte aligned");
  Q36_REQUIRE(a->num_slots >= 1 && (int64_t)a->num_slots * kKVH * kDD < ((int64_t)1 << 31),
              "q36_attn_decode: num_slots=%lld out of range", (long long)a->num_slots);
  Q36_REQUIRE(a->pt_stride >= 1, "q36_attn_decode: pt_stride=%d", a->pt_stride);
  Q36_REQUIRE(!a->out_loc || (a->k_new && a->v_new), "q36_attn_decode: out_loc needs k_new and v_new");
  Q36_REQUIRE((a->gate == nullptr) == (a->oq == nullptr) && (a->oq == nullptr) == (a->oqs == nullptr),
              "q36_attn_decode: gate, oq and oqs go together");
  Q36_REQUIRE(!a->oq || ((reinterpret_cast<uintptr_t>(a->gate) & 7u) == 0 &&
                         (reinterpret_cast<uintptr_t>(a->oq) & 3u) == 0 && (reinterpret_cast<uintptr_t>(a->oqs) & 3u) == 0),
              "q36_attn_decode: gate must be 8-byte, oq and oqs 4-byte aligned");
  const bool one = a->NT <= 2;  // one row tile, two workgroups a CU
  const int cus = decode_cus(), resident = (one ? kDecWPE1 : 1) * cus;
  const int max_steps = table_steps(a->pt_stride);
  // Where no length the table can hold makes the dealing good, the splits are fixed here, by the rule that the kernel
  // applies to the lengths, and neither the dealing nor a combine that may find nothing cut is paid for.  Measured, us
  // a call (dealt, fixed): 84 x 1 row over 191 keys 11.1, 9.0; 56 x 1 over 646 16.0, 15.3; 117 x 3 over 131 .. 187 16.4, 14.2;
  // on the other side 95 x 2 over 750 .. 2445 43.0, 48.6; 46 x 4 over 650 .. 3800 37.2, 49.1.
  const int so = decode_splits(a->B, 0);
  const int even = so <= (one ? 4 : 2) && (int64_t)a->B * kKVH * so <= resident ? so : 0;
  const auto fixed = [&] {
    const int s = even_table(one ? 1 : 2, even, max_steps);
    return (int64_t)a->B * kKVH * s <= resident && a->workspace_bytes >= decode_ws_bytes(a->B, std::max(s, 1)) ? s : 0;
  };
  const int s0 = a->splits > 0 ? a->splits : fixed();
  // balanced unless a split count was asked for (or the workspace holds only the equal splits', or the
  // line's length might not fit 31 bits)
  const bool bal = s0 == 0 && a->workspace_bytes >= decode_bal_bytes(a->B) &&
                   (int64_t)a->B * ((int64_t)max_steps + ovh(2)) < (1 << 30);
  const int S = bal ? 0 : decode_splits(a->B, s0);
  const size_t need = bal ? decode_bal_bytes(a->B) : decode_ws_bytes(a->B, S);
  Q36_REQUIRE(a->workspace_bytes >= need, "q36_attn_decode: workspace of %zu bytes < %zu required", a->workspace_bytes,
              need);
  hipStream_t st = static_cast<hipStream_t>(stream);
  char* ws = static_cast<char*>(a->workspace);
  const int T = a->B * a->NT;
  if (a->out_loc)
    kv_scatter_kernel<<<(T * 64 + 255) / 256, 256, 0, st>>>(static_cast<const uint8_t*>(a->k_new),
                                                            static_cast<const uint8_t*>(a->v_new), a->out_loc, T, a->num_slots,
                                                            static_cast<uint8_t*>(a->k_cache),
                                                            static_cast<uint8_t*>(a->v_cache));
  const int slots = bal ? 2 * cus : a->B * kKVH * S;  // of kDRows rows
  // balanced: as many workgroups per KV head as the chip holds at once, and no more than pieces of a
  // table of this width; a table so narrow that every request is dealt whole needs no combine
  const int nocut = table_uncut(max_steps);
  const int shares = deal_groups(a->B, max_steps, resident / kKVH);
  DecodeDev d{a->B, a->NT, a->pt_stride, S, shares, shares / a->B, even, max_steps,
              static_cast<const uint16_t*>(a->q), static_cast<const uint8_t*>(a->k_cache),
              static_cast<const uint8_t*>(a->v_cache), (int64_t)a->num_slots * kKVH * kDD, a->page_table, a->seqlens,
              a->scale * 1.44269504088896340736f, reinterpret_cast<float*>(ws),
              reinterpret_cast<float*>(ws + align_up(sizeof(float) * (size_t)slots * kDRows * kDD, 256)),
              reinterpret_cast<int2*>(ws + decode_slots_bytes(slots)),
              static_cast<uint16_t*>(a->out), static_cast<const uint16_t*>(a->gate), static_cast<uint8_t*>(a->oq),
              a->oqs};
  const unsigned grid = kKVH * (unsigned)(bal ? shares : a->B * S);
  if (one)
    decode_split_kernel<1, kDecNS1, kDecWPE1><<<grid, 256, 0, st>>>(d);
  else
    decode_split_kernel<2, kDecNS2, 1><<<grid, 256, 0, st>>>(d);
  if (bal ? !nocut : S > 1) {
    // waves per query row by the pieces an average request has
    const int rows = T * kQH, slot_rows = one ? 16 : kDRows, per = bal ? shares / a->B : S;
    if (per >= 32)
      decode_combine_kernel<16><<<rows, 1024, 0, st>>>(d, slot_rows);
    else if (per >= 3)
      decode_combine_kernel<4><<<rows, 256, 0, st>>>(d, slot_rows);
    else
      decode_combine_few_kernel<<<T, 256, 0, st>>>(d, slot_rows);
  }
  return check_launch("q36_attn_decode");
}
