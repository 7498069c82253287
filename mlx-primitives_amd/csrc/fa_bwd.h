// Shared declarations of the attention backward kernels (fa_bwd.hip: 16-bit,
// fa_bwd32.hip: float32).
#pragma once

#include "mpx_common.h"

namespace mpx {

struct BwdParams {
  const void* q;
  const void* k;
  const void* v;
  const void* o;
  const void* dout;
  const float* lse;   // (B, H, Sq) log2 units, +inf for rows without keys
  float* dvec;        // (B, H, Sq) workspace
  void* dq;
  void* dk;
  void* dv;
  int64_t q_sb, q_sh, q_ss, k_sb, k_sh, k_ss, v_sb, v_sh, v_ss, o_sb, o_sh, o_ss;
  int64_t do_sb, do_sh, do_ss, dq_sb, dq_sh, dq_ss, dk_sb, dk_sh, dk_ss, dv_sb, dv_sh, dv_ss;
  int B, H, H_kv, kv_group, Sq, Sk;  // K/V (and dK/dV) carry H_kv = H / kv_group heads
  int win_left, win_right;  // -1 = unbounded (causal: win_right = 0)
  float scale, c;           // c = scale * log2(e)
  // Dropout of the forward (the DROP kernels only): keep threshold and seed
  // words of the keep-mask hash, and the 1 / (1 - p) of the kept weights.
  uint32_t drop_thresh, seed0, seed1;
  float drop_scale;
  // Key-parallel work of a K/V head cut into kv_parts parts of its query heads
  // (1: none): each part's dK and dV go to dkv_part as float32 sums, (B, H_kv,
  // part, Sk, D) dK first, which fa_bwd_dkv_sum_kernel adds up.
  float* dkv_part;
  int kv_parts;
  // Stored dS^T (the stored-dS schedule only): ds_tot blocks per query head.
  void* ds;
  int64_t ds_tot;
};

constexpr int kBwdWaves = 4;    // waves per workgroup (one per SIMD)
constexpr int kBwdOwn = 32 * kBwdWaves;  // rows (or keys) a workgroup owns
constexpr int kBwdTile = 64;    // streamed rows per step

// Stored dS^T: per query head, 2 KB blocks of 32 keys x 32 queries (16-bit).
// Key tile kt (kBwdOwn keys, four key blocks) owns the blocks of the 32-row
// query blocks t0 .. t0 + nt - 1 that its keys' masks reach, query block
// major, key block minor; its first block is 4 * (sum of nt over the key
// tiles before it). Blocks that a key block and a query block do not share
// (outside both window edges, keys past Sk) are never written or read.
constexpr int kDsBlockBytes = 2048;

__host__ __device__ inline void ds_key_tile(int Sq, int Sk, int win_left, int win_right, int kt,
                                            int& t0, int& nt) {
  const int k0 = kt * kBwdOwn;
  const int k_last = (k0 + kBwdOwn < Sk ? k0 + kBwdOwn : Sk) - 1;
  const int q_lo = win_right >= 0 ? (k0 - win_right > 0 ? k0 - win_right : 0) : 0;
  const int q_hi = win_left >= 0 ? (k_last + win_left + 1 < Sq ? k_last + win_left + 1 : Sq) : Sq;
  t0 = q_lo / 32;
  nt = q_hi > q_lo ? (q_hi - 1) / 32 - t0 + 1 : 0;
}

// The query heads of part `part` of a K/V head, counted within its group: as
// even as the parts divide it, the first ones a head longer.
__device__ __forceinline__ void part_heads(const BwdParams& p, int part, int& first, int& n) {
  const int least = p.kv_group / p.kv_parts, more = p.kv_group - least * p.kv_parts;
  first = part * least + min(part, more);
  n = least + (part < more ? 1 : 0);
}

// One key's dK (times scale) and dV (times mul_v) as float32 sums of a part of
// the K/V head's query heads (BwdParams::dkv_part).
// WANT_K / WANT_V: the outputs that the caller has.
template <int NDB, bool WANT_K = true, bool WANT_V = true>
__device__ __forceinline__ void store_part(const BwdParams& p, int bhk, int part, int key, int g,
                                           const f32x16 (&dk)[NDB], const f32x16 (&dv)[NDB],
                                           float mul_v) {
  constexpr int D = 32 * NDB;
  const int64_t plane = (int64_t)p.B * p.H_kv * p.kv_parts * p.Sk * D;
  float* row = p.dkv_part + (((int64_t)bhk * p.kv_parts + part) * p.Sk + key) * D + 4 * g;
#pragma unroll
  for (int db = 0; db < NDB; ++db)
#pragma unroll
    for (int e4 = 0; e4 < 4; ++e4) {
      f32x4 a, c;
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        a[i] = dk[db][4 * e4 + i] * p.scale;
        c[i] = dv[db][4 * e4 + i] * mul_v;
      }
      if constexpr (WANT_K) *(f32x4*)(row + db * 32 + 8 * e4) = a;
      if constexpr (WANT_V) *(f32x4*)(row + plane + db * 32 + 8 * e4) = c;
    }
}

// Order of a joint launch (dQ and dK/dV tiles of one backward in one grid).
// The heads go in chunks of chunk_heads (batch, K/V head)s, chunk_wgs
// workgroups each. Within a chunk, entry i of the order covers the workgroups
// first[i] .. first[i + 1] - 1: tile code >> 2 of kind code & 3, dQ of a query
// tile (one per query head) or dK and dV, dK or dV of a key tile (one per K/V
// head and part).
enum BwdKind { kTileDq = 0, kTileDkDv = 1, kTileDk = 2, kTileDv = 3 };
constexpr int kMaxOrder = 128;
struct BwdOrder {
  int n, chunk_heads, chunk_wgs;
  int first[kMaxOrder + 1];
  uint16_t code[kMaxOrder];
};

// One workgroup's part of a joint launch: its kind and tile, its (batch, K/V
// head) and its part (dK/dV) or query head of the group (dQ).
struct BwdWork {
  int kind, tile, bhk, sub;
};

__device__ __forceinline__ BwdWork joint_work(const BwdOrder& order) {
  const int chunk = blockIdx.x / order.chunk_wgs, wg = blockIdx.x - chunk * order.chunk_wgs;
  int lo = 0, hi = order.n;  // first[lo] <= wg < first[hi]
  while (hi - lo > 1) {
    const int mid = (lo + hi) >> 1;
    if (order.first[mid] <= wg)
      lo = mid;
    else
      hi = mid;
  }
  // K/V heads fastest: with a multiple of 8 heads in a chunk every entry starts
  // on XCD 0, and a K/V head and its query heads stay on XCD head % 8 through
  // all their tiles.
  const int code = order.code[lo], i = wg - order.first[lo], sub = i / order.chunk_heads;
  return {code & 3, code >> 2, chunk * order.chunk_heads + (i - sub * order.chunk_heads), sub};
}

// The order of p's tiles of `own` rows or keys by cost, products per row of
// the streamed side (dQ: 3; dK and dV: 4, dK: 3, dV: 2, for every query head
// of the part), largest first. `split`: dK and dV as tiles of their own (float32
// at D >= 128). The caller has checked that the tiles of a head fit an order.
void make_order(const BwdParams& p, int own, bool split, BwdOrder& order);

// The float32 backward (rowsum, dQ, dK/dV kernels) for D in {64, 128}, with
// the forward's dropout when drop is set, enqueued on st; defined in
// fa_bwd32.hip.
hipError_t launch_bwd32(const BwdParams& p, int D, bool drop, hipStream_t st);

// Whether the float32 backward runs as one joint launch.
bool bwd32_joint(int B, int H, int Sq, int Sk, int D);

}  // namespace mpx
