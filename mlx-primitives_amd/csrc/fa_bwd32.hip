// Attention backward in float32 for gfx950: v_mfma_f32_32x32x2f32 (true fp32
// products), head_dim 64 or 128. Same gradients and decomposition as the
// 16-bit kernels (fa_bwd.hip): Dvec = rowsum(dO * O); a query-parallel dQ
// kernel and a key-parallel dK/dV kernel that recompute S and dP from the
// forward's row log-sum-exp. The reference differentiates its float32 tiled
// path with mx.grad (mlx_primitives/attention/flash.py:257-316;
// tests/attention/test_flash.py:338-362, tests/parity/pytorch/
// test_attention_parity.py:107-163 run float32).
//
// 32x32x2 f32 layouts (lane = j + 32 g): A lane holds element (row j, k = g),
// B (k = g, column j), C element e of the lane holds row 8 (e/4) + 4 g + e%4,
// column j. Products over head dims take their two k values from one 16-byte
// read (dims 8 jj + 4 g + t4, t4 < 4). Products over a C block's rows (dQ^T +=
// K^T dS^T, dV^T += dO^T P, dK^T += Q^T dS) step through the 16 C elements:
// element e is the B operand of its step directly (k = g <-> row 8 (e/4) + 4 g
// + e%4), and the A operand is one scalar LDS read of that row. Tiles of 32
// rows are staged through registers into LDS rows padded to D + 4 floats
// (16-byte row reads conflict-free).
#include "fa_bwd.h"

#include <algorithm>
#include <cmath>

namespace mpx {

constexpr int kB32Tile = 32;  // streamed rows per step

template <int D>
__global__ __launch_bounds__(256) void fa_bwd32_dvec_kernel(BwdParams p) {
  constexpr int LPR = D / 4;  // lanes per row, 4 floats each
  const int64_t rows = (int64_t)p.B * p.H * p.Sq;
  const int64_t row = ((int64_t)blockIdx.x * 256 + threadIdx.x) / LPR;
  const int l = threadIdx.x % LPR;
  float acc = 0.f;
  if (row < rows) {
    const int i = (int)(row % p.Sq);
    const int64_t bh = row / p.Sq;
    const int b = (int)(bh / p.H), h = (int)(bh % p.H);
    const float* o = (const float*)p.o + b * p.o_sb + h * p.o_sh + (int64_t)i * p.o_ss;
    const float* d = (const float*)p.dout + b * p.do_sb + h * p.do_sh + (int64_t)i * p.do_ss;
    const f32x4 ov = *(const f32x4*)(o + 4 * l);
    const f32x4 dv = *(const f32x4*)(d + 4 * l);
    acc = ov[0] * dv[0] + ov[1] * dv[1] + ov[2] * dv[2] + ov[3] * dv[3];
  }
#pragma unroll
  for (int off = LPR / 2; off >= 1; off >>= 1) acc += __shfl_xor(acc, off, 64);
  if (row < rows && l == 0) p.dvec[row] = acc;
}

// 32 KG rows of a float32 (rows, D) slice through 256 threads: global ->
// registers (rows past `rows` re-read the last one) -> LDS rows of stride D + 4.
template <int D, int KG = 1>
struct Stage32 {
  static constexpr int CPR = D / 4, PER_T = KG * kB32Tile * CPR / 256, RS = D + 4;
  f32x4 r[PER_T];
  __device__ __forceinline__ void load(const float* base, int64_t row_stride, int row0,
                                       int rows) {
#pragma unroll
    for (int i = 0; i < PER_T; ++i) {
      const int c = threadIdx.x + 256 * i;
      const int row = min(row0 + c / CPR, rows - 1);
      r[i] = *(const f32x4*)(base + (int64_t)row * row_stride + (c % CPR) * 4);
    }
  }
  __device__ __forceinline__ void store(float* lds) const {
#pragma unroll
    for (int i = 0; i < PER_T; ++i) {
      const int c = threadIdx.x + 256 * i;
      *(f32x4*)(lds + (c / CPR) * RS + (c % CPR) * 4) = r[i];
    }
  }
};

// Row of a float32 tensor as B-operand fragments: f[jj] = dims 8 jj + 4 g .. +3.
template <int D>
__device__ __forceinline__ void load_row32(const float* row, int g, f32x4 (&f)[D / 8]) {
#pragma unroll
  for (int jj = 0; jj < D / 8; ++jj) f[jj] = *(const f32x4*)(row + 8 * jj + 4 * g);
}

// Accumulator set (lane = output row, C rows = dims) times mul, stored as one
// float32 row.
template <int NDB>
__device__ __forceinline__ void store_row32(float* row, int g, const f32x16 (&acc)[NDB],
                                            float mul) {
#pragma unroll
  for (int db = 0; db < NDB; ++db)
#pragma unroll
    for (int e4 = 0; e4 < 4; ++e4)
      *(f32x4*)(row + db * 32 + 8 * e4 + 4 * g) =
          (f32x4){acc[db][4 * e4] * mul, acc[db][4 * e4 + 1] * mul, acc[db][4 * e4 + 2] * mul,
                  acc[db][4 * e4 + 3] * mul};
}

// Row (within a 32-row tile) that C element e of a lane in half g stands for.
__device__ __forceinline__ constexpr int crow(int e, int g) {
  return 8 * (e >> 2) + 4 * g + (e & 3);
}

// ---------------------------------------------------------------------------
// dQ: a workgroup owns 128 query rows of one (batch, head), wave w rows +32w;
// per 32-key tile: S^T = K Q^T, dP^T = V dO^T, dS^T = P^T (dP^T - Dvec),
// dQ^T += K^T dS^T.
// ---------------------------------------------------------------------------
// D = 256: one LDS stage, the next tile loaded after the barrier that ends the
// current one: a tile in flight under the compute, for a second stage, has no
// registers left (491 to 512 are used).
template <int D>
constexpr int kStages32 = D > 128 ? 1 : 2;
// LDS floats: [stage][K, V (or Q, dO)][32 KG rows], then lse and Dvec rows per stage.
template <int D, int KG>
constexpr int kLds32 = kStages32<D> * 2 * KG * kB32Tile * (D + 4) + 2 * 2 * KG * kB32Tile;

// KG key groups: the workgroup's waves are 4 / KG row groups of 32 (so it owns
// 128 / KG rows), and wave group kg takes tile KG t + kg of step t; the groups'
// sums meet in LDS at the end. One wave's chain of tiles bounds small calls
// (each tile is 96 products of 64 cycles at D = 64, on one wave per SIMD), and
// this halves it.
template <int KG>
struct Groups32 {
  int rg, kg;  // row group, key group of the wave
  __device__ __forceinline__ Groups32(int wave) {
    constexpr int NR = kBwdWaves / KG;
    rg = KG == 1 ? wave : wave % NR;
    kg = KG == 1 ? 0 : wave / NR;
  }
};

// Adds the accumulators of wave groups 1 .. KG - 1 to those of group 0 (lds is
// free: every wave is past its last read).
template <int KG, int NDB>
__device__ __forceinline__ void sum_groups32(float* lds, const Groups32<KG>& gr, int lane,
                                             f32x16 (&acc)[NDB]) {
  if constexpr (KG > 1) {
    constexpr int NR = kBwdWaves / KG;
    f32x4* const at = (f32x4*)lds + lane;
    __syncthreads();
    if (gr.kg > 0) {
#pragma unroll
      for (int db = 0; db < NDB; ++db)
#pragma unroll
        for (int e4 = 0; e4 < 4; ++e4)
          at[(((gr.kg - 1) * NR + gr.rg) * NDB * 4 + 4 * db + e4) * 64] =
              (f32x4){acc[db][4 * e4], acc[db][4 * e4 + 1], acc[db][4 * e4 + 2],
                      acc[db][4 * e4 + 3]};
    }
    __syncthreads();
    if (gr.kg == 0) {
#pragma unroll
      for (int k = 1; k < KG; ++k)
#pragma unroll
        for (int db = 0; db < NDB; ++db)
#pragma unroll
          for (int e4 = 0; e4 < 4; ++e4) {
            const f32x4 x = at[(((k - 1) * NR + gr.rg) * NDB * 4 + 4 * db + e4) * 64];
#pragma unroll
            for (int i = 0; i < 4; ++i) acc[db][4 * e4 + i] += x[i];
          }
    }
  }
}

template <int D, bool DROP, int KG>
__device__ __forceinline__ void bwd32_dq_tile(const BwdParams& p, float* smem, int bh, int qt) {
  constexpr int NQ4 = D / 8, NDB = D / 32, RS = D + 4, TILE = KG * kB32Tile * RS;
  constexpr int NSTG = kStages32<D>, OWN = kBwdOwn / KG;
  float(*lds)[2][TILE] = (float(*)[2][TILE])smem;  // [stage][K, V]
  const int b = bh / p.H, h = bh % p.H;
  const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int j = lane & 31, g = lane >> 5;
  const Groups32<KG> gr(wave);
  const int q0 = qt * OWN, wq0 = q0 + gr.rg * 32, myq = wq0 + j;
  const int qrow = min(myq, p.Sq - 1);

  const int kvh = h / p.kv_group;
  const float* Q = (const float*)p.q + b * p.q_sb + h * p.q_sh;
  const float* K = (const float*)p.k + b * p.k_sb + kvh * p.k_sh;
  const float* V = (const float*)p.v + b * p.v_sb + kvh * p.v_sh;
  const float* dO = (const float*)p.dout + b * p.do_sb + h * p.do_sh;
  f32x4 qf[NQ4], df[NQ4];
  load_row32<D>(Q + (int64_t)qrow * p.q_ss, g, qf);
  load_row32<D>(dO + (int64_t)qrow * p.do_ss, g, df);
  const int64_t rix = (int64_t)bh * p.Sq + qrow;
  const float lse = myq < p.Sq ? p.lse[rix] : INFINITY;
  const float dvc = p.dvec[rix];
  // Dropout: this row's key of the forward's keep-mask hash.
  const u32 drop_rk = DROP ? drop_row_key((u32)((int64_t)bh * p.Sq + myq), p.seed0) : 0u;
  const int kv_first = p.win_left >= 0 ? myq - p.win_left : -(1 << 30);
  const int kv_last = min(p.win_right >= 0 ? myq + p.win_right : (1 << 30), p.Sk - 1);

  const int q_last = min(q0 + OWN, p.Sq) - 1;
  const int kv_lo = p.win_left >= 0 ? max(0, q0 - p.win_left) : 0;
  const int kv_hi = p.win_right >= 0 ? min(p.Sk, q_last + p.win_right + 1) : p.Sk;
  // (steps of KG tiles)
  const int t0 = kv_lo / kB32Tile;
  const int n_t = kv_hi > kv_lo ? ((kv_hi - 1) / kB32Tile - t0) / KG + 1 : 0;

  f32x16 dq[NDB];
#pragma unroll
  for (int db = 0; db < NDB; ++db) dq[db] = (f32x16){};

  Stage32<D, KG> kst, vst;
  if (n_t > 0) {
    kst.load(K, p.k_ss, t0 * kB32Tile, p.Sk);
    vst.load(V, p.v_ss, t0 * kB32Tile, p.Sk);
    kst.store(lds[0][0]);
    vst.store(lds[0][1]);
  }
  __syncthreads();
  for (int t = 0; t < n_t; ++t) {
    const int S = NSTG == 1 ? 0 : t & 1;
    const int kvs = (t0 + KG * t) * kB32Tile;  // the step's first key
    if (NSTG == 2 && t + 1 < n_t) {
      kst.load(K, p.k_ss, kvs + KG * kB32Tile, p.Sk);
      vst.load(V, p.v_ss, kvs + KG * kB32Tile, p.Sk);
    }
    const int kv0 = kvs + gr.kg * kB32Tile;
    const bool skip = wq0 >= p.Sq || (KG > 1 && kv0 >= p.Sk) ||
                      (p.win_right >= 0 && kv0 > wq0 + 31 + p.win_right) ||
                      (p.win_left >= 0 && kv0 + kB32Tile - 1 < wq0 - p.win_left);
    const bool full = kv0 + kB32Tile <= p.Sk &&
                      (p.win_right < 0 || kv0 + kB32Tile - 1 <= wq0 + p.win_right) &&
                      (p.win_left < 0 || kv0 >= wq0 + 31 - p.win_left);
    if (!skip) {
      const float* Kt = lds[S][0] + gr.kg * kB32Tile * RS;
      const float* Vt = lds[S][1] + gr.kg * kB32Tile * RS;
      f32x16 sb = {}, dpb = {};
      const f32x4* kp = (const f32x4*)(Kt + j * RS) + g;
      const f32x4* vp = (const f32x4*)(Vt + j * RS) + g;
#pragma unroll
      for (int jj = 0; jj < NQ4; ++jj) {
        const f32x4 ka = kp[2 * jj], va = vp[2 * jj];
#pragma unroll
        for (int t4 = 0; t4 < 4; ++t4) {
          sb = mfma32x32x2f32(ka[t4], qf[jj][t4], sb);
          dpb = mfma32x32x2f32(va[t4], df[jj][t4], dpb);
        }
      }
      if (!full) {
#pragma unroll
        for (int e = 0; e < 16; ++e) {
          const int key = kv0 + crow(e, g);
          sb[e] = (key >= kv_first) & (key <= kv_last) ? sb[e] : -INFINITY;
        }
      }
      if constexpr (DROP) {
        // dS = P (dP keep / (1 - p) - Dvec); elements 2 e2, 2 e2 + 1 hold keys
        // kv0 + crow(2 e2, g) + {0, 1}, the hash's key pair
        // kv0 / 2 + 4 (e2 / 2) + 2 g + e2 % 2.
        const u32 pair0 = drop_pair_key((u32)(kv0 >> 1) + 2u * g, p.seed1);
#pragma unroll
        for (int e2 = 0; e2 < 8; ++e2) {
          const u32 bits = drop_bits(drop_rk, pair0 + (u32)(4 * (e2 >> 1) + (e2 & 1)) * 0x85EBCA77u);
          dpb[2 * e2] = (bits & 0xffffu) >= p.drop_thresh ? dpb[2 * e2] * p.drop_scale : 0.f;
          dpb[2 * e2 + 1] = bits >= (p.drop_thresh << 16) ? dpb[2 * e2 + 1] * p.drop_scale : 0.f;
        }
      }
      f32x16 ds;
#pragma unroll
      for (int e = 0; e < 16; ++e) ds[e] = fast_exp2(sb[e] * p.c - lse) * (dpb[e] - dvc);
#pragma unroll
      for (int db = 0; db < NDB; ++db)
#pragma unroll
        for (int e = 0; e < 16; ++e)
          dq[db] = mfma32x32x2f32(Kt[crow(e, g) * RS + db * 32 + j], ds[e], dq[db]);
    }
    if (t + 1 < n_t) {
      if constexpr (NSTG == 1) {
        __syncthreads();
        kst.load(K, p.k_ss, kvs + KG * kB32Tile, p.Sk);
        vst.load(V, p.v_ss, kvs + KG * kB32Tile, p.Sk);
      }
      kst.store(lds[NSTG == 1 ? 0 : S ^ 1][0]);
      vst.store(lds[NSTG == 1 ? 0 : S ^ 1][1]);
    }
    __syncthreads();
  }
  static_assert(KG == 1 || (KG - 1) * (kBwdWaves / KG) * NDB * 1024 <= kLds32<D, KG>, "LDS");
  sum_groups32<KG>(smem, gr, lane, dq);
  if (gr.kg == 0 && myq < p.Sq)
    store_row32<NDB>((float*)p.dq + b * p.dq_sb + h * p.dq_sh + (int64_t)myq * p.dq_ss, g, dq,
                     p.scale);
}

template <int D, bool DROP = false>
__global__ __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(1, 1)))
void fa_bwd32_dq_kernel(BwdParams p) {
  __shared__ __align__(16) float lds[kLds32<D, 1>];
  const int n_qt = (p.Sq + kBwdOwn - 1) / kBwdOwn;
  bwd32_dq_tile<D, DROP, 1>(p, lds, blockIdx.x % (p.B * p.H),
                            n_qt - 1 - (int)(blockIdx.x / (p.B * p.H)));
}

// ---------------------------------------------------------------------------
// dK, dV: a workgroup owns 128 keys of one (batch, K/V head), wave w keys
// +32w; per 32-row Q tile (every query head of the group): S = Q K^T,
// dP = dO V^T, P = exp2(S c - lse), dS = P (dP - Dvec), dV^T += dO^T P,
// dK^T += Q^T dS. WANT_K / WANT_V select the outputs: at D = 128 K, V and both
// accumulator sets do not fit one wave's registers, so dK and dV run as two
// kernels (the dV one recomputes S and needs neither dP nor V).
// ---------------------------------------------------------------------------
template <int D, bool WANT_K, bool WANT_V, bool DROP, int KG>
__device__ __forceinline__ void bwd32_dkdv_tile(const BwdParams& p, float* smem, int bhk, int part,
                                                int kt) {
  constexpr int NQ4 = D / 8, NDB = D / 32, RS = D + 4, TILE = KG * kB32Tile * RS;
  constexpr int NSTG = kStages32<D>, OWN = kBwdOwn / KG, ROWS = KG * kB32Tile;
  float(*lds)[2][TILE] = (float(*)[2][TILE])smem;  // [stage][Q, dO]
  float(*lse_lds)[ROWS] = (float(*)[ROWS])(smem + NSTG * 2 * TILE);
  float(*dvc_lds)[ROWS] = lse_lds + 2;
  const int b = bhk / p.H_kv, hk = bhk % p.H_kv;
  const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int j = lane & 31, g = lane >> 5;
  const Groups32<KG> gr(wave);
  const int k0 = kt * OWN, wk0 = k0 + gr.rg * 32, mykey = wk0 + j;
  const int krow = min(mykey, p.Sk - 1);
  const int q_first = p.win_right >= 0 ? mykey - p.win_right : -(1 << 30);
  const int q_last = p.win_left >= 0 ? mykey + p.win_left : (1 << 30);
  // Dropout: this key's pair key of the forward's keep-mask hash and the half
  // of the hash that decides it.
  const u32 drop_pk = DROP ? drop_pair_key((u32)mykey >> 1, p.seed1) : 0u;
  const u32 drop_hm = (mykey & 1) ? 0xffff0000u : 0xffffu;
  const u32 drop_ht = (mykey & 1) ? p.drop_thresh << 16 : p.drop_thresh;

  const float* K = (const float*)p.k + b * p.k_sb + hk * p.k_sh;
  const float* V = (const float*)p.v + b * p.v_sb + hk * p.v_sh;
  f32x4 kf[NQ4], vf[NQ4];
  load_row32<D>(K + (int64_t)krow * p.k_ss, g, kf);
  if constexpr (WANT_K) load_row32<D>(V + (int64_t)krow * p.v_ss, g, vf);

  const int k_last = min(k0 + OWN, p.Sk) - 1;
  const int q_lo = p.win_right >= 0 ? max(0, k0 - p.win_right) : 0;
  const int q_hi = p.win_left >= 0 ? min(p.Sq, k_last + p.win_left + 1) : p.Sq;
  // (steps of KG tiles of one head)
  const int t0 = q_lo / kB32Tile;
  const int n_t = q_hi > q_lo ? ((q_hi - 1) / kB32Tile - t0) / KG + 1 : 0;
  int h0, heads;
  part_heads(p, part, h0, heads);
  h0 += hk * p.kv_group;
  const int n_steps = n_t * heads;

  f32x16 dk[NDB], dv[NDB];
#pragma unroll
  for (int db = 0; db < NDB; ++db) {
    dk[db] = (f32x16){};
    dv[db] = (f32x16){};
  }

  Stage32<D, KG> qst, dst;
  float lse_r = 0.f, dvc_r = 0.f;
  auto load = [&](int u) __attribute__((always_inline)) {
    const int h = h0 + u / n_t;
    const int row0 = (t0 + KG * (u % n_t)) * kB32Tile;
    qst.load((const float*)p.q + b * p.q_sb + h * p.q_sh, p.q_ss, row0, p.Sq);
    dst.load((const float*)p.dout + b * p.do_sb + h * p.do_sh, p.do_ss, row0, p.Sq);
    if (threadIdx.x < ROWS) {
      const int r = row0 + threadIdx.x;
      const int64_t rix = ((int64_t)b * p.H + h) * p.Sq + r;
      lse_r = r < p.Sq ? p.lse[rix] : INFINITY;
      dvc_r = r < p.Sq ? p.dvec[rix] : 0.f;
    }
  };
  auto store = [&](int S) __attribute__((always_inline)) {
    qst.store(lds[S][0]);
    dst.store(lds[S][1]);
    if (threadIdx.x < ROWS) {
      lse_lds[S][threadIdx.x] = lse_r;
      dvc_lds[S][threadIdx.x] = dvc_r;
    }
  };
  if (n_steps > 0) {
    load(0);
    store(0);
  }
  __syncthreads();
  for (int u = 0; u < n_steps; ++u) {
    const int S = NSTG == 1 ? 0 : u & 1;
    if (NSTG == 2 && u + 1 < n_steps) load(u + 1);
    const int qr0 = (t0 + KG * (u % n_t) + gr.kg) * kB32Tile;
    const bool skip = wk0 >= p.Sk || (KG > 1 && qr0 >= p.Sq) ||
                      (p.win_right >= 0 && wk0 > qr0 + kB32Tile - 1 + p.win_right) ||
                      (p.win_left >= 0 && wk0 + 31 < qr0 - p.win_left);
    const bool full = (p.win_right < 0 || wk0 + 31 <= qr0 + p.win_right) &&
                      (p.win_left < 0 || wk0 >= qr0 + kB32Tile - 1 - p.win_left);
    if (!skip) {
      const float* Qt = lds[S][0] + gr.kg * kB32Tile * RS;
      const float* Dt = lds[S][1] + gr.kg * kB32Tile * RS;
      const float* lsv = lse_lds[S] + gr.kg * kB32Tile;
      const float* dvv = dvc_lds[S] + gr.kg * kB32Tile;
      f32x16 sb = {}, dpb = {};
      const f32x4* qp = (const f32x4*)(Qt + j * RS) + g;
      const f32x4* dp = (const f32x4*)(Dt + j * RS) + g;
#pragma unroll
      for (int jj = 0; jj < NQ4; ++jj) {
        const f32x4 qa = qp[2 * jj], da = dp[2 * jj];
#pragma unroll
        for (int t4 = 0; t4 < 4; ++t4) {
          sb = mfma32x32x2f32(qa[t4], kf[jj][t4], sb);
          if constexpr (WANT_K) dpb = mfma32x32x2f32(da[t4], vf[jj][t4], dpb);
        }
      }
      if (!full) {
#pragma unroll
        for (int e = 0; e < 16; ++e) {
          const int q = qr0 + crow(e, g);
          sb[e] = (q >= q_first) & (q <= q_last) ? sb[e] : -INFINITY;
        }
      }
      f32x16 pr, ds;
#pragma unroll
      for (int e4 = 0; e4 < 4; ++e4) {
        const f32x4 lv = *(const f32x4*)(lsv + 8 * e4 + 4 * g);
        const f32x4 dv4 = *(const f32x4*)(dvv + 8 * e4 + 4 * g);
#pragma unroll
        for (int i = 0; i < 4; ++i) {
          const int e = 4 * e4 + i;
          pr[e] = fast_exp2(sb[e] * p.c - lv[i]);
          if constexpr (DROP) {
            // Row qr0 + crow(e, g) of this step's head (u / n_t of the group).
            const u32 rk = drop_row_key(
                (u32)(((int64_t)b * p.H + h0 + u / n_t) * p.Sq + qr0 + crow(e, g)),
                p.seed0);
            const bool keep = drop_keep(drop_bits(rk, drop_pk), drop_hm, drop_ht);
            if constexpr (WANT_K) ds[e] = pr[e] * ((keep ? dpb[e] * p.drop_scale : 0.f) - dv4[i]);
            pr[e] = keep ? pr[e] : 0.f;
          } else {
            if constexpr (WANT_K) ds[e] = pr[e] * (dpb[e] - dv4[i]);
          }
        }
      }
#pragma unroll
      for (int db = 0; db < NDB; ++db)
#pragma unroll
        for (int e = 0; e < 16; ++e) {
          const int r = crow(e, g) * RS + db * 32 + j;
          if constexpr (WANT_V) dv[db] = mfma32x32x2f32(Dt[r], pr[e], dv[db]);
          if constexpr (WANT_K) dk[db] = mfma32x32x2f32(Qt[r], ds[e], dk[db]);
        }
    }
    if (u + 1 < n_steps) {
      if constexpr (NSTG == 1) {
        __syncthreads();
        load(u + 1);
      }
      store(NSTG == 1 ? 0 : S ^ 1);
    }
    __syncthreads();
  }
  if constexpr (WANT_K) sum_groups32<KG>(smem, gr, lane, dk);
  if constexpr (WANT_V) sum_groups32<KG>(smem, gr, lane, dv);
  if (gr.kg != 0 || mykey >= p.Sk) return;
  if (p.kv_parts > 1) {
    store_part<NDB, WANT_K, WANT_V>(p, bhk, part, mykey, g, dk, dv, DROP ? p.drop_scale : 1.f);
  } else {
    if constexpr (WANT_K)
      store_row32<NDB>((float*)p.dk + b * p.dk_sb + hk * p.dk_sh + (int64_t)mykey * p.dk_ss, g,
                       dk, p.scale);
    if constexpr (WANT_V)
      store_row32<NDB>((float*)p.dv + b * p.dv_sb + hk * p.dv_sh + (int64_t)mykey * p.dv_ss, g,
                       dv, DROP ? p.drop_scale : 1.f);
  }
}

template <int D, bool WANT_K, bool WANT_V, bool DROP = false>
__global__ __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(1, 1)))
void fa_bwd32_dkdv_kernel(BwdParams p) {
  __shared__ __align__(16) float lds[kLds32<D, 1>];
  const int heads = p.B * p.H_kv, i = blockIdx.x % (heads * p.kv_parts);
  bwd32_dkdv_tile<D, WANT_K, WANT_V, DROP, 1>(p, lds, i % heads, i / heads,
                                              (int)(blockIdx.x / (heads * p.kv_parts)));
}

// dQ and dK/dV tiles in one launch, one tile of 64 rows or keys per workgroup,
// the longest first.
template <int D, bool DROP>
__global__ __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(1, 1)))
void fa_bwd32_joint_kernel(BwdParams p, BwdOrder order) {
  // (133 KB at D = 128: no kernel here has more. 353 registers, none spilled.)
  static_assert(kLds32<D, 2> * 4 <= 160 * 1024, "LDS of a CU");
  __shared__ __align__(16) float lds[kLds32<D, 2>];
  const BwdWork w = joint_work(order);
  if (w.kind == kTileDq) {
    bwd32_dq_tile<D, DROP, 2>(p, lds, w.bhk * p.kv_group + w.sub, w.tile);
  } else if constexpr (D >= 128) {
    if (w.kind == kTileDk)
      bwd32_dkdv_tile<D, true, false, DROP, 2>(p, lds, w.bhk, w.sub, w.tile);
    else
      bwd32_dkdv_tile<D, false, true, DROP, 2>(p, lds, w.bhk, w.sub, w.tile);
  } else {
    bwd32_dkdv_tile<D, true, true, DROP, 2>(p, lds, w.bhk, w.sub, w.tile);
  }
}

// dK (blockIdx.y == 0) or dV = the parts' sums added up: four dims of one key
// per thread.
template <int D>
__global__ __launch_bounds__(256) void fa_bwd32_dkv_sum_kernel(BwdParams p) {
  const int64_t n = (int64_t)p.B * p.H_kv * p.Sk * (D / 4);
  const int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x;
  if (i >= n) return;
  const int d = (int)(i % (D / 4)) * 4;
  const int64_t row = i / (D / 4), bhk = row / p.Sk;
  const int key = (int)(row - bhk * p.Sk), b = (int)(bhk / p.H_kv), hk = (int)(bhk % p.H_kv);
  const float* src = p.dkv_part + ((bhk * p.kv_parts + (int64_t)p.B * p.H_kv * p.kv_parts *
                                    blockIdx.y) * p.Sk + key) * D + d;
  f32x4 sum = *(const f32x4*)src;
  for (int k = 1; k < p.kv_parts; ++k) sum += *(const f32x4*)(src + (int64_t)k * p.Sk * D);
  float* dst = blockIdx.y == 0
                   ? (float*)p.dk + b * p.dk_sb + hk * p.dk_sh + (int64_t)key * p.dk_ss
                   : (float*)p.dv + b * p.dv_sb + hk * p.dv_sh + (int64_t)key * p.dv_ss;
  *(f32x4*)(dst + d) = sum;
}

// Below 2048 tiles of 64 rows over both sides: the two (at D = 128 three)
// launches of 128-row tiles then leave SIMDs empty or end on a few long waves.
// Causal backward of (batch, S, heads, D), launches of their own against one:
// (2, 1024, 12, 64) 266 -> 133 us, (1, 512, 8, 64) 138 -> 46, (2, 1024, 12,
// 128) 576 -> 277, (1, 2048, 16, 128), 1536 tiles, 1125 -> 654; (2, 2048, 16,
// 64), 2048 tiles, 565 against 598, (4, 4096, 16, 64) 4237 against 4516 (half
// the rows a workgroup means twice the streamed tiles).
bool bwd32_joint(int B, int H, int Sq, int Sk, int D) {
  constexpr int own = kBwdOwn / 2;
  const int n_qt = (Sq + own - 1) / own, n_kt = (Sk + own - 1) / own;
  const int per_kv = D >= 128 ? 2 : 1;  // dK and dV tiles
  return D <= 128 && n_qt < kMaxOrder && n_kt < kMaxOrder &&
         n_qt + per_kv * n_kt <= kMaxOrder && (long)B * H * (n_qt + per_kv * n_kt) < 2048;
}

template <int D>
void launch_sum32(const BwdParams& p, hipStream_t st) {
  const long n = (long)p.B * p.H_kv * p.Sk * (D / 4);
  hipLaunchKernelGGL((fa_bwd32_dkv_sum_kernel<D>), dim3((unsigned)((n + 255) / 256), 2), dim3(256),
                     0, st, p);
}

template <int D, bool DROP>
hipError_t launch_bwd32_d(const BwdParams& p, hipStream_t st) {
  const int64_t rows = (int64_t)p.B * p.H * p.Sq;
  hipLaunchKernelGGL((fa_bwd32_dvec_kernel<D>), dim3((unsigned)((rows * (D / 4) + 255) / 256)),
                     dim3(256), 0, st, p);
  if constexpr (D <= 128) {
    if (bwd32_joint(p.B, p.H, p.Sq, p.Sk, D)) {
      constexpr int own = kBwdOwn / 2;
      BwdOrder order;
      make_order(p, own, D >= 128, order);
      const long wgs = (long)(p.B * p.H_kv / order.chunk_heads) * order.chunk_wgs;
      hipLaunchKernelGGL((fa_bwd32_joint_kernel<D, DROP>), dim3((unsigned)wgs), dim3(256), 0, st, p,
                         order);
      if (p.kv_parts > 1) launch_sum32<D>(p, st);
      return hipGetLastError();
    }
  }
  const int n_qt = (p.Sq + kBwdOwn - 1) / kBwdOwn, n_kt = (p.Sk + kBwdOwn - 1) / kBwdOwn;
  hipLaunchKernelGGL((fa_bwd32_dq_kernel<D, DROP>), dim3(p.B * p.H * n_qt), dim3(256), 0, st, p);
  const dim3 grid_kv(p.B * p.H_kv * p.kv_parts * n_kt);
  if constexpr (D >= 128) {
    hipLaunchKernelGGL((fa_bwd32_dkdv_kernel<D, true, false, DROP>), grid_kv, dim3(256), 0, st, p);
    hipLaunchKernelGGL((fa_bwd32_dkdv_kernel<D, false, true, DROP>), grid_kv, dim3(256), 0, st, p);
  } else {
    hipLaunchKernelGGL((fa_bwd32_dkdv_kernel<D, true, true, DROP>), grid_kv, dim3(256), 0, st, p);
  }
  if (p.kv_parts > 1) launch_sum32<D>(p, st);
  return hipGetLastError();
}

template <bool DROP>
hipError_t launch_bwd32_drop(const BwdParams& p, int D, hipStream_t st) {
  if (D == 64) return launch_bwd32_d<64, DROP>(p, st);
  if (D == 256) return launch_bwd32_d<256, DROP>(p, st);
  return launch_bwd32_d<128, DROP>(p, st);
}

hipError_t launch_bwd32(const BwdParams& p, int D, bool drop, hipStream_t st) {
  return drop ? launch_bwd32_drop<true>(p, D, st) : launch_bwd32_drop<false>(p, D, st);
}

}  // namespace mpx
