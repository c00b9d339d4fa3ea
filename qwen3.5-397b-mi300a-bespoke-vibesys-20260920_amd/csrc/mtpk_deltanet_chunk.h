// The gated delta rule over many steps (a prompt's rows), 64 steps at a time.
//
// One step is S <- e^g S, u = beta (v - S^T k), S <- S + k u^T, out = S^T q, and t of them in a row
// are t dependent passes over S: on 64 heads of 128 x 128 they take 1.5 us a step (1500 steps:
// 2286 us with outputs, 1637 us without; this form 178 and 117 us) with 128 one-wave workgroups on
// the whole chip. Inside a
// chunk of C = 64 steps that starts from S0, with G_i the running sum of g,
//   u_i = beta_i (v_i - e^(G_i) S0^T k_i - sum_{j<i} e^(G_i - G_j) (k_i . k_j) u_j)
// is a unit lower triangular system (I + L) U = beta Y, Y = V - e^G (K S0), and
//   out_i = e^(G_i) S0^T q_i + sum_{j<=i} e^(G_i - G_j) (q_i . k_j) u_j
//   S     = e^(G_C) S0 + K^T (e^(G_C - G_j) u_j)
// are matrix products. The parts without S0 (T = (I + L)^-1 beta and the masked q . k) are made for
// every chunk at once (k_dn_chunk_prep); what is left per chunk (k_dn_chunk_scan) is serial only in
// S0: t / 64 steps of matrix products on v_mfma_f32_16x16x4_f32, all in fp32. G is summed and
// differenced in fp64: e^(G_i - G_j) of neighbouring steps must not lose the digits that a long
// chunk's large |G| would cost it in fp32.
//
// A masked element is a product with zero there, so a NaN or infinity in one step's row, given or by
// overflow, would reach the outputs of earlier steps of its chunk. The prep therefore checks each
// chunk (|v| at most kDnLargest, |k|^2 at most 1.01, g <= 0, which takes in -infinity, and beta in [0, 1]:
// what the layer produces) and the scan the state that it starts from (no value above
// kDnLargest): then nothing overflows, as k does not lengthen the state and a call has at most 2^22
// steps. A (row, head) with any other chunk, or 32 columns with any other state, are left to the step-by-step
// form, launched behind the scan, whose workgroups return at once when there is nothing to do.
#pragma once

#include "mtpk_device.h"

namespace mtpk {

constexpr int kDnChunk = 64;      // steps per chunk (C)
constexpr int kDnChunkDk = 128;   // the only k_dim of this form
constexpr int kDnScanCols = 32;   // state columns per scan workgroup
constexpr int kDnScanTiles = kDnScanCols / 16;
constexpr float kDnLargest = 1e30f;  // of v and of the first state; the sums of 2^22 steps of it are finite
constexpr int kDnKkRow = kDnChunk + 4;  // LDS row of a 64 x 64 matrix, padded

__device__ inline f32x4_t mfma16x16x4(float a, float b, f32x4_t c) {
  return __builtin_amdgcn_mfma_f32_16x16x4f32(a, b, c, 0, 0, 0);
}

// The workspace of one call. Matrices lie in 16 x 16 tiles of 64 x 16 bytes, lane (gq, c) holding row
// c, columns 4 gq .. 4 gq + 3 of its tile: the A operand of four products, read as one contiguous
// KB. (Read from row-major memory in that lane order, every lane quad touches four lines, and the
// scan ran at the L1's 14k tag lookups a chunk instead of its 4k.) Per (row, q/k head, chunk): k
// [4 step tiles][8], q the same (calls with outputs) and k transposed [8 k_dim tiles][4]; per (row,
// head, chunk): T [4][4], the masked q . k [4][4] (calls with outputs; both lower triangular, the
// tiles above the diagonal are not written), e^(G_i) and e^(G_C - G_i) [64] each, and a word that
// is nonzero when the chunk is not for this form. Per (row, head, scan workgroup): a word that is
// nonzero when the scan left its columns.
struct DnChunkWs {
  float* kr;
  float* qr;   // null without outputs
  float* kc;
  float* tm;
  float* am;   // null without outputs
  float* eg;
  float* dg;
  int32_t* odd;
  int32_t* left;
};
constexpr int kDnTile = 256;                  // floats of a tile
constexpr int kDnRowTiles = 32, kDnSqTiles = 16;  // tiles of a [64][128] and of a [64][64] matrix

// A piece of a call's steps whose scratch would pass the workspace: its first step (`lengths` count
// from the call's first), and in verify calls, whose pool keeps its values, a [heads][k_dim][v_dim]
// matrix set that carries the one row's state from piece to piece. A whole call has {0, null}.
struct DnPiece {
  int t0;
  float* carry;
};

// Steps of the piece that row `row` runs.
__device__ inline int dn_steps(const int64_t* lengths, int row, int t, int t0) {
  return lengths ? (int)min(max(lengths[row] - t0, (int64_t)0), (int64_t)t) : t;
}

// e^x of an fp64 exponent, to fp32 accuracy: rounding x to fp32 alone would cost |x| roundings.
__device__ inline float dn_exp(double x) {
  const float hi = (float)x;
  const float e = expf(hi);
  return fmaf(e, (float)(x - hi), e);
}

// c + a b for 16 x 16 tiles: a with lane (gq, c) holding row c, columns 4 gq + j; b and the result
// with lane (gq, c) holding rows 4 gq + j of column c.
__device__ inline f32x4_t dn_mma(f32x4_t a, f32x4_t b, f32x4_t acc) {
#pragma unroll
  for (int j = 0; j < 4; ++j) acc = mfma16x16x4(a[j], b[j], acc);
  return acc;
}

// The 16 x 16 x 128 product of a row tile and a column tile, in four partial sums (shorter runs of
// roundings than one sum of 128).
__device__ inline f32x4_t dn_dot(const u32x4_t* a, const u32x4_t* b) {
  f32x4_t p[4];
#pragma unroll
  for (int i = 0; i < 4; ++i) p[i] = f32x4_t{0.f, 0.f, 0.f, 0.f};
#pragma unroll
  for (int u = 0; u < 8; ++u)
    p[u & 3] = dn_mma(__builtin_bit_cast(f32x4_t, a[u]), __builtin_bit_cast(f32x4_t, b[u]), p[u & 3]);
  return (p[0] + p[1]) + (p[2] + p[3]);
}

// One workgroup of 4 waves per (row, q/k head, chunk). Wave w multiplies the 16 k rows of tile w
// and the 16 q rows of tile 3 - w with the k rows of the tiles at or before them (5 products of 16
// x 16 x 128 each), both matrices going to LDS, and copies its share of k and q into tiles; then each
// wave takes v heads of this q/k head: the decays, the two masked matrices, and the inverse T of
// (I + L). The four diagonal blocks are inverted side by side by forward substitution (lane
// (block, column)), and the tiles below them are
//   T[r][c] = -D[r] sum_{c<=m<r} L[r][m] T[m][c],  D[r] = T[r][r],
// 64 MFMAs; a product of T^T with the identity then leaves each tile in the order in which it is
// stored. (Substitution over all 64 rows, lane j holding column j, reads every L value back from
// LDS as a broadcast: 57 us a launch at 1500 steps of 64 heads, one workgroup per CU.)
template <bool OUT>
__global__ __launch_bounds__(256) void k_dn_chunk_prep(
    int t, int heads, int qk_heads, int dv, int nch, const float* __restrict__ q,
    const float* __restrict__ k, const float* __restrict__ v, const float* __restrict__ g,
    const float* __restrict__ beta, const int64_t* __restrict__ lengths, DnChunkWs ws, int t0) {
  constexpr int C = kDnChunk, DK = kDnChunkDk;
  __shared__ __attribute__((aligned(16))) float kk[C][kDnKkRow];
  __shared__ __attribute__((aligned(16))) float qk[OUT ? C : 1][kDnKkRow];
  constexpr int kDRow = 20, kDBlock = 16 * kDRow + 8;  // a diagonal block in LDS, padded against bank conflicts
  __shared__ __attribute__((aligned(16))) float diag[4][4 * kDBlock];
  __shared__ __attribute__((aligned(16))) double gs[4][C];
  __shared__ __attribute__((aligned(16))) float bs[4][C];
  int id = blockIdx.x;
  const int ch = id % nch;
  id /= nch;
  const int kh = id % qk_heads, row = id / qk_heads;
  const int rep = heads / qk_heads;
  const int n = dn_steps(lengths, row, t, t0);
  const int c0 = ch * C;
  if (c0 >= n) return;  // uniform: the scan does not visit this chunk
  const int tid = threadIdx.x, w = uniform(tid / kWave), lane = tid & (kWave - 1);
  const int gq = lane >> 4, c = lane & 15;
  // rows at or past n read as zeros (past the end of the buffer)
  const uint32_t stride = (uint32_t)qk_heads * DK * 4u, vstride = (uint32_t)heads * (uint32_t)dv * 4u;
  const rsrc_t rk = make_rsrc(k + (int64_t)row * t * qk_heads * DK, (uint32_t)n * stride);
  const rsrc_t rq = make_rsrc(q + (int64_t)row * t * qk_heads * DK, (uint32_t)n * stride);
  const rsrc_t rv = make_rsrc(v + (int64_t)row * t * heads * dv, (uint32_t)n * vstride);
  // element (step 16 tile + c, k index 16 u + 4 gq + j): the four j are one 16-byte load, and the
  // products of step (u, j) take that k index from both operands
  const uint32_t off = (uint32_t)(c0 + c) * stride + (uint32_t)kh * (DK * 4) + (uint32_t)gq * 16u;
  const int64_t kslab = ((int64_t)row * qk_heads + kh) * nch + ch;
  u32x4_t ka[8], qa[8];
#pragma unroll
  for (int u = 0; u < 8; ++u) {
    ka[u] = buf16(rk, off + (uint32_t)(16 * w) * stride + 64u * u);
    if (OUT) qa[u] = buf16(rq, off + (uint32_t)(16 * (3 - w)) * stride + 64u * u);
  }
  float kt[2][16];  // k_dim tiles 2 w and 2 w + 1: element (16 m + c, step 16 u + 4 gq + j)
#pragma unroll
  for (int u = 0; u < 4; ++u)
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      const uint32_t o = (uint32_t)(c0 + 16 * u + 4 * gq + j) * stride + (uint32_t)(kh * DK + 32 * w + c) * 4u;
#pragma unroll
      for (int m = 0; m < 2; ++m)
        kt[m][4 * u + j] = __builtin_bit_cast(float, __builtin_amdgcn_raw_buffer_load_b32(rk, (int)(o + 64u * m), 0, 0));
    }
  for (int b = 0; b < 4; ++b) {
    if (b > w && (!OUT || b > 3 - w)) continue;  // uniform over the wave
    u32x4_t kb[8];
#pragma unroll
    for (int u = 0; u < 8; ++u) kb[u] = buf16(rk, off + (uint32_t)(16 * b) * stride + 64u * u);
    if (b <= w) {
      const f32x4_t acc = dn_dot(ka, kb);
#pragma unroll
      for (int i = 0; i < 4; ++i) kk[16 * w + 4 * gq + i][16 * b + c] = acc[i];
    }
    if (OUT && b <= 3 - w) {
      const f32x4_t acc = dn_dot(qa, kb);
#pragma unroll
      for (int i = 0; i < 4; ++i) qk[16 * (3 - w) + 4 * gq + i][16 * b + c] = acc[i];
    }
  }
  {
    f32x4_t* const kr = reinterpret_cast<f32x4_t*>(ws.kr + kslab * (kDnRowTiles * kDnTile));
    f32x4_t* const kc = reinterpret_cast<f32x4_t*>(ws.kc + kslab * (kDnRowTiles * kDnTile));
#pragma unroll
    for (int u = 0; u < 8; ++u) kr[(w * 8 + u) * kWave + lane] = __builtin_bit_cast(f32x4_t, ka[u]);
    if (OUT) {
      f32x4_t* const qr = reinterpret_cast<f32x4_t*>(ws.qr + kslab * (kDnRowTiles * kDnTile));
#pragma unroll
      for (int u = 0; u < 8; ++u) qr[((3 - w) * 8 + u) * kWave + lane] = __builtin_bit_cast(f32x4_t, qa[u]);
    }
#pragma unroll
    for (int m = 0; m < 2; ++m)
#pragma unroll
      for (int u = 0; u < 4; ++u)
        kc[((2 * w + m) * 4 + u) * kWave + lane] =
            f32x4_t{kt[m][4 * u], kt[m][4 * u + 1], kt[m][4 * u + 2], kt[m][4 * u + 3]};
  }
  __syncthreads();
  for (int hh = w; hh < rep; hh += 4) {
    const int head = kh * rep + hh;
    const int64_t slab = ((int64_t)row * heads + head) * nch + ch;
    const bool live = c0 + lane < n;
    const int64_t hv = ((int64_t)row * t + c0 + (live ? lane : 0)) * heads + head;
    const float gl = live ? g[hv] : 0.f, bl = live ? beta[hv] : 0.f;
    // e^-1000 is 0 in fp32, and a finite sum keeps G_i - G_j defined
    double gsum = gl < -1000.f ? -1000.f : gl;
#pragma unroll
    for (int o = 1; o < kWave; o <<= 1) {
      const double up = __shfl_up(gsum, o, kWave);
      if (lane >= o) gsum += up;
    }
    gs[w][lane] = gsum;
    bs[w][lane] = bl;
    auto own_lds = [&]() {  // the wave reads back only what it wrote
      ring_fence();
      __builtin_amdgcn_s_waitcnt(0xC07F);
      ring_fence();
    };
    own_lds();
    ws.eg[slab * C + lane] = dn_exp(gsum);
    ws.dg[slab * C + lane] = dn_exp(gs[w][C - 1] - gsum);
    // v of the chunk's steps, read for its check alone (the scan then finds it in cache); the check
    // comes after the matrices, which hide its latency
    constexpr int kAhead = 16;  // 4 steps of 64 values a load
    auto load_v = [&](u32x4_t* vv, int d) {
#pragma unroll
      for (int e = 0; e < kAhead; ++e)
        vv[e] = buf16(rv, (uint32_t)(c0 + 4 * e + gq) * vstride + (uint32_t)(head * dv + d + 4 * c) * 4u);
    };
    u32x4_t v0[kAhead];
    load_v(v0, 0);
    f32x4_t* const am = reinterpret_cast<f32x4_t*>(ws.am + slab * (kDnSqTiles * kDnTile));
    f32x4_t lt[4][4];  // the tiles of L below the diagonal ones
    float* const dw = diag[w];
#pragma unroll
    for (int rt = 0; rt < 4; ++rt) {
      const int i = 16 * rt + c;
      const double gi = gs[w][i];
      const float bi = bs[w][i];
#pragma unroll
      for (int ct = 0; ct <= rt; ++ct) {
        f32x4_t lv, av;
        const int j0 = 16 * ct + 4 * gq;
        const f32x4_t kv = *reinterpret_cast<const f32x4_t*>(&kk[i][j0]);
        const f32x4_t qv = *reinterpret_cast<const f32x4_t*>(&qk[OUT ? i : 0][j0]);
#pragma unroll
        for (int e = 0; e < 4; ++e) {
          const float d = dn_exp(fmin(gi - gs[w][j0 + e], 0.0));
          lv[e] = j0 + e < i ? bi * d * kv[e] : 0.f;
          av[e] = j0 + e <= i ? d * qv[e] : 0.f;
        }
        if (ct == rt)
          *reinterpret_cast<f32x4_t*>(&dw[rt * kDBlock + c * kDRow + 4 * gq]) = lv;
        else
          lt[rt][ct] = lv;
        if (OUT) am[(rt * 4 + ct) * kWave + lane] = av;
      }
    }
    own_lds();
    // column c of block gq: D[i] = [i == c] - sum_{m<i} L[i][m] D[m]
    float dc[16];
#pragma unroll
    for (int i = 0; i < 16; ++i) {
      float acc = c == i ? 1.f : 0.f;
#pragma unroll
      for (int m4 = 0; m4 < (i + 3) / 4; ++m4) {
        const f32x4_t lr = *reinterpret_cast<const f32x4_t*>(&dw[gq * kDBlock + i * kDRow + 4 * m4]);
#pragma unroll
        for (int e = 0; e < 4; ++e)
          if (4 * m4 + e < i) acc = fmaf(-lr[e], dc[4 * m4 + e], acc);
      }
      dc[i] = acc;
    }
    own_lds();
#pragma unroll
    for (int i = 0; i < 16; ++i) dw[gq * kDBlock + i * kDRow + c] = dc[i];
    own_lds();
    const f32x4_t zero = {0.f, 0.f, 0.f, 0.f};
    f32x4_t tt[4][4];
#pragma unroll
    for (int rt = 0; rt < 4; ++rt) {
#pragma unroll
      for (int j = 0; j < 4; ++j) tt[rt][rt][j] = dw[rt * kDBlock + (4 * gq + j) * kDRow + c];
      const f32x4_t da = *reinterpret_cast<const f32x4_t*>(&dw[rt * kDBlock + c * kDRow + 4 * gq]);
#pragma unroll
      for (int ct = 0; ct < rt; ++ct) {
        f32x4_t acc = zero;
#pragma unroll
        for (int m = ct; m < rt; ++m) acc = dn_mma(lt[rt][m], tt[m][ct], acc);
        tt[rt][ct] = -dn_mma(da, acc, zero);
      }
    }
    f32x4_t* const tm = reinterpret_cast<f32x4_t*>(ws.tm + slab * (kDnSqTiles * kDnTile));
    f32x4_t one;  // the identity as a right operand
#pragma unroll
    for (int j = 0; j < 4; ++j) one[j] = 4 * gq + j == c ? 1.f : 0.f;
#pragma unroll
    for (int ct = 0; ct < 4; ++ct) {
      const f32x4_t bc = *reinterpret_cast<const f32x4_t*>(&bs[w][16 * ct + 4 * gq]);
#pragma unroll
      for (int rt = ct; rt < 4; ++rt) tm[(rt * 4 + ct) * kWave + lane] = dn_mma(tt[rt][ct], one, zero) * bc;
    }
    uint32_t most = 0;  // bits of the largest |v|; NaN and infinity lie above every number
    for (int d = 0; d < dv; d += kWave) {
      if (d > 0) load_v(v0, d);
#pragma unroll
      for (int e = 0; e < kAhead; ++e)
#pragma unroll
        for (int x = 0; x < 4; ++x) most = max(most, v0[e][x] & 0x7fffffffu);
    }
    const bool fine =
        gl <= 0.f && bl >= 0.f && bl <= 1.f && kk[lane][lane] <= 1.01f && most <= f32_bits(kDnLargest);
    const bool odd = __ballot(fine) != ~0ull;
    if (lane == 0) ws.odd[slab] = odd;
    own_lds();
  }
}

// Lane (gq, c)'s four values of tile `tile` of a [tile][lane] exchange area.
__device__ inline f32x4_t dn_tile(const f32x4_t* area, int tile, int lane) { return area[tile * kWave + lane]; }

// One workgroup of 8 waves per (row, head, 32 state columns), chunk after chunk. A wave owns a
// 16-column tile of the state's columns and one 16-row tile of the chunk's steps; S, Y and U pass
// between the four waves of a column tile through LDS in the MFMA result layout (lane (gq, c): rows
// 4 gq + i of column c), which is also the layout of the B operand that each next product reads.
// The A operands (k rows, q rows, k columns, T and the masked q . k) come from the prep's tiles,
// each reloaded for the next chunk as soon as it is used up, so nothing waits for a
// load that was not issued a whole chunk earlier. 128 MFMAs a wave and chunk (80 without outputs):
// 82 us of matrix time at 1500 steps of 64 heads, of the scan's 147 us (92 without outputs); the
// rest is the exchange behind the three barriers of a chunk.
template <bool OUT, bool COMMIT>
__global__ __launch_bounds__(256 * kDnScanTiles, 2) void k_dn_chunk_scan(
    float* __restrict__ state, int64_t slots_total, const int64_t* __restrict__ slot, int t,
    int heads, int qk_heads, int dv, int nch, const float* __restrict__ v,
    const int64_t* __restrict__ lengths, float* __restrict__ out, DnChunkWs ws, int bhs, DnPiece piece) {
  constexpr int C = kDnChunk, DK = kDnChunkDk;
  constexpr int NT = kDnScanTiles;
  __shared__ f32x4_t ss[NT][8 * kWave], sy[NT][4 * kWave], su[NT][4 * kWave], sd[NT][4 * kWave];
  __shared__ int over[4 * NT];
  // the column blocks of one head are bhs apart: with bhs a multiple of 8 they share an XCD's L2
  const int bh = blockIdx.x % bhs, cb = blockIdx.x / bhs;
  const int row = bh / heads, head = bh - row * heads, kh = head / (heads / qk_heads);
  const int tid = threadIdx.x, wave = uniform(tid / kWave), lane = tid & (kWave - 1);
  const int nt = wave >> 2, w = wave & 3, w2 = 3 - w;
  const int gq = lane >> 4, c = lane & 15;
  const int col = cb * kDnScanCols + 16 * nt + c;
  const int n = dn_steps(lengths, row, t, piece.t0);
  const int64_t s_idx = slot ? slot[row] : row;
  int32_t* const left = ws.left + (int64_t)bh * (dv / kDnScanCols) + cb;
  if (s_idx < 0 || s_idx >= slots_total) {  // no such slot: zero outputs, no state access
    if (OUT && w == 0)
      for (int st = gq; st < t; st += 4) out[(((int64_t)row * t + st) * heads + head) * dv + col] = 0.f;
    if (tid == 0) *left = 0;
    return;  // uniform over the workgroup
  }
  const int used = (n + C - 1) / C;
  const int64_t slab0 = (int64_t)bh * nch;
  bool odd = false;
  for (int i = lane; i < used; i += kWave) odd |= ws.odd[slab0 + i] != 0;
  const bool given = __ballot(odd) != 0ull;  // uniform: the step-by-step form takes it
  if (given || used == 0) {
    if (tid == 0) *left = given;
    return;
  }

  const uint32_t vstride = (uint32_t)heads * (uint32_t)dv * 4u;
  const rsrc_t rv = make_rsrc(v + (int64_t)row * t * heads * dv, (uint32_t)n * vstride);
  const rsrc_t ro = make_rsrc(OUT ? out + (int64_t)row * t * heads * dv : v, OUT ? (uint32_t)n * vstride : 0u);
  float* const pool = state + ((s_idx * heads + head) * DK) * (int64_t)dv + col;
  float* const kept = piece.carry ? piece.carry + (int64_t)head * DK * dv + col : pool;  // one row
  const float* const sp = piece.t0 > 0 ? kept : pool;

  f32x4_t s[8], own[2];  // every tile of this column tile's S (B operand), and the two it updates
#pragma unroll
  for (int m = 0; m < 8; ++m)
#pragma unroll
    for (int i = 0; i < 4; ++i) s[m][i] = sp[(int64_t)(16 * m + 4 * gq + i) * dv];
#pragma unroll
  for (int m = 0; m < 2; ++m)
#pragma unroll
    for (int i = 0; i < 4; ++i) own[m][i] = sp[(int64_t)(16 * (2 * w + m) + 4 * gq + i) * dv];

  u32x4_t ka[8], qa[8], kt[2][4], ta[4], aa[4];
  float va[4], eg[4], dg[4], eq[4], egc;
  const int64_t kslab0 = ((int64_t)row * qk_heads + kh) * nch;
  constexpr uint32_t kRowB = kDnRowTiles * kDnTile * 4u, kSqB = kDnSqTiles * kDnTile * 4u, kTileB = kDnTile * 4u;
  const uint32_t lane16 = (uint32_t)lane * 16u;
  auto load_rows = [&](int ch) {  // the operands of the products with S0
    const rsrc_t rk = make_rsrc(ws.kr + (kslab0 + ch) * (kDnRowTiles * kDnTile), kRowB);
#pragma unroll
    for (int u = 0; u < 8; ++u) ka[u] = buf16(rk, lane16 + (uint32_t)(w * 8 + u) * kTileB);
    if (OUT) {
      const rsrc_t rq = make_rsrc(ws.qr + (kslab0 + ch) * (kDnRowTiles * kDnTile), kRowB);
#pragma unroll
      for (int u = 0; u < 8; ++u) qa[u] = buf16(rq, lane16 + (uint32_t)(w2 * 8 + u) * kTileB);
    }
#pragma unroll
    for (int i = 0; i < 4; ++i)
      va[i] = __builtin_bit_cast(float, __builtin_amdgcn_raw_buffer_load_b32(
          rv, (int)((uint32_t)(ch * C + 16 * w + 4 * gq + i) * vstride + (uint32_t)(head * dv + col) * 4u), 0, 0));
    const float* const e = ws.eg + (slab0 + ch) * C;
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      eg[i] = e[16 * w + 4 * gq + i];
      if (OUT) eq[i] = e[16 * w2 + 4 * gq + i];
    }
  };
  // tiles above the diagonal read as zeros (out of range, no memory access)
  auto load_sq = [&](u32x4_t* x, const float* m, int ch, int rt) {
    const rsrc_t r = make_rsrc(m + (slab0 + ch) * (kDnSqTiles * kDnTile), kSqB);
#pragma unroll
    for (int u = 0; u < 4; ++u)
      x[u] = buf16(r, (lane16 + (uint32_t)(rt * 4 + u) * kTileB) | ((uint32_t)(u > rt) << 31));
  };
  auto load_t = [&](int ch) {
    load_sq(ta, ws.tm, ch, w);
    const float* const d = ws.dg + (slab0 + ch) * C;
#pragma unroll
    for (int i = 0; i < 4; ++i) dg[i] = d[16 * w + 4 * gq + i];
  };
  auto load_cols = [&](int ch) {  // k by columns, and the masked q . k
    egc = ws.eg[(slab0 + ch) * C + C - 1];
    const rsrc_t rk = make_rsrc(ws.kc + (kslab0 + ch) * (kDnRowTiles * kDnTile), kRowB);
#pragma unroll
    for (int m = 0; m < 2; ++m)
#pragma unroll
      for (int u = 0; u < 4; ++u) kt[m][u] = buf16(rk, lane16 + (uint32_t)((2 * w + m) * 4 + u) * kTileB);
    if (OUT) load_sq(aa, ws.am, ch, w2);
  };
  // in the order in which every chunk reloads them, so that the loop's waits count alike
  ring_fence();
  load_rows(0);
  ring_fence();
  load_t(0);
  ring_fence();
  load_cols(0);
  ring_fence();
  uint32_t most = 0;
#pragma unroll
  for (int m = 0; m < 8; ++m)
#pragma unroll
    for (int i = 0; i < 4; ++i) most = max(most, f32_bits(s[m][i]) & 0x7fffffffu);
  const bool large = __ballot(most > f32_bits(kDnLargest)) != 0ull;
  if (lane == 0) over[wave] = large;
  auto barrier = [&]() {  // LDS only: the next chunk's loads stay in flight
    ring_fence();
    __builtin_amdgcn_s_waitcnt(0xC07F);
    __builtin_amdgcn_s_barrier();
    ring_fence();
  };
  barrier();
  int any = 0;
#pragma unroll
  for (int i = 0; i < 4 * NT; ++i) any |= over[i];
  if (tid == 0) *left = any;
  if (any) return;  // uniform over the workgroup
  int ch = 0;  // used >= 1: a bottom-tested loop keeps the loads above in front of it
#pragma clang loop unroll(disable)
  do {
    const int nx = min(ch + 1, used - 1);  // past the end: the last chunk again, unused
    // Y = V - e^G (K S0), this wave's 16 steps; then Q S0 of its 16 output steps
    // (sums of 128 in four parts: shorter runs of roundings)
    const f32x4_t zero = {0.f, 0.f, 0.f, 0.f};
    f32x4_t xp[4] = {zero, zero, zero, zero}, o = zero;
#pragma unroll
    for (int u = 0; u < 8; ++u)
#pragma unroll
      for (int j = 0; j < 4; ++j) xp[u & 3] = mfma16x16x4(bits_f32(ka[u][j]), s[u][j], xp[u & 3]);
    const f32x4_t x = (xp[0] + xp[1]) + (xp[2] + xp[3]);
    f32x4_t y;
#pragma unroll
    for (int i = 0; i < 4; ++i) y[i] = va[i] - eg[i] * x[i];
    sy[nt][w * kWave + lane] = y;
    if (OUT) {
      f32x4_t op[4] = {zero, zero, zero, zero};
#pragma unroll
      for (int u = 0; u < 8; ++u)
#pragma unroll
        for (int j = 0; j < 4; ++j) op[u & 3] = mfma16x16x4(bits_f32(qa[u][j]), s[u][j], op[u & 3]);
      o = (op[0] + op[1]) + (op[2] + op[3]);
#pragma unroll
      for (int i = 0; i < 4; ++i) o[i] *= eq[i];
    }
    ring_fence();
    load_rows(nx);
    barrier();
    // U = T Y
    f32x4_t uu = zero;
#pragma unroll
    for (int u = 0; u < 4; ++u) {
      const f32x4_t yv = dn_tile(sy[nt], u, lane);
#pragma unroll
      for (int j = 0; j < 4; ++j) uu = mfma16x16x4(bits_f32(ta[u][j]), yv[j], uu);
    }
    if (OUT) su[nt][w * kWave + lane] = uu;
    f32x4_t du;
#pragma unroll
    for (int i = 0; i < 4; ++i) du[i] = dg[i] * uu[i];
    sd[nt][w * kWave + lane] = du;
    ring_fence();
    load_t(nx);
    barrier();
    // S = e^(G_C) S0 + K^T (e^(G_C - G) U), state rows 32 w .. 32 w + 31
#pragma unroll
    for (int m = 0; m < 2; ++m)
#pragma unroll
      for (int i = 0; i < 4; ++i) own[m][i] *= egc;
#pragma unroll
    for (int u = 0; u < 4; ++u) {
      const f32x4_t dv4 = dn_tile(sd[nt], u, lane);
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        own[0] = mfma16x16x4(bits_f32(kt[0][u][j]), dv4[j], own[0]);
        own[1] = mfma16x16x4(bits_f32(kt[1][u][j]), dv4[j], own[1]);
      }
    }
    ss[nt][(2 * w) * kWave + lane] = own[0];
    ss[nt][(2 * w + 1) * kWave + lane] = own[1];
    if (OUT) {
      f32x4_t au = zero;
#pragma unroll
      for (int u = 0; u < 4; ++u) au = dn_mma(__builtin_bit_cast(f32x4_t, aa[u]), dn_tile(su[nt], u, lane), au);
      o += au;
#pragma unroll
      for (int i = 0; i < 4; ++i)  // steps at or past n lie past the end of the buffer: not stored
        __builtin_amdgcn_raw_buffer_store_b32(
            f32_bits(o[i]), ro,
            (int)((uint32_t)(ch * C + 16 * w2 + 4 * gq + i) * vstride + (uint32_t)(head * dv + col) * 4u), 0, 0);
    }
    ring_fence();
    load_cols(nx);
    barrier();
#pragma unroll
    for (int m = 0; m < 8; ++m) s[m] = dn_tile(ss[nt], m, lane);
  } while (++ch < used);
  if (COMMIT) {
#pragma unroll
    for (int m = 0; m < 2; ++m)
#pragma unroll
      for (int i = 0; i < 4; ++i) kept[(int64_t)(16 * (2 * w + m) + 4 * gq + i) * dv] = own[m][i];
  }
}

}  // namespace mtpk
