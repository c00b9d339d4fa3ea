// Causal GQA attention of many query rows per kv head (a prompt, or the next piece of one) over
// the paged cache of mtpk_attention.hip.
//
// The rows of a kv head are taken token by token (row r = step r / group, q head r % group), 128
// to a workgroup, 32 to a wave, so a workgroup's rows span few positions and it reads only the keys
// up to its last one. Both products are transposed, so that a lane
// holds one query row:
//   S^T = K Q^T   v_mfma_f32_32x32x16_bf16, A = 32 keys from LDS, B = Q (registers)
//   O^T += V^T P^T  A = V^T from LDS (the cache's own layout), B = P
// Row m of a K tile is its key with bits 2 and 3 of m swapped: then the S^T values that a lane gets
// (query row l % 32, rows 8 i + 4 (l / 32) + 0..3 of the tile) are 8 adjacent keys of each 16, which
// is the B operand of O^T with V^T read 16 bytes at a time, so P never leaves its registers. The
// row maximum needs one exchange with lane l ^ 32, and the rescaling of O is a lane's own factor.
// The reference exponent of a row moves with its maximum, as in the decode form, so that the largest
// P is exactly 1: error against 64 bits at 2047 rows 3.07e-3 in both forms, and nearly all outputs
// the same bits (moved only once a score lay 2^8 above it, P of the largest key was a rounded
// value: 3.13e-3, at 103 us). Tiles of 32 keys go straight to LDS, one tile ahead, in two
// buffers with one barrier per tile; their 16-byte pieces are permuted on the way (by the key, or by
// the channel) so that the reads fall on all banks.
//
// 115 us at 2047 rows of 32 heads of 256 on 2 kv heads (69 GFLOP: 0.60 PFLOP/s) against 382 us for
// the decode form, which runs every row group over all keys with 16 rows a wave. What is
// left: the heaviest workgroup's 64 tiles one after another (products, softmax, rescaling, products),
// whose CU partner ends early. Two teams of four waves on alternate tiles in one workgroup halved
// that chain but run in lockstep, matrix unit and softmax taking turns: slower by a quarter.
#pragma once

#include "mtpk_device.h"

namespace mtpk {

typedef float f32x16_t __attribute__((ext_vector_type(16)));
typedef uint32_t u32x2_t __attribute__((ext_vector_type(2)));

constexpr int kPromptRows = 128;  // query rows per workgroup
constexpr int kPromptKeys = 32;   // keys per tile

// The row groups' order: heaviest first; where every workgroup is resident at once (two per CU),
// the second half of the ids lightest first instead, so that a CU's two add up evenly.
__device__ inline int prompt_row_group(int rank, int row_groups, int paired) {
  const int half = (row_groups + 1) / 2;
  return paired && rank >= half ? rank - half : row_groups - 1 - rank;
}

// Keys [0, end) that row group `rg` sees.
__device__ __host__ inline int prompt_keys_end(int bp, int rg, int rows, int group) {
  const int last = rg * kPromptRows + kPromptRows - 1;
  return bp + (last < rows ? last : rows - 1) / group + 1;
}

// Bits 2 and 3 of a tile's key or row index swapped.
__device__ inline int prompt_swap(int i) { return (i & ~12) | ((i & 4) << 1) | ((i & 8) >> 1); }

// The change of place of a K row's pieces: the rows 0..3 and 0..7 that one LDS cycle reads, of either
// half of the wave, then lie in different bank groups.
__device__ inline int prompt_flip(int row) { return ((row & 3) << 1) | (row >> 2 & 1); }

template <int HD>
__global__ __launch_bounds__(256, 2) void k_prompt_attention(
    AttnIO io, const uint16_t* __restrict__ k_pool, const uint16_t* __restrict__ v_pool,
    int64_t pool_rows, const int32_t* __restrict__ table, int table_stride,
    const int64_t* __restrict__ base_pos, int t, int heads, int kvh, int bk, float scale_log2,
    int n_split, int row_groups, int paired, int wide, float* __restrict__ part_o, float* __restrict__ part_ml) {
  constexpr int KS = HD / 16, NT = HD / 32, PK = HD / 8;  // k steps, d tiles, 16-byte pieces of a key
  constexpr int kTile = kPromptKeys * HD * 2;             // bytes of a K (or V) tile
  constexpr int kLoads = kTile / 1024 / 4;                // 1 KB loads per wave and tensor
  static_assert(kLoads >= 1, "a tile splits over four waves");
  __shared__ __attribute__((aligned(16))) uint8_t smem[4 * kTile];  // two buffers of (K, V)
  const int group = heads / kvh, R = group * t;
  const int rg = prompt_row_group((int)blockIdx.x / bk, row_groups, paired);
  const int bkh = (int)blockIdx.x % bk, kh = bkh % kvh, b = bkh / kvh;
  const int sp = blockIdx.y;
  const int tid = threadIdx.x, wave = uniform(tid / kWave), lane = tid & (kWave - 1);
  const int h = lane >> 5, c = lane & 31;
  const int bp = uniform((int)base_pos[b]);
  int k0, k1;
  attn_split_range(prompt_keys_end(bp, rg, R, group), n_split, sp, k0, k1);
  k0 = uniform(k0);
  k1 = uniform(k1);
  if (k0 >= k1) return;  // uniform: an empty split writes nothing (the merge skips it)

  const int r = kPromptRows * rg + 32 * wave + c;
  const int qpos = r < R ? bp + r / group : -1;
  // the tiles at or past the first row's position are masked row by row
  const int first_pos = bp + kPromptRows * rg / group;
  bf16x8_t q[KS];
  {  // rows past R read row 0 and see no key
    const int rq = r < R ? r : 0;
    const uint16_t* const qrow = io.q + io.qr.at(b, kh * group + rq % group, rq / group) + 8 * h;
    u32x4_t d[KS];
#pragma unroll
    for (int s = 0; s < KS; ++s) d[s] = ld16(qrow + 16 * s);
#pragma unroll
    for (int s = 0; s < KS; ++s) {
      asm volatile("" : "+v"(d[s]));  // landed before the loop: its waits count the tiles' loads alone
      q[s] = as_bf16x8(d[s]);
    }
  }
  const int32_t* const trow = table + (int64_t)b * table_stride;
  // Tile at key0 (this wave's block of it is p) into a buffer: K as [key][piece ^ prompt_flip(row)], V as
  // [block][channel][piece ^ (channel / 4 & 1)]. Each block is a buffer of its own that ends with the
  // last key below k1 (V: with the block), so a lane's offsets are the same for every tile and keys
  // past k1, or of a block outside the pool, read as zeros.
  uint32_t koff[kLoads];
#pragma unroll
  for (int j = 0; j < kLoads; ++j) {
    const int key = (wave * kLoads + j) * (64 / PK) + lane / PK;  // an instruction's keys lie in one block
    koff[j] = (uint32_t)((((key & (kAttnBlock - 1)) * kvh + kh) * HD + ((lane % PK) ^ prompt_flip(prompt_swap(key))) * 8) * 2);
  }
  // channel 32 i + lane / 2 of the block's load i, i.e. one offset plus 1 KB per load
  const uint32_t voff = (uint32_t)(kh * HD * 32 + (wave & 1) * (kLoads * 1024) + (lane >> 1) * 32 +
                                   (((lane & 1) ^ (lane >> 3 & 1)) * 16));
  const int64_t slab = (int64_t)kAttnBlock * kvh * HD;  // elements of a block, K or V
  const int half = wave >> 1;  // the tile's block that this wave loads
  auto stage = [&](int buf, int key0, int p) {
    p = uniform(p);
    const bool ok = p >= 0 && (int64_t)(p + 1) * kAttnBlock <= pool_rows;
    const int left = uniform(ok ? k1 - key0 - kAttnBlock * half : 0);  // keys below k1 from the block's first
    const int64_t at = (int64_t)uniform(ok ? p : 0) * slab;
    const rsrc_t rk = make_rsrc(k_pool + at, (uint32_t)uniform(max(min(left, kAttnBlock), 0) * kvh * HD * 2));
    const rsrc_t rv = make_rsrc(v_pool + at, left > 0 ? (uint32_t)(kAttnBlock * kvh * HD * 2) : 0u);
    uint8_t* const to = smem + buf + wave * (kLoads * 1024);
#pragma unroll
    for (int j = 0; j < kLoads; ++j) {
      __builtin_amdgcn_raw_ptr_buffer_load_lds(rk, (lds_void_t*)(to + j * 1024), 16, (int)koff[j], 0, 0, 0);
      __builtin_amdgcn_raw_ptr_buffer_load_lds(rv, (lds_void_t*)(to + kTile + j * 1024), 16, (int)(voff + 1024u * j), 0, 0, 0);
    }
  };

  float m = -INFINITY, l = 0.f;
  f32x16_t o[NT];
#pragma unroll
  for (int dt = 0; dt < NT; ++dt)
#pragma unroll
    for (int i = 0; i < 16; ++i) o[dt][i] = 0.f;
  // this lane's K pieces: 2 s + h of tile row c, whose place is that of piece h with bits of s flipped
  const uint32_t kat = (uint32_t)(prompt_swap(c) * HD * 2 + ((h ^ prompt_flip(c)) * 16));
  // and its V^T keys: 8 h .. 8 h + 7 of each block, channel 32 dt + c
  const uint32_t vat = (uint32_t)(kTile + c * 32 + (h ^ (c >> 2 & 1)) * 16);

  auto block = [&](int key0) { return sload(trow, min(key0 / kAttnBlock + half, table_stride - 1)); };
  stage(0, k0, block(k0));
  int next = block(k0 + kPromptKeys);
  int buf = 0;  // byte offset of the tile's buffer
  for (int key0 = k0; key0 < k1; key0 += kPromptKeys, buf ^= 2 * kTile) {
    ring_fence();
    vmcnt_wait<0>();  // this tile, issued a tile ago
    __builtin_amdgcn_s_barrier();
    ring_fence();
    if (key0 + kPromptKeys < k1) {
      stage(buf ^ (2 * kTile), key0 + kPromptKeys, next);  // last read a tile ago, before the barrier
      next = block(key0 + 2 * kPromptKeys);
    }
    ring_fence();
    const uint32_t ka = (uint32_t)buf + kat, va = (uint32_t)buf + vat;
    if (key0 + kPromptKeys > k1) {  // uniform: the last tile, partly past k1: V there becomes zeros (P is zero there)
      for (int i = tid; i < 2 * HD; i += 256) {
        const int blk = i / HD, d = i % HD;
        for (int e = 0; e < kAttnBlock; ++e)
          if (key0 + kAttnBlock * blk + e >= k1)
            *reinterpret_cast<uint16_t*>(smem + buf + kTile + i * 32 + (((e >> 3) ^ (d >> 2 & 1)) * 16) + (e & 7) * 2) = 0;
      }
      __syncthreads();
    }
    f32x16_t s;
#pragma unroll
    for (int i = 0; i < 16; ++i) s[i] = 0.f;
    // operands come from LDS four products ahead (fenced: the compiler would read each one just
    // before its product and wait out the LDS latency 32 times a tile: 152 against 132 us with the rest as it was)
    u32x4_t f[4];
    auto kfrag = [&](int i) { return lds16(smem + (ka ^ (32u * (i & 3))) + 128 * (i >> 2)); };
    auto vfrag = [&](int i) { return lds16(smem + va + (i % NT) * 1024 + (i / NT) * (HD * 32)); };
#pragma unroll
    for (int i = 0; i < 4; ++i) f[i] = kfrag(i);
    ring_fence();
#pragma unroll
    for (int i = 0; i < KS; ++i) {
      s = __builtin_amdgcn_mfma_f32_32x32x16_bf16(as_bf16x8(f[i & 3]), q[i], s, 0, 0, 0);
      f[i & 3] = i + 4 < KS ? kfrag(i + 4) : vfrag(i + 4 - KS);
      ring_fence();
    }
    if (key0 + kPromptKeys > first_pos) {  // uniform: some key may lie past some row
#pragma unroll
      for (int i = 0; i < 16; ++i) {
        const int key = key0 + 16 * (i >> 3) + 8 * h + (i & 7);
        if (key > qpos || key >= k1) s[i] = -INFINITY;
      }
    }
    float tm = s[0];
#pragma unroll
    for (int i = 1; i < 16; ++i) tm = fmaxf(tm, s[i]);
    tm = fmaxf(tm, __shfl_xor(tm, 32, kWave));
    const float mn = fmaxf(m, tm * scale_log2);
    if (__ballot(mn > m) != 0ull) {  // uniform over the wave
      const float alpha = mn == -INFINITY ? 1.f : exp2f(m - mn);
      m = mn;
      l *= alpha;
#pragma unroll
      for (int dt = 0; dt < NT; ++dt)
#pragma unroll
        for (int i = 0; i < 16; ++i) o[dt][i] *= alpha;
    }
    const float ms = m == -INFINITY ? 0.f : m;  // a row with no key so far: every e below is 0
    bf16x8_t p[2];
    float part[4] = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int i = 0; i < 16; ++i) {
      const float e = __builtin_amdgcn_exp2f(fmaf(s[i], scale_log2, -ms));  // in [0, 1]; 0 below 2^-126
      part[i & 3] += e;
      p[i >> 3][i & 7] = (__bf16)e;
    }
    l += (part[0] + part[1]) + (part[2] + part[3]);
#pragma unroll
    for (int i = 0; i < KS; ++i) {
      o[i % NT] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(as_bf16x8(f[i & 3]), p[i / NT], o[i % NT], 0, 0, 0);
      if (i + 4 < KS) f[i & 3] = vfrag(i + 4);
      ring_fence();
    }
  }
  l += __shfl_xor(l, 32, kWave);
  const int row = 32 * wave + c;
  // o[dt][4 i + e] is channel 32 dt + 8 i + 4 h + e of the row
  if (n_split == 1) {
    // Through LDS into whole bf16 rows: a lane holds 8 bytes here and there of its row, and stored
    // (and the gate read) like that, every instruction would touch 64 lines. 16-byte pieces at
    // [row][piece ^ row].
    constexpr int kFlip = PK - 1 < 15 ? PK - 1 : 15;
    const float inv = 1.f / l;
    __syncthreads();  // the last tile's reads are done
#pragma unroll
    for (int dt = 0; dt < NT; ++dt)
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        const int d = 32 * dt + 8 * i + 4 * h;
        uint32_t w[2];
#pragma unroll
        for (int e = 0; e < 2; ++e)
          w[e] = (uint32_t)f32_to_bf16(o[dt][4 * i + 2 * e] * inv) |
                 ((uint32_t)f32_to_bf16(o[dt][4 * i + 2 * e + 1] * inv) << 16);
        *reinterpret_cast<u32x2_t*>(smem + row * (HD * 2) + ((d >> 3) ^ (row & kFlip)) * 16 + (d & 4) * 2) = u32x2_t{w[0], w[1]};
      }
    __syncthreads();
#pragma unroll 2
    for (int i = tid; i < kPromptRows * PK; i += 256) {  // 8 channels each
      const int rl = i / PK, p = i % PK, ro = kPromptRows * rg + rl;
      if (ro >= R) break;
      const int st = ro / group, hq = kh * group + ro % group;
      u32x4_t w = lds16(smem + rl * (HD * 2) + (p ^ (rl & kFlip)) * 16);
      uint16_t* const orow = io.out + io.orow.at(b, hq, st) + 8 * p;
      if (io.gate) {
        const uint16_t* const grow = io.gate + io.gr.at(b, hq, st) + 8 * p;
        u32x4_t g;
        if (wide) {
          g = ld16(grow);
        } else {
#pragma unroll
          for (int e = 0; e < 4; ++e) g[e] = grow[2 * e] | ((uint32_t)grow[2 * e + 1] << 16);
        }
#pragma unroll
        for (int e = 0; e < 4; ++e)
          w[e] = (uint32_t)attn_gated(true, (uint16_t)(g[e] & 0xffffu), bits_f32(w[e] << 16)) |
                 ((uint32_t)attn_gated(true, (uint16_t)(g[e] >> 16), bits_f32(w[e] & 0xffff0000u)) << 16);
      }
      if (wide) {  // uniform: output and gate rows on 16-byte boundaries
        *reinterpret_cast<u32x4_t*>(orow) = w;
      } else {
#pragma unroll
        for (int e = 0; e < 4; ++e) {
          orow[2 * e] = (uint16_t)(w[e] & 0xffffu);
          orow[2 * e + 1] = (uint16_t)(w[e] >> 16);
        }
      }
    }
  } else {
    if (kPromptRows * rg + row >= R) return;
    const int64_t pr = (((int64_t)bkh * row_groups + rg) * n_split + sp) * kPromptRows + row;
    float* const po = part_o + pr * HD;
#pragma unroll
    for (int dt = 0; dt < NT; ++dt)
#pragma unroll
      for (int i = 0; i < 4; ++i)
        *reinterpret_cast<f32x4_t*>(po + 32 * dt + 8 * i + 4 * h) =
            f32x4_t{o[dt][4 * i], o[dt][4 * i + 1], o[dt][4 * i + 2], o[dt][4 * i + 3]};
    if (h == 0) {
      part_ml[pr * 2] = m;
      part_ml[pr * 2 + 1] = l;
    }
  }
}

}  // namespace mtpk
