// Routed MXFP4 MoE over a prompt's rows: units of up to 64 tokens of one expert. Included by
// mtpk_moe.hip.
//
// The 16-token units read and decode an expert's weights once per 16 of its tokens, which over a
// prompt is several times (2048 rows of 10 of 512 experts: 1547 units, gate_up 999 us and down
// 586 us where the weights alone are 3.4 GB, about 550 us). Here a decoded weight fragment feeds up
// to four token tiles. 8 waves stage the unit's activation rows, each wave streams its own weight
// rows from HBM to registers:
//   gate_up  item = (unit, 128 intermediate rows); a wave has 16 gate rows and the matching up rows
//   down     item = (half a unit, 512 hidden rows); a wave has four tiles of 16 rows. Two planes
//            make a staged row twice as long, and four tiles of 64 tokens would spill.
// Measured at 2048 rows: gate_up 671 us, down 519 us, the whole call 1604 -> 1259 us. The sums run in
// the order of k_moe_gate_up_lds and k_moe_down_lds: the same bits (not k_moe_gate_up's split form,
// which takes calls of few units). N is a multiple of 512: every item has all of its weight rows.
// What bounds it is the weight stream as long as most experts have one unit. Token rows go straight
// to LDS (256 k a chunk, no registers), so that 128 VGPRs leave two workgroups a CU and one's item
// start hides behind the other's stream. The weights are the A operand: a lane ends with
// four consecutive output columns of one token, stored together.
#pragma once

constexpr int kWideTokens = 64;  // tokens of a unit
constexpr int kWideWaves = 8;
constexpr int kWideThreads = kWideWaves * kWave;
constexpr int kWideBuf = kWideTokens * 512;  // a chunk: 64 rows of 256 k, or 32 of two planes

// lds_barrier, and no LDS read moves above it: what lies there came by direct-to-LDS loads.
__device__ inline void wide_barrier() {
  lds_barrier();
  __asm__ volatile("" ::: "memory");
}

// A staged row's 16-byte piece p lies at slot p ^ (row & 15): the 16 lanes that read one piece of 16
// rows take 16 different slots of 256 bytes (rows are 512 or 1024 bytes apart, so unswizzled they would all
// meet on the same four banks). A direct-to-LDS load writes 64 slots in order, so the swizzle is in
// the address that each lane loads from.
template <bool UP>
__global__ __launch_bounds__(kWideThreads, 4) void k_moe_wide(
    const uint16_t* __restrict__ x, uint32_t x_bytes, int64_t x_plane, int K,
    const uint8_t* __restrict__ wq, const uint8_t* __restrict__ ws, int N, UnitSrc src, int top_k,
    uint16_t* __restrict__ inter, int64_t inter_plane, float* __restrict__ y) {
  constexpr int S = UP ? 2 : 4;        // weight streams of a wave (gate and up, or four tiles)
  constexpr int TPC = 2;               // trips of 128 k per staged chunk
  constexpr int NPL = UP ? 1 : 2;      // bf16 planes of a staged row
  constexpr int kTurns = UP ? 8 : 2;   // 4-trip turns: K <= 4096, K <= 1024
  constexpr int kRow = NPL * 512;      // LDS bytes of a staged row
  constexpr int kLoads = NPL;          // staging loads of a wave per 16 token rows
  constexpr int kHalves = UP ? 1 : 2;  // items of one unit and weight group
  constexpr int kScalePieces = S * 16 * kTurns / kWave;
  constexpr int kItemTiles = UP ? kWideWaves : kWideWaves * S;
  static_assert(S * 16 * kTurns * 16 * kWideWaves <= kWideBuf, "layout");
  __shared__ __attribute__((aligned(16))) uint8_t xs[2 * kWideBuf];
  const int ngroup = N / (16 * kItemTiles);
  const int n_items = min(sload(src.n_units, 0), src.max_units) * ngroup * kHalves;
  const int tid = threadIdx.x, wave = uniform(tid / kWave);
  const int nb = K >> 5, ntrip = nb >> 2, nchunk = ntrip / TPC, segs = nb >> 4;
  const uint32_t row_bytes = (uint32_t)(K >> 1);
  const int rows = UP ? 2 * N : N;  // weight rows of one expert
  const uint32_t exp_bytes = (uint32_t)rows * row_bytes;
  const rsrc_t rx = make_rsrc(x, x_bytes);
  const int whole = (int)gridDim.x - (int)gridDim.x % (ngroup * kHalves);
  const int alternate = whole > 0 ? whole : INT32_MAX;
  for (int item = blockIdx.x; item < n_items; item += gridDim.x) {
    // Down's two halves of a unit and weight group are ngroup items apart: on one XCD when that is a
    // multiple of 8, close in time, sharing its L2. Which comes first alternates with the grid's
    // rounds: many units have an empty second half, and a workgroup would meet only those (without
    // it down took 629 us at 2048 rows, 519 with, and 167 against 108 at 64).
    const int uh = item / ngroup, q = item - uh * ngroup, u = uh / kHalves;
    const int past = ((uh + item / alternate) & (kHalves - 1)) * (kWideTokens / kHalves);
    const int e = sload(src.units, 3 * u), first = sload(src.units, 3 * u + 1) + past;
    const int cnt = min(sload(src.units, 3 * u + 2) - past, kWideTokens / kHalves);
    if (cnt <= 0) continue;  // uniform over the workgroup
    int lane = tid & (kWave - 1);
    __asm__ volatile("" : "+v"(lane));  // an item's addresses are made anew: kept, they would spill
    const MoeLane ln = moe_lane(lane);
    const uint32_t sel01 = lane_byte_sel01(ln.g);
    // where this lane's pieces 4 g + h of its token row (tile 0, trip 0, plane 0) lie
    uint32_t ha[4];
#pragma unroll
    for (int h = 0; h < 4; ++h) ha[h] = (uint32_t)(ln.c * kRow + (((4 * ln.g + h) ^ ln.c) << 4));
    const int tile0 = UP ? q * kWideWaves + wave : (q * kWideWaves + wave) * S;
    const rsrc_t rw = make_rsrc(wq + (int64_t)e * exp_bytes, exp_bytes);
    const rsrc_t rs = make_rsrc(ws + (int64_t)e * rows * nb, (uint32_t)rows * (uint32_t)nb);
    auto stream_row = [&](int r) { return UP ? r * N + tile0 * 16 : (tile0 + r) * 16; };  // first row of stream r

    auto run = [&](auto nt_c) {
      constexpr int NT = decltype(nt_c)::value;  // token tiles of this unit
      // Few token tiles leave registers and LDS for deeper prefetch: weights LA chunks ahead, token
      // rows SA chunks ahead (64 rows 352 -> 339 us, 2048 rows 1371 -> 1336 us).
      constexpr int LA = UP && NT <= 2 ? 2 : 1, SA = NT * NPL <= 2 ? 2 : 1;
      constexpr int kBuf = NT * 16 * kRow;
      static_assert((SA + 1) * kBuf <= 2 * kWideBuf && SA * kBuf <= kWideBuf && SA <= LA + 1, "");
      // Staging: a wave's load moves two rows of 512 bytes, or one of 1024, whose address is then
      // uniform but for the piece (and rows 8 apart differ by one bit of the swizzle).
      constexpr int NL = NT * kLoads;
      uint32_t sx[NL];
      uint32_t vx = 0;
      if constexpr (UP) {
#pragma unroll
        for (int j = 0; j < NL; ++j) {
          const int r = 16 * j + 2 * wave + (lane >> 5);
          const int a = src.sorted[first + min(r, cnt - 1)];
          const uint32_t at = (uint32_t)(a / top_k) * (uint32_t)K * 2u + (uint32_t)((lane & 31) ^ (r & 15)) * 16u;
          sx[j] = r < cnt ? at : kOutOfRange;
        }
      } else {
        const int piece = lane ^ wave;
        vx = (uint32_t)(piece >> 5) * (uint32_t)x_plane * 2u + (uint32_t)(piece & 31) * 16u;
#pragma unroll
        for (int j = 0; j < NL; ++j) {
          const int r = 8 * j + wave, a = sload(src.sorted, first + min(r, cnt - 1));
          sx[j] = r < cnt ? (uint32_t)a * (uint32_t)K * 2u : kOutOfRange;
        }
      }
      auto stage = [&](int c, int b) {  // chunk c at byte b of xs; past the last chunk: zeros, unread
        const uint32_t bad = (uint32_t)!(c < nchunk) << 31;
#pragma unroll
        for (int j = 0; j < NL; ++j) {
          const uint32_t at = (sx[j] + (uint32_t)c * 512u) | bad;
          buf16_lds(rx, UP ? at : (vx ^ (uint32_t)(j & 1) * 128u) + at,
                    xs + b + (8 * j + wave) * 1024);
        }
      };
      const uint32_t vrow = (uint32_t)ln.c * row_bytes + (uint32_t)ln.g * 16u;
      u32x4_t ring[LA * TPC][S];
      auto issue = [&](int s, int tr) {
        const uint32_t bad = (uint32_t)!(tr < ntrip) << 31;
#pragma unroll
        for (int r = 0; r < S; ++r)
          ring[s][r] = buf16(rw, (vrow + (uint32_t)tr * 64u) | bad, (uint32_t)stream_row(r) * row_bytes);
      };
      // The wave's scale rows come in with full-line loads and pass through its slice of xs's upper half;
      // a lane keeps the bytes of its group, four trips a dword.
      u32x4_t sl[kScalePieces];
#pragma unroll
      for (int k = 0; k < kScalePieces; ++k) {
        const int idx = k * kWave + lane, rr = idx / segs, sg = idx - rr * segs;
        const uint32_t bad = (uint32_t)!(rr < 16 * S) << 31;
        int r0 = stream_row(0);
#pragma unroll
        for (int r = 1; r < S; ++r) r0 = (rr >> 4) == r ? stream_row(r) : r0;
        sl[k] = buf16(rs, ((uint32_t)(r0 + (rr & 15)) * (uint32_t)nb + (uint32_t)sg * 16u) | bad);
      }
      ring_fence();
#pragma unroll
      for (int b = 0; b < SA; ++b) stage(b, b * kBuf);
      ring_fence();
#pragma unroll
      for (int s = 0; s < LA * TPC; ++s) issue(s, s);
      ring_fence();
      uint32_t sd[S][kTurns];
      {
        uint8_t* scr = xs + kWideBuf + wave * (kScalePieces * kWave * 16);
#pragma unroll
        for (int k = 0; k < kScalePieces; ++k) lds16_store(scr + (k * kWave + lane) * 16, sl[k]);
        ring_fence();
        __builtin_amdgcn_s_waitcnt(0xC07F);  // the wave reads back only its own slice
#pragma unroll
        for (int r = 0; r < S; ++r)
#pragma unroll
          for (int T = 0; T < kTurns; ++T)
            sd[r][T] = T < segs ? pick_lane_bytes(lds16(scr + (r * 16 + ln.c) * nb + 16 * T), sel01, kLaneByteSelC)
                                : 0u;
      }
      f32x4_t acc[S][NT];
#pragma unroll
      for (int r = 0; r < S; ++r)
#pragma unroll
        for (int t = 0; t < NT; ++t) acc[r][t] = f32x4_t{0.f, 0.f, 0.f, 0.f};
      vmcnt_wait<LA * S * TPC + (SA - 1) * NL>();  // chunk 0; the rest stays in flight
      wide_barrier();
      int here = 0, ahead = SA * kBuf;  // the buffers of chunks c and c + SA
      auto chunk = [&](int c, auto half_c) {
        constexpr int half = decltype(half_c)::value;
        // every wave has left chunk c - 1 (or its scale slice), whose buffer takes chunk c + SA
        stage(c + SA, ahead);
        ring_fence();
        const uint8_t* buf = xs + here;
#pragma unroll
        for (int s = 0; s < TPC; ++s) {
          u32x4_t* w = ring[half % LA * TPC + s];
          BlockScale fs[S];
#pragma unroll
          for (int r = 0; r < S; ++r) fs[r] = block_scale(sd[r][0] >> (8 * (half * TPC + s)));
#pragma unroll
          for (int h = 0; h < 4; ++h) {
            bf16x8_t b[S];
#pragma unroll
            for (int r = 0; r < S; ++r) b[r] = decode8(w[r][h], fs[r]);
#pragma unroll
            for (int t = 0; t < NT; ++t)
#pragma unroll
              for (int p = 0; p < NPL; ++p) {
                const bf16x8_t a = as_bf16x8(lds16(buf + ha[h] + t * 16 * kRow + s * 256 + p * 512));
#pragma unroll
                for (int r = 0; r < S; ++r) acc[r][t] = mfma16x16x32(b[r], a, acc[r][t]);
              }
            ring_fence();  // one step's decodes and LDS reads at a time: 128 VGPRs
          }
          issue(half % LA * TPC + s, (c + LA) * TPC + s);
          ring_fence();
        }
        // chunk c + 1 has landed: only the SA - 1 later chunks and the refills behind it may be out
        vmcnt_wait<S * TPC + (SA - 1) * (NL + S * TPC)>();
        wide_barrier();
        here = here == SA * kBuf ? 0 : here + kBuf;
        ahead = ahead == SA * kBuf ? 0 : ahead + kBuf;
      };
      int c = 0;  // nchunk is even
#pragma clang loop unroll(disable)
      do {
        chunk(c, std::integral_constant<int, 0>{});
        chunk(c + 1, std::integral_constant<int, 1>{});
#pragma unroll
        for (int r = 0; r < S; ++r)  // the next turn's scales (an index would put them in scratch)
#pragma unroll
          for (int T = 1; T < kTurns; ++T) sd[r][T - 1] = sd[r][T];
      } while ((c += 2) < nchunk);
      if (SA > 1) {  // the zeros past the last chunk, before the next item takes their buffers
        vmcnt_wait<0>();
        wide_barrier();
      }

      __asm__ volatile("" : "+v"(lane));
      const MoeLane out = moe_lane(lane);
#pragma unroll
      for (int t = 0; t < NT; ++t) {
        if (16 * t + out.c >= cnt) continue;
        const int64_t om = src.sorted[first + 16 * t + out.c];
        if (UP) {
          uint16_t hi[4], lo[4];
#pragma unroll
          for (int i = 0; i < 4; ++i) {
            const float gt = acc[0][t][i];
            split_bf16(gt / (1.f + __expf(-gt)) * acc[1][t][i], &hi[i], &lo[i]);
          }
          uint16_t* d = inter + om * N + tile0 * 16 + 4 * out.g;
          *reinterpret_cast<uint2*>(d) = make_uint2(hi[0] | (uint32_t)hi[1] << 16, hi[2] | (uint32_t)hi[3] << 16);
          *reinterpret_cast<uint2*>(d + inter_plane) =
              make_uint2(lo[0] | (uint32_t)lo[1] << 16, lo[2] | (uint32_t)lo[3] << 16);
        } else {
#pragma unroll
          for (int r = 0; r < S; ++r)
            *reinterpret_cast<f32x4_t*>(y + om * N + (tile0 + r) * 16 + 4 * out.g) = acc[r][t];
        }
      }
    };
    if (cnt <= 16) {
      run(std::integral_constant<int, 1>{});
    } else if (!UP || cnt <= 32) {
      run(std::integral_constant<int, 2>{});
    } else if (cnt <= 48) {
      if constexpr (UP) run(std::integral_constant<int, 3>{});
    } else {
      if constexpr (UP) run(std::integral_constant<int, 4>{});
    }
  }
}
