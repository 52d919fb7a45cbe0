// W4A16 GEMM for many token rows (prompt chunks): square register tiles, two K streams.
//
// Arithmetic, fp32 summation order (splits, even and odd streams) and results: w4a16.hpp; every
// output has the bits of the streaming kernel's (w4a16_ws.hpp).
//
// Bound: the matrix cores and what feeds them.  The streaming kernel's waves cover all of a tile's
// rows and 16 or 32 channels, so each activation fragment read from LDS feeds two MFMAs and the
// LDS reads take as long as the MFMAs; and it hands the splits of narrow layers over through
// memory (M = 1024, N = 4096: 64 MB written and read back).  Here a workgroup of 8 waves owns 128
// rows x 128 channels, waves 0-3 the even stream and 4-7 the odd one, each stream a 2 x 2 grid of
// 64 x 64 tiles: four activation fragments and four weight fragments feed 16 MFMAs.  The splits of
// K are summed one after the other by the same workgroup, in the order the streaming kernel's last
// workgroup adds them, with nothing handed over.
//
// Measured (us over distinct weights, streaming -> here): M = 1024, N = K = 4096 81 -> 48, N = 4096, K =
// 14336 178 -> 139, M = 1500, N = K = 5120 131 -> 101.  The weight loads stay in L2, where the other
// M-chunks of the channel tile find them (M = 1024, K = 14336, on one layer's weights: 142 -> 134 from
// non-temporal loads).  Unsplit layers stay with the streaming kernel, which runs them at the same rate
// (0.75 to 0.85 PFLOP/s).  Counters at M = 1024, K = 14336: the matrix cores are busy 36 % of the launch;
// a wave issues VALU work, mostly the dequantization, a quarter of its time (two waves a SIMD) and waits
// 38 % of it for an issue slot and 28 % for memory and LDS (profiles/many_row_gemms_counters.md).  Also
// tried: the next fragment dequantized between the MFMAs of this one, wave priorities by stream and
// around the MFMAs, weights two blocks ahead: no gain.
//
//  * A stream walks its 128-wide K blocks, a block a chunk: the 256 bytes of each activation row
//    land in one of the stream's two LDS slots by LDS DMA, 16-byte pieces XOR-swizzled by row;
//    packed weights and scales go to registers one block ahead.  A weight fragment is
//    dequantized by the two waves that share its channels.
//  * The activations of the next MFMA step are read while this one's MFMAs issue.  One barrier per
//    chunk, ahead of its last step: every wave has read the chunk by then and the next one has
//    landed, so the chunk after that is requested into the slot just freed.
//  * At the end of a split partner waves of the two streams exchange half of their tiles through
//    LDS, and each adds up and stores the other half.
//  * The activation DMAs are inline asm the compiler does not count; every wait on them is explicit.
#pragma once
#include "w4a16.hpp"

namespace specq {

template <int LAYOUT, bool WIDE>
__device__ __forceinline__ void w4a16_deep_entry(W4A16Params p) {
  constexpr int FM = 4, FN = 4, BM = 128, BN = 128;
  constexpr int NSC = W4Nsc<LAYOUT>::value;
  constexpr int SLOT = BM * 256;           // activation bytes of a block
  constexpr int A_L = SLOT / 4096;         // 1 KB DMAs per wave and block
  constexpr int XCH = 4 * SLOT;            // the hand-over region: half of the odd waves' tiles
  constexpr int NW = 2;                    // weight ring, in blocks
  __shared__ __attribute__((aligned(1024))) uint8_t lds[XCH + 4 * FM * FN / 2 * 1024];
  tl_mark(p.tl, p.tl_cap, 0);  // diagnostics build: workgroup start

  int mc, tile;
  deep_tile_of(deep_order((int)blockIdx.x, p.m_chunks * p.n_tiles), p.m_chunks, p.n_tiles, mc, tile);
  const int M = p.M, m0 = uniform(mc) * BM;
  if (m0 >= M) return;  // the grid may cover more rows than there are
  const int ltile = w4_select_member(p, uniform(tile));
  const int lane = lane_id(), wv = uniform(wave_id()), g = lane >> 4, r = lane & 15;
  const int h = wv >> 2, w = wv & 3, wm = w & 1, wn = w >> 1;
  const int n0 = ltile * BN + wn * FN * 16;

  // The stream's chunks: chunk q of split s is block s * bps + 2 q + h, none past the split's end.
  const int cps = (p.bps + 1) >> 1, nchunks = p.splits * cps;
  struct Cursor { int q, first; };  // chunk within the split, the split's first block
  auto next = [&](Cursor& c) __attribute__((always_inline)) {
    if (++c.q == cps) { c.q = 0; c.first += p.bps; }
  };
  auto live = [&](const Cursor& c) { return 2 * c.q + h < min(p.bps, p.nblocks - c.first); };
  auto block = [&](const Cursor& c) { return c.first + 2 * c.q + h; };

  // ---- Activation DMA i of a block: rows 4 (w A_L + i) .. + 3, lane l piece (l % 16) ^ (row % 16)
  // of the row's 256 bytes (layout 0: 128 bytes at K and 128 at K + K/2).  WIDE: a tile's rows may span
  // more than the 4 GiB of a resource, so each DMA has one of its own from its first row on and a lane's
  // 32-bit offset covers that DMA's four rows only (row strides up to 1 GiB).
  const int m_rows = min(BM, M - m0);
  const uint8_t* a0 = reinterpret_cast<const uint8_t*>(p.A + (int64_t)m0 * p.lda);
  const int64_t a_bytes = ((int64_t)(m_rows - 1) * p.lda + p.K) * 2;
  constexpr int kBlockBytes = LAYOUT == 0 ? 128 : 256;
  uint32_t a_off[A_L];
#pragma unroll
  for (int i = 0; i < A_L; ++i) {
    const int row = 4 * (w * A_L + i) + g, c = r ^ (row & 15);
    a_off[i] = (uint32_t)(WIDE ? g : row) * (uint32_t)p.lda * 2 +
               (LAYOUT == 0 ? (c < 8 ? 16 * c : p.K + 16 * (c - 8)) : 16 * c);
  }
  const uint32_t lds0 = (uint32_t)(uintptr_t)(lds_ptr_t)lds + (uint32_t)(h * 2 * SLOT + w * A_L * 1024);
  auto dma = [&](const Cursor& c, int slot) __attribute__((always_inline)) {
    const int64_t k = (int64_t)block(c) * kBlockBytes;
#pragma unroll
    for (int i = 0; i < A_L; ++i) {
      const v4i rs = WIDE ? deep_rows_rsrc<4>(a0, 4 * (w * A_L + i), live(c) ? m_rows : 0, 2 * p.lda, k, 2 * (int64_t)p.K)
                          : deep_rsrc(a0 + k, deep_extent(live(c) ? a_bytes - k : 0));
      deep_dma(rs, a_off[i], lds0 + (uint32_t)(slot * SLOT + i * 1024));
    }
  };
  const uint8_t* a_rd = lds + h * 2 * SLOT + (wm * FM * 16 + r) * 256;
  int pc[4];  // LDS position of the lane's piece of MFMA step u
#pragma unroll
  for (int u = 0; u < 4; ++u) pc[u] = 16 * ((LAYOUT == 0 ? ((u < 2 ? 0 : 8) + 2 * g + (u & 1)) : 4 * g + u) ^ r);
  auto read_a = [&](int slot, int u, v8h (&af)[FM]) __attribute__((always_inline)) {
#pragma unroll
    for (int t = 0; t < FM; ++t) af[t] = *reinterpret_cast<const v8h*>(a_rd + slot * SLOT + t * 4096 + pc[u]);
  };

  W4Weights<FN, LAYOUT, true> wt;  // read by every M-chunk
  wt.init(p, n0);
  v4i wq[NW][FN];
  uint32_t sv[NW][FN][NSC];

  v4f acc[FN][FM], tot[FN / 2][FM];
#pragma unroll
  for (int i = 0; i < FN; ++i)
#pragma unroll
    for (int j = 0; j < FM; ++j) acc[i][j] = v4f{0.f, 0.f, 0.f, 0.f};

  // Even + odd of the split just finished, set in or added to tot: each wave passes half of its
  // channel fragments to its partner in the other stream and keeps the sums of the other half (even
  // waves the lower).  acc starts again from zero.
  float* xch = reinterpret_cast<float*>(lds + XCH) + w * (FN / 2 * FM * 256) + lane * 4;
  auto combine = [&](bool first) __attribute__((always_inline)) {
    static_for<0, 2>([&](auto hc) __attribute__((always_inline)) {
      constexpr int keep = decltype(hc)::value, i0 = keep * (FN / 2);  // stream that keeps these sums
      if (h != keep) {
#pragma unroll
        for (int i = 0; i < FN / 2; ++i)
#pragma unroll
          for (int j = 0; j < FM; ++j) *reinterpret_cast<v4f*>(xch + (i * FM + j) * 256) = acc[i0 + i][j];
      }
      wg_barrier_lds();
      if (h == keep) {
#pragma unroll
        for (int i = 0; i < FN / 2; ++i)
#pragma unroll
          for (int j = 0; j < FM; ++j) {
            const v4f s = acc[i0 + i][j] + *reinterpret_cast<const v4f*>(xch + (i * FM + j) * 256);
            tot[i][j] = first ? s : tot[i][j] + s;
          }
      }
      wg_barrier_lds();
    });
#pragma unroll
    for (int i = 0; i < FN; ++i)
#pragma unroll
      for (int j = 0; j < FM; ++j) acc[i][j] = v4f{0.f, 0.f, 0.f, 0.f};
  };

  // Chunk c requests the weights of chunk c + 1 at its top and, after its barrier, the activations
  // of chunk c + 2.
  Cursor cur = {0, 0}, cw = {0, 0}, ca = {0, 0};  // chunk c, next weights, next activations
  wt.issue(block(cw), live(cw), wq[0], sv[0]);
  next(cw);
  dma(ca, 0);
  next(ca);
  dma(ca, 1);
  next(ca);
  // Block c's weights have landed.  The compiler waits here for the loads it counts, which are the
  // newest in flight, so everything older has landed too; later uses need no wait of its own, which
  // would take the activation DMAs issued since for its loads.
  auto landed = [&](v4i (&q)[FN], uint32_t (&s)[FN][NSC]) __attribute__((always_inline)) {
    wait_vmcnt<0>();
#pragma unroll
    for (int i = 0; i < FN; ++i) {
      asm volatile("" : "+v"(q[i]));
#pragma unroll
      for (int j = 0; j < NSC; ++j) asm volatile("" : "+v"(s[i][j]));
    }
  };
  v8h af[2][FM];
  landed(wq[0], sv[0]);
  wg_barrier();
  tl_mark(p.tl, p.tl_cap, 1);  // diagnostics build: first chunks landed
  read_a(0, 0, af[0]);

  for (int c0 = 0; c0 < nchunks; c0 += NW) {
    static_for<0, NW>([&](auto cc) __attribute__((always_inline)) {
      constexpr int ri = decltype(cc)::value;
      const int c = c0 + ri;
      if (c >= nchunks) return;
      wt.issue(block(cw), live(cw), wq[ri ^ 1], sv[ri ^ 1]);
      next(cw);
      __builtin_amdgcn_sched_barrier(0);
      const int b = block(cur);
      static_for<0, 4>([&](auto uc) __attribute__((always_inline)) {
        constexpr int u = decltype(uc)::value;
        if constexpr (u == 3) {
          landed(wq[ri ^ 1], sv[ri ^ 1]);  // ... and this wave's activations of chunk c + 1
          wg_barrier_lds();                // every wave's have, and every wave has read this slot
          dma(ca, ri);
          next(ca);
          read_a(ri ^ 1, 0, af[0]);
        } else {
          read_a(ri, u + 1, af[(u + 1) & 1]);
        }
        __builtin_amdgcn_sched_barrier(0);
#pragma unroll
        for (int i = 0; i < FN; ++i) {
          const v8h wf = wt.frag(b, i, u, wq[ri], sv[ri]);
#pragma unroll
          for (int j = 0; j < FM; ++j) acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x32_f16(wf, af[u & 1][j], acc[i][j], 0, 0, 0);
        }
        __builtin_amdgcn_sched_barrier(0);
      });
      if (cur.q == cps - 1) combine(cur.first == 0);
      next(cur);
    });
  }
  wait_vmcnt<0>();  // the DMAs past the end (zeros) have landed too
  tl_mark(p.tl, p.tl_cap, 2);  // diagnostics build: main loop done
#pragma unroll
  for (int i = 0; i < FN / 2; ++i)
#pragma unroll
    for (int j = 0; j < FM; ++j) {
      const int m = m0 + wm * FM * 16 + 16 * j + r, n = n0 + 16 * (h * (FN / 2) + i) + 4 * g;
      if (m < M && n < p.N) w4_store4(p, m, n, tot[i][j]);
    }
  tl_mark(p.tl, p.tl_cap, 3);          // diagnostics build: stores issued
  tl_mark_drained(p.tl, p.tl_cap, 4);  // ... and completed
}

template <int LAYOUT>
__global__ __launch_bounds__(512) void w4a16_deep_kernel(W4A16Params p) { w4a16_deep_entry<LAYOUT, false>(p); }
template <int LAYOUT>
__global__ __launch_bounds__(512) void w4a16_deep_wide_kernel(W4A16Params p) { w4a16_deep_entry<LAYOUT, true>(p); }

// Defined in the instantiation unit (`wide`: the kernel for rows that span more than 4 GiB within a tile).
const void* w4a16_deep_fn(int layout, bool wide = false);

}  // namespace specq
