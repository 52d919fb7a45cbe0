// W8A8 / W4A8 GEMM for many token rows (prompt chunks): both operands staged in LDS, square
// register tiles.
//
// Same arithmetic as w8a8_ws.hpp: INT8 x INT8 products summed exactly in INT32 (any order gives
// the same bits), then (acc * sa[m]) * sw[n] in fp32 and one RNE cast to fp16.
//
// Bound: the matrix cores.  Past a few hundred rows the weight-streaming schedule
// (w8a8_ws.hpp: 304 rows x 128 channels, each wave 304 x 32) reads 19 activation fragments from
// LDS for 38 MFMAs, so its LDS reads alone take as long as its MFMAs.  Here the 4 waves of a
// workgroup form a 2 x 2 grid of (16 FM) x (16 FN) tiles: at FM = FN = 8 a wave reads 16
// fragments for 64 MFMAs, every byte of both operands crosses L2 -> CU once per 256 x 256 tile,
// and 256 accumulator registers leave room for two sets of operands.
//
// Measured (us over distinct weights and, in brackets, on one; streaming -> here; INT8 weights unless
// said): M = 2048, N = 28672, K = 4096 334 -> 222 (332 -> 210, 2.3 POPS), N = 4096, K = 14336 137 -> 108 (137 ->
// 102); M = 1024, N = K = 4096 30.6 -> 24.3 (32.6 -> 24.0); INT4 weights, M = 1024, N = 27648, K = 5120 195 -> 135
// (195 -> 124).  Counters at M = 2048: the matrix cores are busy 46 to 50 % of the launch, a wave waits 41 %
// of its time for an issue slot and 17 % for memory, LDS and barriers, and the clock is 1.9 GHz under
// this load (profiles/many_row_gemms_counters.md).  Also tried: 64-byte K steps in a ring twice as
// deep (218 -> 264 and slower at every large tile), splits of K over workgroups for few tiles (slower
// than the streaming kernel at M <= 517), 256 x 128 tiles (slower than 128 x 256).
//
//  * K is walked in chunks of 128 bytes (two MFMA K steps) on a ring of NSL LDS slots, filled by
//    LDS DMA (buffer_load ... lds).  Activation rows land as 128 bytes with their 16-byte pieces
//    XOR-swizzled (piece c of row m in position c ^ (m / 2 % 8)), so 16 consecutive rows read
//    at one K offset touch every LDS bank once.  The packed weight fragments are copied as
//    they are: MFMA operand order, one contiguous 1 KB (INT4: 512 B) per fragment.
//  * Operands of the next K step are read from LDS while the MFMAs of this one issue.  One
//    barrier per chunk, in its middle: the wave has read the chunk's second step by then and
//    the next chunk has landed, so the chunk NSL ahead is requested into the slot just freed.
//  * Nothing is masked in the loop: rows past M and fragments past N feed only outputs that are
//    never stored, K past the end meets the zero padding of the packed weight, and what lies
//    past either buffer's end is an out-of-range buffer read (zero).
//  * The DMAs are inline asm the compiler does not count; every wait on them is explicit.
//  * 256 x 256 tiles fill whole rounds of CUs; a last round of at most half the CUs runs each of
//    its tiles as two 128 x 256 halves (M = 2048, N = 28672: 246 -> 218 us).  Fewer tiles than
//    that run at 64 or 128 rows x 128 channels, up to three workgroups per CU (kDeep*).
//  * Workgroup b runs on XCD b mod 8: each XCD takes a contiguous run of tiles, M-chunks
//    fastest in blocks of 8, so the workgroups running together on it share weights and
//    activations in its L2.
#pragma once
#include "w8a8.hpp"

namespace specq {

template <int FM, int FN, int NSL, int WL>
struct W8A8DeepCfg {
  static constexpr int BM = 32 * FM, BN = 32 * FN;
  static constexpr int KC = 128;
  static constexpr int FB = W8A8WFragBytes<WL>::value;   // bytes of a weight fragment
  static constexpr int ASLOT = BM * KC;                  // activation bytes of a chunk
  static constexpr int WSLOT = 2 * (BN / 16) * FB;       // weight bytes of a chunk
  static constexpr int SLOT = ASLOT + WSLOT;             // LDS ring slot: activations, then weights
  static constexpr int EPI = 4 * (16 * FM) * (16 * FN) * 2;  // the waves' fp16 tiles
  static constexpr int LDS = NSL * SLOT > EPI ? NSL * SLOT : EPI;
  static constexpr int A_L = ASLOT / 4096, W_L = WSLOT / 4096;  // 1 KB DMAs per wave and chunk
  static constexpr int PER = A_L + W_L;
  static_assert(NSL >= 2 && LDS <= 160 * 1024 && (NSL - 1) * PER <= 63, "tile");
};

// One 32 FM x 32 FN tile: rows m0.., channel tile `tile` (launch-wide) of BN channels.  WIDE: a tile's
// rows may span more than the 4 GiB of a resource, so each activation DMA has one of its own from its
// first row on and a lane's 32-bit offset covers that DMA's eight rows only (row strides up to 512 MiB).
// The scalar arithmetic of that between the MFMAs costs 5 % (MLP block of M = 2048, hidden 4096, 14336
// channels: 366 -> 383 us) and a branch in one kernel its registers, so it is a kernel of its own.
template <int FM, int FN, int NSL, int WL, bool WIDE>
__device__ __forceinline__ void w8a8_deep_body(W8A8Params p, uint8_t* lds, int m0, int tile) {
  using C = W8A8DeepCfg<FM, FN, NSL, WL>;
  constexpr int BM = C::BM, BN = C::BN, FB = C::FB;
  const int M = p.M;
  const int ltile = w8a8_select_member(p, tile);
  const int lane = lane_id(), w = uniform(wave_id()), g = lane >> 4, r = lane & 15;
  const int wm = w & 1, wn = w >> 1;
  const int nbase = ltile * BN;

  // ---- DMA addresses.  Activation DMA i of wave w covers rows 8 (w A_L + i) .. + 7 of the tile; weight
  // DMA f covers 1 KB of the chunk's fragments, step-major.  Wave w issues A_L and W_L of them.
  const int m_rows = min(BM, M - m0);
  const int8_t* a0 = p.A + (int64_t)m0 * p.lda;
  const int64_t a_bytes = (int64_t)(m_rows - 1) * p.lda + p.K;
  const int ntiles = (p.N + 15) / 16, ksteps = (p.K + 63) / 64;
  const int64_t step_bytes = (int64_t)ntiles * FB;
  const int8_t* w0 = p.W + (int64_t)(nbase / 16) * FB;
  const int64_t w_bytes = ksteps * step_bytes - (int64_t)(nbase / 16) * FB;
  uint32_t a_off[C::A_L], w_off[C::W_L];
#pragma unroll
  for (int i = 0; i < C::A_L; ++i) {
    const int row = 8 * (w * C::A_L + i) + (lane >> 3);
    a_off[i] = (uint32_t)(WIDE ? lane >> 3 : row) * (uint32_t)p.lda + 16 * ((lane & 7) ^ ((row >> 1) & 7));
  }
#pragma unroll
  for (int i = 0; i < C::W_L; ++i) {
    const int byte = (w * C::W_L + i) * 1024;                 // within the chunk's fragments
    constexpr int SB = (BN / 16) * FB;                        // bytes of one K step of them
    w_off[i] = (uint32_t)((byte / SB) * (int)step_bytes + byte % SB + 16 * lane);
  }
  const uint32_t lds0 = (uint32_t)(uintptr_t)(lds_ptr_t)lds;
  auto dma_a = [&](int c, int slot, int i) __attribute__((always_inline)) {
    const int64_t k = (int64_t)c * C::KC;
    const v4i rs = WIDE ? deep_rows_rsrc<8>(a0, 8 * (w * C::A_L + i), m_rows, p.lda, k, p.K)
                        : deep_rsrc(a0 + k, deep_extent(a_bytes - k));
    deep_dma(rs, a_off[i], lds0 + (uint32_t)(slot * C::SLOT + (w * C::A_L + i) * 1024));
  };
  auto dma_w = [&](int c, int slot, int i) __attribute__((always_inline)) {
    const int64_t o = 2 * step_bytes * c;
    deep_dma(deep_rsrc(w0 + o, deep_extent(w_bytes - o)), w_off[i],
             lds0 + (uint32_t)(slot * C::SLOT + C::ASLOT + (w * C::W_L + i) * 1024));
  };

  v4i acc[FN][FM];
#pragma unroll
  for (int t = 0; t < FN; ++t)
#pragma unroll
    for (int u = 0; u < FM; ++u) acc[t][u] = v4i{0, 0, 0, 0};

  // ---- Operand reads: activation fragment u and weight fragment t of step s of a slot.
  const uint8_t* a_rd[2];
#pragma unroll
  for (int s = 0; s < 2; ++s)
    a_rd[s] = lds + (wm * FM * 16 + r) * C::KC + 16 * ((4 * s + g) ^ (r >> 1));
  const uint8_t* w_rd = lds + C::ASLOT + wn * FN * FB + lane * (FB / 64);
  using WFrag = W8A8WFrag<WL>;
  auto read_a = [&](int slot, int s, int u) __attribute__((always_inline)) {
    return *reinterpret_cast<const v4i*>(a_rd[s] + slot * C::SLOT + u * 16 * C::KC);
  };
  auto read_w = [&](int slot, int s, int t) __attribute__((always_inline)) {
    return *reinterpret_cast<const WFrag*>(w_rd + slot * C::SLOT + (s * (BN / 16) + t) * FB);
  };

  const int nchunks = (ksteps + 1) / 2;
  static_for<0, NSL>([&](auto cc) __attribute__((always_inline)) {
    constexpr int c = decltype(cc)::value;
#pragma unroll
    for (int i = 0; i < C::A_L; ++i) dma_a(c, c, i);
#pragma unroll
    for (int i = 0; i < C::W_L; ++i) dma_w(c, c, i);
  });
  v4i a0f[FM], a1f[FM];
  WFrag w0f[FN], w1f[FN];
  wait_vmcnt<(NSL - 1) * C::PER>();  // chunk 0 has landed
  wg_barrier();
  tl_mark(p.tl, p.tl_cap, 1);  // diagnostics build: first chunk landed
#pragma unroll
  for (int u = 0; u < FM; ++u) a0f[u] = read_a(0, 0, u);
#pragma unroll
  for (int t = 0; t < FN; ++t) w0f[t] = read_w(0, 0, t);

  // Chunk c, in slot c mod NSL.  Group t of a K step: a share of the next step's operand reads
  // (and, in the second step, of the DMAs of chunk c + NSL), then the FM MFMAs of weight
  // fragment t.
  int slot = 0;
  for (int c = 0; c < nchunks; ++c) {
    const int next = slot + 1 == NSL ? 0 : slot + 1;
    static_for<0, FN>([&](auto tc) __attribute__((always_inline)) {
      constexpr int t = decltype(tc)::value;
      w1f[t] = read_w(slot, 1, t);
      static_for<t * FM / FN, (t + 1) * FM / FN>([&](auto uc) __attribute__((always_inline)) {
        a1f[decltype(uc)::value] = read_a(slot, 1, decltype(uc)::value);
      });
      __builtin_amdgcn_sched_barrier(0);
      const v4i wf = w8a8_wop(w0f[t]);
#pragma unroll
      for (int u = 0; u < FM; ++u) acc[t][u] = __builtin_amdgcn_mfma_i32_16x16x64_i8(wf, a0f[u], acc[t][u], 0, 0, 0);
      __builtin_amdgcn_sched_barrier(0);
    });
    wait_vmcnt<(NSL - 2) * C::PER>();  // this wave's DMAs of chunk c + 1 have landed
    wg_barrier_lds();                  // ... every wave's have, and every wave has read this slot
    static_for<0, FN>([&](auto tc) __attribute__((always_inline)) {
      constexpr int t = decltype(tc)::value;
      static_for<t * C::A_L / FN, (t + 1) * C::A_L / FN>([&](auto ic) __attribute__((always_inline)) {
        dma_a(c + NSL, slot, decltype(ic)::value);
      });
      static_for<t * C::W_L / FN, (t + 1) * C::W_L / FN>([&](auto ic) __attribute__((always_inline)) {
        dma_w(c + NSL, slot, decltype(ic)::value);
      });
      w0f[t] = read_w(next, 0, t);
      static_for<t * FM / FN, (t + 1) * FM / FN>([&](auto uc) __attribute__((always_inline)) {
        a0f[decltype(uc)::value] = read_a(next, 0, decltype(uc)::value);
      });
      __builtin_amdgcn_sched_barrier(0);
      const v4i wf = w8a8_wop(w1f[t]);
#pragma unroll
      for (int u = 0; u < FM; ++u) acc[t][u] = __builtin_amdgcn_mfma_i32_16x16x64_i8(wf, a1f[u], acc[t][u], 0, 0, 0);
      __builtin_amdgcn_sched_barrier(0);
    });
    slot = next;
  }
  W8A8EpiScales<FM, FN> es;
  es.load(p, M, m0 + wm * FM * 16, nbase + wn * FN * 16, true);
  wait_vmcnt<0>();   // the DMAs past the end (zeros) have landed too
  wg_barrier_lds();  // every wave is done with the slots
  tl_mark(p.tl, p.tl_cap, 2);  // diagnostics build: main loop done
  if constexpr (WL == 2) w8a8_unscale16(acc);

  // Each wave's fp16 tile goes through its own part of LDS (row-major, 16-byte pieces
  // XOR-swizzled by row), so that a lane stores 16 contiguous bytes of an output row.
  constexpr int PIECES = FN * 2, ROWB = PIECES * 16;  // pieces and bytes per tile row
  uint8_t* ct = lds + w * (FM * 16 * ROWB);
#pragma unroll
  for (int t = 0; t < FN; ++t)
#pragma unroll
    for (int u = 0; u < FM; ++u) {
      const int row = u * 16 + r, pc = (2 * t + (g >> 1)) ^ (row & (PIECES - 1));
      *reinterpret_cast<v4h*>(ct + row * ROWB + pc * 16 + (g & 1) * 8) = w8a8_cvt4(acc[t][u], es.a[u], es.w[t]);
    }
  wait_lgkm0();  // only this wave reads its tile
  const bool v16 = ((uintptr_t)p.C % 16 == 0) & (p.ldc % 8 == 0);
#pragma unroll
  for (int i = 0; i < FM * 16 * PIECES / 64; ++i) {
    const int q = i * 64 + lane, row = q / PIECES, pc = q % PIECES;
    const int m = m0 + wm * FM * 16 + row, n = nbase + wn * FN * 16 + pc * 8;
    if (m < M && n < p.N) {
      const v8h v = *reinterpret_cast<const v8h*>(ct + row * ROWB + ((pc ^ (row & (PIECES - 1))) * 16));
      _Float16* dst = reinterpret_cast<_Float16*>(p.C + (int64_t)m * p.ldc + n);
      if (v16 && n + 7 < p.N) {
        *reinterpret_cast<v8h*>(dst) = v;
      } else {
#pragma unroll
        for (int e = 0; e < 8; ++e)
          if (n + e < p.N) dst[e] = v[e];
      }
    }
  }
  tl_mark(p.tl, p.tl_cap, 3);          // diagnostics build: stores issued
  tl_mark_drained(p.tl, p.tl_cap, 4);  // ... and completed
}

template <int FM, int FN, int NSL, int WL, bool WIDE>
__device__ __forceinline__ void w8a8_deep_entry(const W8A8Params& p) {
  __shared__ __attribute__((aligned(1024))) uint8_t lds[W8A8DeepCfg<FM, FN, NSL, WL>::LDS];
  tl_mark(p.tl, p.tl_cap, 0);  // diagnostics build: workgroup start
  int mc, tile;
  deep_tile_of(deep_order((int)blockIdx.x, p.m_chunks * p.n_tiles), p.m_chunks, p.n_tiles, mc, tile);
  const int m0 = uniform(mc) * (32 * FM);
  if (m0 < p.M) w8a8_deep_body<FM, FN, NSL, WL, WIDE>(p, lds, m0, uniform(tile));  // the grid may cover more rows
}

// 256 x 256 tiles, those from p.whole on as two 128 x 256 halves each.
template <int WL, bool WIDE>
__device__ __forceinline__ void w8a8_deep_mix_entry(const W8A8Params& p) {
  constexpr int L0 = W8A8DeepCfg<8, 8, 2, WL>::LDS, L1 = W8A8DeepCfg<4, 8, 3, WL>::LDS;
  __shared__ __attribute__((aligned(1024))) uint8_t lds[L0 > L1 ? L0 : L1];
  tl_mark(p.tl, p.tl_cap, 0);  // diagnostics build: workgroup start
  const int id = (int)blockIdx.x;
  int mc, tile;
  if (id < p.whole) {
    deep_tile_of(deep_order(id, p.whole), p.m_chunks, p.n_tiles, mc, tile);
    const int m0 = uniform(mc) * 256;
    if (m0 < p.M) w8a8_deep_body<8, 8, 2, WL, WIDE>(p, lds, m0, uniform(tile));
  } else {
    const int idx = deep_order(id - p.whole, 2 * (p.m_chunks * p.n_tiles - p.whole));
    deep_tile_of(p.whole + idx / 2, p.m_chunks, p.n_tiles, mc, tile);
    const int m0 = uniform(mc) * 256 + (idx & 1) * 128;
    if (m0 < p.M) w8a8_deep_body<4, 8, 3, WL, WIDE>(p, lds, m0, uniform(tile));
  }
}

template <int FM, int FN, int NSL, int WL>
__global__ __launch_bounds__(256) void w8a8_deep_kernel(W8A8Params p) { w8a8_deep_entry<FM, FN, NSL, WL, false>(p); }
template <int WL>
__global__ __launch_bounds__(256) void w8a8_deep_mix_kernel(W8A8Params p) { w8a8_deep_mix_entry<WL, false>(p); }
template <int FM, int FN, int NSL, int WL>
__global__ __launch_bounds__(256) void w8a8_deep_wide_kernel(W8A8Params p) { w8a8_deep_entry<FM, FN, NSL, WL, true>(p); }
template <int WL>
__global__ __launch_bounds__(256) void w8a8_deep_mix_wide_kernel(W8A8Params p) { w8a8_deep_mix_entry<WL, true>(p); }

// Tiles of the dispatch (api_w8a8.hip prices them), in order of the rows they are for.
enum DeepTile { kDeep64, kDeep128, kDeep128Pair, kDeepMix, kDeepTiles };
constexpr int kDeepRows[kDeepTiles] = {64, 128, 128, 256};       // token rows
constexpr int kDeepChannels[kDeepTiles] = {128, 128, 128, 256};  // channels

// Defined in the instantiation unit: the kernel of a tile for a weight layout (`wide`: the one for rows
// that span more than 4 GiB within a tile), or null.
const void* w8a8_deep_fn(int tile, int layout, bool wide = false);

}  // namespace specq
