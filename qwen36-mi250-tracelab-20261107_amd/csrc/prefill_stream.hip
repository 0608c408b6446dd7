// Grouped MFMA GEMM for prefill-sized batches on gfx950 with e4m3 weights streamed through
// registers (subsystems a8, a9, a6): the routed experts' launches that prefill_stream_takes.
// prefill_gemm.hip has the other ones (bf16 weights, many rows per expert, other K).
//
// Same contract as k_expert_gemm (expert_gemm.hip) and the reference's grouped kernels
// (engine/fast/moe_prefill.py:156-257): for the sorted rows of ONE expert in a tile,
//   SWIGLU: act[r, n]       = bf16(bf16(silu(bf16 g)) * bf16 u)
//   PLAIN:  out[orow(r), n] = bf16(act_or_x[r] . W[e, n])
// with e4m3 weights and per-output-row fp32 scales on the fp32 accumulator. It takes tables of
// routed experts' tiles (op[0]; a shared expert's tiles are passed over), K a multiple of 128 from
// 256 on, outputs in multiples of 16, tensors under 4 GiB.
//
// Split. A workgroup of 8 waves takes blocks of 256 weight rows and up to 160 token rows of a
// tile; a wave owns 32 rows of a block (two 16-row MFMA blocks; SWIGLU: 16 gate rows and
// the matching 16 up rows, paired in registers by the epilogue) against every token row.
// * A weight row is used by one wave only, so weights go from HBM straight into that wave's
//   registers in the MFMA A layout (lane: row l % 16, 16 bytes at 16 (l / 16); 64 contiguous
//   bytes of each of 16 rows per load), a ring of R chunks of 64 k. The launch is bound by
//   this stream and by the stores that share the memory with it; registers hold more of it in
//   flight than LDS could. (bf16 weights in this form measured slower than staged where expert
//   popularity is skewed: a block of 1111 tokens, Zipf(1.1) routing, 457 against 438 µs.)
// * Token rows are used by all waves: global -> LDS DMA (no registers on the way) in phases of
//   R chunks, two stages: the next phase is requested at the start of the current one, and one
//   barrier separates them.
// vmcnt retires in order; every phase issues the same loads, so every wait is a constant and
// waiting for a phase's token rows never drains younger weight loads.
//
// Measured (block, H = 2048, I = 512, E = 256, top-8, µs) against the kernel staged through LDS
// before it: 1111 / 2048 tokens 312 / 358 -> 289 / 320; Zipf(1.1) routing at 600 / 1111 / 2500 /
// 4096 tokens 310 / 356 / 433 / 541 -> 289 / 330 / 417 / 545. 160-row parts for every batch: 64-row
// ones gain 3 % at 1111 tokens with uniform routing and lose 13 % with Zipf.
//
// LDS layout of a chunk: row r's 128 bytes at 128 r; 16-byte unit q of row r sits at physical unit
// p(q) ^ (r & 7), p(2 kq + h) = 4 h + kq: a lane's 16 weight bytes are k = 16 kq .. + 15, fed as two
// k-steps of 8 bytes, so k-step h's lane group kq reads logical unit 2 kq + h, and its fragment
// reads (16 rows, one unit) are bank-conflict free.
//
// The body is compiled per number of 16-token blocks (NB), so that a part-filled tile loads,
// reads and multiplies only the blocks it has.
#include <stdint.h>
#include <stdlib.h>

#include <mutex>

#include "moe_common.h"
#include "expert_gemm.h"
#include "lds_dma.h"

namespace moe {

namespace {
constexpr int kPKC = 64;            // k per chunk
constexpr int kPRowBytes = kPKC * 2;             // bytes of a staged token row
constexpr int kPBlkBytes = 16 * kPRowBytes;      // a 16-token block of a stage: 2 KiB
// Cache policy of the results' stores. gate_up's go through the L2 at once (sc1): the launch
// ends with little left to write back (T = 1111: 226 -> 215 us). down's rows are completed in
// the L2 by two waves each and stay there until then (156 against 170 us at T = 4096 with sc1,
// 232 non-temporal).
template <int MODE>
constexpr int kStorePolicy = MODE == kModeSwiglu ? 16 : 0;
constexpr int kXcds = 8;            // XCDs of an MI355X (round-robin dispatch)
constexpr int kCus = 256;
constexpr int kWaves = 8;
constexpr int kMaxBlocks = 10;                   // 16-token blocks of a part of a tile
constexpr int kPartRows = 16 * kMaxBlocks;
constexpr int kRows = 32 * kWaves;               // weight rows per block
// output rows per block
template <int MODE>
constexpr int kOut = MODE == kModeSwiglu ? kRows / 2 : kRows;
}  // namespace

// The NB token fragments (16 rows each, 2 KiB apart) at LDS byte address addr, waited for.
// One asm block, so no fragment register is visible before its data has arrived.
template <int NB>
struct TokenFrags;
template <>
struct TokenFrags<4> {
  static __device__ __forceinline__ void read(uint32_t addr, u32x4v (&f)[4]) {
    asm volatile(
               "ds_read_b128 %0, %4 offset:0\n\t"
               "ds_read_b128 %1, %4 offset:2048\n\t"
               "ds_read_b128 %2, %4 offset:4096\n\t"
               "ds_read_b128 %3, %4 offset:6144\n\t"
               "s_waitcnt lgkmcnt(0)"
               : "=&v"(f[0]), "=&v"(f[1]), "=&v"(f[2]), "=&v"(f[3])
               : "v"(addr));
  }
};
template <>
struct TokenFrags<6> {
  static __device__ __forceinline__ void read(uint32_t addr, u32x4v (&f)[6]) {
    asm volatile(
               "ds_read_b128 %0, %6 offset:0\n\t"
               "ds_read_b128 %1, %6 offset:2048\n\t"
               "ds_read_b128 %2, %6 offset:4096\n\t"
               "ds_read_b128 %3, %6 offset:6144\n\t"
               "ds_read_b128 %4, %6 offset:8192\n\t"
               "ds_read_b128 %5, %6 offset:10240\n\t"
               "s_waitcnt lgkmcnt(0)"
               : "=&v"(f[0]), "=&v"(f[1]), "=&v"(f[2]), "=&v"(f[3]), "=&v"(f[4]), "=&v"(f[5])
               : "v"(addr));
  }
};
template <>
struct TokenFrags<8> {
  static __device__ __forceinline__ void read(uint32_t addr, u32x4v (&f)[8]) {
    asm volatile(
               "ds_read_b128 %0, %8 offset:0\n\t"
               "ds_read_b128 %1, %8 offset:2048\n\t"
               "ds_read_b128 %2, %8 offset:4096\n\t"
               "ds_read_b128 %3, %8 offset:6144\n\t"
               "ds_read_b128 %4, %8 offset:8192\n\t"
               "ds_read_b128 %5, %8 offset:10240\n\t"
               "ds_read_b128 %6, %8 offset:12288\n\t"
               "ds_read_b128 %7, %8 offset:14336\n\t"
               "s_waitcnt lgkmcnt(0)"
               : "=&v"(f[0]), "=&v"(f[1]), "=&v"(f[2]), "=&v"(f[3]), "=&v"(f[4]), "=&v"(f[5]), "=&v"(f[6]), "=&v"(f[7])
               : "v"(addr));
  }
};
template <>
struct TokenFrags<10> {
  static __device__ __forceinline__ void read(uint32_t addr, u32x4v (&f)[10]) {
    asm volatile(
               "ds_read_b128 %0, %10 offset:0\n\t"
               "ds_read_b128 %1, %10 offset:2048\n\t"
               "ds_read_b128 %2, %10 offset:4096\n\t"
               "ds_read_b128 %3, %10 offset:6144\n\t"
               "ds_read_b128 %4, %10 offset:8192\n\t"
               "ds_read_b128 %5, %10 offset:10240\n\t"
               "ds_read_b128 %6, %10 offset:12288\n\t"
               "ds_read_b128 %7, %10 offset:14336\n\t"
               "ds_read_b128 %8, %10 offset:16384\n\t"
               "ds_read_b128 %9, %10 offset:18432\n\t"
               "s_waitcnt lgkmcnt(0)"
               : "=&v"(f[0]), "=&v"(f[1]), "=&v"(f[2]), "=&v"(f[3]), "=&v"(f[4]), "=&v"(f[5]), "=&v"(f[6]), "=&v"(f[7]), "=&v"(f[8]), "=&v"(f[9])
               : "v"(addr));
  }
};

// Wait until at most N of this wave's loads are in flight, then the workgroup's barrier.
template <int N>
__device__ __forceinline__ void wait_barrier() {
  asm volatile("s_waitcnt vmcnt(%0)\n\ts_barrier" ::"n"(N) : "memory");
}

// Keeps the loads before it ahead of those after it: the waits count them in issue order.
__device__ __forceinline__ void issue_fence() { asm volatile("" ::: "memory"); }

__device__ __forceinline__ u32x4v ld_weight(const char* p) {
  return __builtin_nontemporal_load(reinterpret_cast<const u32x4v*>(p));
}

// Stores a block's results: lane (kq, lr) holds rows 4 kq .. + 3 of token column lr of each
// 16-token block.
// Two token blocks at a time, exchanged between lane rows so that a lane holds 8
// consecutive results of one token (16-byte stores, half as many), always all of them: those
// of rows past the tile or the weights go past the buffer's end, where they are dropped. The
// weights of the next block are in flight meanwhile, and their waits count the stores.
template <int MODE, int NB, class OutRow>
__device__ __forceinline__ void prefill_epilogue(const GemmArgs& args, int e, int r0, int r1,
                                                 int rb, int wave, int lr, int kq, OutRow out_row,
                                                 const f32x4_t (&acc)[2][NB]) {
  const GemmOperand& op = args.op[0];
  constexpr int kA = MODE == kModeSwiglu ? 1 : 2;  // 16-row groups of results
  const float* sc = op.scale ? op.scale + (long long)e * op.sstride : nullptr;
  const int nw = MODE == kModeSwiglu ? rb * (kRows / 2) + wave * 16 : rb * kRows + wave * 32;
  const int n0 = nw + 4 * kq;
  float scl[2][4] = {{1.f, 1.f, 1.f, 1.f}, {1.f, 1.f, 1.f, 1.f}};
  if (sc) {
#pragma unroll
    for (int a = 0; a < 2; ++a)
#pragma unroll
      for (int i = 0; i < 4; ++i)
        scl[a][i] = sc[MODE == kModeSwiglu ? n0 + i + (a ? (int)op.s_up_off : 0)
                                           : min(n0 + a * 16 + i, op.N - 1)];
  }
  // the lane's 4 results of group a and block b, as two pairs
  auto results = [&](int a, int b, uint32_t (&o)[2]) __attribute__((always_inline)) {
#pragma unroll
    for (int i = 0; i < 4; i += 2) {
      if (MODE == kModeSwiglu) {
        const uint32_t g = pack_bf2_rne(acc[0][b][i] * scl[0][i], acc[0][b][i + 1] * scl[0][i + 1]);
        const uint32_t u = pack_bf2_rne(acc[1][b][i] * scl[1][i], acc[1][b][i + 1] * scl[1][i + 1]);
        const uint32_t s = pack_bf2_rne(silu_fast(bf_lo(g)), silu_fast(bf_hi(g)));
        o[i / 2] = pack_bf2_rne(bf_lo(s) * bf_lo(u), bf_hi(s) * bf_hi(u));
      } else {
        o[i / 2] = pack_bf2_rne(acc[a][b][i] * scl[a][i], acc[a][b][i + 1] * scl[a][i + 1]);
      }
    }
  };
  const __amdgpu_buffer_rsrc_t obuf = __builtin_amdgcn_make_buffer_rsrc(
      op.out, 0, args.out_bytes, 0x00020000);
  const uint32_t ld = (uint32_t)(op.ld_out * 2);
#pragma unroll
  for (int b = 0; b < NB; b += 2) {
    __builtin_amdgcn_sched_barrier(0);  // one pair's results live at a time
    const int blk = b + (kq & 1);
    const int row = out_row(blk, b);
    const bool live = r0 + blk * 16 + lr < r1;
#pragma unroll
    for (int a = 0; a < kA; ++a) {
      uint32_t p[2], q[2];
      results(a, b, p);
      results(a, b + 1, q);
      u32x4v v;
#pragma unroll
      for (int i = 0; i < 2; ++i) {
        const auto x = __builtin_amdgcn_permlane16_swap(p[i], q[i], false, false);
        v[i] = x[0];
        v[i + 2] = x[1];
      }
      const int n = nw + a * 16 + (kq >> 1) * 8;
      const uint32_t off = (uint32_t)row * ld + (uint32_t)n * 2;
      __builtin_amdgcn_raw_buffer_store_b128(v, obuf, live && n < op.N ? off : 0xfffffff0u, 0,
                                             kStorePolicy<MODE>);
    }
  }
}

// One workgroup's product: weight rows of blocks rb0 .. rb0 + nblk - 1 (expert e) against sorted
// rows [r0, r1), r1 - r0 <= 16 NB. R: chunks per phase and ring depth; K / 64 is a multiple of
// R, at least 2 R. RES: K = 128 R, both phases stay in LDS for all blocks.
template <int MODE, int NB, int R, bool RES>
__device__ __forceinline__ void prefill_body(const GemmArgs& args, int e, int r0, int r1, int rb0,
                                             int nblk, char* lds) {
  constexpr int W = kWaves;
  constexpr int kLA = 2;                      // weight loads per chunk: one per row block
  constexpr int kLB = 2 * NB * R / W;         // token DMA loads of a wave per phase
  constexpr int kSub = NB * kPBlkBytes;       // a chunk of the token rows in LDS
  constexpr int kStage = R * kSub;            // a phase
  static_assert(kLB * W == 2 * NB * R && W % R == 0, "whole DMA groups per wave");
  const GemmOperand& op = args.op[0];
  const int tid = threadIdx.x;
  const int lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int lr = lane & 15;
  const int kq = lane >> 4;

  // ---- token rows of this wave's DMA loads: chunk wave % R of the phase, 8-row groups
  // wave / R + (W / R) i. The order lookups go first, the weights (which need no lookup)
  // right behind them.
  const int sub = wave % R;
  const int grow = lane >> 3;
  const int pq = (lane & 7) ^ grow;
  const int unit = 2 * (pq & 3) + (pq >> 2);
  int trow[kLB];
#pragma unroll
  for (int i = 0; i < kLB; ++i)
    trow[i] = min(r0 + (wave / R + (W / R) * i) * 8 + grow, r1 - 1);
  // gate_up rows are pairs in sorted order, whose tokens order gives; down rows are sorted rows
  if (MODE == kModeSwiglu) {
#pragma unroll
    for (int i = 0; i < kLB; ++i) trow[i] = args.order[trow[i]];
  }
  const int row_div = MODE == kModeSwiglu ? args.topk : 1;

  // The output rows. Down's pairs are looked up once: lane 16 m + l holds row l of 16-row
  // block 4 i + m.
  int orow[(NB + 3) / 4];
  if (MODE == kModePlain) {
#pragma unroll
    for (int i = 0; i < (NB + 3) / 4; ++i) orow[i] = args.order[min(r0 + i * 64 + lane, r1 - 1)];
  }
  // of row lr of block b, one of the constant group of four blocks that holds b0
  auto out_row = [&](int b, int b0) __attribute__((always_inline)) {
    if (MODE == kModeSwiglu) return r0 + b * 16 + lr;
    return __shfl(orow[b0 / 4], (b & 3) * 16 + lr);
  };

  // ---- this lane's two weight rows of a block: wave-uniform bases, 32-bit lane offsets (the
  // launcher checks that an expert's rows span less than 2 GiB)
  const char* const wbase = reinterpret_cast<const char*>(op.w) + (long long)e * op.estride;
  const char* const wbase1 = wbase + (MODE == kModeSwiglu ? op.up_off : 0);
  uint32_t woff[2];
  auto weight_rows = [&](int rb) __attribute__((always_inline)) {
#pragma unroll
    for (int a = 0; a < 2; ++a) {
      int row;
      if (MODE == kModeSwiglu)
        row = rb * (kRows / 2) + wave * 16 + lr;
      else  // the last block may be partial
        row = min(rb * kRows + wave * 32 + a * 16 + lr, op.N - 1);
      woff[a] = rb < 0 ? 0u : (uint32_t)row * (uint32_t)op.ldw + (uint32_t)(kq * 16);
    }
  };
  const int nch = op.K / kPKC;
  u32x4v ring[R][2];
  auto issue_a = [&](int slot, int c) __attribute__((always_inline)) {
#pragma unroll
    for (int a = 0; a < 2; ++a)
      ring[slot][a] = ld_weight((a ? wbase1 : wbase) + c * kPKC + woff[a]);
    issue_fence();
  };
  // The DMA is the buffer form: its counter is one the compiler can count loads in order with
  // (after a global -> LDS load it waits for every load in flight before it uses any of the
  // weight registers). 32-bit offsets: the launcher checks the input's size.
  uint32_t toff[kLB];
  auto issue_b = [&](int stage, int phase, bool any) __attribute__((always_inline)) {
    const __amdgpu_buffer_rsrc_t tbuf = __builtin_amdgcn_make_buffer_rsrc(
        const_cast<uint16_t*>(op.in), 0, any ? args.in_bytes : 0, 0x00020000);
#pragma unroll
    for (int i = 0; i < kLB; ++i)
      dma16_buffer(tbuf,
                   lds + stage * kStage + sub * kSub + (wave / R + (W / R) * i) * 1024, toff[i],
                   (phase * R + sub) * kPRowBytes);
    issue_fence();
  };

  f32x4_t acc[2][NB];
  auto clear = [&]() __attribute__((always_inline)) {
#pragma unroll
    for (int a = 0; a < 2; ++a)
#pragma unroll
      for (int b = 0; b < NB; ++b) acc[a][b] = f32x4_t{0.f, 0.f, 0.f, 0.f};
  };
  // fragment read offsets of k-steps 0 and 1: row lr of a block, physical unit 4 h + kq
  const uint32_t lbase = lds_addr(lds) + (uint32_t)(lr * kPRowBytes);
  const uint32_t roff[2] = {lbase + (uint32_t)((kq ^ (lr & 7)) * 16),
                            lbase + (uint32_t)(((4 + kq) ^ (lr & 7)) * 16)};
  auto mma = [&](int slot, uint32_t at) __attribute__((always_inline)) {
#pragma unroll
    for (int h = 0; h < 2; ++h) {
      u32x4v f[NB];
      TokenFrags<NB>::read(roff[h] + at, f);
#pragma unroll
      for (int a = 0; a < 2; ++a) {
        const u32x4v w = h ? widen8(ring[slot][a].z, ring[slot][a].w)
                           : widen8(ring[slot][a].x, ring[slot][a].y);
#pragma unroll
        for (int b = 0; b < NB; ++b) acc[a][b] = mfma_frag(w, f[b], acc[a][b]);
      }
      // the products stay ahead of the requests that refill their weight registers
      __builtin_amdgcn_sched_barrier(0);
    }
  };
  auto epilogue = [&](int rb) __attribute__((always_inline)) {
    prefill_epilogue<MODE, NB>(args, e, r0, r1, rb, wave, lr, kq, out_row, acc);
  };

  weight_rows(rb0);
  clear();
  const int nph = nch / R;
  const int rot = prefill_start_chunk(e, nch, op.ldw) / R;  // whole phases: R divides 4
  auto phase_of = [&](int p) __attribute__((always_inline)) {  // p < nph
    p += rot;
    return p >= nph ? p - nph : p;
  };
  const int ph0 = phase_of(0);
  issue_a(0, ph0 * R);
#pragma unroll
  for (int i = 0; i < kLB; ++i)
    toff[i] = (uint32_t)(trow[i] / row_div) * (uint32_t)(op.ld_in * 2) + (uint32_t)(unit * 16);
  issue_b(0, ph0, true);
#pragma unroll
  for (int c = 1; c < R; ++c) issue_a(c, ph0 * R + c);
  if constexpr (RES) {
    issue_b(1, phase_of(1), true);
    wait_barrier<(R - 1) * kLA + kLB>();
  } else {
    wait_barrier<(R - 1) * kLA>();
  }
  // A phase multiplies the R chunks at LDS offset `at` and requests the next phase's
  // operands, so that the counts are the same in every phase; the walk's last phase requests
  // nothing from the buffer and one line of the weights. At its end the next phase's token
  // rows have landed (younger: this phase's weight requests) and every wave is past this one.
  auto phase = [&](int at, int stage, int next, bool more, bool sync) __attribute__((always_inline)) {
    if constexpr (!RES) issue_b(stage, next, more);
#pragma unroll
    for (int q = 0; q < R; ++q) {
      mma(q, at + q * kSub);
      issue_a(q, next * R + q);
    }
    if (sync) wait_barrier<R * kLA>();
  };
  // Phase f of the walk: token stage f & 1 (RES: the two stages hold all of K, requested
  // once). A block's first phase follows the stores of the block before it, whose number is
  // a constant: hence the code of its own (the first block's is before the loop).
  int f = 0;
  phase(0, 1, phase_of(1), true, true);
  for (int rb = rb0;;) {
    for (int p = 1; p + 1 < nph; ++p) {
      ++f;
      phase((f & 1) * kStage, (f + 1) & 1, phase_of(p + 1), true, !RES);
    }
    const bool more = rb + 1 < rb0 + nblk;
    weight_rows(more ? rb + 1 : -1);
    ++f;
    phase((RES ? 1 : f & 1) * kStage, (f + 1) & 1, ph0, more, !RES);
    epilogue(rb);
    if (!more) break;
    ++rb;
    clear();
    ++f;
    phase((RES ? 0 : f & 1) * kStage, (f + 1) & 1, phase_of(1), true, !RES);
  }
}

template <int MODE, int R, bool RES>
__global__ __launch_bounds__(64 * kWaves)
__attribute__((amdgpu_waves_per_eu(2))) void k_prefill_stream(GemmArgs args) {
  extern __shared__ uint4 smem[];  // two phases of up to kMaxBlocks 16-token blocks

  // XCD-aware order: workgroup b runs on XCD b % 8, so the workgroups of one tile get ids 8
  // apart (same XCD, dispatched together) and share the tile's token rows in that XCD's L2
  // instead of fetching them once per XCD.
  const int ng = (args.nrb + args.nblk - 1) / args.nblk;  // workgroups per tile
  const int xcd = blockIdx.x & (kXcds - 1);
  const int j = blockIdx.x / kXcds;
  int tile = (j / ng) * kXcds + xcd;
  const int rb = (j - (j / ng) * ng) * args.nblk;
  // nsub parts of kPartRows rows per table tile, all the first parts before the second ones
  // (alternating, the parts would follow the XCDs and the rarer ones leave theirs idle)
  const int sub = tile / args.MTgrid;
  tile -= sub * args.MTgrid;
  if (sub >= args.nsub || tile >= args.table[3 * args.MT]) return;
  const int e = args.table[tile];
  if (e >= args.E) return;  // a shared expert's tile
  const int t0 = args.table[args.MT + tile];
  // the table holds the expert's end row; this tile is its next tile_rows at most
  const int t1 = min(args.table[2 * args.MT + tile], t0 + args.tile_rows);
  const int r0 = t0 + sub * kPartRows;
  const int r1 = min(t1, r0 + kPartRows);
  if (r0 >= r1) return;
  const int nblk = min(args.nblk, args.nrb - rb);
  char* lds = reinterpret_cast<char*>(smem);
  const int nb = (r1 - r0 + 15) >> 4;
#define NB_CASE(NB)                                                   \
  if (NB == kMaxBlocks || nb <= NB) {                                 \
    prefill_body<MODE, NB, R, RES>(args, e, r0, r1, rb, nblk, lds);   \
    return;                                                           \
  }
  NB_CASE(4)
  NB_CASE(6)
  NB_CASE(8)
  NB_CASE(10)
#undef NB_CASE
}

namespace {

// The kernel's dynamic LDS above the default limit, allowed once per device and kernel.
hipError_t allow_lds(const void* fn, int which, int bytes) {
  static std::mutex mu;
  static uint64_t done[5] = {};  // [kernel], bit d: device d
  int dev = 0;
  hipError_t err = hipGetDevice(&dev);
  if (err != hipSuccess) return err;
  if (dev < 0 || dev >= 64) return hipErrorInvalidDevice;
  std::lock_guard<std::mutex> lock(mu);
  if (done[which] >> dev & 1) return hipSuccess;
  err = hipFuncSetAttribute(fn, hipFuncAttributeMaxDynamicSharedMemorySize, bytes);
  if (err == hipSuccess) done[which] |= uint64_t(1) << dev;
  return err;
}

template <int MODE, int R, bool RES>
hipError_t launch_one(GemmArgs a, int tiles, int which, hipStream_t st) {
  constexpr int bytes = 2 * R * kMaxBlocks * kPBlkBytes;
  a.nrb = (a.op[0].N + kOut<MODE> - 1) / kOut<MODE>;
  // Row blocks per workgroup: down's token rows are staged once for all of them and the next
  // block's weights stream through the epilogue of one (T = 777 / 1111 / 2048 / 4096, e4m3: 75 /
  // 81 / 93 / 146 µs with 4, 77 / 82 / 96 / 132 with 2, 81 / 87 / 102 / 139 with 1). gate_up
  // gains nothing that the coarser work units do not cost (144 / 206 against 138 / 223 with 2).
  // One block per workgroup where two, at a tile per expert, would leave the last of their
  // rounds over the chip a fifth or more idle (16 experts of 2048 x 1408, 88 rows each, 45 µs with 2
  // and 26 with 1; 64 of 3072 x 1536 at 48 rows 1.10 and 1.03 of the staged kernel's time). Not so
  // with a short K where one round of two fills half the chip and more: a block's other launches use
  // the rest (2 / 1 blocks, 520 and 1000 tokens: 32 experts of 2048 x 512, top-4, 105, 121 / 115, 127 µs;
  // 16 of 4096 x 512, top-2, 153, 159 / 158, 173; 85 of 768 x 512 89, 96 / 91, 97; but 128 of 512 x 512
  // 91, 100 / 89, 96).
  const long long two = (long long)a.E * ((a.nrb + 1) / 2), one = (long long)a.E * a.nrb;
  const bool idle = 8 * ((two + kCus - 1) / kCus) > 5 * ((one + kCus - 1) / kCus);
  a.nblk = MODE == kModePlain && (!idle || (RES && two >= kCus / 2 && two <= kCus)) ? 2 : 1;
  const long long ng = (a.nrb + a.nblk - 1) / a.nblk;
  const long long grid = (long long)((tiles + kXcds - 1) / kXcds) * kXcds * ng;
  if (grid > 0x7fffffffLL) return hipErrorInvalidValue;
  const auto fn = &k_prefill_stream<MODE, R, RES>;
  const hipError_t err = allow_lds(reinterpret_cast<const void*>(fn), which, bytes);
  if (err != hipSuccess) return err;
  hipLaunchKernelGGL((k_prefill_stream<MODE, R, RES>), dim3((unsigned)grid), dim3(64 * kWaves), bytes,
                     st, a);
  return hipGetLastError();
}

long long in_bytes(const GemmArgs& a) { return (a.op[0].in_map ? a.T : a.P) * a.op[0].ld_in * 2; }
long long out_bytes(const GemmArgs& a) { return a.P * a.op[0].ld_out * 2; }

}  // namespace

// K in whole phases, at least two per block; 32-bit offsets into the tensors; and a number of rows
// per expert between the lines at which the staged kernel is the faster one.
// For other K (64, 128 and odd multiples of 64) and tensors past 4 GiB (down's from 131072 tokens
// of the model) a form of this kernel with one chunk in flight measured slower than the staged
// kernel: down at 777 tokens, K = 320 / 576, 85 / 138 against 75 / 103 µs; gate_up at 4096 tokens,
// K = 128, 45 against 42; the experts at 140000 tokens 12.8 against 9.6 ms.
bool prefill_stream_takes(int mode, const GemmArgs& a) {
  const GemmOperand& o = a.op[0];
  if (o.K % (2 * kPKC) || o.K < 4 * kPKC) return false;
  if (in_bytes(a) > 0xffffff00LL || out_bytes(a) > 0xffffff00LL ||
      (long long)o.N * o.ldw * 2 > 0x7fffffffLL)
    return false;
  const auto at_most = [](int v, int most) { return v < most ? v : most; };
  long long least;
  if (mode == kModeSwiglu)
    least = o.K & (o.K - 1) ? at_most(o.K / 32, 96) : o.N <= 512 ? 16 : at_most(o.N / 32, 24);
  else
    least = o.K <= 512 ? 0 : o.K / 32;
  return a.P >= least * a.E && a.P <= (long long)kStreamRowsPerExpert * a.E;
}

hipError_t launch_prefill_stream(int mode, const GemmArgs& a_in, int max_tiles, hipStream_t st) {
  GemmArgs a = a_in;
  a.tile_rows = prefill_tile_rows();
  a.nsub = (a.tile_rows + kPartRows - 1) / kPartRows;
  a.MTgrid = max_tiles;
  const int tiles = max_tiles * a.nsub;
  a.in_bytes = (unsigned)in_bytes(a);
  a.out_bytes = (unsigned)out_bytes(a);
  // phases of four chunks where K has whole ones, else of two; down with all of K in two phases
  // (K = 512) keeps both in LDS
  const int K = a.op[0].K;
  const bool four = K % (4 * kPKC) == 0 && K >= 8 * kPKC;
  if (mode == kModeSwiglu)
    return four ? launch_one<kModeSwiglu, 4, false>(a, tiles, 0, st)
                : launch_one<kModeSwiglu, 2, false>(a, tiles, 1, st);
  if (!four) return launch_one<kModePlain, 2, false>(a, tiles, 2, st);
  return K == 8 * kPKC ? launch_one<kModePlain, 4, true>(a, tiles, 3, st)
                       : launch_one<kModePlain, 4, false>(a, tiles, 4, st);
}

}  // namespace moe
