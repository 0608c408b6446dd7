// Arguments of the expert-grouped MFMA GEMM (expert_gemm.hip).
#pragma once
#include <hip/hip_runtime.h>
#include <stdint.h>

namespace moe {

constexpr int kModePlain = 0;   // out = bf16(acc * scale)
constexpr int kModeSwiglu = 1;  // out = bf16(bf16(silu(bf16 g)) * bf16 u), gate/up row pairs

constexpr int kRoleRouter = 0;
constexpr int kRoleGateUp = 1;
constexpr int kRoleDown = 2;

// One weight family: the routed experts (op[0]) or the virtual expert id E (op[1],
// the shared expert or the router), whose rows map 1:1 to tokens (row r -> token r - P).
struct GemmOperand {
  const void* w;        // expert 0, output row 0 (SWIGLU: gate row 0); bf16 or fp8 elements
  long long estride;    // elements between experts
  long long up_off;     // SWIGLU: elements from gate row n to up row n
  long long ldw;        // elements per weight row
  const float* scale;   // per-output-row fp32 scales (fp8) or null
  long long sstride;    // scales per expert
  long long s_up_off;   // SWIGLU: scale index of up row 0
  int K, N;             // reduction length; output rows (SWIGLU: gate rows)
  const uint16_t* in;   // B operand rows (bf16)
  long long ld_in;
  uint16_t* out;        // bf16 output rows
  long long ld_out;
  int in_map;           // routed: 1 -> B row = token of pair order[r]; 0 -> B row = r
  int out_map;          // routed: 1 -> out row = pair order[r]; 0 -> out row = r
  int fp8;              // weights are OCP e4m3fn bytes (else bf16)
};

struct GemmArgs {
  GemmOperand op[2];
  const int* table;  // tile table, or null: virtual-expert tiles over rows P .. P + T
  int MT;            // table capacity (max tiles)
  const int* order;  // sorted row -> pair
  int topk, P, E, T;
  int nrb;           // weight-row blocks per tile (set by the launcher)
  int MTgrid;        // tiles the grid covers (set by the launcher)
  int tile_rows, nsub, nblk;  // rows per table tile, parts a tile is taken in, row blocks per
                              // workgroup (set by the streaming kernel's launcher)
  unsigned in_bytes, out_bytes;  // of op[0]'s input and output (set by the same)
  int shared_first;  // the table's last shared_first tiles run first (set by the launcher)
};

// Launches k_expert_gemm over max_tiles tiles of at most bm (16, 32, 64 or 128) sorted rows.
// Both operands of one launch must have the same weight type.
// hipErrorInvalidValue: no kernel configuration fits the operands' shapes.
// Whether a launch may mix fp8 routed tiles with bf16 shared-expert tiles (MOE_MIXED=0: no;
// then the caller splits them into two launches).
bool mixed_enabled();
hipError_t launch_expert_gemm(int mode, int role, int bm, const GemmArgs& a, int max_tiles,
                              hipStream_t st);

// Where the prefill kernels (bf16: gate_up's; e4m3: both projections') start their walk over the
// nch = K / 64 chunks of expert e's weight rows of row_bytes (it wraps around). Workgroups run nearly
// in step, and the rows of the model lie 4 KiB apart: all reading the same columns at once keeps
// few memory channels busy. Start by expert / one start for all, a block's µs: bf16, K = 2048 at 64 /
// 128 experts and 700 tokens 144 / 225 against 158 / 246, K = 4096 252 / 398 against 277 / 433; e4m3,
// K = 4096 206 / 308 against 219 / 336. Shorter rows gain nothing (bf16 K = 1536 182 / 182, e4m3
// K = 2048 286 / 286) or lose, since the experts then read a token's columns at different times (bf16
// K = 1024 at 64 / 256 experts 101 / 219 against 98 / 209). The start is the expert's own and, for one
// weight type, the same in every kernel that runs the projection above 512 tokens, so that a row's result
// does not depend on its batch there; whole groups of four chunks, the streaming kernel's phases.
__host__ __device__ inline bool prefill_starts_by_expert(int nch, long long row_bytes) {
  return row_bytes >= 4096 && nch % 4 == 0;
}
__host__ __device__ inline int prefill_start_chunk(int e, int nch, long long row_bytes) {
  return prefill_starts_by_expert(nch, row_bytes) ? e % (nch / 4) * 4 : 0;
}

// Prefill batches. launch_prefill_gemm (prefill_gemm.hip) takes tables of prefill_tile_rows()
// sorted rows per tile and passes on to prefill_stream.hip the e4m3 launches that one takes.
int prefill_tile_rows();
bool prefill_fits(int mode, const GemmOperand& op);
hipError_t launch_prefill_gemm(int mode, const GemmArgs& a, int max_tiles, hipStream_t st);
// A routed e4m3 launch (op[0], a table, prefill_fits operands): whether it takes the streaming
// kernel, and that kernel's launch. The streaming kernel reads a row block's weights once per
// 160 rows of an expert, the one staged through LDS once per 256: the line is the average number
// of rows per expert from which many experts need a second pass. A block (H = 2048, I = 512,
// E = 256, top-8) of 3072 / 3584 / 4096 / 4608 / 5120 tokens, streaming against staged, µs: uniform
// routing 369 / 397 / 440 / 498 / 591 against 403 / 435 / 464 / 491 / 519; Zipf(1.1) routing
// 462 / 489 / 547 / 600 / 631 against 467 / 488 / 518 / 563 / 591.
// With few rows per expert the staged kernel is the faster one again, except for down with K up to 512.
// The line is 16 to 24 rows (N / 32) for gate_up where K is a power of two, else K / 32 (at most 96), and
// K / 32 for down:
// streaming / staged, µs, uniform routing, 256 experts at 8 / 16 / 24 / 32 / 48 rows each. gate_up of hidden x
// intermediate 2048 x 512 133 / 134 / 135 / 135 / 138 against 121 / 127 / 137 / 140 / 154, 4096 x 1024 452 / 456 /
// 457 / 462 / 475 against 403 / 424 / 448 / 467 / 506, 3072 x 512 191 / 193 / 196 / 198 / 203 against 172 / 177 / 183 /
// 187 / 206 (64 / 100 rows 212 / 239 against 217 / 259); down of 2048 x 512 76 / 82 / 87 / 89 / 89 against 88 / 91 /
// 99 / 104 / 120, 2048 x 1024 139 / 140 / 145 / 148 / 146 against 136 / 142 / 152 / 160 / 171, 4096 x 1024 282 / 303 /
// 311 / 317 / 323 against 257 / 270 / 290 / 307 / 334, 2048 x 1536 200 / 208 / 203 / 222 / 227 against 184 / 191 / 201 /
// 211 / 226. Over 1359 shapes and batches (hidden 256 to 7168, intermediate 256 to 2048, 16 to 512 experts, 8 to
// 100 rows) the projections so chosen take 0.957 and 0.906 of the staged kernel's time. (16, not 20: at 18 and 20
// rows a block of the model takes 271 / 272 against 272 / 276 beside its other launches, with Zipf(1.1)
// routing 289 / 291 against 291 / 298.)
constexpr int kStreamRowsPerExpert = 128;
bool prefill_stream_takes(int mode, const GemmArgs& a);
hipError_t launch_prefill_stream(int mode, const GemmArgs& a, int max_tiles, hipStream_t st);

}  // namespace moe
