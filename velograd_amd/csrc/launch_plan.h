// Launch plans of the fused RMSNorm + residual kernels (host-only C++, no HIP dependency), so
// the planner can be compiled and checked on a CPU (tests/plan_check.cpp, under ASan/UBSan).
//
// A row of `dim` elements is cut into 16-byte chunks (8 bf16/fp16 or 4 fp32 elements).  The
// register-resident kernels give each row `tpr` threads (whole wave64s) and each thread NV
// chunks, c = lane + k * tpr for k < NV, so that consecutive lanes touch consecutive 16-byte
// chunks (coalesced 1 KiB per wave instruction).  Rows whose length is not a multiple of the
// chunk and misaligned rows go in chunks from any element (plan_any_rows, plan_bwd_ring_any,
// plan_bwd_rope_ring_any, plan_rope_tiles) or, short ones, element by element; rows too long for
// registers, and the few that these rules leave, use the generic looping kernels.
#ifndef VELOGRAD_LAUNCH_PLAN_H
#define VELOGRAD_LAUNCH_PLAN_H

#include <stddef.h>
#include <stdint.h>

#ifndef VG_HOST_DEVICE
#define VG_HOST_DEVICE
#endif

namespace vg_plan {

constexpr int kWave = 64;
constexpr int kMaxWavesPerRow = 16;  // 1024 threads per row at most
// 16-byte chunks per thread in the register-resident path.  Capped at 4: the one-wave-per-row
// forward with 8 chunks per thread (191 VGPRs) made an illegal memory access on MI355X although
// its launch plan was correct (checked on the CPU by intercepting the launch); until that is
// understood, NV 5..8 are neither planned nor compiled.
constexpr int kMaxNV = 4;
constexpr int kGenericBlock = 256;
// The generic backward sums a slot's dweight columns in dynamic LDS (dim floats) for rows of up
// to kGenericLdsCols elements (64 KiB of LDS a workgroup, less its static row-sum buffers), else
// in its partial row in global memory.  Returns the launch's dynamic LDS bytes.
constexpr int kGenericLdsCols = 16000;
VG_HOST_DEVICE constexpr size_t generic_bwd_lds_bytes(int64_t dim, bool dweight) {
  return dweight && dim > 0 && dim <= kGenericLdsCols ? (size_t)dim * sizeof(float) : 0;
}

// Workgroup size bound of the register-resident kernels, so that a thread's packed chunks fit
// its VGPR budget (512 VGPRs per SIMD lane shared by the block's waves on that SIMD):
// NV <= 2 -> 1024 threads (128 VGPRs), NV 3..4 -> 512 (256).
VG_HOST_DEVICE constexpr int max_block_for_nv(int nv) { return nv <= 2 ? 1024 : 512; }

// The same bound for the backward with the fused inverse RoPE of grad_y: its rotation state
// (cos and sin per pair) takes more VGPRs, so NV 1 -> 1024 threads (95 VGPRs used),
// NV 2 and 3 -> 512 (256); with NV 4 the kernel would spill, so those rows take the generic
// kernel.
VG_HOST_DEVICE constexpr int max_block_for_nv_rope(int nv) {
  return nv <= 1 ? 1024 : (nv <= 3 ? 512 : 0);
}

struct RowPlan {
  bool vec;    // register-resident path
  int nv;      // 16-byte chunks per thread
  int tpr;     // threads per row
  int groups;  // rows per workgroup
  int block;   // threads per workgroup = tpr * groups
};

// Automatic orders in which chunks-per-thread values are tried (measured on MI355X, bf16 rows of
// 4096 and 8192): the forward with a residual (two streams read, two written) is fastest with
// one chunk per thread (more waves per row, all of a row's loads in one instruction per lane);
// without one (x read, y written) with two, since one 16-byte load per lane leaves too few
// bytes in flight (16384 x 4096: 44.5 us against 51.0 us, the plain copy's speed); the
// persistent backward with two (it keeps the next row's chunks in flight too, so it trades
// waves for bytes per lane).
constexpr int kFwdOrder[kMaxNV] = {1, 2, 3, 4};
constexpr int kFwdOrderOneStream[kMaxNV] = {2, 4, 3, 1};
// The quantised epilogues (fp8 per row, MXFP8, MXFP4) reduce each row twice (sum of squares,
// then amax), so fewer waves per row pay off there: two chunks per thread against one ran
// 76.9 / 301.5 / 39.9 us against 79.6 / 335.0 / 42.5 us for the per-row fp8 forward at configs
// C / D / B (and MXFP4 at D 280 against 314); four chunks were within 1% at C and D and 2-3%
// slower at B.
constexpr int kFwdOrderEpilogue[kMaxNV] = {2, 4, 3, 1};
constexpr int kBwdOrder[kMaxNV] = {2, 3, 4, 1};
// The backward with the fused RoPE gradient prefers one chunk per thread: its rotation state
// then fits 1024-thread workgroups (16384 x 4096 bf16: 84.0 us against 89.7 us at two chunks
// in 768-thread workgroups).
constexpr int kBwdOrderRope[kMaxNV] = {1, 2, 3, 4};

// Register-resident layout for rows of `dim` elements of `elem_bytes` bytes, or the generic
// plan when the row does not split into 16-byte chunks or does not fit in registers.
// `prefer_nv` (1..kMaxNV, 0 = automatic) is tried first, then `auto_order`; the first choice
// whose idle lanes stay under 1/8 wins, else the least idle one.
inline RowPlan plan_rows(int64_t dim, int elem_bytes, bool aligned, int prefer_nv,
                         const int (&auto_order)[kMaxNV]) {
  RowPlan p{false, 0, kGenericBlock, 1, kGenericBlock};
  if (elem_bytes != 2 && elem_bytes != 4) return p;
  const int V = 16 / elem_bytes;
  if (!aligned || dim <= 0 || dim % V != 0) return p;
  const int64_t chunks = dim / V;
  int order[1 + kMaxNV];
  int n = 0;
  if (prefer_nv >= 1 && prefer_nv <= kMaxNV) order[n++] = prefer_nv;
  for (int i = 0; i < kMaxNV; ++i)
    if (auto_order[i] != prefer_nv) order[n++] = auto_order[i];
  int best_nv = 0, best_wpr = 0;
  int64_t best_waste = -1;
  for (int i = 0; i < n; ++i) {
    const int nv = order[i];
    const int64_t wpr = (chunks + (int64_t)kWave * nv - 1) / ((int64_t)kWave * nv);
    if (wpr * kWave > max_block_for_nv(nv)) continue;
    const int64_t slots = wpr * kWave * nv;
    const int64_t waste = slots - chunks;
    if (waste * 8 <= slots) {
      best_nv = nv;
      best_wpr = (int)wpr;
      break;
    }
    if (best_waste < 0 || waste < best_waste) {
      best_waste = waste;
      best_nv = nv;
      best_wpr = (int)wpr;
    }
  }
  if (best_nv == 0) return p;
  p.vec = true;
  p.nv = best_nv;
  p.tpr = best_wpr * kWave;
  p.groups = p.tpr >= 256 ? 1 : 256 / p.tpr;
  p.block = p.tpr * p.groups;
  return p;
}

// Rows that the chunked layout does not fit (lengths that are no whole number of 16-byte chunks,
// streams that start anywhere): fwd_vec_kernel's any-alignment form takes them from one chunk up,
// laid out over the dim / V whole chunks a row can hold.  Two chunks a thread where a row has
// enough for that without a residual or with a quantised output (the orders above), else up to
// kAnyTwoChunks chunks (two waves); longer rows one chunk a thread up to the workgroup bound.
// Measured with a residual (bf16, 16384 rows; one chunk and h stored early / two chunks and h stored
// late, us): 1001 26.8 / 25.3, 1535 40.0 / 38.7, 2047 51.6 / 50.0, but in three waves, alone in their
// workgroup, 2201 51.1 / 54.5, 2562 58.6 / 62.7, 3002 66.3 / 70.6, 3076 69.7 / 74.7 (rows of
// 8n + 4 elements in 8-byte halves 72.0), 4095 95.6 / 98.4, fp32 1281 58.6 / 62.1, 1537 72.6 / 76.8,
// 8192 x 4099 90.0 / 93.2.
constexpr int kAnyTwoChunks = 256;
// Without a residual and with y in the activation dtype, rows of more chunks than this keep the
// generic kernel, whose 256-thread workgroups leave a CU more rows to overlap than one row group of
// eight to sixteen waves.  Measured (8192 rows; generic kernel / any-row form, us): bf16 4099 32.0 /
// 27.3, 6149 41.9 / 39.9, 7001 46.0 / 45.8, 7503 48.3 / 50.4, 8191 50.2 / 53.0, 10003 63.3 / 70.5,
// 14001 89.1 / 100.7; fp32 3501 41.0 / 41.1, 4095 47.5 / 48.3, 5001 57.7 / 61.5, 8191 95.1 / 98.2.  A
// few rows, which leave CUs idle either way, wait for one pass instead of two: 256 rows bf16 8191 5.5
// / 4.7, 14001 8.5 / 6.1; 512 rows 6.5 / 6.0, 9.6 / 9.4; 768 rows 7.6 / 7.9, 11.5 / 13.5; fp32 8191 at
// 512 rows 9.4 / 8.5, 768 11.7 / 13.0.
constexpr int kAnyOneStreamChunks = 896;
constexpr int64_t kAnyOneStreamRows = 512;
// `residual`: the forward adds one; `quantised`: y is stored as fp8 or MX codes.
inline RowPlan plan_any_rows(int64_t rows, int64_t dim, int elem_bytes, bool residual,
                             bool quantised) {
  RowPlan p{false, 0, kGenericBlock, 1, kGenericBlock};
  if (elem_bytes != 2 && elem_bytes != 4) return p;
  const int V = 16 / elem_bytes;
  if (dim < V) return p;
  const int64_t chunks = dim / V;
  if (!residual && !quantised && chunks > kAnyOneStreamChunks && rows > kAnyOneStreamRows) return p;
  const bool two = chunks > kWave && (!residual || quantised || chunks <= kAnyTwoChunks);
  const int nv = two || chunks > max_block_for_nv(1) ? 2 : 1;
  const int64_t tpr = (chunks + (int64_t)kWave * nv - 1) / ((int64_t)kWave * nv) * kWave;
  if (tpr > max_block_for_nv(nv)) return p;
  p.vec = true;
  p.nv = nv;
  p.tpr = (int)tpr;
  p.groups = p.tpr >= 256 ? 1 : 256 / p.tpr;
  p.block = p.tpr * p.groups;
  return p;
}

// Workgroups go to the XCDs round robin by block index: block b of n takes the work item that
// gives each XCD runs of 2^run_log2 consecutive items (a run's blocks are 8 apart); the last
// n % (8 << run_log2) blocks keep their own index.  A permutation of 0..n-1.
constexpr int kXcdsLog2 = 3;
VG_HOST_DEVICE inline uint32_t xcd_item(uint32_t b, uint32_t n, int run_log2) {
  const int span_log2 = kXcdsLog2 + run_log2;
  const uint32_t span = b >> span_log2;
  if (span >= n >> span_log2) return b;
  const uint32_t r = b & ((1u << span_log2) - 1);
  return (span << span_log2) + ((r & ((1u << kXcdsLog2) - 1)) << run_log2) + (r >> kXcdsLog2);
}

// log2 of the workgroups of consecutive rows that one XCD takes in the one-shot forwards (the
// kernels' xcd_item): about 256 KiB of each stream, 64 workgroups at most.  Consecutive blocks go
// to different XCDs, so rows by block index spread every 64 KiB of a stream over all eight; runs
// keep an XCD's requests on neighbouring pages and let the lines that two ragged rows share meet
// in one L2.  The forward is bound by HBM; measured (bf16, alternating processes, best of 3 to 6;
// rows by block index / runs of 8, 16, 32 and 64 workgroups, us): 16384 x 4096 86.1 / 86.0, 86.8,
// 84.1, 89.5; 16384 x 8192 172.1 / 170.3, 169.5, 168.7, 168.8; 32768 x 2048 86.7 / 88.8, 86.6,
// 88.4, 84.3; 32768 x 768 35.0 / 34.1, 34.0, 33.6, 33.6; 16384 x 4095 (generic kernel) 100.6 /
// 97.8, 97.3, 95.8, 94.8; fp32 8192 x 4096 87.5 / 87.9, 86.6, 85.6, 84.7.  256 KiB is the best or
// within 2% of it in each.  Two chunks a thread (one process, the same buffers in turn; by block
// index / runs of 128, 256 and 512 KiB): 8192 x 16384 176.7 / 174.5, 174.1, 175.8; fp8 16384 x 4096
// 76.2 / 76.1, 75.7, 76.8, 4096 x 4096 22.8 / 22.5, 22.5, 22.8, 32768 x 1024 39.5 / 39.4, 39.2,
// 40.1; MXFP8 16384 x 4096 77.6 / 77.5, 76.5, 78.7; MXFP4 16384 x 4096 71.8 / 71.3, 71.0, 71.4;
// without a residual 16384 x 4096 44.9 / 44.8, 44.9, 45.9.
constexpr int64_t kXcdRunBytes = 256 << 10;
constexpr int kXcdRunMaxLog2 = 6;
// Rows of more than kXcdGenericRowBytes in the generic kernel, which reads them twice, go by block
// index: 4096 rows, by block index / in runs, us: bf16 without a residual 9001 (twice the rows) 58.6
// / 57.7, 11005 37.8 / 38.5, 14001 45.3 / 47.3, 32768 103.8 / 106.9, with one 20000 135.6 / 139.0,
// 32768 231.0 / 234.5; fp32 5001 (twice) 58.9 / 57.9, 16384 108.6 / 112.3; MXFP8 20000 2621 / 2710.
constexpr int64_t kXcdGenericRowBytes = 20 << 10;
inline int xcd_run_log2(int64_t row_bytes, int groups, bool generic = false) {
  if (generic && row_bytes > kXcdGenericRowBytes) return 0;
  const int64_t wg = row_bytes * groups > 0 ? row_bytes * groups : 1;
  int n = 0;
  while (n < kXcdRunMaxLog2 && (wg << (n + 1)) * 3 <= kXcdRunBytes * 4) ++n;
  return n;
}

// Where the register-resident forward stores h: after the row reduction, beside y, when a row
// takes at most kLateHMaxTpr threads; before it otherwise.  Measured on MI355X (bf16, A/B in
// one process, batched launches over rotating buffer sets, 6 rounds): after is faster at dim
// 2048 (86.6 against 87.5 us for 32768 rows) and 4096 (86.0 against 86.8 us at 16384 rows;
// 44.9 against 45.2 at 8192), equal at 3072 (65.2 / 65.1 us), slower at 5120 (110.7 against
// 109.5) and 8192 (179.1 against 172.7).
constexpr int kLateHMaxTpr = 512;

inline bool fwd_late_h(const RowPlan& p) { return p.vec && p.tpr <= kLateHMaxTpr; }

// The facts the kernels' indexing relies on; the C entry points refuse to launch a plan that
// breaks one of them.
inline bool row_plan_valid(const RowPlan& p, int64_t dim, int elem_bytes) {
  if (!p.vec)
    return p.tpr == kGenericBlock && p.groups == 1 && p.block == kGenericBlock;
  if (elem_bytes != 2 && elem_bytes != 4) return false;
  const int V = 16 / elem_bytes;
  return dim > 0 && dim % V == 0 && p.nv >= 1 && p.nv <= kMaxNV && p.tpr >= kWave &&
         p.tpr % kWave == 0 && p.groups >= 1 && p.block == p.tpr * p.groups &&
         p.block <= max_block_for_nv(p.nv) && (int64_t)p.nv * p.tpr * V >= dim;
}

// Backward launch: row layout, row groups per workgroup, persistent grid size and dynamic LDS.
// The register-resident kernel packs as many row groups into a workgroup as its size bound
// allows (capped by `max_block`), because the groups' dweight columns are combined in LDS and
// each workgroup writes one partial row: fewer, larger workgroups mean fewer partial rows for
// stage 2.  The grid targets `waves_per_cu` resident waves on each of `cus` compute units.
struct BwdPlan {
  RowPlan rp;
  int64_t wgs;       // workgroups = dweight partial rows
  size_t lds_bytes;  // dynamic LDS of the group combine
  bool ring = false; // the ring-pipelined kernel (plan_bwd_ring) instead of bwd_vec_kernel
  // the ring over rows of 8-byte alignment with a half chunk at their end (plan_bwd_ring8): rp
  // lays out the row's whole chunks (dim - 4 elements)
  bool x8 = false;
  // the ring over rows of any length and alignment (plan_bwd_ring_any)
  bool any = false;
  // the element-strided ring (plan_bwd_ring_elem): elements per lane, 0 when not planned
  int elem_m = 0;
  // with the RoPE gradient: bwd_vec_kernel's plain plan, each pair's rotation evaluated directly
  // where g is decoded (rows too wide for the RoPE walk's bound)
  bool rope_direct = false;
};

// The ring-pipelined backward (bwd_ring_kernel): a ring of kRingPrefetch + 1 row buffers per
// thread, so two rows are in flight while one reduces, in a branch-free steady loop.  It takes
// rows of whole 16-byte chunks over whole waves (dim <= nv * tpr * V, at most 1/8 of the chunk
// slots idle, or for 2-byte rows of one chunk per thread a partly idle last wave; idle lanes
// reload the row's last chunk, so no branch guards a load), at most two
// chunks per thread, and workgroups of at most kRingBlock threads (its launch bound: 256 VGPRs a lane for
// the three row buffers), one per CU, so each row slot walks twice as many rows as in the
// 1024-thread persistent kernel.  Measured on MI355X at 16384 x 4096 bf16: 69.2 us against 72.4.
constexpr int kRingBlock = 512;
constexpr int kRingMaxNV = 2;
constexpr int kRingPrefetch = 2;

inline BwdPlan plan_bwd(int64_t rows, int64_t dim, int elem_bytes, bool aligned, int cus,
                        int prefer_nv, int max_block, int waves_per_cu,
                        const int (&order)[kMaxNV] = kBwdOrder) {
  BwdPlan b;
  b.rp = plan_rows(dim, elem_bytes, aligned, prefer_nv, order);
  RowPlan& p = b.rp;
  if (p.vec) {
    int mb = max_block_for_nv(p.nv);
    if (max_block < mb) mb = max_block;
    p.groups = mb / p.tpr;
    if (p.groups < 1) p.groups = 1;
    p.block = p.tpr * p.groups;
  }
  const int64_t wgs_needed = rows > 0 ? (rows + p.groups - 1) / p.groups : 1;
  int64_t wg_per_cu = waves_per_cu / (p.block / kWave);
  if (wg_per_cu < 1) wg_per_cu = 1;
  int64_t wgs = (int64_t)(cus > 0 ? cus : 1) * wg_per_cu;
  if (wgs > wgs_needed) wgs = wgs_needed;
  if (wgs < 1) wgs = 1;
  b.wgs = wgs;
  b.lds_bytes = (p.vec && p.groups > 1) ? (size_t)dim * sizeof(float) : 0;
  return b;
}

// Whether a row plan suits the ring-pipelined backward (see kRingBlock).
// Rows may leave lanes idle (whole waves over fewer chunks), at most 1/8 of the row group's
// chunk slots, or for 2-byte rows of one chunk per thread any part of the last wave: the
// kernel's idle-lane variant (kRingTail) reloads the row's last chunk there.  Measured on
// MI355X (bf16, 16384 rows, alternating processes, two runs each), one-chunk row groups with a
// partly idle last wave against the plans before them (two or three chunks per thread in
// bwd_vec_kernel): 640 19.1 against 20.6 us, 768 19.5 against 21.9, 1152 29.6 against 32.4, 1280
// 30.2 against 34.0.
inline bool ring_eligible(const RowPlan& p, int64_t dim, int elem_bytes) {
  if (!p.vec || (elem_bytes != 2 && elem_bytes != 4)) return false;
  const int V = 16 / elem_bytes;
  const int64_t slots = (int64_t)p.nv * p.tpr;
  if (dim % V != 0) return false;
  const int64_t chunks = dim / V;
  return p.nv >= 1 && p.nv <= kRingMaxNV && p.tpr <= kRingBlock && chunks >= 1 &&
         slots >= chunks && slots - chunks < p.tpr &&
         ((p.nv == 1 && elem_bytes == 2) ? slots - chunks < kWave : (slots - chunks) * 8 <= slots);
}

// Whether the ring's idle-lane variant is planned for rows that leave lanes idle (whole rows
// always take the ring).  Measured on MI355X against bwd_vec_kernel (16384 rows, backward only,
// two alternating processes each, best of 3 batched rounds): faster everywhere except (a) rows
// of one chunk per thread in 320-thread row groups, whose workgroup alone on its CU holds five
// waves (2240 bf16: 56.1 us against 51.4; 1120 fp32 56.6 against 50.7), and (b) rows of two
// chunks per thread in row groups of 448 or 512 threads that are not whole 128-byte lines (bf16
// 7160: 131.0 against 125.4, 7176: 132.2 against 127.7, 8184: 150.2 against 148.3), where the
// workgroup's seven or eight waves hold the ring while bwd_vec_kernel keeps twice the waves;
// whole lines there still pay (6272 bf16: 105.8 against 112.9).  Elsewhere, e.g. bf16 4000:
// 71.3 against 73.4, 5000 87.0 against 91.9, 3576 63.2 against 75.8, fp32 2240 74.4 against
// 84.9.
inline bool ring_tail_pays(const RowPlan& p, int64_t dim, int elem_bytes) {
  const int64_t chunks = dim / (16 / elem_bytes);
  if ((int64_t)p.nv * p.tpr == chunks) return true;
  if (p.nv == 1) return (kRingBlock / p.tpr) * p.tpr >= 6 * kWave;
  return p.tpr < 448 || (dim * elem_bytes) % 128 == 0;
}

// Plan of the ring-pipelined backward: row groups packed into workgroups of up to kRingBlock
// threads, one workgroup per CU.  `ring` is false (and the plan unusable) when the row layout
// does not suit it; the caller then plans bwd_vec_kernel.
// `max_block` (at most kRingBlock) bounds the workgroup and `wgs_per_cu` (1 or 2) sets the
// resident workgroups per CU: two 256-thread workgroups per CU hold the same waves as one of 512
// (the ring's registers allow eight waves per CU) without sharing a barrier.
// Without a preference (`prefer_nv` 0), for 2-byte dtypes a ring row group of one chunk per
// thread comes first where it is planned (rows of up to kRingBlock chunks), else the backward's
// order: one chunk per thread in row groups of up to 512 threads beat two in half as many (no
// LDS combine of the row groups' dweight columns when one row group fills the workgroup).
// Measured on MI355X (16384 rows, alternating processes): the bench's config C backward
// 67.3-67.5 us against 68.6-68.7 in three runs each (the step 6094-6098 GB/s against
// 6062-6070), and with batched launches (best of 3 rounds, two runs each) bf16 1024 22.0 against
// 23.5, 1536 30.2 against 36.7, 2048 37.5 against 38.6, 3584 60.1 against 62.7, 4000 68.0
// against 71.5, 4096 68.2 against 69.4, 512, 768, 2560 and 3072 equal.  fp32 rows keep two
// chunks per thread first: one ran 1024 in 39.7 against 37.5 us, 1536 62.2 against 53.4, 2048
// 74.1 against 68.2.  Nor do one-chunk row groups of 320 or 384 threads come first (one
// workgroup of five or six waves a CU): bf16 3000 ran 59.4-59.6 us against 55.8-56.0 with two
// chunks per thread in two 192-thread row groups, 3072 55.6-56.0 against 54.7, and 2560
// 52.6-53.0 against 52.0-52.3 in bwd_vec_kernel; 448-thread ones stay first (3500 70.9-71.6
// against 72.2-72.6, 3584 60.9-62.1 against 62.5-62.7; 3200 within 1%).
// Walks of more than kRingOneChunkMaxIters rows per slot keep the backward's order: one chunk per
// thread halves the row slots, and its walks of 256 rows ran slower than two chunks' walks of 128
// (bf16 65536 x 4096: 265.9-268.3 us against 259.7-260.0; 131072 x 2048: 267.2-269.0 against
// 260.9), while walks of up to 192 rows kept its lead (49152 x 4096: 193.4 against 194.3; 32768
// x 4096: 128.5-128.7 against 130.7-131.2).
constexpr int64_t kRingOneChunkMaxIters = 192;

inline BwdPlan plan_bwd_ring(int64_t rows, int64_t dim, int elem_bytes, bool aligned, int cus,
                             int prefer_nv, int max_block = kRingBlock, int wgs_per_cu = 1) {
  if (max_block > kRingBlock) max_block = kRingBlock;
  if (wgs_per_cu < 1) wgs_per_cu = 1;
  if (wgs_per_cu > 2) wgs_per_cu = 2;
  // The ring's launch over row layout `rp`: `ring` false when the layout does not suit it.
  auto complete = [&](const RowPlan& rp) {
    BwdPlan b;
    b.rp = rp;
    b.wgs = 0;
    b.lds_bytes = 0;
    b.ring = ring_eligible(rp, dim, elem_bytes) && rp.tpr <= max_block &&
             ring_tail_pays(rp, dim, elem_bytes);
    if (!b.ring) return b;
    int wpc = wgs_per_cu;
    if (rp.tpr * wpc > kRingBlock) wpc = 1;  // a row group fills the CU's waves
    RowPlan& p = b.rp;
    p.groups = max_block / p.tpr;
    if (p.groups * wpc * p.tpr > kRingBlock) p.groups = kRingBlock / (wpc * p.tpr);
    p.block = p.tpr * p.groups;
    const int64_t wgs_needed = rows > 0 ? (rows + p.groups - 1) / p.groups : 1;
    int64_t wgs = cus > 0 ? (int64_t)cus * wpc : 1;
    if (wgs > wgs_needed) wgs = wgs_needed;
    b.wgs = wgs;
    b.lds_bytes = p.groups > 1 ? (size_t)dim * sizeof(float) : 0;
    return b;
  };
  if (prefer_nv == 0 && elem_bytes == 2) {
    // one chunk per thread in whole waves, the last one partly idle where the chunks end there
    RowPlan one = plan_rows(dim, elem_bytes, aligned, 1, kBwdOrder);
    if (aligned && dim % 8 == 0 && dim / 8 <= kRingBlock) {
      const int t = (int)((dim / 8 + kWave - 1) / kWave) * kWave;
      one = RowPlan{true, 1, t, 1, t};
    }
    if (one.vec && one.nv == 1 && one.tpr != 320 && one.tpr != 384) {
      const BwdPlan b = complete(one);
      const int64_t slots = b.wgs * b.rp.groups;
      if (b.ring && (rows + slots - 1) / slots <= kRingOneChunkMaxIters) return b;
    }
  }
  return complete(plan_rows(dim, elem_bytes, aligned, prefer_nv, kBwdOrder));
}

// The ring over rows of a 2-byte dtype whose streams start on 8-byte boundaries only and hold
// dim = 8 * n + 4 elements (hidden sizes such as 4100, whose rows alternate between the two
// halves of a 16-byte line): the ring's plan for the n whole chunks (dim - 4 elements, each
// moved as two 8-byte halves), the row's last 4 elements an extra half chunk of the row group's
// lane 0, the group combine over all dim columns.  One chunk per thread: the extra chunk's ring
// buffers and sums fit beside one chunk's, not beside two (the planner asks plan_bwd_ring for
// one, so rows of up to kRingBlock whole chunks, dim <= 4100 bf16, take it).
inline BwdPlan plan_bwd_ring8(int64_t rows, int64_t dim, int elem_bytes, int cus,
                              int max_block = kRingBlock, int wgs_per_cu = 1) {
  BwdPlan b;
  b.rp = RowPlan{false, 0, kGenericBlock, 1, kGenericBlock};
  b.wgs = 0;
  b.lds_bytes = 0;
  if (elem_bytes != 2 || dim < 12 || dim % 8 != 4) return b;
  b = plan_bwd_ring(rows, dim - 4, elem_bytes, true, cus, 1, max_block, wgs_per_cu);
  if (!b.ring || b.rp.nv != 1) {
    b.ring = false;
    return b;
  }
  b.x8 = true;
  b.lds_bytes = b.rp.groups > 1 ? (size_t)dim * sizeof(float) : 0;
  return b;
}

// The ring over rows that the chunked layout does not fit (bwd_ring_kernel's kRingAny), the row's
// last chunk overlapping the one before it: one chunk a thread, two where that leaves a workgroup of
// five or six waves (2503 bf16: 48.9 us, 72 element by element), for fp32 rows of more than two waves
// (601: 26.9 against 31.9 us, 2047 72.7 against 77.2, but with grad_h 401 26.6 against 23.3) and
// past kRingBlock chunks.
inline BwdPlan plan_bwd_ring_any(int64_t rows, int64_t dim, int elem_bytes, int cus) {
  BwdPlan b;
  b.rp = RowPlan{false, 0, kGenericBlock, 1, kGenericBlock};
  b.wgs = 0;
  b.lds_bytes = 0;
  if (elem_bytes != 2 && elem_bytes != 4) return b;
  const int V = 16 / elem_bytes;
  if (dim < V) return b;
  const int64_t chunks = (dim + V - 1) / V;
  const int64_t waves = (chunks + kWave - 1) / kWave;
  const bool two = chunks > kRingBlock || waves == 5 || waves == 6 || (elem_bytes == 4 && waves > 2);
  const int nv = two ? 2 : 1;
  const int64_t tpr = (waves + nv - 1) / nv * kWave;
  if (tpr > kRingBlock) return b;
  RowPlan& p = b.rp;
  p.vec = true;
  p.nv = nv;
  p.tpr = (int)tpr;
  p.groups = kRingBlock / p.tpr;
  p.block = p.tpr * p.groups;
  const int64_t wgs_needed = rows > 0 ? (rows + p.groups - 1) / p.groups : 1;
  const int64_t wgs = cus > 0 ? (int64_t)cus : 1;
  b.wgs = wgs < wgs_needed ? wgs : wgs_needed;
  b.lds_bytes = p.groups > 1 ? (size_t)dim * sizeof(float) : 0;
  b.any = true;
  b.ring = true;
  return b;
}

// Element-strided rows (fwd_elem_kernel, bwd_ring_elem_kernel) for rows the chunked kernels
// cannot take (odd lengths, streams that start anywhere in a 16-byte line): M elements a lane,
// 4 for rows of up to 512 elements, else 8 (0: a row longer than kRingElemMaxM * kRingBlock
// elements), row groups of whole waves packed into workgroups of up to kRingBlock threads.
// Eight elements a lane in half the lanes (more row groups a workgroup) ran the backward at bf16
// 16384 x 1535 in 42.3 us against 55.5 with four, 2047 49.4 against 60.5, 1001 30.0 against
// 31.8, and 3001 and 4095 alike.
constexpr int kRingElemMaxM = 8;

constexpr int elem_per_lane(int64_t dim) {
  if (dim <= 0 || dim > (int64_t)kRingElemMaxM * kRingBlock) return 0;
  return dim > 512 ? 8 : 4;
}

inline RowPlan plan_elem_rows(int64_t dim) {
  RowPlan p{false, 0, kGenericBlock, 1, kGenericBlock};
  const int m = elem_per_lane(dim);
  if (m == 0) return p;
  const int64_t lanes = (dim + m - 1) / m;
  p.tpr = (int)((lanes + kWave - 1) / kWave) * kWave;
  p.groups = kRingBlock / p.tpr;
  p.block = p.tpr * p.groups;
  return p;
}

// Whether a backward over rows that the chunked layout does not fit goes element by element rather
// than in chunks from any element (plan_bwd_ring_any).  2-byte rows of up to 512 elements are one
// wave of chunks, eight row groups a workgroup, whose combine alone costs a short tensor more than
// the chunks save; up to 256 elements both have eight.  Measured (bf16; elements / chunks, us): 193
// at 128 rows 7.2 / 8.0, 16384 13.4 / 14.2, 49152 24.3 / 24.6; 257 at 64 rows 6.5 / 8.1, 2048 8.5 /
// 10.0, 4096 10.4 / 10.3, 16384 18.0 / 14.4; 511 at 128 rows 7.0 / 8.4, 3072 10.3 / 11.4, 6144 12.6 /
// 13.0, 8192 13.6 / 13.7, 10240 15.3 / 14.1; 513 at 64 rows 7.7 / 7.0.
constexpr int kAnyOneWaveRowsPerCu = 32;
inline bool bwd_elem_first(int64_t rows, int64_t dim, int elem_bytes, bool has_gh, int cus) {
  if (elem_bytes == 4) return dim <= (has_gh ? 192 : 512);
  return dim <= 256 || (dim <= 512 && rows < (int64_t)kAnyOneWaveRowsPerCu * cus);
}

// The element-strided ring backward: plan_elem_rows' row groups, one workgroup per CU.
inline BwdPlan plan_bwd_ring_elem(int64_t rows, int64_t dim, int elem_bytes, int cus) {
  BwdPlan b;
  b.rp = RowPlan{false, 0, kGenericBlock, 1, kGenericBlock};
  b.wgs = 0;
  b.lds_bytes = 0;
  const int m = elem_per_lane(dim);
  if ((elem_bytes != 2 && elem_bytes != 4) || m == 0) return b;
  b.rp = plan_elem_rows(dim);
  const RowPlan& p = b.rp;
  const int64_t wgs_needed = rows > 0 ? (rows + p.groups - 1) / p.groups : 1;
  int64_t wgs = cus > 0 ? (int64_t)cus : 1;
  if (wgs > wgs_needed) wgs = wgs_needed;
  b.wgs = wgs;
  b.lds_bytes = p.groups > 1 ? (size_t)dim * sizeof(float) : 0;
  b.elem_m = m;
  return b;
}

// The ring-pipelined backward with the fused RoPE gradient (bwd_rope_ring_kernel): whole rows
// of one 16-byte chunk per thread where a row has at most kRingBlock chunks (its rotation state
// and tables keep it at 128 VGPRs), else of two (rows of up to 2 * kRingBlock chunks; 256
// VGPRs), row groups packed into workgroups of up to kRingBlock threads, rope_ring_wgs_per_cu of
// them per CU.  `ring` is false when the row layout does not suit it.  Where a slot's walk does not just
// advance by the slot count or return to its first position (rope_walk_ok), the kernel evaluates its
// angles afresh at each sequence it enters.
constexpr int kRopeRingMaxWgsPerCu = 2;

// One chunk per thread: one workgroup per CU when it fills kRingBlock threads (eight waves),
// else two (a 320- to 448-thread workgroup alone would leave the CU five to seven waves).
// Measured on MI355X (bf16, A/B in one process, 4 rounds): one 512-thread workgroup per CU
// against two runs 16384 x 4096 in 71.8 us against 79.0 (and 72.0 against 79.2 as 8 sequences of
// 2048), 8192 x 4096 in 41.7 against 45.1 and 32768 x 2048 in 71.8 against 77.6 (half the partial
// rows, and twice as many rows per walk over the same resident waves); 384-thread workgroups
// (16384 x 3072) run 61.5 us two per CU against 63.4 alone.  Two chunks per thread hold up to
// 256 VGPRs, so one workgroup per CU.
inline int rope_ring_wgs_per_cu(int nv, int block) {
  return nv == 1 && block < kRingBlock ? kRopeRingMaxWgsPerCu : 1;
}

inline BwdPlan plan_bwd_rope_ring(int64_t rows, int64_t dim, int elem_bytes, bool aligned,
                                  int cus) {
  BwdPlan b;
  b.rp = RowPlan{false, 0, kGenericBlock, 1, kGenericBlock};
  b.wgs = 0;
  b.lds_bytes = 0;
  if ((elem_bytes != 2 && elem_bytes != 4) || !aligned || dim <= 0) return b;
  const int V = 16 / elem_bytes;
  if (dim % V != 0) return b;
  const int64_t chunks = dim / V;
  const int nv = chunks <= kRingBlock ? 1 : 2;
  if (chunks % ((int64_t)nv * kWave) != 0 || chunks > (int64_t)nv * kRingBlock) return b;
  RowPlan& p = b.rp;
  p.vec = true;
  p.nv = nv;
  p.tpr = (int)(chunks / nv);
  p.groups = kRingBlock / p.tpr;
  p.block = p.tpr * p.groups;
  const int64_t wgs_needed = rows > 0 ? (rows + p.groups - 1) / p.groups : 1;
  int64_t wgs = (int64_t)(cus > 0 ? cus : 1) * rope_ring_wgs_per_cu(nv, p.block);
  if (wgs > wgs_needed) wgs = wgs_needed;
  b.wgs = wgs;
  // per thread and pair (V / 2 pairs a chunk): with one chunk the double frequency and the float
  // step and first rotations, 24 bytes; with two the float step rotation, 8 bytes; then, with
  // several row groups, their dweight combine
  const int pairs = nv * (V / 2);
  const size_t per_pair = nv == 1 ? sizeof(double) + 4 * sizeof(float) : 2 * sizeof(float);
  b.lds_bytes = (size_t)p.block * pairs * per_pair +
                (p.groups > 1 ? (size_t)dim * sizeof(float) : 0);
  b.ring = true;
  return b;
}

// The same over rows that the chunked layout does not fit or fills only in part (even lengths from
// one chunk up, any alignment; bwd_rope_ring_kernel's ANY, the last chunk overlapping the one
// before it).
inline BwdPlan plan_bwd_rope_ring_any(int64_t rows, int64_t dim, int elem_bytes, int cus) {
  BwdPlan b;
  b.rp = RowPlan{false, 0, kGenericBlock, 1, kGenericBlock};
  b.wgs = 0;
  b.lds_bytes = 0;
  if ((elem_bytes != 2 && elem_bytes != 4) || dim < 16 / elem_bytes || dim % 2 != 0) return b;
  const int V = 16 / elem_bytes;
  const int64_t chunks = (dim + V - 1) / V;
  const int nv = chunks <= kRingBlock ? 1 : 2;
  const int64_t tpr = (chunks + (int64_t)nv * kWave - 1) / ((int64_t)nv * kWave) * kWave;
  if (tpr > kRingBlock) return b;
  // the plan of the whole row group, its combine over the row's own columns
  b = plan_bwd_rope_ring(rows, tpr * nv * V, elem_bytes, true, cus);
  if (!b.ring) return b;
  if (b.rp.groups > 1) b.lds_bytes -= (size_t)(tpr * nv * V - dim) * sizeof(float);
  // fp32's step rotations are double, in the place of the first rotations with one chunk a thread;
  // with two, those or the 2-byte rows' frequencies come on top
  if (nv == 2) b.lds_bytes += (size_t)b.rp.block * nv * (V / 2) * sizeof(double);
  b.any = true;
  return b;
}

// The turns a position of RoPE pair i, the first of a lane's chunk: `first` at the pair that begins the
// row's aligned chunk of `pairs` around it, then the double ratio from pair to pair (as the lane goes on
// to its next ones).  So the pairs that the row's last chunk shares with the one before it, where it
// begins inside that, have the same bits in both lanes, and so have the columns that both store.
template <typename First>
VG_HOST_DEVICE inline double rope_first_turns(int i, int pairs, double ratio, First first) {
  double g = first(i - i % pairs);
  for (int t = i % pairs; t > 0; --t) g *= ratio;
  return g;
}

// Rows a float rotation of the ring's walk is advanced before its angles are evaluated afresh.
// `each_row`: the rows whose other kernel, the generic one, evaluates every angle at its row.  Four
// rows keep their dweight as near its 64-bit value (fp16 8192 x 2050, generic / 16 / 4 rows: off by
// 2.0e-7 / 2.5e-7 / 1.8e-7 of it) at little cost (31.1 us both; 8192 x 4098, two chunks a thread, 53.2 /
// 57.8).
constexpr int rope_ring_anchor(bool each_row) { return each_row ? 4 : 16; }

// Whether such rows of a short tensor stay in the generic kernel: the ring's set-up of each pair's
// rotation and its combine of many row groups outlast a few short rows.  Measured (generic / ring, us):
// bf16 74 at 16 rows 5.6 / 9.2, 512 7.8 / 9.8, 1024 10.1 / 10.0; 510 at 512 9.5 / 10.6, 1024 13.0 / 10.9;
// 514 at 64 rows 7.8 / 8.9, 256 8.0 / 9.2, 512 10.4 / 9.6; 2050 at 1 row 9.6 / 8.2; fp32 130 at 64 rows
// 6.5 / 7.2, 512 8.4 / 7.6; 258 at 16 rows 5.9 / 6.9, 128 8.1 / 7.1; 514 at 16 rows 6.7 / 6.6.
inline bool rope_bwd_generic_first(int64_t rows, int64_t dim, int elem_bytes, int cus) {
  const int64_t V = 16 / elem_bytes, waves = ((dim + V - 1) / V + kWave - 1) / kWave;
  if (waves == 1) return elem_bytes == 2 ? rows < 4 * (int64_t)cus : rows <= cus;
  return waves == 2 && rows <= (elem_bytes == 2 ? cus : cus / 4);
}

// Whether `slots` row slots walking `rows` rows (slot s: rows s, s + slots, ...) see positions
// (row % seq) that only advance by `slots` or return to the walk's first one: slots is a
// multiple or a divisor of seq, or no walk reaches the end of a sequence.
inline bool rope_walk_ok(int64_t rows, int64_t slots, int64_t seq) {
  if (rows <= 0 || slots <= 0 || seq <= 0) return false;
  if (seq % slots == 0 || slots % seq == 0) return true;
  const int64_t iters = (rows + slots - 1) / slots;
  return iters <= seq / slots;  // iters * slots <= seq
}

// Whether a plan suits bwd_rope_ring_kernel (the facts its indexing relies on).
inline bool rope_ring_eligible(const RowPlan& p, int64_t dim, int elem_bytes) {
  if (!p.vec || (elem_bytes != 2 && elem_bytes != 4)) return false;
  return (p.nv == 1 || p.nv == 2) && p.tpr % kWave == 0 &&
         (int64_t)p.nv * p.tpr * (16 / elem_bytes) == dim && p.block == p.tpr * p.groups &&
         p.block <= kRingBlock;
}

// Backward plan with the fused inverse RoPE: the same layout under max_block_for_nv_rope, or the
// generic plan where a row group does not fit that bound.
inline BwdPlan plan_bwd_rope(int64_t rows, int64_t dim, int elem_bytes, bool aligned, int cus,
                             int prefer_nv, int max_block, int waves_per_cu) {
  RowPlan rp = plan_rows(dim, elem_bytes, aligned, prefer_nv, kBwdOrderRope);
  if (rp.vec && max_block_for_nv_rope(rp.nv) < rp.tpr) {
    // the first chunk count whose row group fits the RoPE walk's bound (rows of 1536 chunks:
    // three chunks per thread in 512 threads, not two in 768)
    rp.vec = false;
    for (int nv = 1; nv <= kMaxNV && !rp.vec; ++nv) {
      const RowPlan q = plan_rows(dim, elem_bytes, aligned, nv, kBwdOrderRope);
      if (q.vec && q.nv == nv && q.tpr <= max_block_for_nv_rope(nv)) rp = q;
    }
    if (!rp.vec) {
      // no chunk count fits the walk (rows of more than 1536 chunks): the plain plan with each
      // pair's rotation evaluated where g is decoded, preferring four chunks per thread (248
      // VGPRs in 512-thread rows; two chunks in 1024-thread rows spill), else the generic kernel
      BwdPlan d = plan_bwd(rows, dim, elem_bytes, aligned, cus, 4, max_block, waves_per_cu);
      if (d.rp.vec) {
        d.rope_direct = true;
        return d;
      }
      return plan_bwd(rows, dim, elem_bytes, false, cus, prefer_nv, max_block,
                      waves_per_cu);  // generic
    }
    prefer_nv = rp.nv;
  }
  int mb = max_block;
  if (rp.vec) {
    const int bound = max_block_for_nv_rope(rp.nv);
    if (bound < mb) mb = bound;
  }
  return plan_bwd(rows, dim, elem_bytes, aligned, cus, prefer_nv, mb, waves_per_cu,
                  kBwdOrderRope);
}

// Tiles of the norm + RoPE forward (fwd_rope_tile_kernel): row groups of one chunk a thread up to
// the workgroup bound (the row's last chunk may overlap the one before it), else of two; tiles of
// up to rope_tile_most rows, halved while they leave fewer than kRopeTileMinWgs workgroups (bf16 dim
// 4096, tiles of 1 / 2 / 4, us: 64 rows 3.5 / 3.9 / 4.5, 512 4.8 / 4.4 / 5.0, 2048 11.7 / 8.8 / 8.1) or
// are longer than what they cut.  A tile's rows are consecutive positions of one sequence, or, of
// sequences shorter than a tile (decode steps), one position of consecutive sequences, so that its
// rotations still serve all of its rows (bf16, cut to the sequence / across sequences, us: 16384 x
// 4096 in sequences of 1 72.5 / 46.2, of 2 54.2 / 48.1, of 3 62.0 / 46.6, 65536 x 768 of 1 70.4 /
// 34.8).  `rp.vec` false: a row shorter than a chunk or longer than the registers hold.
//
// With a residual its loads double the registers, and two chunks a thread or fp32's double rotations
// do so again: tiles of 1 / 2 / 4 there, us: bf16 16384 x 4096 - / 88.2 / 91.6, 8192 x 16384 188 / 205 /
// 259, 4096 x 12288 70.9 / 76.5; fp32 8192 x 2048 44.8 / 45.8, 8192 x 4096 90.8 / 93.1, 4096 x 8192
// 90.2 / 94.9, 16384 x 1024 45.5 / 45.1.
constexpr int rope_tile_most(int elem_bytes, int nv, bool residual) {
  return !residual ? 4 : elem_bytes == 4 || nv == 2 ? 1 : 2;
}
struct RopeTilePlan {
  RowPlan rp;
  int tile;     // rows a tile
  bool across;  // of consecutive sequences, at one position
  int64_t wgs;  // workgroups, rp.groups tiles each
};
constexpr int64_t kRopeTileMinWgs = 256;

inline RopeTilePlan plan_rope_tiles(int64_t rows, int64_t dim, int elem_bytes, int64_t seq,
                                    bool residual) {
  RopeTilePlan t{RowPlan{false, 0, kGenericBlock, 1, kGenericBlock}, 1, false, 0};
  if ((elem_bytes != 2 && elem_bytes != 4) || rows < 1 || seq < 1) return t;
  const int V = 16 / elem_bytes;
  if (dim < V) return t;
  const int64_t chunks = (dim + V - 1) / V;
  const int nv = chunks > max_block_for_nv(1) ? 2 : 1;
  const int64_t tpr = (chunks + (int64_t)kWave * nv - 1) / ((int64_t)kWave * nv) * kWave;
  if (tpr > max_block_for_nv(nv)) return t;
  RowPlan& p = t.rp;
  p.vec = true;
  p.nv = nv;
  p.tpr = (int)tpr;
  p.groups = p.tpr >= 256 ? 1 : 256 / p.tpr;
  p.block = p.tpr * p.groups;
  t.tile = rope_tile_most(elem_bytes, nv, residual);
  t.across = seq < t.tile;
  const int64_t cut = t.across ? rows / seq : seq;  // what the tiles cut, rows / cut times
  auto wgs = [&](int r) { return (rows / cut * ((cut + r - 1) / r) + p.groups - 1) / p.groups; };
  while (t.tile > 1 && (t.tile > cut || wgs(t.tile) < kRopeTileMinWgs)) t.tile /= 2;
  t.wgs = wgs(t.tile);
  return t;
}

// The rows of tile i, r of them at most: first, first + step, ..., n of them, the first at position
// pos and the others at the next ones or (`across`) at the same.  Tiles past the last one give the
// last (ok false).
struct RopeTile {
  uint32_t first, step, pos;
  int n;
  bool ok;
};
VG_HOST_DEVICE inline RopeTile rope_tile(uint32_t i, uint32_t rows, uint32_t seq, int r,
                                         bool across) {
  const uint32_t outer = rows / seq;
  const uint32_t cut = across ? outer : seq, other = across ? seq : outer;
  const uint32_t per = (cut + r - 1) / r;
  RopeTile t;
  t.ok = i < per * other;
  if (!t.ok) i = per * other - 1;
  // consecutive tiles hold neighbouring rows: across, the positions of the same sequences
  const uint32_t q = i / (across ? other : per);
  const uint32_t m = i - q * (across ? other : per);
  const uint32_t at = (across ? q : m) * r;  // in what is cut
  t.pos = across ? m : at;
  t.first = across ? at * seq + m : q * seq + at;
  t.step = across ? seq : 1;
  t.n = (int)(cut - at < (uint32_t)r ? cut - at : (uint32_t)r);
  return t;
}

// Workspace of the backward's dweight partial rows.  The plan depends on the element size, on
// pointer alignment and on whether the RoPE gradient is fused, which a size query does not know,
// so this is the largest need over every plan the backward can pick for (rows, dim).
inline size_t bwd_workspace_bytes(int64_t rows, int64_t dim, int cus, int prefer_nv,
                                  int max_block, int waves_per_cu, int ring_block = kRingBlock,
                                  int ring_wgs_per_cu = 1) {
  if (rows <= 0 || dim <= 0 || cus <= 0) return 0;
  int64_t most = 0;
  const int sizes[2] = {2, 4};
  for (int si = 0; si < 2; ++si) {
    for (int al = 0; al < 2; ++al) {
      const int64_t n =
          plan_bwd(rows, dim, sizes[si], al != 0, cus, prefer_nv, max_block, waves_per_cu).wgs;
      if (n > most) most = n;
      const int64_t nr = plan_bwd_rope(rows, dim, sizes[si], al != 0, cus, prefer_nv, max_block,
                                       waves_per_cu).wgs;
      if (nr > most) most = nr;
      const BwdPlan rg = plan_bwd_ring(rows, dim, sizes[si], al != 0, cus, prefer_nv,
                                       ring_block, ring_wgs_per_cu);
      if (rg.ring && rg.wgs > most) most = rg.wgs;
      const BwdPlan rr = plan_bwd_rope_ring(rows, dim, sizes[si], al != 0, cus);
      if (rr.ring && rr.wgs > most) most = rr.wgs;
      const BwdPlan rra = plan_bwd_rope_ring_any(rows, dim, sizes[si], cus);
      if (rra.ring && rra.wgs > most) most = rra.wgs;
      const BwdPlan r8 = plan_bwd_ring8(rows, dim, sizes[si], cus, ring_block, ring_wgs_per_cu);
      if (r8.ring && r8.wgs > most) most = r8.wgs;
      const BwdPlan re = plan_bwd_ring_elem(rows, dim, sizes[si], cus);
      if (re.elem_m > 0 && re.wgs > most) most = re.wgs;
      const BwdPlan ra = plan_bwd_ring_any(rows, dim, sizes[si], cus);
      if (ra.ring && ra.wgs > most) most = ra.wgs;
    }
  }
  return (size_t)most * (size_t)dim * sizeof(float);
}

}  // namespace vg_plan

#endif  // VELOGRAD_LAUNCH_PLAN_H
