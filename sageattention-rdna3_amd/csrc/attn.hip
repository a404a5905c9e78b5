// Fused flash attention for gfx950 (CDNA4, wave64 MFMA): the INT8 quantized
// path and the direct fp16/bf16 path, one kernel template.  The kernels and
// their host code live in attn_body.inc, compiled here in three block shapes;
// this file holds the C entry points, which pick the shape per launch.  The
// mapping below describes the 256-row shape (8 waves); the 128-row shapes have
// 4 waves and two blocks per CU, or 8 waves in two key groups.
//
// Math (csrc/attn_gfx11.cu of the reference):
//   INT8   (:409-825)   s_ij = float(sum_d q8[i,d] * k8[j,d]) * (q_scale[i/32] * k_scale[j/16])
//   direct (:1465-1885) s_ij = fp32(sum_d q[i,d] * k[j,d]) * fl(sm_scale * log2 e)  (fp16 or bf16 Q/K)
// in the log2 domain (INT8: Q was pre-scaled by sm_scale*log2 e), causal mask
// j > i (top-left) and j >= Sk, online softmax with exp2, P rounded to fp16
// (RNE), O += P.V_T with fp32 accumulation (V_T fp16 in both paths), out =
// O * (1/l) cast to fp16/bf16.
//
// Mapping onto CDNA4:
//   * block = 8 waves x 32 query rows (BM = 256), one block per CU, two waves
//     per SIMD; KV tiles of BN = 64 keys shared by all 8 waves through LDS;
//   * S^T = K . Q^T: A = K rows from LDS, B = the wave's Q^T fragment held in
//     registers for the whole kernel (v_mfma_i32_32x32x32_i8, or
//     v_mfma_f32_32x32x16_f16/bf16 for the direct path: both take 32 bytes of
//     each row per MFMA).  The 32x32 accumulator puts one query per lane
//     column (lane & 31), so the row softmax is 32 in-lane values plus one
//     permlane32 swap;
//   * O^T = V^T . P^T with v_mfma_f32_32x32x16_f16: B = P^T taken straight
//     from the S^T accumulators (no LDS round trip), A = V_T rows from LDS.
//     K rows sit in LDS with bits 2 and 3 of the key index swapped, which
//     makes accumulator register r of lane half h hold key 16(r/8) + 8h + r%8:
//     exactly the 8 consecutive keys the PV operand wants from that lane;
//   * software pipeline inside every wave: step j runs the softmax of tile j
//     (VALU) interleaved with the MFMAs of P_{j-1}.V_{j-1} and S_{j+1} =
//     K_{j+1}.Q^T, so each wave keeps the matrix core and the VALU busy at
//     once and the two waves of a SIMD fill each other's gaps.  A single wave
//     issues VALU at half the SIMD's rate, so both waves of a SIMD carry
//     softmax work all the time (no MFMA-only / VALU-only roles).  S and P are
//     rewritten in place: the chunk order reads each before overwriting it;
//   * online softmax with a lazy reference max: the max moves only when a row
//     max grows by more than 2^8; O is then rescaled at the top of the next
//     step, after the P.V MFMAs that still used the old max.  The unmasked
//     loop tests each lane's tile sum of p against 2^8 after the exponentials
//     instead of taking the max first, and redoes the rare tile that fails
//     with the max moved (TileSoftmaxSum);
//   * K/V tiles stream into a 3-stage LDS ring with buffer_load ... lds
//     (no staging registers), issued two steps ahead; loads past the block's
//     last key read as zero through the descriptor's record count.  The
//     direct path reads K (and Q) straight from the caller's strided tensors;
//   * causal: the KV loop stops at the block's last row, masks only on tail /
//     diagonal tiles;
//   * work items (a q-block, or a key range of one for split launches) go to
//     XCDs in contiguous ranges (consecutive q-blocks of a head share an XCD's
//     L2 for K/V), heaviest causal blocks first; with more items than CUs a
//     persistent grid of one block per CU walks a static snake schedule
//     instead of relying on the hardware dispatcher (see attn_fwd_kernel);
//   * the epilogue stages each wave's output rows in LDS and writes whole
//     rows; non-causal launches that leave CUs idle can split key ranges,
//     merged by attn_merge_kernel with the partial LSEs.
#include <algorithm>
#include <atomic>
#include <cfloat>
#include <cmath>
#include <type_traits>
#include <utility>

#include "attn_device.h"

namespace sage {

// The kernels and their host code in three block shapes (attn_body.inc):
//   * w8: 8 waves x 32 query rows = 256-row q-blocks, one block per CU;
//   * w4: 4 waves x 32 query rows = 128-row q-blocks, two blocks per CU, whose
//     waves do not share barriers, so one block's prologue, epilogue and
//     barrier waits overlap the other's key loop; each block loads its own K/V
//     tiles (twice the L2->LDS traffic of w8);
//   * g2: 2 key groups x 4 waves x 32 query rows = 128-row q-blocks, one block
//     per CU: the groups take every other key tile of the same rows and merge
//     in LDS.  A launch with at most one 128-row q-block per CU has two waves
//     per SIMD this way and half the key steps; in w4 the lone block's one wave
//     per SIMD issues alone (a D = 64 direct step 1.9k cycles, against 3.0k for
//     two tiles in g2).
// The 128-row shapes run the D = 64 non-causal launches (direct and INT8) and
// the causal launches with few q-blocks (small_blocks; key_groups picks w4 or
// g2), w8 all others.  Same-box timings of w4
// against w8 (identical outputs): D = 64 non-causal -7% to -27% (the direct
// kernel at B1 H20 S1024: 21.3 -> 15.6 us; INT8 at B1 H10 S4096: 65.9 -> 56.2
// us); causal launches of one or more full rounds +2% to +6% and D = 128
// non-causal launches with key splits +3% to +4% (the doubled tile traffic),
// so those stay on w8.  w4 / g2, whole sageattn, bf16, same box: INT8 causal B1 H8 S4096 D128 65.1 / 60.9 us,
// H4 S8192 107.8 / 97.4, D64 H8 S6144 68.0 / 59.4; direct causal B1 H16 S2048
// D128 40.7 / 37.6, H8 S1024 24.1 / 22.8, D64 H16 S2048 27.8 / 24.5; paired
// causal: direct H32 S2048 D128 54.0 / 52.9, D64 33.7 / 30.8, INT8 H16 S4096
// D128 82.0 / 80.9; non-causal as at kMinGroupTiles below.
// The stamps build (build.py --stamps, SAGE_STAMPS=1) adds per-wave cycle
// stamps to the attention kernels (attn_body.inc, StampField) and the two
// functions below that read them; the default build has neither.
#ifndef SAGE_STAMPS
#define SAGE_STAMPS 0
#endif
#if SAGE_STAMPS
constexpr int kStampBlocks = 2048;  // blocks whose waves record (8 waves each at most)
constexpr int kStampStride = 32;    // uint64 fields per wave record
__device__ uint64_t g_stamps[kStampBlocks * 8 * kStampStride];
#endif

namespace w8 {
constexpr int kBM = 256;
constexpr int kWaves = 8;
constexpr int kGroups = 1;
constexpr int kBlocksPerCu = 1;
constexpr bool kSmallShape = false;
#include "attn_body.inc"
}  // namespace w8

namespace w4 {
constexpr int kBM = 128;
constexpr int kWaves = 4;
constexpr int kGroups = 1;
constexpr int kBlocksPerCu = 2;
constexpr bool kSmallShape = true;
#include "attn_body.inc"
}  // namespace w4

namespace g2 {
constexpr int kBM = 128;
constexpr int kWaves = 4;
constexpr int kGroups = 2;
constexpr int kBlocksPerCu = 1;
constexpr bool kSmallShape = true;
#include "attn_body.inc"
}  // namespace g2

// A lone 128-row block on a CU takes this fraction of a 256-row block's time
// per key tile step.  Fitted to 4-wave blocks (MI355X, B1 H32 S2048 causal: the
// D = 128 direct kernel 0.97 against 1.38 us; the Q-fused INT8 kernel's paired
// launches at B1 H16 S4096 and B1 H32 S2048: 0.77).  The g2 blocks that run
// instead are 1-17% faster, so a launch taken by these factors gains, and a few
// that would gain are left in w8 (below).
constexpr double kLoneHalfBlockTileDirect = 0.70;
constexpr double kLoneHalfBlockTileI8 = 0.77;

// Whether a launch runs 128-row q-blocks (in w4 or g2, by key_groups): D = 64
// non-causal launches, and causal ones.  128 rows for causal launches whose
// 256-row q-blocks would fill at most half the CUs (their 128-row q-blocks then
// fill twice as many, one block per CU); w8 for launches of more than a round.
// A causal launch also runs 128 rows when its 256-row q-blocks fill at most one
// round and the causal cost model rates the 128-row q-blocks faster: with one
// block resident per CU they run as a persistent grid in which the snake
// schedule gives each block a heavy and a light q-block.  (The model walks w4's
// schedule, which is g2's: both have 128 rows and, causal, one block per CU.)
// Whole sageattn, w8 / 128 rows as g2, causal, B1, bf16, same box: half a round
// INT8 H8 S4096 D128 91.1 / 60.9 us, direct H8 S1024 D128 31.5 / 22.8, H16 S2048
// 54.0 / 37.6; one round direct D128 H32 S2048 59.5 / 52.9, H24 54.0 / 45.6, D64
// H32 S2048 38.7 / 30.8, H20 S3072 52.8 / 46.5, INT8 H16 S4096 D128 97.8 / 80.9,
// D64 72.0 / 55.9, H12 S4096 D128 92.4 / 74.4.  The model rightly keeps H32 S1536
// D128 direct in w8 (46.0 / 53.7: a block would get two heavy q-blocks), and
// INT8 S3072 wrongly (H12-H20 D64 57.9 / 51.2, D128 76.0 / 72.2).
bool small_blocks(int64_t head_dim, int is_causal, int64_t batch, int64_t q_heads, int64_t q_len, int64_t kv_len,
                  bool direct) {
  if (is_causal == 0) return head_dim == 64;
  const int64_t qblocks = batch * q_heads * ((q_len + 255) / 256);
  if (qblocks <= 0) return false;
  if (qblocks * 2 <= device_cus()) return true;
  if (qblocks > device_cus()) return false;
  const double f = direct ? kLoneHalfBlockTileDirect : kLoneHalfBlockTileI8;
  if (head_dim == 64)
    return f * w4::causal_blocks_cost<64, w4::kQkBf16>(batch * q_heads, q_len, kv_len) <
           w8::causal_blocks_cost<64, w8::kQkBf16>(batch * q_heads, q_len, kv_len);
  return f * w4::causal_blocks_cost<128, w4::kQkBf16>(batch * q_heads, q_len, kv_len) <
         w8::causal_blocks_cost<128, w8::kQkBf16>(batch * q_heads, q_len, kv_len);
}

// Whether a launch of 128-row q-blocks runs in g2 instead of w4: a causal one
// (their blocks are alone on a CU in either shape) whose heaviest q-block has
// more key tiles than kMaxLoneTiles*, and a non-causal one whose items (q-blocks,
// or key pieces of split ones) fit one per CU and have at least kMinGroupTiles.
// Causal, whole call, w4 / g2, MI355X: direct fp16 B1 H8 S64 D64 5.8 / 6.9 us,
// D128 7.5 / 8.8; S128 D128 9.6 / 10.3; S320 D64 8.4 / 8.8, D128 11.0 / 11.5; S384
// even, S1024 D64 +7% in w4; INT8 fp16 S64 -15%, S320 D128 19.5 / 22.4, S512 -3% to
// -11%, S640 -4% to +1%, S1280 D64 +6%.  Non-causal: with more items than CUs w4 hosts two blocks
// a CU, which share no barrier (B1 H10 S4096 D64, 512 items: w4 60 us, g2 65);
// with few tiles the merge and the doubled prologue outweigh the halved steps.
// Whole call, w4 / g2, B1 H20 Sq1024 D64 (160 items; 80 to 240 items alike):
// direct fp16 4 tiles 7.9 / 8.7 us, 8 10.2 / 10.7, 12 12.5 / 12.5, 14 13.8 /
// 13.4, 16 14.9 / 14.4, 24 19.6 / 18.1, 32 24.1 / 21.8; bf16 16 15.9 / 15.0;
// INT8 fp16 8 17.3 / 17.4, 16 22.1 / 21.2, 48 41.3 / 36.2.  Even at 12; from 16
// on g2 gains in every kind.  Per piece of split items the same: H10, 2 or 3
// pieces of 10 tiles 17.4 / 18.3, 3 of 16 29.3 / 28.9 (INT8).
constexpr int64_t kMaxLoneTilesDirect = 5;
constexpr int64_t kMaxLoneTilesI8 = 8;
constexpr int64_t kMinGroupTiles = 16;
bool key_groups(int is_causal, int64_t head_dim, int64_t batch, int64_t q_heads, int64_t q_len, int64_t kv_len,
                bool direct, int num_splits, int64_t ws_bytes) {
  if (is_causal != 0) {
    const int64_t tiles = cdiv(std::min(cdiv(q_len, w4::kBM) * w4::kBM, kv_len), w4::kBN);
    return tiles > (direct ? kMaxLoneTilesDirect : kMaxLoneTilesI8);
  }
  const int64_t qblocks = batch * q_heads * cdiv(q_len, w4::kBM);
  if (qblocks <= 0 || qblocks > device_cus()) return false;
  const w4::SplitPlan sp = w4::plan_splits(!direct, qblocks, kv_len, head_dim, false, num_splits, ws_bytes);
  return sp.nfull + (qblocks - sp.nfull) * sp.nsplit <= device_cus() &&
         cdiv(kv_len, w4::kBN) >= kMinGroupTiles * sp.nsplit;
}

}  // namespace sage


using namespace sage;

// Scratch of sage_attn_i8_fwd_qfused_noalloc (the key splits' partial outputs
// and LSEs): device memory the library holds until the process ends, one copy
// per GPU.  The name is a host-side stand-in for host code; kernels get the
// device address that hipGetSymbolAddress returns for the current device.
// 64 MiB holds the automatic plans of about 95% of shapes (a sweep of B 1-4,
// H 1-64, S 256-40k, D 64/128 on 256 CUs: 4.5% need more, up to 161 MiB),
// among them every 256-piece plan of 256-row D = 128 q-blocks (33.8 MB).
constexpr int64_t kScratchBytes = int64_t{64} << 20;
static __device__ __align__(256) char scratch[kScratchBytes];

namespace {
// The current device's address of `scratch`, looked up once per device (with
// that device current) and kept; null with the error recorded if the runtime
// cannot give it.
void* scratch_address(const char* fn) {
  constexpr int kDevs = 64;
  static std::atomic<void*> cache[kDevs];
  int dev = 0;
  hipError_t e = hipGetDevice(&dev);
  if (e != hipSuccess || dev < 0 || dev >= kDevs) {
    (void)hipGetLastError();
    set_error(SAGE_ERR_HIP, "%s: no current device (%s)", fn, e != hipSuccess ? hipGetErrorString(e) : "out of range");
    return nullptr;
  }
  void* ptr = cache[dev].load(std::memory_order_acquire);
  if (ptr != nullptr) return ptr;
  e = hipGetSymbolAddress(&ptr, HIP_SYMBOL(scratch));
  if (e != hipSuccess || ptr == nullptr) {
    (void)hipGetLastError();
    set_error(SAGE_ERR_HIP, "%s: hipGetSymbolAddress(scratch) failed: %s", fn, hipGetErrorString(e));
    return nullptr;
  }
  cache[dev].store(ptr, std::memory_order_release);
  return ptr;
}

// attn_fwd of the block shape the launch runs (the arguments include head_dim and is_causal again)
template <typename... Args>
int run_attn(int64_t head_dim, int is_causal, int64_t batch, int64_t q_heads, int64_t q_len, int64_t kv_len, int qk,
             int num_splits, int64_t ws_bytes, Args... args) {
  const bool direct = qk == w8::kQkF16 || qk == w8::kQkBf16 || qk == w8::kQkF16V || qk == w8::kQkBf16V;
  if (!small_blocks(head_dim, is_causal, batch, q_heads, q_len, kv_len, direct)) return w8::attn_fwd(qk, args...);
  return key_groups(is_causal, head_dim, batch, q_heads, q_len, kv_len, direct, num_splits, ws_bytes)
             ? g2::attn_fwd(qk, args...)
             : w4::attn_fwd(qk, args...);
}

// The plan of the shape the launch runs and its workspace bytes (or a negative status).
int64_t split_plan(bool quantized, int64_t batch, int64_t q_heads, int64_t q_len, int64_t kv_len, int64_t head_dim,
                   int is_causal, int num_splits, int64_t* whole, int* splits) {
  int64_t r;
  if (small_blocks(head_dim, is_causal, batch, q_heads, q_len, kv_len, !quantized)) {
    w4::SplitPlan sp;
    r = w4::attn_split_plan(quantized, batch, q_heads, q_len, kv_len, head_dim, is_causal, num_splits, &sp);
    *whole = sp.nfull;
    *splits = static_cast<int>(sp.nsplit);
  } else {
    w8::SplitPlan sp;
    r = w8::attn_split_plan(quantized, batch, q_heads, q_len, kv_len, head_dim, is_causal, num_splits, &sp);
    *whole = sp.nfull;
    *splits = static_cast<int>(sp.nsplit);
  }
  return r;
}
}  // namespace

extern "C" int sage_attn_i8_fwd(const int8_t* q_i8, const int8_t* k_i8, const void* value_t, void* out,
                                const float* q_scale, const float* k_scale, int out_dtype,
                                int64_t batch, int64_t q_heads, int64_t kv_heads,
                                int64_t q_len, int64_t kv_len, int64_t head_dim,
                                int64_t o_stride_b, int64_t o_stride_h, int64_t o_stride_n,
                                int is_causal, void* stream) {
  clear_error();
  return run_attn(head_dim, is_causal, batch, q_heads, q_len, kv_len, w8::kQkI8, 1, 0, q_i8, k_i8, value_t, out, nullptr,
                  q_scale, k_scale, out_dtype, batch, q_heads, kv_heads, q_len, kv_len, head_dim,
                  q_heads * q_len * head_dim, q_len * head_dim, head_dim, kv_heads * kv_len * head_dim,
                  kv_len * head_dim, head_dim, 0, 0, 0, o_stride_b, o_stride_h, o_stride_n, is_causal, 0.0, 1, nullptr,
                  0, stream, "sage_attn_i8_fwd");
}

extern "C" int sage_attn_i8_fwd_lse(const int8_t* q_i8, const int8_t* k_i8, const void* value_t, void* out,
                                    float* lse, const float* q_scale, const float* k_scale, int out_dtype,
                                    int64_t batch, int64_t q_heads, int64_t kv_heads,
                                    int64_t q_len, int64_t kv_len, int64_t head_dim,
                                    int64_t o_stride_b, int64_t o_stride_h, int64_t o_stride_n,
                                    int is_causal, void* stream) {
  clear_error();
  return run_attn(head_dim, is_causal, batch, q_heads, q_len, kv_len, w8::kQkI8, 1, 0, q_i8, k_i8, value_t, out, lse, q_scale,
                  k_scale, out_dtype, batch, q_heads, kv_heads, q_len, kv_len, head_dim, q_heads * q_len * head_dim,
                  q_len * head_dim, head_dim, kv_heads * kv_len * head_dim, kv_len * head_dim, head_dim, 0, 0, 0,
                  o_stride_b, o_stride_h, o_stride_n, is_causal, 0.0, 1, nullptr, 0, stream, "sage_attn_i8_fwd_lse");
}

extern "C" int sage_attn_direct_fwd(const void* query, const void* key, const void* value_t, void* out, float* lse,
                                    int dtype, int64_t batch, int64_t q_heads, int64_t kv_heads,
                                    int64_t q_len, int64_t kv_len, int64_t head_dim,
                                    int64_t q_stride_b, int64_t q_stride_h, int64_t q_stride_n,
                                    int64_t k_stride_b, int64_t k_stride_h, int64_t k_stride_n,
                                    int64_t o_stride_b, int64_t o_stride_h, int64_t o_stride_n,
                                    int is_causal, double sm_scale, int num_splits, void* workspace,
                                    int64_t workspace_bytes, void* stream) {
  clear_error();
  return run_attn(head_dim, is_causal, batch, q_heads, q_len, kv_len,
                  dtype == SAGE_DTYPE_BF16 ? w8::kQkBf16 : w8::kQkF16, num_splits,
                  workspace != nullptr ? workspace_bytes : 0, query, key, value_t, out, lse, nullptr, nullptr,
                  dtype, batch, q_heads, kv_heads, q_len, kv_len, head_dim, q_stride_b, q_stride_h, q_stride_n,
                  k_stride_b, k_stride_h, k_stride_n, 0, 0, 0, o_stride_b, o_stride_h, o_stride_n, is_causal, sm_scale,
                  num_splits, workspace, workspace_bytes, stream, "sage_attn_direct_fwd");
}

extern "C" int sage_attn_direct_fwd_vrows(const void* query, const void* key, const void* value, void* out,
                                          float* lse, int dtype, int64_t batch, int64_t q_heads, int64_t kv_heads,
                                          int64_t q_len, int64_t kv_len, int64_t head_dim,
                                          int64_t q_stride_b, int64_t q_stride_h, int64_t q_stride_n,
                                          int64_t k_stride_b, int64_t k_stride_h, int64_t k_stride_n,
                                          int64_t v_stride_b, int64_t v_stride_h, int64_t v_stride_n,
                                          int64_t o_stride_b, int64_t o_stride_h, int64_t o_stride_n,
                                          int is_causal, double sm_scale, int num_splits, void* workspace,
                                          int64_t workspace_bytes, void* stream) {
  clear_error();
  return run_attn(head_dim, is_causal, batch, q_heads, q_len, kv_len, w8::kQkF16V, num_splits,
                  workspace != nullptr ? workspace_bytes : 0, query, key, value, out, lse, nullptr,
                  nullptr, dtype, batch, q_heads, kv_heads, q_len, kv_len, head_dim, q_stride_b, q_stride_h,
                  q_stride_n, k_stride_b, k_stride_h, k_stride_n, v_stride_b, v_stride_h, v_stride_n, o_stride_b,
                  o_stride_h, o_stride_n, is_causal, sm_scale, num_splits, workspace, workspace_bytes, stream,
                  "sage_attn_direct_fwd_vrows");
}

extern "C" int sage_attn_i8_fwd_qfused(const void* query, const int8_t* k_i8, const void* value_t, void* out,
                                       float* lse, const float* k_scale, int dtype,
                                       int64_t batch, int64_t q_heads, int64_t kv_heads,
                                       int64_t q_len, int64_t kv_len, int64_t head_dim,
                                       int64_t q_stride_b, int64_t q_stride_h, int64_t q_stride_n,
                                       int64_t o_stride_b, int64_t o_stride_h, int64_t o_stride_n,
                                       int is_causal, double sm_scale, int num_splits, void* workspace,
                                       int64_t workspace_bytes, void* stream) {
  clear_error();
  return run_attn(head_dim, is_causal, batch, q_heads, q_len, kv_len, w8::kQkI8F, num_splits,
                  workspace != nullptr ? workspace_bytes : 0, query, k_i8, value_t, out, lse,
                  nullptr, k_scale, dtype, batch, q_heads, kv_heads, q_len, kv_len, head_dim, q_stride_b, q_stride_h,
                  q_stride_n, kv_heads * kv_len * head_dim, kv_len * head_dim, head_dim, 0, 0, 0, o_stride_b,
                  o_stride_h, o_stride_n, is_causal, sm_scale, num_splits, workspace, workspace_bytes, stream,
                  "sage_attn_i8_fwd_qfused");
}

extern "C" int sage_attn_i8_fwd_qfused_vrows(const void* query, const int8_t* k_i8, const void* value, void* out,
                                             float* lse, const float* k_scale, int dtype,
                                             int64_t batch, int64_t q_heads, int64_t kv_heads,
                                             int64_t q_len, int64_t kv_len, int64_t head_dim,
                                             int64_t q_stride_b, int64_t q_stride_h, int64_t q_stride_n,
                                             int64_t v_stride_b, int64_t v_stride_h, int64_t v_stride_n,
                                             int64_t o_stride_b, int64_t o_stride_h, int64_t o_stride_n,
                                             int is_causal, double sm_scale, int num_splits, void* workspace,
                                             int64_t workspace_bytes, void* stream) {
  clear_error();
  return run_attn(head_dim, is_causal, batch, q_heads, q_len, kv_len, w8::kQkI8FV, num_splits,
                  workspace != nullptr ? workspace_bytes : 0, query, k_i8, value, out, lse,
                  nullptr, k_scale, dtype, batch, q_heads, kv_heads, q_len, kv_len, head_dim, q_stride_b, q_stride_h,
                  q_stride_n, kv_heads * kv_len * head_dim, kv_len * head_dim, head_dim, v_stride_b, v_stride_h,
                  v_stride_n, o_stride_b, o_stride_h, o_stride_n, is_causal, sm_scale, num_splits, workspace,
                  workspace_bytes, stream, "sage_attn_i8_fwd_qfused_vrows");
}

extern "C" int sage_attn_direct_fwd_vrows_bf16(const void* query, const void* key, const void* value, void* out,
                                               float* lse, int64_t batch, int64_t q_heads, int64_t kv_heads,
                                               int64_t q_len, int64_t kv_len, int64_t head_dim,
                                               int64_t q_stride_b, int64_t q_stride_h, int64_t q_stride_n,
                                               int64_t k_stride_b, int64_t k_stride_h, int64_t k_stride_n,
                                               int64_t v_stride_b, int64_t v_stride_h, int64_t v_stride_n,
                                               int64_t o_stride_b, int64_t o_stride_h, int64_t o_stride_n,
                                               int is_causal, double sm_scale, int num_splits, void* workspace,
                                               int64_t workspace_bytes, void* stream) {
  clear_error();
  return run_attn(head_dim, is_causal, batch, q_heads, q_len, kv_len, w8::kQkBf16V, num_splits,
                  workspace != nullptr ? workspace_bytes : 0, query, key, value, out, lse, nullptr,
                  nullptr, SAGE_DTYPE_BF16, batch, q_heads, kv_heads, q_len, kv_len, head_dim, q_stride_b, q_stride_h,
                  q_stride_n, k_stride_b, k_stride_h, k_stride_n, v_stride_b, v_stride_h, v_stride_n, o_stride_b,
                  o_stride_h, o_stride_n, is_causal, sm_scale, num_splits, workspace, workspace_bytes, stream,
                  "sage_attn_direct_fwd_vrows_bf16");
}

extern "C" int sage_attn_i8_fwd_qfused_noalloc(const void* query, const int8_t* k_i8, const void* value_t, void* out,
                                               float* lse, const float* k_scale, int dtype,
                                               int64_t batch, int64_t q_heads, int64_t kv_heads,
                                               int64_t q_len, int64_t kv_len, int64_t head_dim,
                                               int64_t q_stride_b, int64_t q_stride_h, int64_t q_stride_n,
                                               int64_t o_stride_b, int64_t o_stride_h, int64_t o_stride_n,
                                               int is_causal, double sm_scale, int num_splits, void* stream) {
  static const char* const fn = "sage_attn_i8_fwd_qfused_noalloc";
  clear_error();
  // a forced split count must fit the scratch (an automatic plan is chosen within it)
  if (num_splits > 1 && is_causal == 0) {
    int64_t whole = 0;
    int splits = 0;
    const int64_t need = split_plan(true, batch, q_heads, q_len, kv_len, head_dim, 0, num_splits, &whole, &splits);
    if (need < 0) return static_cast<int>(need);
    if (need > kScratchBytes)
      return set_error(SAGE_ERR_UNSUPPORTED, "%s: %d key splits need %lld bytes of scratch, beyond its %lld", fn,
                       num_splits, static_cast<long long>(need), static_cast<long long>(kScratchBytes));
  }
  // only a launch that may split touches the scratch (causal launches, unsplit
  // ones and empty ones never do)
  void* ws = nullptr;
  if (is_causal == 0 && num_splits != 1 && batch > 0 && q_len > 0 && kv_len > 0) {
    ws = scratch_address(fn);
    if (ws == nullptr) return SAGE_ERR_HIP;
  }
  return run_attn(head_dim, is_causal, batch, q_heads, q_len, kv_len, w8::kQkI8F, num_splits,
                  ws != nullptr ? kScratchBytes : 0, query, k_i8, value_t, out, lse,
                  nullptr, k_scale, dtype, batch, q_heads, kv_heads, q_len, kv_len, head_dim, q_stride_b, q_stride_h,
                  q_stride_n, kv_heads * kv_len * head_dim, kv_len * head_dim, head_dim, 0, 0, 0, o_stride_b,
                  o_stride_h, o_stride_n, is_causal, sm_scale, num_splits, ws, ws != nullptr ? kScratchBytes : 0,
                  stream, fn);
}

extern "C" int64_t sage_attn_workspace_bytes(int quantized, int64_t batch, int64_t q_heads, int64_t q_len,
                                             int64_t kv_len, int64_t head_dim, int is_causal, int num_splits) {
  clear_error();
  int64_t whole = 0;
  int splits = 0;
  return split_plan(quantized != 0, batch, q_heads, q_len, kv_len, head_dim, is_causal, num_splits, &whole, &splits);
}

extern "C" int sage_attn_split_plan(int quantized, int64_t batch, int64_t q_heads, int64_t q_len, int64_t kv_len,
                                    int64_t head_dim, int is_causal, int num_splits, int64_t* whole_qblocks,
                                    int* splits) {
  clear_error();
  if (whole_qblocks == nullptr || splits == nullptr)
    return set_error(SAGE_ERR_INVALID_ARG, "sage_attn_split_plan: null output pointer");
  const int64_t r =
      split_plan(quantized != 0, batch, q_heads, q_len, kv_len, head_dim, is_causal, num_splits, whole_qblocks, splits);
  return r < 0 ? static_cast<int>(r) : SAGE_OK;
}

#if SAGE_STAMPS
// Stamps build only: copy `bytes` of the wave records (kStampStride uint64
// fields per wave, block-major) to host memory / clear them.
extern "C" int sage_stamps_read(void* host, size_t bytes) {
  if (bytes > sizeof(sage::g_stamps)) return SAGE_ERR_INVALID_ARG;
  return hipMemcpyFromSymbol(host, HIP_SYMBOL(sage::g_stamps), bytes, 0, hipMemcpyDeviceToHost) == hipSuccess
             ? SAGE_OK
             : SAGE_ERR_HIP;
}
extern "C" int sage_stamps_clear(void) {
  void* ptr = nullptr;
  if (hipGetSymbolAddress(&ptr, HIP_SYMBOL(sage::g_stamps)) != hipSuccess) return SAGE_ERR_HIP;
  return hipMemset(ptr, 0, sizeof(sage::g_stamps)) == hipSuccess ? SAGE_OK : SAGE_ERR_HIP;
}
#endif
