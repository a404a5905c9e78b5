// Compiled host layer of `sageattn` (the reference's sageattention/core.py:40-213):
// shapes and strides, the output / LSE / intermediate allocations from the
// caller's torch allocator, and the launches through the C ABI of
// libsage_mi355x.so, in one Python call, because for the short and
// cross-attention shapes the GPU work of a call (~9 us) is smaller than what
// the same steps cost as Python (~10 us on top of the launches).  A plain
// fp16/bf16 call is checked and dispatched here too (sageattn_plain); any other
// goes through the Python function, which holds the reference's assertions
// with their messages, its fp32 handling and the direct/INT8 dispatch with its
// environment overrides, and enters at sageattn_fwd.
//
// The module calls no HIP API itself: every launch goes through the C ABI on
// the stream handle the caller passes (the current stream of the tensors'
// device), and torch allocates on that same stream, so temporaries released
// here return to the caching allocator in stream order.
#include <c10/core/impl/VirtualGuardImpl.h>
#include <torch/extension.h>

#include <cmath>
#include <cstdint>
#include <cstdlib>
#include <sstream>
#include <string>

#include "sageattn_mi355x.h"

namespace py = pybind11;

namespace {

// A negative status of the C ABI, raised in Python as the exception type the
// package registers (sageattention._capi.SageError: function, status, message).
struct SageStatus {
  const char* fn;
  int code;
  std::string msg;
};

// set by set_error_type(); RuntimeError until then.  A plain reference that is
// never released: a py::object here would be decremented by a static
// destructor after the interpreter has finalised.
PyObject* g_error_type = nullptr;

void check(const char* fn, int rc) {
  if (rc != SAGE_OK) {
    const char* m = sage_last_error();
    throw SageStatus{fn, rc, m != nullptr ? m : ""};
  }
}

// (B, H, N, D) sizes and (b, h, n) strides in elements of a 4-D tensor;
// layout 1 = HND [B,H,N,D], 0 = NHD [B,N,H,D] (reference csrc/attn_gfx11.cu:32-33)
struct Dims {
  int64_t b, h, n, d;
  int64_t sb, sh, sn;
};

Dims bhnd(const at::Tensor& t, int64_t layout) {
  const auto s = t.sizes();
  const auto st = t.strides();
  if (layout == 1) return {s[0], s[1], s[2], s[3], st[0], st[1], st[2]};
  return {s[0], s[2], s[1], s[3], st[0], st[2], st[1]};
}

// t, or a copy that meets the 16-byte access contract (16-byte aligned base,
// batch/head/token strides multiples of 8 elements)
at::Tensor vector_ready(const at::Tensor& t) {
  const auto st = t.strides();
  if (reinterpret_cast<uintptr_t>(t.data_ptr()) % 16 == 0 && st[0] % 8 == 0 && st[1] % 8 == 0 && st[2] % 8 == 0)
    return t;
  return t.is_contiguous() ? t.clone() : t.contiguous();
}

std::string shape_str(const at::Tensor& t) {
  std::ostringstream s;
  s << "(";
  for (int64_t i = 0; i < t.dim(); ++i) s << (i ? ", " : "") << t.size(i);
  s << ")";
  return s.str();
}

// The key-split workspace of a non-causal launch (undefined when it runs
// unsplit); num_splits is already within [0, SAGE_MAX_KV_SPLITS].
at::Tensor split_workspace(bool quantized, const Dims& q, int64_t kv_len, bool causal, int64_t num_splits,
                           const at::Tensor& like, int64_t* bytes) {
  *bytes = 0;
  if (causal) return at::Tensor();
  const int64_t n = sage_attn_workspace_bytes(quantized ? 1 : 0, q.b, q.h, q.n, kv_len, q.d, 0,
                                              static_cast<int>(num_splits));
  if (n < 0) check("sage_attn_workspace_bytes", static_cast<int>(n));
  if (n == 0) return at::Tensor();
  *bytes = n;
  return at::empty({n}, like.options().dtype(at::kByte));
}

void* ptr(const at::Tensor& t) { return t.defined() ? t.data_ptr() : nullptr; }

// INT8 path, fp16 inputs: V is read in place (sage_attn_i8_fwd_qfused_vrows,
// the same output bit for bit) instead of through a V_T pass up to this many
// query rows per kv head.  The pass saved is proportional to the V of a head,
// the cost (twice the LDS reads per P.V MFMA, ~3% of the kernel) to its V times
// the query rows that read it.  Whole call on MI355X, V_T / in place: B1 H16
// S4096 D128 causal 85.6 / 79.2 us, non-causal 118.1 / 114.8; B1 H8 S7000 D64
// causal 69.8 / 67.4; B1 H10 S4096 D64 61.1 / 60.0; H24 S6000 D64 226.0 /
// 224.5; B1 H5 S7423 D128 149.6 / 151.2; Hq32 Hkv8 S16384 D128 causal (65536
// rows) 1554 / 1566.
constexpr int64_t kVRowsMaxQueries = 6144;
constexpr int64_t kVRowsMaxQueriesCausal = 8192;

// Few query rows per kv head against the key range: one pass over K and V in
// place for the rows of all its query heads (sage_attn_few_fwd).  The general
// path quantises K and transposes V first (INT8), pads each query head to 128
// or 256 rows and reads K/V once per query head.  The few-queries kernel packs
// the rows into 32-row tiles, two of them a block ("row group"), and runs one
// 4-wave block per CU (its rings fill the LDS), where the general kernel hosts
// two 128-row blocks a CU at D = 64; every row group reads K/V again (INT8:
// and quantises K again).  Whole call on MI355X, general / few in us, D64 fp16,
// D128 bf16, H the (kv) heads of all batches; the lines below were drawn over
// 4700 shapes of 4 to 1024 kv heads, 1 to 8 query heads each, 1 to 256 queries
// and 32 to 16384 keys.  One pass over K and V pays most where the general path
// makes several: INT8 B8 Hq32 Hkv8 Sq1 Sk8192 D128 226 / 56, Hq64 Hkv8 Sq1
// Sk8192 D64 33 / 25, H8 Sq256 Sk8192 D128 42 / 36.  More row tiles than these
// lose: 16 (Sq512) 46 / 53; direct 4 of 128-row heads (H16 Sk2048 D128) 20 / 22.
constexpr int64_t kFewMaxTiles = 8;
constexpr int64_t kFewMaxTilesDirect = 3;   // direct path, heads of more than kFewShortHead rows
constexpr int64_t kFewShortHead = 64;
constexpr int64_t kCus = 256;               // MI355X

bool few_pays(int64_t b, int64_t hq, int64_t hkv, int64_t sq, int64_t sk, int64_t d, bool direct) {
  if (sq <= 0 || sk <= 0 || sq > 32 * kFewMaxTiles) return false;
  const int64_t group = hq / hkv;
  const int64_t units = group * ((sq + 31) / 32);  // 32-token groups of the heads, never cut by a tile
  const int64_t per_tile = 32 / std::min<int64_t>(sq, 32);
  const int64_t tiles = (units + per_tile - 1) / per_tile;
  if (tiles > (direct && sq > kFewShortHead ? kFewMaxTilesDirect : kFewMaxTiles)) return false;
  // blocks of either kernel and the rounds over the CUs they take (before key splits)
  const int64_t row_groups = tiles > 1 ? (tiles + 1) / 2 : 1;
  const int64_t rows = d == 64 ? 128 : 256, per_cu = d == 64 ? 2 : 1;
  const int64_t q_blocks = group * ((sq + rows - 1) / rows);
  const int64_t few_blocks = b * hkv * row_groups, gen_blocks = b * hkv * q_blocks;
  const int64_t few_rounds = (few_blocks + kCus - 1) / kCus;
  const int64_t gen_rounds = (gen_blocks + per_cu * kCus - 1) / (per_cu * kCus);
  if (direct) {
    // more rounds than the general kernel: H1024 Sq64 Sk64 D64 12.0 / 22.2, Sq96 Sk64 12.8 / 42.0, Sq1 Sk1024 50.5 /
    // 55.0; Sq96 Sk64 D128 31.0 / 65.4.  As many or fewer: H256 Sq1 Sk256 D64 8.5 / 6.6; Hq128 Hkv32 Sq1 Sk1024 D128
    // 29.8 / 11.6
    if (few_rounds > gen_rounds) return false;
    // several row tiles against one key tile of the general kernel (two where the launch has several rounds): half of
    // a block's waves have no key tile.  H64 Sq64 Sk64 D64 5.4 / 6.1, D128 7.9 / 9.0; Sk256 D128 13.0 / 10.9
    if (tiles > 1 && few_rounds == gen_rounds && sk <= (few_rounds > 1 ? 128 : 64)) return false;
    // few ungrouped heads and long keys: the general kernel's key splits fill the CUs as well, and merge faster.  H8
    // Sq1 Sk4096 D64 11.5 / 14.2, Sq64 Sk1024 10.3 / 11.2; H64 Sq64 Sk1024 15.8 / 14.1; H8 Sq64 Sk4096 D128 18.3 / 22.2
    if (group == 1 && gen_blocks <= (d == 64 ? 32 : 8) &&
        sk > (d == 64 ? (tiles > 1 ? 1000 : 2000) : (tiles > 1 ? 3000 : sk)))
      return false;
  } else {
    // K quantised by each of 4 row groups, and more rounds: H128 Sq256 Sk2048 D128 89 / 102; Hq1024 Hkv256 Sq64 Sk512
    // D64 36 / 51.  Two row groups: from 4 times the rounds, H512 Sq128 Sk512 D64 34 / 57, H256 Sk2048 D128 125 / 100
    if (row_groups > 2 && few_rounds > gen_rounds) return false;
    if (row_groups == 2 && few_rounds >= 4 * gen_rounds) return false;
    // ... in one round, where the general kernel reads K/V half as often and the keys are long: H64 Sq256 Sk8192 D128
    // 146 / 184, Sk2048 60 / 55
    if (row_groups > 2 && row_groups >= 2 * q_blocks && sk >= 4096 && 2 * few_blocks >= kCus) return false;
    // little K and V and few query heads in all: the merge of up to 32 key splits outweighs the quantisation pass.  H4
    // Sq1 Sk8192 D64 20.7 / 23.7, Sq128 22.4 / 29.5; H4 Sq1 Sk5000 19.0 / 16.2, Hq64 Hkv8 Sq1 Sk8192 33.2 / 24.7
    if (d == 64 && sk > 6144 && few_blocks * sk <= 65536 && gen_blocks <= 16) return false;
  }
  return true;
}

bool few_queries(const Dims& q, const Dims& k, const Dims& v, bool direct) {
  if (!few_pays(q.b, q.h, k.h, q.n, k.n, q.d, direct)) return false;
  constexpr int64_t kPastEnd = 24 * 32;  // keys past the last that the kernel's loads address (they read as zero)
  return k.sn >= q.d && v.sn >= q.d && (k.n + kPastEnd) * k.sn * 2 <= UINT32_MAX &&
         (k.n + kPastEnd) * v.sn * 2 <= UINT32_MAX && q.b * q.h <= INT32_MAX / SAGE_FEW_MAX_ROWS;
}

// Direct path, bf16 inputs: whether the kernel reads V in place.  Every block
// then converts its V tiles to fp16, about 24 (D = 64) or 30 (D = 128) ns per
// million query-key pairs of the launch; the V_T pass saved is a launch and
// twice V's bytes, about 1.9 us + 0.35 us per MB of V.  Fitted to 630 shapes of
// 256 to 8192 queries and 77 to 6144 keys (the side taken is at most 3%
// slower).  Whole call on MI355X, V_T / in place in us: D128 H16 Sq4096 Sk512
// 27.9 / 25.0, causal H32 S2048 58.4 / 52.0; D64 H20 S1024 17.2 / 14.7, causal
// H32 S4096 90.7 / 83.1; H32 Sq5529 Sk6144 296 / 315, Hq32 Hkv8 290 / 312,
// causal S5000 210 / 217, B2 Hq32 Hkv4 Sq8192 Sk2048 298 / 323.  (fp16 needs no
// conversion and is at most 1.5% slower in place.)
bool bf16_v_in_place(int64_t b, int64_t hq, int64_t hkv, int64_t sq, int64_t sk, int64_t d, bool causal) {
  const double n = static_cast<double>(std::min(sq, sk)), rows = static_cast<double>(sq), keys = static_cast<double>(sk);
  const double pairs = causal ? n * (n + 1) / 2 + (rows - n) * keys : rows * keys;  // of a head
  const double convert_us = static_cast<double>(b * hq) * pairs * (d == 64 ? 24e-9 : 30e-9);
  const double pass_us = 1.9 + 0.35e-6 * static_cast<double>(b * hkv * sk * d * 2);
  return convert_us < pass_us;
}

py::object sageattn_fwd(at::Tensor q, at::Tensor k, at::Tensor v, int64_t layout, bool is_causal, double sm_scale,
                        bool return_lse, bool smooth_k, bool direct, int64_t num_splits, int64_t stream_handle) {
  if (q.dim() != 4 || k.dim() != 4 || v.dim() != 4) throw py::value_error("q, k and v must be 4-D tensors");
  if (num_splits < 0 || num_splits > SAGE_MAX_KV_SPLITS) {
    std::ostringstream s;
    s << "num_splits must be in [0, " << SAGE_MAX_KV_SPLITS << "], got " << num_splits;
    throw py::value_error(s.str());
  }
  q = vector_ready(q);
  k = vector_ready(k);
  v = vector_ready(v);
  const Dims qd = bhnd(q, layout);
  Dims kd = bhnd(k, layout);
  if (k.sizes() != v.sizes() || kd.b != qd.b || kd.d != qd.d)
    throw py::value_error("incompatible shapes q=" + shape_str(q) + " k=" + shape_str(k) + " v=" + shape_str(v));
  if (qd.h % kd.h != 0)
    throw py::value_error("number of query heads (" + std::to_string(qd.h) + ") must be a multiple of kv heads (" +
                          std::to_string(kd.h) + ")");
  const Dims vd = bhnd(v, layout);
  const int dtype = q.scalar_type() == at::kBFloat16 ? SAGE_DTYPE_BF16 : SAGE_DTYPE_F16;
  void* stream = reinterpret_cast<void*>(stream_handle);
  const int64_t B = qd.b, Hq = qd.h, Sq = qd.n, D = qd.d, Hkv = kd.h, Sk = kd.n;
  const int64_t np = sage_v_layout_padded_len(Sk);

  at::Tensor o = at::empty_like(q);
  const Dims od = bhnd(o, layout);
  at::Tensor lse;
  if (return_lse) lse = at::empty({B, Hq, Sq}, q.options().dtype(at::kFloat));

  if (!is_causal && num_splits == 0 && !(smooth_k && !direct) && few_queries(qd, kd, vd, direct)) {
    const int64_t ws_bytes = sage_attn_few_workspace_bytes(B, Hq, Hkv, Sq, Sk, D);
    if (ws_bytes < 0) check("sage_attn_few_workspace_bytes", static_cast<int>(ws_bytes));
    at::Tensor ws;
    if (ws_bytes > 0) ws = at::empty({ws_bytes}, q.options().dtype(at::kByte));
    check("sage_attn_few_fwd",
          sage_attn_few_fwd(direct ? 0 : 1, q.data_ptr(), k.data_ptr(), v.data_ptr(), o.data_ptr(),
                            static_cast<float*>(ptr(lse)), dtype, B, Hq, Hkv, Sq, Sk, D, qd.sb, qd.sh, qd.sn, kd.sb,
                            kd.sh, kd.sn, vd.sb, vd.sh, vd.sn, od.sb, od.sh, od.sn, sm_scale, ptr(ws), ws_bytes,
                            stream));
  } else if (direct) {
    // the direct kernel reads Q and K in place (core.py:141-164); K rows must not overlap
    if (kd.sn < D) {
      k = k.contiguous();
      kd = bhnd(k, layout);
    }
    int64_t ws_bytes = 0;
    at::Tensor ws = split_workspace(false, qd, Sk, is_causal, num_splits, q, &ws_bytes);
    // V read in place: one launch, the same output bit for bit as the V_T path (kept for V rows that overlap or
    // span more than 32-bit offsets, and for bf16 where the conversion costs more).  Whole call on MI355X, V_T / in
    // place: fp16 D64 causal B1 H32 S2048 37.5 / 29.8 us, H20 S3072 50.4 / 43.6, H16 S6144 142 / 133; D64 non-causal B1
    // H20 S1536 23.9 / 19.8, S2304 43.8 / 39.8
    const bool v_rows = vd.sn >= D && (Sk + 5 * SAGE_VT_ALIGN) * vd.sn * 2 <= UINT32_MAX &&
                        (dtype == SAGE_DTYPE_F16 || bf16_v_in_place(B, Hq, Hkv, Sq, Sk, D, is_causal));
    if (v_rows && dtype == SAGE_DTYPE_BF16) {
      check("sage_attn_direct_fwd_vrows_bf16",
            sage_attn_direct_fwd_vrows_bf16(q.data_ptr(), k.data_ptr(), v.data_ptr(), o.data_ptr(),
                                            static_cast<float*>(ptr(lse)), B, Hq, Hkv, Sq, Sk, D, qd.sb, qd.sh, qd.sn,
                                            kd.sb, kd.sh, kd.sn, vd.sb, vd.sh, vd.sn, od.sb, od.sh, od.sn,
                                            is_causal ? 1 : 0, sm_scale, static_cast<int>(num_splits), ptr(ws),
                                            ws_bytes, stream));
    } else if (v_rows && dtype == SAGE_DTYPE_F16) {
      check("sage_attn_direct_fwd_vrows",
            sage_attn_direct_fwd_vrows(q.data_ptr(), k.data_ptr(), v.data_ptr(), o.data_ptr(),
                                       static_cast<float*>(ptr(lse)), dtype, B, Hq, Hkv, Sq, Sk, D, qd.sb, qd.sh,
                                       qd.sn, kd.sb, kd.sh, kd.sn, vd.sb, vd.sh, vd.sn, od.sb, od.sh, od.sn,
                                       is_causal ? 1 : 0, sm_scale, static_cast<int>(num_splits), ptr(ws), ws_bytes,
                                       stream));
    } else {
      // V transform: fp16 V_T [B,Hkv,D,ceil64(Sk)] zero padded (reference core.py:145-152,171-180)
      at::Tensor vt = at::empty({B, Hkv, D, np}, q.options().dtype(at::kHalf));
      check("sage_v_layout",
            sage_v_layout(v.data_ptr(), vt.data_ptr(), dtype, B, Hkv, Sk, D, vd.sb, vd.sh, vd.sn, stream));
      check("sage_attn_direct_fwd",
            sage_attn_direct_fwd(q.data_ptr(), k.data_ptr(), vt.data_ptr(), o.data_ptr(),
                                 static_cast<float*>(ptr(lse)), dtype, B, Hq, Hkv, Sq, Sk, D, qd.sb, qd.sh, qd.sn,
                                 kd.sb, kd.sh, kd.sn, od.sb, od.sh, od.sn, is_causal ? 1 : 0, sm_scale,
                                 static_cast<int>(num_splits), ptr(ws), ws_bytes, stream));
    }
  } else {
    // K quantisation and the V transform in one launch; Q is quantised inside
    // the attention kernel (the q_int8 and q_scale of quant_qk_int8, so the
    // same output, without the int8 Q round trip).  smooth_k: K minus its mean
    // (reference mean_seq, csrc/attn_gfx11.cu:1937-1972), the mean's chunk
    // sums in a launch before, finished by the quantisation blocks.  fp16 V
    // with few enough query rows stays where it is: K quantisation alone, and
    // the kernel that reads V in place
    const bool smooth = smooth_k && Sk > 0;
    const bool v_rows = dtype == SAGE_DTYPE_F16 && !smooth && vd.sn >= D &&
                        Hq / Hkv * Sq <= (is_causal ? kVRowsMaxQueriesCausal : kVRowsMaxQueries) &&
                        (Sk + 5 * SAGE_VT_ALIGN) * vd.sn * 2 <= UINT32_MAX;
    at::Tensor k8 = at::empty({B, Hkv, Sk, D}, q.options().dtype(at::kChar));
    at::Tensor ks = at::empty({B, Hkv, (Sk + SAGE_K_GROUP - 1) / SAGE_K_GROUP}, q.options().dtype(at::kFloat));
    at::Tensor vt;
    if (!v_rows) vt = at::empty({B, Hkv, D, np}, q.options().dtype(at::kHalf));
    if (smooth) {
      const int64_t mb = sage_k_mean_workspace_bytes(B, Hkv, Sk, D);
      if (mb < 0) check("sage_k_mean_workspace_bytes", static_cast<int>(mb));
      at::Tensor mws = at::empty({(std::max<int64_t>(mb, 4) + 3) / 4}, q.options().dtype(at::kFloat));
      check("sage_prep_kv_i8_smooth",
            sage_prep_kv_i8_smooth(k.data_ptr(), v.data_ptr(), nullptr, mws.data_ptr(),
                                   static_cast<int8_t*>(k8.data_ptr()), static_cast<float*>(ks.data_ptr()),
                                   vt.data_ptr(), dtype, B, Hkv, Sk, D, kd.sb, kd.sh, kd.sn, vd.sb, vd.sh, vd.sn,
                                   stream));
    } else if (v_rows) {
      check("sage_quant_qk_i8",
            sage_quant_qk_i8(nullptr, k.data_ptr(), nullptr, nullptr, nullptr, static_cast<int8_t*>(k8.data_ptr()),
                             static_cast<float*>(ks.data_ptr()), dtype, B, Hkv, Hkv, 0, Sk, D, 0, 0, 0, kd.sb, kd.sh,
                             kd.sn, 1.0, stream));
    } else {
      check("sage_prep_kv_i8",
            sage_prep_kv_i8(k.data_ptr(), v.data_ptr(), nullptr, static_cast<int8_t*>(k8.data_ptr()),
                            static_cast<float*>(ks.data_ptr()), vt.data_ptr(), dtype, B, Hkv, Sk, D, kd.sb, kd.sh,
                            kd.sn, vd.sb, vd.sh, vd.sn, stream));
    }
    // return_lse: the reference returns a zero placeholder (core.py:203-211);
    // the fused kernel writes the real log-sum-exp of each row
    int64_t ws_bytes = 0;
    at::Tensor ws = split_workspace(true, qd, Sk, is_causal, num_splits, q, &ws_bytes);
    if (v_rows) {
      check("sage_attn_i8_fwd_qfused_vrows",
            sage_attn_i8_fwd_qfused_vrows(q.data_ptr(), static_cast<const int8_t*>(k8.data_ptr()), v.data_ptr(),
                                          o.data_ptr(), static_cast<float*>(ptr(lse)),
                                          static_cast<const float*>(ks.data_ptr()), dtype, B, Hq, Hkv, Sq, Sk, D,
                                          qd.sb, qd.sh, qd.sn, vd.sb, vd.sh, vd.sn, od.sb, od.sh, od.sn,
                                          is_causal ? 1 : 0, sm_scale, static_cast<int>(num_splits), ptr(ws), ws_bytes,
                                          stream));
    } else {
      check("sage_attn_i8_fwd_qfused",
            sage_attn_i8_fwd_qfused(q.data_ptr(), static_cast<const int8_t*>(k8.data_ptr()), vt.data_ptr(),
                                    o.data_ptr(), static_cast<float*>(ptr(lse)),
                                    static_cast<const float*>(ks.data_ptr()), dtype, B, Hq, Hkv, Sq, Sk, D, qd.sb,
                                    qd.sh, qd.sn, od.sb, od.sh, od.sn, is_causal ? 1 : 0, sm_scale,
                                    static_cast<int>(num_splits), ptr(ws), ws_bytes, stream));
    }
  }
  if (return_lse) return py::make_tuple(o, lse);
  return py::cast(o);
}

// The reference's choice between the direct and the INT8 path with its default
// thresholds (sageattention/core.py:113-139; core.use_direct_path has the
// environment overrides too).
bool default_direct(int64_t head_dim, int64_t q_len, int64_t kv_len, bool causal, bool hnd) {
  if (head_dim == 64) {
    if (causal || q_len < kv_len) return kv_len <= 6144;
    return kv_len <= (hnd ? 2048 : 3072);
  }
  return kv_len <= (q_len * 2 < kv_len ? 4096 : 2048);
}

// The whole call where nothing is unusual: fp16/bf16 tensors that pass every
// check of sageattn on the current device, and none of its environment
// variables set.  None otherwise, and the Python function goes through its
// steps (and raises what fails).  Those steps cost 3.5 us a call, as much as
// the launches of the short calls; these checks 0.3 us.
py::object sageattn_plain(at::Tensor q, at::Tensor k, at::Tensor v, bool hnd, bool is_causal,
                          std::optional<double> sm_scale, bool return_lse, bool smooth_k, int64_t stream_handle) {
  const auto dt = q.scalar_type();
  if ((dt != at::kHalf && dt != at::kBFloat16) || k.scalar_type() != dt || v.scalar_type() != dt || !q.is_cuda() ||
      k.device() != q.device() || v.device() != q.device() || q.dim() != 4 || k.dim() != 4 || v.dim() != 4)
    return py::none();
  const int64_t d = q.size(3);
  if ((d != 64 && d != 128) || q.stride(3) != 1 || k.stride(3) != 1 || v.stride(3) != 1 || q.stride(0) % 8 != 0 ||
      q.stride(1) % 8 != 0 || q.stride(2) % 8 != 0)
    return py::none();
  for (const char* name :
       {"SAGEATTN_KV_SPLITS", "SAGEATTN_DIRECT_THRESHOLD_D64", "SAGEATTN_DIRECT_THRESHOLD_D64_CAUSAL",
        "SAGEATTN_DIRECT_THRESHOLD_D64_CROSS", "SAGEATTN_DIRECT_THRESHOLD_D128", "SAGEATTN_DIRECT_THRESHOLD_D128_CROSS"})
    if (std::getenv(name) != nullptr) return py::none();
  if (c10::impl::VirtualGuardImpl(c10::DeviceType::CUDA).getDevice().index() != q.device().index()) return py::none();
  const int seq = hnd ? 2 : 1;
  const bool direct = default_direct(d, q.size(seq), k.size(seq), is_causal, hnd);
  return sageattn_fwd(q, k, v, hnd ? 1 : 0, is_causal, sm_scale ? *sm_scale : std::pow(static_cast<double>(d), -0.5),
                      return_lse, smooth_k, direct, 0, stream_handle);
}

}  // namespace

PYBIND11_MODULE(TORCH_EXTENSION_NAME, m) {
  m.doc() = "Compiled host layer of sageattn over the libsage_mi355x C ABI";
  m.def("abi_version", []() { return sage_abi_version(); });
  m.def("set_error_type", [](py::object t) {
    PyObject* old = g_error_type;
    g_error_type = t.inc_ref().ptr();
    Py_XDECREF(old);
  });
  m.def("sageattn_fwd", &sageattn_fwd, py::arg("q"), py::arg("k"), py::arg("v"), py::arg("tensor_layout"),
        py::arg("is_causal"), py::arg("sm_scale"), py::arg("return_lse"), py::arg("smooth_k"), py::arg("direct"),
        py::arg("num_splits"), py::arg("stream"));
  m.def("sageattn_plain", &sageattn_plain, py::arg("q"), py::arg("k"), py::arg("v"), py::arg("hnd"),
        py::arg("is_causal"), py::arg("sm_scale"), py::arg("return_lse"), py::arg("smooth_k"), py::arg("stream"));
  m.def("few_pays", &few_pays, py::arg("batch"), py::arg("q_heads"), py::arg("kv_heads"), py::arg("q_len"),
        py::arg("kv_len"), py::arg("head_dim"), py::arg("direct"));
  m.def("bf16_v_in_place", &bf16_v_in_place, py::arg("batch"), py::arg("q_heads"), py::arg("kv_heads"), py::arg("q_len"),
        py::arg("kv_len"), py::arg("head_dim"), py::arg("is_causal"));
  m.def("default_direct", &default_direct, py::arg("head_dim"), py::arg("q_len"), py::arg("kv_len"),
        py::arg("is_causal"), py::arg("hnd"));
  py::register_exception_translator([](std::exception_ptr p) {
    try {
      if (p) std::rethrow_exception(p);
    } catch (const SageStatus& e) {
      if (g_error_type != nullptr && g_error_type != Py_None) {
        py::object type = py::reinterpret_borrow<py::object>(g_error_type);
        py::object err = type(e.fn, e.code, e.msg);
        PyErr_SetObject(g_error_type, err.ptr());
      } else {
        PyErr_SetString(PyExc_RuntimeError, (std::string(e.fn) + ": " + e.msg).c_str());
      }
    }
  });
}
