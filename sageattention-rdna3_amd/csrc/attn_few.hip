// Attention of few queries over long key ranges, for gfx950: the rows of all
// query heads of a kv head share one pass over its K and V, read from the
// caller's tensors in place.
//
// The general path spends such a call on work the queries do not need: K
// quantisation and V_T write and re-read the whole K/V (10 bytes per element
// of K and V moved where 4 are read here), every query head of a group reads
// K/V again, and 255 of a 256-row q-block's rows are padding.  At B8 Hq32
// Hkv8 Sq1 Sk8192 D128 bf16 that took 74 us of prologue and 152 us of
// attention, for K/V that a plain copy reads in 55 us; this kernel takes 55.8
// us in all (4.81 TB/s of K and V).
//
// What bounds this kernel: the HBM reads of K and V (INT8 kind: with the
// quantisation of K, ~7 VALU per element, close behind).  Mapping:
//   * the query rows of a kv head (group x Sq) are packed into 32-column
//     tiles, RT of them per block; a column belongs to one Q scale group (32
//     tokens of a head), and no scale group is cut by a tile;
//   * S^T = K.Q^T and O^T = V^T.P^T with the layouts of attn_body.inc (K row m
//     of the operand is key kperm(m), so P feeds the P.V operand from the
//     accumulator), but every wave owns whole 32-key tiles: K and V stream
//     into a wave-private LDS ring, with no barrier in the key loop.  A ring
//     slot is refilled as soon as it has been read, so 4 waves x 32 KB keep
//     about 100 KB a CU in flight;
//   * INT8 kind: the K scale groups are 16 keys, half a tile: a lane holds half
//     a key row, the group's absmax is 4 DPP steps and a lane swap, and the
//     int8 values are made in registers with the quantiser's arithmetic, so
//     they equal sage_prep_kv_i8's;
//   * V is read through the transposing LDS reads and (bf16) converted to fp16
//     per operand;
//   * the 4 waves' partial results merge in LDS; key splits (one block per CU
//     in all) merge in a second small launch.
#include <algorithm>
#include <cfloat>
#include <cmath>

#include "attn_device.h"

namespace sage {
namespace {

constexpr int kFewWaves = 4;
constexpr int kFewThreads = kFewWaves * 64;
constexpr int kTileKeys = 32;
constexpr int kFewMaxSplits = 64;
constexpr float kFewRescale = 8.0f;  // the reference max moves when a tile max exceeds it by more (log2 units)

struct FewParams {
  const void* q;
  const void* k;
  const void* v;
  void* out;
  float* lse;  // [B,Hq,Sq] or null
  int64_t q_sb, q_sh, q_sn, k_sb, k_sh, v_sb, v_sh, o_sb, o_sh, o_sn;
  uint32_t k_pitch, v_pitch;  // bytes between K / V rows
  float sc;                   // direct kind: |fl(sm_scale * log2 e)|
  float qpre;                 // INT8 kind: fl(fl(sm_scale) * log2 e)
  uint32_t q_xor;             // direct kind: 0x80008000 negates Q
  int32_t hq, hkv, sq, sk, group;
  int32_t u_rows;             // rows of a unit: min(Sq, 32)
  int32_t upt;                // units per 32-column tile
  int32_t upb;                // units per query head: ceil(Sq / 32)
  int32_t units;              // units per kv head
  int32_t rgroups;            // row groups (RT tiles each) per kv head
  int32_t tiles;              // key tiles: ceil(Sk / 32)
  int32_t nsplit, items;      // items = B * Hkv * nsplit * rgroups
  FastDiv d_rg, d_split, d_hkv, d_upb, d_u;
  float* part;      // [B*Hkv*rgroups][nsplit][RT*32][D] partial outputs, each normalised
  float* part_lse;  // [B*Hkv*rgroups][nsplit][RT*32]
};

template <int D>
struct FewCfg {
  static constexpr int kRow = 2 * D;                         // bytes of a K or V row
  static constexpr int kTileBytes = kTileKeys * kRow;        // one K or V tile
  static constexpr int kLoads = kTileBytes / 1024;           // its 1 KB LDS-direct loads
  static constexpr int kStages = D == 128 ? 2 : 4;           // 32 KB a wave
  static constexpr int kWaveBytes = kStages * 2 * kTileBytes;
  static constexpr int kInFlight = (2 * kStages - 1) * kLoads;  // loads issued after the tile that is waited for
  static constexpr int kDB = D / 32;
  static_assert(kInFlight < 64, "vmcnt counts to 63");
};

// column c of row tile `tile` of kv head: its query head (within the group) and token; false past the last
__device__ __forceinline__ bool few_row(const FewParams& p, int tile, int c, int& g, int& tok) {
  const int ut = div_by(c, p.d_u);
  const int unit = tile * p.upt + ut;
  g = div_by(unit, p.d_upb);
  tok = (unit - g * p.upb) * 32 + (c - ut * p.u_rows);
  return ut < p.upt && unit < p.units && tok < p.sq;
}

template <int N>
__device__ __forceinline__ void wait_vm() {
  asm volatile("s_waitcnt vmcnt(%0)" ::"n"(N) : "memory");
}

__device__ __forceinline__ float max_abs3(float m, float a, float b) {
  return __builtin_fmaxf(m, __builtin_fmaxf(__builtin_fabsf(a), __builtin_fabsf(b)));
}

template <int D, bool I8, bool BF16, int RT>
__global__ __launch_bounds__(kFewThreads, 1) void few_attn_kernel(FewParams p) {
  using C = FewCfg<D>;
  constexpr int kSteps = I8 ? D / 32 : D / 16;  // QK MFMAs of a tile
  using SAcc = std::conditional_t<I8, int16_t_, float16_t_>;
  __shared__ __align__(16) char smem[kFewWaves * C::kWaveBytes];
  __shared__ float row_stat[kFewWaves][RT][2][64];  // (m, l) per lane; before the loop, row maxima
  static_assert(kFewWaves * RT * C::kDB * 4 * 1024 <= kFewWaves * C::kWaveBytes, "the merge exceeds the ring");

  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int lane = threadIdx.x & 63;
  const int m = lane & 31, hh = lane >> 5;
  // blocks of one XCD take consecutive items (row groups of a key range share its L2)
  int item;
  {
    const int per = p.items / kXcds, rem = p.items % kXcds;
    const int xcd = blockIdx.x % kXcds, slot = blockIdx.x / kXcds;
    item = xcd * per + min(xcd, rem) + slot;
  }
  const int ks_id = div_by(item, p.d_rg);  // (b, hk, split)
  const int rg = item - ks_id * p.rgroups;
  const int bhk = div_by(ks_id, p.d_split);
  const int split = ks_id - bhk * p.nsplit;
  const int b = div_by(bhk, p.d_hkv);
  const int hk = bhk - b * p.hkv;
  const int t0 = div_by(split * p.tiles, p.d_split), t1 = div_by((split + 1) * p.tiles, p.d_split);
  const int kv_end = min(t1 * kTileKeys, p.sk);

  // ---- the wave's tile loads: tiles t0 + wave + 4 i, slot i % kStages; rows
  // past kv_end read as zero through the record count
  const char* kbase = static_cast<const char*>(p.k) + 2 * (static_cast<int64_t>(b) * p.k_sb + hk * p.k_sh);
  const char* vbase = static_cast<const char*>(p.v) + 2 * (static_cast<int64_t>(b) * p.v_sb + hk * p.v_sh);
  const auto rk = make_rsrc(kbase, static_cast<uint32_t>(kv_end - 1) * p.k_pitch + C::kRow);
  const auto rv = make_rsrc(vbase, static_cast<uint32_t>(kv_end - 1) * p.v_pitch + C::kRow);
  char* const ring = smem + wave * C::kWaveBytes;
  uint32_t k_off[C::kLoads], v_off[C::kLoads];
#pragma unroll
  for (int i = 0; i < C::kLoads; ++i) {
    const int byte = i * 1024 + lane * 16;
    const int row = byte / C::kRow, pos = (byte % C::kRow) / 16;
    k_off[i] = static_cast<uint32_t>(row) * p.k_pitch + (pos ^ swz<C::kRow>(row)) * 16;
    v_off[i] = static_cast<uint32_t>(row) * p.v_pitch + (pos ^ swz_vrow<D>(row)) * 16;
  }
  auto issue_k = [&](int i, int slot) __attribute__((always_inline)) {
    const uint32_t key = static_cast<uint32_t>((t0 + wave + kFewWaves * i) * kTileKeys);
#pragma unroll
    for (int x = 0; x < C::kLoads; ++x)
      lds_direct_load16(rk, ring + slot * 2 * C::kTileBytes + x * 1024, k_off[x], key * p.k_pitch);
  };
  auto issue_v = [&](int i, int slot) __attribute__((always_inline)) {
    const uint32_t key = static_cast<uint32_t>((t0 + wave + kFewWaves * i) * kTileKeys);
#pragma unroll
    for (int x = 0; x < C::kLoads; ++x)
      lds_direct_load16(rv, ring + (slot * 2 + 1) * C::kTileBytes + x * 1024, v_off[x], key * p.v_pitch);
  };

  // ---- Q^T operands: lane (m, hh) holds column m of each row tile
  int4_t qf[RT][kSteps];
  float qs[RT];
  {
    uint32_t w[RT][D / 32][8];
#pragma unroll
    for (int rt = 0; rt < RT; ++rt) {
      int g, tok;
      const bool ok = few_row(p, rg * RT + rt, m, g, tok);
      const uint16_t* qp = static_cast<const uint16_t*>(p.q) + static_cast<int64_t>(b) * p.q_sb +
                           static_cast<int64_t>(hk * p.group + g) * p.q_sh + static_cast<int64_t>(tok) * p.q_sn;
#pragma unroll
      for (int x = 0; x < D / 32; ++x) {
#pragma unroll
        for (int h = 0; h < 2; ++h) {
          // INT8: elements 32x + 16hh + 8h .. of the row; direct: 32x + 16h + 8hh ..
          uint4 t = make_uint4(0, 0, 0, 0);
          if (ok) t = *reinterpret_cast<const uint4*>(qp + 32 * x + (I8 ? 16 * hh + 8 * h : 16 * h + 8 * hh));
          w[rt][x][4 * h + 0] = t.x;
          w[rt][x][4 * h + 1] = t.y;
          w[rt][x][4 * h + 2] = t.z;
          w[rt][x][4 * h + 3] = t.w;
        }
      }
    }
#pragma unroll
    for (int i = 0; i < C::kStages; ++i) {
      issue_k(i, i);
      issue_v(i, i);
    }
    if constexpr (I8) {
#pragma clang fp contract(off)
      // absmax of each row, then of its scale group: the u_rows columns of its unit
      const float pre = p.qpre;
#pragma unroll
      for (int rt = 0; rt < RT; ++rt) {
        float mx = 0.0f;
#pragma unroll
        for (int x = 0; x < D / 32; ++x) {
#pragma unroll
          for (int k = 0; k < 8; ++k) {
            const float2_t f = unpack2<BF16>(w[rt][x][k]);
            mx = max_abs3(mx, f.x, f.y);
          }
        }
        row_stat[wave][rt][0][lane] = xhalf_max(mx);
      }
      asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
      const int c0 = min(div_by(m, p.d_u) * p.u_rows, 32 - p.u_rows);
#pragma unroll
      for (int rt = 0; rt < RT; ++rt) {
        float mx = 0.0f;
        for (int c = 0; c < p.u_rows; ++c) mx = __builtin_fmaxf(mx, row_stat[wave][rt][0][c0 + c]);
        const float amax = __builtin_fmaxf(kAmaxFloor, mx * __builtin_fabsf(pre));
        const float inv = 127.0f / amax;
        qs[rt] = amax / 127.0f;
#pragma unroll
        for (int x = 0; x < D / 32; ++x) qf[rt][x] = quant16<BF16>(w[rt][x], inv * pre);
      }
    } else {
#pragma unroll
      for (int rt = 0; rt < RT; ++rt) {
        qs[rt] = p.sc;
#pragma unroll
        for (int x = 0; x < kSteps; ++x) {
          const uint32_t* t = &w[rt][x / 2][4 * (x & 1)];
          qf[rt][x] = int4_t{static_cast<int>(t[0] ^ p.q_xor), static_cast<int>(t[1] ^ p.q_xor),
                             static_cast<int>(t[2] ^ p.q_xor), static_cast<int>(t[3] ^ p.q_xor)};
        }
      }
    }
  }

  float16_t_ o[RT][C::kDB];
  float m_run[RT], l_run[RT];
#pragma unroll
  for (int rt = 0; rt < RT; ++rt) {
    m_run[rt] = -FLT_MAX;  // see the softmax: finite, so that a tile of -inf scores gives p = 0
    l_run[rt] = 0.0f;
#pragma unroll
    for (int db = 0; db < C::kDB; ++db) o[rt][db] = float16_t_{};
  }

  // operand reads.  K: chunk c of LDS row kperm(m); V: the transposing reads of
  // 16-key step t, d block db (lane mapping as in attn_body.inc's OperandMap)
  const int krow = kperm(m);
  const int kread = krow * C::kRow, kswz = swz<C::kRow>(krow);
  uint32_t v_read[C::kDB];
  {
    const int g = lane >> 4, j = lane & 15, u = j >> 2, q = j & 3;
    const int row = 8 * (g >> 1) + u;
#pragma unroll
    for (int db = 0; db < C::kDB; ++db)
      v_read[db] = row * C::kRow + (((4 * db + 2 * (g & 1) + (q >> 1)) ^ swz_vrow<D>(row)) * 16) + 8 * (q & 1);
  }
  auto read_v = [&](const char* vst, int t, int db) __attribute__((always_inline)) {
#if defined(__HIP_DEVICE_COMPILE__)
    const char* a = vst + v_read[db] + 16 * t * C::kRow;
    const uint2 lo = lds_read_tr(a), hi = lds_read_tr(a + 4 * C::kRow);
    uint32_t w[4] = {lo.x, lo.y, hi.x, hi.y};
    if constexpr (BF16) {
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        const float2_t f = unpack2<true>(w[i]);
        w[i] = pack_f16x2(f.x, f.y);
      }
    }
    return make_uint4(w[0], w[1], w[2], w[3]);
#else
    (void)vst, (void)t, (void)db;
    return make_uint4(0, 0, 0, 0);
#endif
  };

  // one key tile from ring slot `slot`; i is the wave's tile count
  auto tile = [&](int i, int slot) __attribute__((always_inline)) {
    const int key0 = (t0 + wave + kFewWaves * i) * kTileKeys;
    const char* kst = ring + slot * 2 * C::kTileBytes;
    const char* vst = kst + C::kTileBytes;
    wait_vm<C::kInFlight>();  // K_i landed
    SAcc s[RT];
    float ks[2] = {1.0f, 1.0f};  // scales of the tile's two key groups
    if constexpr (I8) {
#pragma clang fp contract(off)
      uint32_t w[kSteps][8];
      float mx = 0.0f;
#pragma unroll
      for (int x = 0; x < kSteps; ++x) {
#pragma unroll
        for (int h = 0; h < 2; ++h) {
          const int4_t t = *reinterpret_cast<const int4_t*>(kst + kread + (((4 * x + 2 * hh + h) ^ kswz) * 16));
          w[x][4 * h + 0] = static_cast<uint32_t>(t[0]);
          w[x][4 * h + 1] = static_cast<uint32_t>(t[1]);
          w[x][4 * h + 2] = static_cast<uint32_t>(t[2]);
          w[x][4 * h + 3] = static_cast<uint32_t>(t[3]);
        }
      }
      asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");  // the slot's K is in registers
      issue_k(i + C::kStages, slot);
#pragma unroll
      for (int x = 0; x < kSteps; ++x) {
#pragma unroll
        for (int k = 0; k < 8; ++k) {
          const float2_t f = unpack2<BF16>(w[x][k]);
          mx = max_abs3(mx, f.x, f.y);
        }
      }
      // absmax over the 16 keys of the group: this 16-lane row, both halves
      mx = __builtin_fmaxf(mx, __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(mx), 0xB1, 0xf, 0xf, false)));
      mx = __builtin_fmaxf(mx, __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(mx), 0x4E, 0xf, 0xf, false)));
      mx = __builtin_fmaxf(mx, __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(mx), 0x141, 0xf, 0xf, false)));
      mx = __builtin_fmaxf(mx, __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(mx), 0x140, 0xf, 0xf, false)));
      const float amax = __builtin_fmaxf(kAmaxFloor, xhalf_max(mx));
      const float inv = 127.0f / amax;
      const float scale = amax / 127.0f;
      ks[0] = __int_as_float(__builtin_amdgcn_readlane(__float_as_int(scale), 0));
      ks[1] = __int_as_float(__builtin_amdgcn_readlane(__float_as_int(scale), 16));
#pragma unroll
      for (int x = 0; x < kSteps; ++x) {
        const int4_t a = quant16<BF16>(w[x], inv);
#pragma unroll
        for (int rt = 0; rt < RT; ++rt)
          s[rt] = __builtin_amdgcn_mfma_i32_32x32x32_i8(a, qf[rt][x], x == 0 ? SAcc{} : s[rt], 0, 0, 0);
      }
    } else {
      int4_t a[kSteps];
#pragma unroll
      for (int x = 0; x < kSteps; ++x)
        a[x] = *reinterpret_cast<const int4_t*>(kst + kread + (((2 * x + hh) ^ kswz) * 16));
      asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
      issue_k(i + C::kStages, slot);
#pragma unroll
      for (int x = 0; x < kSteps; ++x) {
#pragma unroll
        for (int rt = 0; rt < RT; ++rt) {
          if constexpr (BF16) {
            s[rt] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(__builtin_bit_cast(bf16x8_t, a[x]),
                                                            __builtin_bit_cast(bf16x8_t, qf[rt][x]),
                                                            x == 0 ? SAcc{} : s[rt], 0, 0, 0);
          } else {
            s[rt] = __builtin_amdgcn_mfma_f32_32x32x16_f16(__builtin_bit_cast(half8_t, a[x]),
                                                           __builtin_bit_cast(half8_t, qf[rt][x]),
                                                           x == 0 ? SAcc{} : s[rt], 0, 0, 0);
          }
        }
      }
    }
    // ---- softmax: register r of lane half hh is key 16(r/8) + 8hh + r%8 of the tile
    const bool ragged = key0 + kTileKeys > p.sk;
    half8_t pf[RT][2];
#pragma unroll
    for (int rt = 0; rt < RT; ++rt) {
      const float sc[2] = {qs[rt] * ks[0], qs[rt] * ks[1]};
      float y[16];
#pragma unroll
      for (int r = 0; r < 16; ++r) y[r] = static_cast<float>(s[rt][r]);
      auto mask = [&]() __attribute__((always_inline)) {
        if (ragged) {
#pragma unroll
          for (int r = 0; r < 16; ++r)
            if (key0 + 16 * (r >> 3) + 8 * hh + (r & 7) >= p.sk) y[r] = -INFINITY;
        }
      };
      mask();
      // the row's largest score: each key group's largest accumulator, scaled (scales are not negative; fmaxf
      // drops the NaN that a scale of 0 makes of a group without a live key)
      float mx = -INFINITY;
#pragma unroll
      for (int g = 0; g < 2; ++g) {
        float gm = y[8 * g];
#pragma unroll
        for (int r = 1; r < 8; ++r) gm = __builtin_fmaxf(gm, y[8 * g + r]);
        mx = __builtin_fmaxf(mx, gm * sc[g]);
      }
      mx = xhalf_max(mx);
      // lazy reference max, as in attn_body.inc: it moves when a row's tile max
      // passes it by more than kFewRescale, so p stays below 2^8.  It starts at
      // the lowest finite value: a row whose scores are all -inf so far (keys
      // masked through K) has p = exp2(-inf) = 0 against it, where -inf would
      // give exp2(-inf + inf), and the first live score moves it
      if (__builtin_amdgcn_ballot_w64(mx > m_run[rt] + kFewRescale) != 0) {
        asm volatile("");  // a real branch
        float m_new = __builtin_fmaxf(m_run[rt], mx);
        if constexpr (I8) m_new = __builtin_ceilf(m_new);
        const float alpha = fast_exp2(m_run[rt] - m_new);
        m_run[rt] = m_new;
        l_run[rt] *= alpha;
#pragma unroll
        for (int db = 0; db < C::kDB; ++db) {
#pragma unroll
          for (int r = 0; r < 16; ++r) o[rt][db][r] *= alpha;
        }
      }
      // score - max in one rounding: scores may be far larger than their differences
#pragma unroll
      for (int r = 0; r < 16; ++r) y[r] = __builtin_fmaf(y[r], sc[r >> 3], -m_run[rt]);
      mask();
      float sum[2] = {0.0f, 0.0f};
      uint32_t pw[8];
#pragma unroll
      for (int r = 0; r < 16; r += 2) {
        const float e0 = fast_exp2(y[r]), e1 = fast_exp2(y[r + 1]);
        sum[0] += e0;
        sum[1] += e1;
        pw[r / 2] = pack_f16x2(e0, e1);
      }
      l_run[rt] += sum[0] + sum[1];
#pragma unroll
      for (int t = 0; t < 2; ++t)
        pf[rt][t] = __builtin_bit_cast(half8_t, make_uint4(pw[4 * t], pw[4 * t + 1], pw[4 * t + 2], pw[4 * t + 3]));
    }
    // ---- O^T += V^T . P^T
    wait_vm<C::kInFlight>();  // V_i landed
#pragma unroll
    for (int t = 0; t < 2; ++t) {
#pragma unroll
      for (int db = 0; db < C::kDB; ++db) {
        const half8_t a = __builtin_bit_cast(half8_t, read_v(vst, t, db));
#pragma unroll
        for (int rt = 0; rt < RT; ++rt)
          o[rt][db] = __builtin_amdgcn_mfma_f32_32x32x16_f16(a, pf[rt][t], o[rt][db], 0, 0, 0);
      }
    }
    asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");  // the slot's V has been read
    issue_v(i + C::kStages, slot);
  };

  const int mine = (t1 - t0 - wave + kFewWaves - 1) / kFewWaves;  // the wave's tiles (may be 0 or less)
  for (int i = 0, slot = 0; i < mine; ++i) {
    tile(i, slot);
    slot = slot == C::kStages - 1 ? 0 : slot + 1;
  }
  wait_vm<0>();  // loads past the end still write this wave's ring
  __syncthreads();

  // ---- merge of the 4 waves: each hands over its O (unnormalised) and row
  // statistics, then merges a quarter of the 16-byte pieces of every row tile.
  // A wave without tiles, or without a live key of the row, has l = 0.
  constexpr int kPieces = C::kDB * 4;  // float4 pieces per lane and row tile
#pragma unroll
  for (int rt = 0; rt < RT; ++rt) {
    row_stat[wave][rt][0][lane] = m_run[rt];
    row_stat[wave][rt][1][lane] = xhalf_sum(l_run[rt]);
#pragma unroll
    for (int x = 0; x < kPieces; ++x) {
      const float16_t_& v = o[rt][x / 4];
      *reinterpret_cast<float4*>(smem + (((wave * RT + rt) * kPieces + x) * 64 + lane) * 16) =
          make_float4(v[4 * (x % 4)], v[4 * (x % 4) + 1], v[4 * (x % 4) + 2], v[4 * (x % 4) + 3]);
    }
  }
  __syncthreads();
#pragma unroll
  for (int rt = 0; rt < RT; ++rt) {
    float mw[kFewWaves], lw[kFewWaves], mm = -INFINITY, l = 0.0f;
#pragma unroll
    for (int w = 0; w < kFewWaves; ++w) {
      lw[w] = row_stat[w][rt][1][lane];
      mw[w] = lw[w] == 0.0f ? -INFINITY : row_stat[w][rt][0][lane];
      mm = __builtin_fmaxf(mm, mw[w]);
    }
    mm = (mm == -INFINITY) ? 0.0f : mm;
#pragma unroll
    for (int w = 0; w < kFewWaves; ++w) {
      mw[w] = fast_exp2(mw[w] - mm);
      l = __builtin_fmaf(lw[w], mw[w], l);
    }
    // no live key: output 0 and LSE -inf; a NaN sum (undefined scores) stays NaN in both
    const float inv = (l == 0.0f) ? 0.0f : 1.0f / l;
    const float lse = row_lse(mm, l);
    int g, tok;
    const bool ok = few_row(p, rg * RT + rt, m, g, tok);
    const int head = hk * p.group + g;
    const int64_t prow = ((static_cast<int64_t>(bhk) * p.rgroups + rg) * p.nsplit + split) * (RT * 32) + rt * 32 + m;
    if (ok && hh == 0 && wave == 0) {
      if (p.nsplit > 1) p.part_lse[prow] = lse;
      else if (p.lse != nullptr) p.lse[(static_cast<int64_t>(b) * p.hq + head) * p.sq + tok] = lse;
    }
#pragma unroll
    for (int y = 0; y < kPieces / kFewWaves; ++y) {
      const int x = wave * (kPieces / kFewWaves) + y;
      float4 acc = make_float4(0.0f, 0.0f, 0.0f, 0.0f);
#pragma unroll
      for (int w = 0; w < kFewWaves; ++w) {
        const float4 v = *reinterpret_cast<const float4*>(smem + (((w * RT + rt) * kPieces + x) * 64 + lane) * 16);
        acc.x = __builtin_fmaf(v.x, mw[w], acc.x);
        acc.y = __builtin_fmaf(v.y, mw[w], acc.y);
        acc.z = __builtin_fmaf(v.z, mw[w], acc.z);
        acc.w = __builtin_fmaf(v.w, mw[w], acc.w);
      }
      const int d = 32 * (x / 4) + 8 * (x % 4) + 4 * hh;
      if (!ok) continue;
      if (p.nsplit > 1) {
        *reinterpret_cast<float4*>(p.part + prow * D + d) = make_float4(acc.x * inv, acc.y * inv, acc.z * inv, acc.w * inv);
      } else {
        uint16_t* op = static_cast<uint16_t*>(p.out) + static_cast<int64_t>(b) * p.o_sb +
                       static_cast<int64_t>(head) * p.o_sh + static_cast<int64_t>(tok) * p.o_sn + d;
        *reinterpret_cast<uint2*>(op) =
            BF16 ? make_uint2(pack_bf16x2(acc.x * inv, acc.y * inv), pack_bf16x2(acc.z * inv, acc.w * inv))
                 : make_uint2(pack_f16x2(acc.x * inv, acc.y * inv), pack_f16x2(acc.z * inv, acc.w * inv));
      }
    }
  }
}

// Merge of the key splits (the formulas of attn_merge_kernel, a NaN LSE
// included): D/4 lanes per query row, which is one (b, query head, token); 8
// splits' loads at a time.
template <int D, bool BF16>
__global__ __launch_bounds__(256) void few_merge_kernel(FewParams p, int rt_rows, int64_t rows, FastDiv d_sq,
                                                        FastDiv d_hq, FastDiv d_group, FastDiv d_upt) {
  constexpr int kLanes = D / 4;
  const int64_t row = static_cast<int64_t>(blockIdx.x) * (256 / kLanes) + threadIdx.x / kLanes;
  if (row >= rows) return;
  const int c = threadIdx.x % kLanes;
  const int bh = div_by(static_cast<int>(row), d_sq);
  const int tok = static_cast<int>(row) - bh * p.sq;
  const int b = div_by(bh, d_hq), head = bh - b * p.hq;
  const int hk = div_by(head, d_group), g = head - hk * p.group;
  // its tile and column (the inverse of few_row)
  const int unit = g * p.upb + tok / 32;
  const int tile = div_by(unit, d_upt);
  const int col = (unit - tile * p.upt) * p.u_rows + tok % 32;
  const int rt_tiles = rt_rows / 32;
  const int rg = tile / rt_tiles;
  const int64_t base = ((static_cast<int64_t>(b) * p.hkv + hk) * p.rgroups + rg) * p.nsplit * rt_rows +
                       (tile - rg * rt_tiles) * 32 + col;
  const float* lp = p.part_lse + base;
  const float* op = p.part + base * D + 4 * c;
  float mx = -INFINITY;
  for (int s = 0; s < p.nsplit; ++s) mx = fmaxf(mx, lp[static_cast<int64_t>(s) * rt_rows]);
  float4 acc = make_float4(0.0f, 0.0f, 0.0f, 0.0f);
  float wsum = 0.0f;
  if (mx == -INFINITY) mx = 0.0f;  // no live key, or only NaN ones: weights 0 or NaN
  for (int s0 = 0; s0 < p.nsplit; s0 += 8) {
    float l[8];
    float4 v[8];
#pragma unroll
    for (int i = 0; i < 8; ++i) {
      const int64_t s = min(s0 + i, p.nsplit - 1);
      l[i] = s0 + i < p.nsplit ? lp[s * rt_rows] : -INFINITY;
      v[i] = *reinterpret_cast<const float4*>(op + s * rt_rows * D);
    }
#pragma unroll
    for (int i = 0; i < 8; ++i) {
      if (s0 + i >= p.nsplit) break;
      const float w = expf(l[i] - mx);
      wsum += w;
      acc.x += w * v[i].x;
      acc.y += w * v[i].y;
      acc.z += w * v[i].z;
      acc.w += w * v[i].w;
    }
  }
  const float inv = wsum == 0.0f ? 0.0f : 1.0f / wsum;
  uint16_t* dst = static_cast<uint16_t*>(p.out) + static_cast<int64_t>(b) * p.o_sb + static_cast<int64_t>(head) * p.o_sh +
                  static_cast<int64_t>(tok) * p.o_sn + 4 * c;
  *reinterpret_cast<uint2*>(dst) =
      BF16 ? make_uint2(pack_bf16x2(acc.x * inv, acc.y * inv), pack_bf16x2(acc.z * inv, acc.w * inv))
           : make_uint2(pack_f16x2(acc.x * inv, acc.y * inv), pack_f16x2(acc.z * inv, acc.w * inv));
  if (c == 0 && p.lse != nullptr) p.lse[row] = wsum == 0.0f ? -INFINITY : mx + logf(wsum);
}

// ---- host side
struct FewPlan {
  int64_t u_rows, upt, upb, units, tiles_q, rt, rgroups, tiles, nsplit, items;
};

// Row packing and key splits of a launch (kv_len > 0, q_len > 0).
FewPlan few_plan(int64_t batch, int64_t q_heads, int64_t kv_heads, int64_t q_len, int64_t kv_len) {
  FewPlan f;
  f.u_rows = std::min<int64_t>(q_len, 32);
  f.upt = 32 / f.u_rows;
  f.upb = cdiv(q_len, 32);
  f.units = q_heads / kv_heads * f.upb;
  f.tiles_q = cdiv(f.units, f.upt);
  f.rt = f.tiles_q > 1 ? 2 : 1;
  f.rgroups = cdiv(f.tiles_q, f.rt);
  f.tiles = cdiv(kv_len, kTileKeys);
  // splits: the least of rounds of one block per CU x (a wave's tiles + the
  // block's fixed time, about kFixedTiles tiles) + the merge
  constexpr double kFixedTiles = 3.0, kMergeTiles = 3.0;
  const int64_t cus = device_cus();
  const int64_t base = batch * kv_heads * f.rgroups;
  double best = 0.0;
  f.nsplit = 1;
  for (int64_t n = 1; n <= kFewMaxSplits && (n == 1 || n * 2 * kFewWaves <= f.tiles); ++n) {
    const double t = static_cast<double>(cdiv(base * n, cus)) *
                         (static_cast<double>(cdiv(cdiv(f.tiles, n), kFewWaves)) + kFixedTiles) +
                     (n > 1 ? kMergeTiles + 0.05 * static_cast<double>(n) : 0.0);
    if (n == 1 || t < best) {
      best = t;
      f.nsplit = n;
    }
  }
  f.items = base * f.nsplit;
  return f;
}

int64_t few_workspace(const FewPlan& f, int64_t batch, int64_t kv_heads, int64_t head_dim) {
  return f.nsplit > 1 ? batch * kv_heads * f.rgroups * f.nsplit * f.rt * 32 * (head_dim + 1) * 4 : 0;
}

template <int D, bool I8, bool BF16>
void few_launch(const FewParams& p, const FewPlan& f, int64_t batch, hipStream_t st) {
  const dim3 grid(static_cast<uint32_t>(f.items)), block(kFewThreads);
  if (f.rt == 1) few_attn_kernel<D, I8, BF16, 1><<<grid, block, 0, st>>>(p);
  else few_attn_kernel<D, I8, BF16, 2><<<grid, block, 0, st>>>(p);
  if (f.nsplit > 1) {
    const int64_t rows = batch * p.hq * p.sq;
    few_merge_kernel<D, BF16><<<dim3(static_cast<uint32_t>(cdiv(rows, 256 / (D / 4)))), dim3(256), 0, st>>>(
        p, static_cast<int>(f.rt * 32), rows, fast_div(p.sq), fast_div(p.hq), fast_div(p.group), fast_div(p.upt));
  }
}

}  // namespace
}  // namespace sage

using namespace sage;

extern "C" int64_t sage_attn_few_workspace_bytes(int64_t batch, int64_t q_heads, int64_t kv_heads, int64_t q_len,
                                                 int64_t kv_len, int64_t head_dim) {
  clear_error();
  if (head_dim != 64 && head_dim != 128)
    return set_error(SAGE_ERR_UNSUPPORTED, "head_dim must be 64 or 128, got %lld", static_cast<long long>(head_dim));
  if (batch < 0 || q_heads <= 0 || kv_heads <= 0 || q_heads % kv_heads != 0 || q_len < 0 || kv_len < 0)
    return set_error(SAGE_ERR_INVALID_ARG, "sage_attn_few_workspace_bytes: bad size");
  if (batch == 0 || q_len == 0 || kv_len == 0) return 0;
  if (batch * q_heads > INT32_MAX / SAGE_FEW_MAX_ROWS || q_len > SAGE_FEW_MAX_ROWS || kv_len > INT32_MAX - 64 * kTileKeys)
    return set_error(SAGE_ERR_UNSUPPORTED, "sage_attn_few_workspace_bytes: sizes beyond the kernel's limits");
  return few_workspace(few_plan(batch, q_heads, kv_heads, q_len, kv_len), batch, kv_heads, head_dim);
}

extern "C" int sage_attn_few_fwd(int quantized, const void* query, const void* key, const void* value, void* out,
                                 float* lse, int dtype, int64_t batch, int64_t q_heads, int64_t kv_heads,
                                 int64_t q_len, int64_t kv_len, int64_t head_dim, int64_t q_stride_b,
                                 int64_t q_stride_h, int64_t q_stride_n, int64_t k_stride_b, int64_t k_stride_h,
                                 int64_t k_stride_n, int64_t v_stride_b, int64_t v_stride_h, int64_t v_stride_n,
                                 int64_t o_stride_b, int64_t o_stride_h, int64_t o_stride_n, double sm_scale,
                                 void* workspace, int64_t workspace_bytes, void* stream) {
  static const char* const fn = "sage_attn_few_fwd";
  clear_error();
  if (dtype != SAGE_DTYPE_F16 && dtype != SAGE_DTYPE_BF16)
    return set_error(SAGE_ERR_INVALID_ARG, "%s: dtype must be SAGE_DTYPE_F16 or SAGE_DTYPE_BF16, got %d", fn, dtype);
  if (head_dim != 64 && head_dim != 128)
    return set_error(SAGE_ERR_UNSUPPORTED, "head_dim must be 64 or 128, got %lld", static_cast<long long>(head_dim));
  if (batch < 0 || q_heads <= 0 || kv_heads <= 0 || q_len < 0 || kv_len <= 0 || workspace_bytes < 0)
    return set_error(SAGE_ERR_INVALID_ARG, "%s: negative or zero size", fn);
  if (q_heads % kv_heads != 0)
    return set_error(SAGE_ERR_INVALID_ARG, "q_heads (%lld) must be a multiple of kv_heads (%lld)",
                     static_cast<long long>(q_heads), static_cast<long long>(kv_heads));
  if (batch == 0 || q_len == 0) return SAGE_OK;
  if (!query || !key || !value || !out) return set_error(SAGE_ERR_INVALID_ARG, "%s: null pointer argument", fn);
  if (!aligned(query, 16) || !aligned(key, 16) || !aligned(value, 16) || !aligned(out, 16) || !aligned(lse, 4))
    return set_error(SAGE_ERR_ALIGNMENT, "%s: query/key/value/out must be 16-byte aligned, lse 4-byte", fn);
  for (int64_t s : {q_stride_b, q_stride_h, q_stride_n, k_stride_b, k_stride_h, v_stride_b, v_stride_h, o_stride_b,
                    o_stride_h, o_stride_n, k_stride_n, v_stride_n}) {
    if (s < 0) return set_error(SAGE_ERR_INVALID_ARG, "%s: strides must be non-negative", fn);
    if (s % 8) return set_error(SAGE_ERR_ALIGNMENT, "%s: strides must be multiples of 16 bytes", fn);
  }
  if (k_stride_n < head_dim || v_stride_n < head_dim)
    return set_error(SAGE_ERR_INVALID_ARG, "%s: K and V rows must not overlap", fn);
  // byte offsets within a head are 32-bit; a wave's loads run up to 5 x 4 tiles past the last
  constexpr int64_t kAhead = 24 * kTileKeys;
  if (batch * q_heads > INT32_MAX / SAGE_FEW_MAX_ROWS || q_len > SAGE_FEW_MAX_ROWS || kv_len > INT32_MAX - 64 * kTileKeys ||
      (kv_len + kAhead) * k_stride_n * 2 > UINT32_MAX || (kv_len + kAhead) * v_stride_n * 2 > UINT32_MAX)
    return set_error(SAGE_ERR_UNSUPPORTED, "%s: sizes beyond the kernel's limits", fn);
  const FewPlan f = few_plan(batch, q_heads, kv_heads, q_len, kv_len);
  const int64_t need = few_workspace(f, batch, kv_heads, head_dim);
  if (need > 0 && (workspace == nullptr || workspace_bytes < need || !aligned(workspace, 16)))
    return set_error(SAGE_ERR_INVALID_ARG, "%s: needs a 16-byte aligned workspace of %lld bytes (got %lld)", fn,
                     static_cast<long long>(need), static_cast<long long>(workspace != nullptr ? workspace_bytes : 0));
  if (f.items * kFewMaxSplits > INT32_MAX || f.tiles * kFewMaxSplits > INT32_MAX)
    return set_error(SAGE_ERR_UNSUPPORTED, "%s: sizes beyond the kernel's limits", fn);

  FewParams p;
  p.q = query;
  p.k = key;
  p.v = value;
  p.out = out;
  p.lse = lse;
  p.q_sb = q_stride_b;
  p.q_sh = q_stride_h;
  p.q_sn = q_stride_n;
  p.k_sb = k_stride_b;
  p.k_sh = k_stride_h;
  p.v_sb = v_stride_b;
  p.v_sh = v_stride_h;
  p.o_sb = o_stride_b;
  p.o_sh = o_stride_h;
  p.o_sn = o_stride_n;
  p.k_pitch = static_cast<uint32_t>(k_stride_n * 2);
  p.v_pitch = static_cast<uint32_t>(v_stride_n * 2);
  const float sc = static_cast<float>(sm_scale) * 1.4426950408889634f;
  p.sc = std::fabs(sc);
  p.qpre = sc;
  p.q_xor = std::signbit(sc) ? 0x80008000u : 0u;
  p.hq = static_cast<int32_t>(q_heads);
  p.hkv = static_cast<int32_t>(kv_heads);
  p.sq = static_cast<int32_t>(q_len);
  p.sk = static_cast<int32_t>(kv_len);
  p.group = static_cast<int32_t>(q_heads / kv_heads);
  p.u_rows = static_cast<int32_t>(f.u_rows);
  p.upt = static_cast<int32_t>(f.upt);
  p.upb = static_cast<int32_t>(f.upb);
  p.units = static_cast<int32_t>(f.units);
  p.rgroups = static_cast<int32_t>(f.rgroups);
  p.tiles = static_cast<int32_t>(f.tiles);
  p.nsplit = static_cast<int32_t>(f.nsplit);
  p.items = static_cast<int32_t>(f.items);
  p.d_rg = fast_div(f.rgroups);
  p.d_split = fast_div(f.nsplit);
  p.d_hkv = fast_div(kv_heads);
  p.d_upb = fast_div(f.upb);
  p.d_u = fast_div(f.u_rows);
  const int64_t prows = f.items * f.rt * 32;
  p.part = f.nsplit > 1 ? static_cast<float*>(workspace) : nullptr;
  p.part_lse = f.nsplit > 1 ? static_cast<float*>(workspace) + prows * head_dim : nullptr;
  hipStream_t st = static_cast<hipStream_t>(stream);
  const bool bf16 = dtype == SAGE_DTYPE_BF16;
  auto launch = [&](auto d) {
    constexpr int D = decltype(d)::value;
    if (quantized != 0) {
      if (bf16) few_launch<D, true, true>(p, f, batch, st);
      else few_launch<D, true, false>(p, f, batch, st);
    } else {
      if (bf16) few_launch<D, false, true>(p, f, batch, st);
      else few_launch<D, false, false>(p, f, batch, st);
    }
  };
  if (head_dim == 128) launch(std::integral_constant<int, 128>{});
  else launch(std::integral_constant<int, 64>{});
  return check_launch(fn);
}
