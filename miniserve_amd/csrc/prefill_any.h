// Chunked prefill for the calls the copying prefill kernel (prefill_mfma.h) does not take:
// an fp32 query, head sizes other than 64 and 128, pages of any length, rows off 16-byte
// boundaries, and every (query, cache) type pair. Matrix cores throughout.
//
// Work split: a workgroup owns 128 query rows of one (sequence, KV head), 32 rows a wave, as
// the copying kernel does (same tasks, same stream-K shares and fold), and NG key groups of 4
// waves take alternate key steps, so that two waves share a SIMD where the head size leaves
// registers and LDS for it (NG = 2 up to 128 dims, else 1). A step of KS keys is loaded by
// the group's threads into registers one step ahead, converted to the query type and
// written to the group's other LDS buffer: one barrier a step.
//
// fp32: S^T and O^T on v_mfma_f32_32x32x2_f32 (64 cycles for 4096 FLOP, 157 TFLOP/s a chip),
// which bounds the kernel: at 128 dims a 32-key step holds 8192 such cycles a wave against
// about 260 of LDS reads and 1000 of softmax. Measured on 2 x 512 queries over 4.6k keys
// (H28/KVH4/D128, 63.9 GFLOP): 579 us with the fold's 11, 110 TFLOP/s, the matrix unit busy in
// 71 % of the kernel's cycles, no bank conflicts.
// The decode partition kernel, which took these calls before at 16 rows a tile and re-reads
// K and V for every tile, measured 913 us. Tried and not kept: two 4-wave workgroups a CU
// instead of two key groups (584 us, twice the partials); group 1 half a step behind group 0
// (741-926 us: a second copy of the loop's products spills); wave priority for either group
// or for the scores, and K operands read a product group ahead (576-581 us).
//
// 16-bit types: v_mfma_f32_32x32x16. The weights are kept in two operands of the query type,
// P = hi + lo, so that P V is summed over products as exact as the result's rounding needs (the
// generic kernel's weights are fp32): 15 to 16 significant bits in bf16, 2^-7 of the result's
// own rounding; 21 or more in fp16, whose lo is scaled by 2^18 and summed on its own, so that a
// weight is held to 2^-42 of the row's largest rather than to fp16's smallest step, 2^-24 (a row
// whose largest weight meets a zero value is made of the small ones). hi is rounded down and lo
// gets 2^-24 of the weight on top, so that neither is below 0 nor is lo 0 beside a weight: an
// infinite value then gives an infinite result, not the NaN of inf - inf or inf * 0. 256 queries
// over 512 to 2304 keys (H24/KVH8/D96 bf16): 30 us against the generic kernel's 182; 4 x 256
// queries over 4096 keys (H32/KVH8/D256): 0.31 ms in bf16, 0.32 in fp16, against 7.5.
//
// Lane layout (both): lane (cc = l % 32, hh = l / 32) holds query row cc. Register v of a
// 32-key score tile is key (v & 3) + 8 (v >> 2) + 4 hh; register v of output tile t is dim
// 32 t + (v & 3) + 8 (v >> 2) + 4 hh. In fp32 a score register is itself the B operand of
// the product with V rows (v & 3) + 8 (v >> 2) and the same + 4.
#pragma once

#include "prefill_mfma.h"

namespace msattn {

// Tasks a stream-K launch of this kernel may hold (its list sits in LDS beside the buffers).
constexpr int kPaSkMaxTasks = 1024;

__host__ __device__ constexpr int pa_capacity(int D) {  // compiled head sizes
  return D <= 32 ? 32 : D <= 64 ? 64 : D <= 96 ? 96 : D <= 128 ? 128 : D <= 192 ? 192 : 256;
}
__host__ __device__ constexpr int pa_groups(int DP) { return DP <= 128 ? 2 : 1; }

// NE elements of a cache row (one 16-byte chunk once converted to T): held as loaded.
template <typename T, typename KT> struct PaChunk {
  static constexpr int NE = 16 / static_cast<int>(sizeof(T));
  static constexpr int NWD = NE * static_cast<int>(sizeof(KT)) / 4;
  uint32_t w[NWD];
  __device__ void clear() {
#pragma unroll
    for (int i = 0; i < NWD; ++i) w[i] = 0u;
  }
  // VEC: the chunk is whole and aligned for vector loads; else its `valid` leading elements
  // load one by one and the others are zeros.
  template <bool VEC>
  __device__ void load(const KT* p, int valid) {
    if constexpr (VEC) {
      if constexpr (NWD >= 4) {
#pragma unroll
        for (int i = 0; i < NWD / 4; ++i) {
          const uint4 x = reinterpret_cast<const uint4*>(p)[i];
          w[4 * i] = x.x; w[4 * i + 1] = x.y; w[4 * i + 2] = x.z; w[4 * i + 3] = x.w;
        }
      } else if constexpr (NWD == 2) {
        const uint2 x = *reinterpret_cast<const uint2*>(p);
        w[0] = x.x; w[1] = x.y;
      } else {
        w[0] = *reinterpret_cast<const uint32_t*>(p);
      }
    } else {
      constexpr int EB = static_cast<int>(sizeof(KT));
      // (opaque, so that the element masks are compared here and not held through the key loop)
      asm volatile("" : "+v"(valid));
#pragma unroll
      for (int e = 0; e < NE; ++e) {
        if (e < valid) {
          uint32_t bits;
          if constexpr (EB == 4) bits = reinterpret_cast<const uint32_t*>(p)[e];
          else if constexpr (EB == 2) bits = reinterpret_cast<const uint16_t*>(p)[e];
          else bits = reinterpret_cast<const uint8_t*>(p)[e];
          w[(e * EB) / 4] |= bits << (8 * ((e * EB) % 4));
        }
      }
    }
  }
  __device__ void floats(float (&f)[NE]) const {
#pragma unroll
    for (int e = 0; e < NE; ++e) {
      if constexpr (sizeof(KT) == 4) {
        f[e] = __uint_as_float(w[e]);
      } else if constexpr (std::is_same<KT, bf16_t>::value) {
        f[e] = __uint_as_float(e & 1 ? w[e / 2] & 0xffff0000u : w[e / 2] << 16);
      } else if constexpr (std::is_same<KT, _Float16>::value) {
        f[e] = static_cast<float>(__builtin_bit_cast(
            _Float16, static_cast<uint16_t>(e & 1 ? w[e / 2] >> 16 : w[e / 2] & 0xffffu)));
      } else {
        const mf_f32x2 x = e & 2 ? __builtin_amdgcn_cvt_pk_f32_fp8(static_cast<int>(w[e / 4]), true)
                                 : __builtin_amdgcn_cvt_pk_f32_fp8(static_cast<int>(w[e / 4]), false);
        f[e] = e & 1 ? x.y : x.x;
      }
    }
  }
  __device__ uint4 as_query_type() const {
    if constexpr (std::is_same<T, KT>::value) {
      return make_uint4(w[0], w[1], w[2], w[3]);
    } else {
      float f[NE];
      floats(f);
      if constexpr (sizeof(T) == 4)
        return make_uint4(__float_as_uint(f[0]), __float_as_uint(f[1]), __float_as_uint(f[2]),
                          __float_as_uint(f[3]));
      else
        return make_uint4(Pack2<T>::pack(f[0], f[1]), Pack2<T>::pack(f[2], f[3]),
                          Pack2<T>::pack(f[4], f[5]), Pack2<T>::pack(f[6], f[7]));
    }
  }
};

template <typename T>
__device__ __forceinline__ void pa_unpack2(uint32_t w, float& a, float& b) {
  if constexpr (std::is_same<T, bf16_t>::value) {
    a = __uint_as_float(w << 16);
    b = __uint_as_float(w & 0xffff0000u);
  } else {
    const mf_h2 h = __builtin_bit_cast(mf_h2, w);
    a = static_cast<float>(h.x);
    b = static_cast<float>(h.y);
  }
}

// Two weights (at least 0) rounded towards zero to T.
template <typename T>
__device__ __forceinline__ uint32_t pa_pack2_down(float a, float b) {
  if constexpr (std::is_same<T, bf16_t>::value)
    return __builtin_amdgcn_perm(__float_as_uint(b), __float_as_uint(a), 0x07060302u);
  else
    return __builtin_bit_cast(uint32_t, __builtin_amdgcn_cvt_pkrtz(a, b));
}

// Four output elements at o (dims d .. d + 3 of a row of D), as one store where VEC.
template <typename T, bool VEC>
__device__ __forceinline__ void pa_store4(T* o, int d, int D, float x, float y, float z, float w) {
  if constexpr (VEC) {
    if (d + 4 > D) return;  // (D is a multiple of 8)
    if constexpr (sizeof(T) == 4)
      *reinterpret_cast<float4*>(o) = make_float4(x, y, z, w);
    else
      *reinterpret_cast<uint2*>(o) = make_uint2(Pack2<T>::pack(x, y), Pack2<T>::pack(z, w));
    return;
  }
  if (d + 0 < D) Elt<T>::store(o + 0, x);
  if (d + 1 < D) Elt<T>::store(o + 1, y);
  if (d + 2 < D) Elt<T>::store(o + 2, z);
  if (d + 3 < D) Elt<T>::store(o + 3, w);
}

// Stream-K set-up: the work list's task offsets into s_pre[0 .. ntasks] (see the copying
// kernel for the list and its heads), this workgroup's share and its first task. s_tmp:
// THREADS / 64 + 1 words. Every thread calls it.
struct PaShare {
  int begin, end, task, share, head;
};
template <int BROWS, int THREADS, int MAXT>
__device__ __forceinline__ PaShare pa_share(const PrefillParams& p, int* s_pre, int* s_tmp) {
  constexpr int kPer = (MAXT + THREADS - 1) / THREADS;
  constexpr int kNW = THREADS / kWave;
  const int tid = threadIdx.x;
  const int lane = tid & (kWave - 1);
  const int wg = __builtin_amdgcn_readfirstlane(tid / kWave);
  int cnt[kPer];
  int sum = 0;
#pragma unroll
  for (int k = 0; k < kPer; ++k) {
    const int t = tid * kPer + k;
    cnt[k] = t < p.ntasks ? pf_task<BROWS>(p, static_cast<unsigned>(t)).iterations() : 0;
    sum += cnt[k];
  }
  const int incl = wave_inclusive_sum(sum);
  if (lane == kWave - 1) s_tmp[wg] = incl;
  __syncthreads();
  int excl = incl - sum;
  for (int k = 0; k < wg; ++k) excl += s_tmp[k];
#pragma unroll
  for (int k = 0; k < kPer; ++k) {
    const int t = tid * kPer + k;
    if (t < p.ntasks) s_pre[t] = excl;
    excl += cnt[k];
  }
  if (tid == THREADS - 1) s_pre[p.ntasks] = excl;
  if (tid == 0) s_tmp[kNW] = 1;
  __syncthreads();
  // Heads unless every task boundary sits on a share boundary of the list without them.
  const int total0 = s_pre[p.ntasks];
  const int shares0 = pf_sk_shares(p.sk_groups, total0);
  const int q = shares0 > 0 && total0 % shares0 == 0 ? total0 / shares0 : 0;
  bool off = q == 0;
#pragma unroll
  for (int k = 0; k < kPer; ++k) {
    const int t = tid * kPer + k;
    if (t < p.ntasks && q > 0) off = off || s_pre[t] % q != 0;
  }
  if (off) s_tmp[kNW] = 0;  // (any writer stores the same value)
  __syncthreads();
  PaShare s;
  s.head = s_tmp[kNW] ? 0 : p.sk_head;
  if (s.head > 0) {
#pragma unroll
    for (int k = 0; k < kPer; ++k) {
      const int t = tid * kPer + k;
      if (t < p.ntasks) s_pre[t] += s.head * t;
    }
    if (tid == THREADS - 1) s_pre[p.ntasks] += s.head * p.ntasks;
  }
  __syncthreads();
  if (blockIdx.x == 0) {  // for the fold launch: the list, then the head size
    for (int t = tid; t <= p.ntasks; t += THREADS) p.sk_pre[t] = s_pre[t];
    if (tid == 0) p.sk_pre[p.ntasks + 1] = s.head;
  }
  // shares dealt to the XCDs in contiguous runs
  const unsigned i = blockIdx.x;
  s.share = p.sk_groups % kXcds == 0
                ? static_cast<int>((i % kXcds) * static_cast<unsigned>(p.sk_groups / kXcds) + i / kXcds)
                : static_cast<int>(i);
  const int total = __builtin_amdgcn_readfirstlane(s_pre[p.ntasks]);
  pf_sk_range(s.share, total, pf_sk_shares(p.sk_groups, total), &s.begin, &s.end);
  int lo = 0, hi = p.ntasks;  // the task holding s.begin: s_pre[lo] <= s.begin < s_pre[hi]
  while (hi - lo > 1) {
    const int mid = (lo + hi) >> 1;
    if (__builtin_amdgcn_readfirstlane(s_pre[mid]) <= s.begin) lo = mid;
    else hi = mid;
  }
  s.task = lo;
  return s;
}

template <typename T, typename KT, int DP, bool VEC>
__global__ __launch_bounds__(pa_groups(DP) * kPfGroupThreads) void prefill_any_kernel(
    const PrefillParams p) {
  constexpr bool F32 = std::is_same<T, float>::value;
  constexpr int NG = pa_groups(DP);
  constexpr int THREADS = NG * kPfGroupThreads;
  constexpr int GT = kPfGroupThreads;      // threads of a key group
  constexpr int KS = F32 ? 32 : 64;        // keys of a group's step
  constexpr int NT = KS / 32;              // 32-key score tiles of it
  constexpr int SPU = 2 * kPfStep / KS;    // steps of a work-list unit (a key-step pair)
  constexpr int NE = 16 / static_cast<int>(sizeof(T));
  constexpr int CPR = DP / NE;             // 16-byte chunks of a staged row
  constexpr int LPT = KS * CPR / GT;
  static_assert(LPT * GT == KS * CPR, "staging split");
  // Row strides (elements): the operand reads of 8 lanes a cycle fall on distinct banks.
  constexpr int RSK = DP + NE;
  constexpr int RSV = F32 ? DP : DP + 16;
  constexpr int ND = DP / 32;
  constexpr int JD = F32 ? DP / 8 : DP / 16;  // K operand chunks of a lane
  constexpr int WROWS = 32;
  // fp16's rest of a weight, scaled: weights are at most 2^8 (kPfSumBound), a rest 2^-3.
  constexpr float kLoScale = std::is_same<T, _Float16>::value ? 0x1p18f : 1.0f;

  constexpr int kKBytes = KS * RSK * static_cast<int>(sizeof(T));
  constexpr int kVBytes = KS * RSV * static_cast<int>(sizeof(T));
  constexpr int kSlot = kKBytes + kVBytes;
  constexpr int kMerge = NG == 2 ? kPfWaves * kWave * (ND * 64 + 8) : 0;
  constexpr int kBuf = NG * 2 * kSlot;
  __shared__ __attribute__((aligned(256))) unsigned char s_mem[kBuf > kMerge ? kBuf : kMerge];
  __shared__ int64_t s_off[NG][3][KS];   // element offsets of a step's tokens, -1: none
  __shared__ uint64_t s_msk[NG][3];      // bit k: token k has a row
  __shared__ int s_pre[kPaSkMaxTasks + 1];
  __shared__ int s_tmp[THREADS / kWave + 1];

  if (threadIdx.x == 0 && blockIdx.x == 0) {
    p.hdr[kHdrKind] = 2;  // this launch (and its fold) writes the output
    p.hdr[kHdrPart] = 2 * kPfStep;
    p.hdr[kHdrWaves] = THREADS / kWave;
    p.hdr[kHdrResidency] = 1;
  }
  const bool sk = p.sk_groups > 0;
  PaShare share{0, 0, 0, 0, 0};
  if (sk) share = pa_share<kPfRows, THREADS, kPaSkMaxTasks>(p, s_pre, s_tmp);
  const int D = p.head_dim;

  for (int seg = 0;; ++seg) {
    const int tid = static_cast<int>(threadIdx.x);
    const int lane = tid & (kWave - 1);
    const int wg = __builtin_amdgcn_readfirstlane(tid / kWave);
    const int grp = NG == 2 ? wg / kPfWaves : 0;  // key group: steps first + grp, + NG, ...
    const int w = wg - grp * kPfWaves;
    const int gtid = tid - grp * GT;
    const int hh = lane >> 5;
    const int cc = lane & 31;
    int it_lo = 0, it_hi = 1 << 24;  // (2^24 units hold 2^31 keys)
    bool full = true;
    unsigned task;
    if (sk) {
      if (share.task >= p.ntasks || share.begin >= share.end) break;
      const int p0 = __builtin_amdgcn_readfirstlane(s_pre[share.task]) + share.head;
      const int p1 = __builtin_amdgcn_readfirstlane(s_pre[share.task + 1]);
      if (p0 >= share.end) break;
      it_lo = share.begin > p0 ? share.begin - p0 : 0;
      it_hi = (share.end < p1 ? share.end : p1) - p0;
      full = it_lo == 0 && it_hi == p1 - p0;
      task = static_cast<unsigned>(share.task++);
    } else {
      if (seg > 0) break;
      const unsigned i = blockIdx.x;
      task = (i % kXcds) * static_cast<unsigned>(p.xcd_per) + i / kXcds;
      if (task >= static_cast<unsigned>(p.rblocks) * static_cast<unsigned>(p.KVH) *
                      static_cast<unsigned>(p.batch))
        break;  // the grid's tail
    }
    const PfTask t = pf_task<kPfRows>(p, task);
    const int b = t.b, kvh = t.kvh, ctx = t.ctx, row0 = t.row0;

    // This lane's query row and its key range [lo_n, hi_n); the wave's rows all see
    // [wave_lo, wave_hi), and none sees a key outside [any_lo, any_hi).
    const int row = row0 + w * WROWS + cc;
    const bool row_ok = row < p.rows_per_kvh;
    int lo_n = 0, hi_n = 0;
    auto out_row = [&]() {  // (recomputed where needed rather than held through the key loop)
      const int i = row / p.G;
      return (static_cast<int64_t>(b) * p.q_len + i) * p.H + kvh * p.G + (row - i * p.G);
    };
    if (row_ok) {
      const int i = row / p.G;
      const int qpos = ctx - p.q_len + i;
      hi_n = p.causal ? min(ctx, qpos + 1) : ctx;
      lo_n = p.window > 0 ? max(0, qpos - p.window + 1) : 0;
      if (hi_n < lo_n) hi_n = lo_n;
    }
    int wave_lo = 0, wave_hi = 0, any_lo = 0, any_hi = 0;
    {
      const int wr0 = row0 + w * WROWS;
      const int wr1 = min(wr0 + WROWS, p.rows_per_kvh) - 1;
      if (wr1 >= wr0) {
        const int qa = ctx - p.q_len + wr0 / p.G;
        const int qz = ctx - p.q_len + wr1 / p.G;
        wave_hi = p.causal ? min(ctx, qa + 1) : ctx;
        wave_lo = p.window > 0 ? max(0, qz - p.window + 1) : 0;
        any_hi = p.causal ? min(ctx, qz + 1) : ctx;
        any_lo = p.window > 0 ? max(0, qa - p.window + 1) : 0;
      }
    }

    // The query row: B operand chunk j = dims (F32: 8 j + 4 hh .. + 3; else 16 j + 8 hh .. + 7).
    uint4 qb[JD];
    {
      const int i = row_ok ? row / p.G : 0;
      const T* qp = static_cast<const T*>(p.q) +
                    (row_ok ? b * p.q_batch + i * p.q_token + (kvh * p.G + (row - i * p.G)) * p.q_head
                            : 0);
#pragma unroll
      for (int j = 0; j < JD; ++j) {
        const int d0 = NE * (2 * j + hh);
        PaChunk<T, T> x;
        x.clear();
        if (row_ok && d0 < D) x.template load<VEC>(qp + d0, D - d0);
        qb[j] = x.as_query_type();
      }
    }
    mf_f32x16 acc[ND];
#pragma unroll
    for (int i = 0; i < ND; ++i) acc[i] = zero16();
    float m_run = -INFINITY, l_run = 0.0f;
    const float masked = p.scale_log2 > 0.0f ? -INFINITY : INFINITY;  // -inf once scaled

    const KT* kbase = static_cast<const KT*>(p.k);
    const KT* vbase = static_cast<const KT*>(p.v);
    const int step0 = t.step_first * (kPfStep / KS);
    const int first = step0 + SPU * it_lo;
    const int end = t.hi_all > t.lo_all
                        ? min(ceil_div(t.hi_all, KS), step0 + SPU * it_hi)
                        : first;

    const int n_it = end > first ? (end - first + NG - 1) / NG : 0;
    const int s_first = first + grp;

    auto kbuf = [&](int s) { return reinterpret_cast<T*>(s_mem + (grp * 2 + s) * kSlot); };
    auto vbuf = [&](int s) { return reinterpret_cast<T*>(s_mem + (grp * 2 + s) * kSlot + kKBytes); };
    // Element offsets of step s's tokens (the group's first wave, a token a lane).
    auto page_id = [&](int s) {
      const int tok = s * KS + lane;
      int phys = -1;
      if (lane < KS && s < end && tok >= t.lo_all && tok < t.hi_all) {
        const int pg = p.bs_shift >= 0 ? tok >> p.bs_shift : tok / p.bs;
        if (pg < p.W) phys = p.table[static_cast<int64_t>(b) * p.W + pg];
      }
      return phys;
    };
    auto put_offsets = [&](int s, int slot, int phys) {
      const int tok = s * KS + lane;
      const bool ok = phys >= 0 && phys < p.num_blocks;
      const int pg = p.bs_shift >= 0 ? tok >> p.bs_shift : tok / p.bs;
      const int64_t off = static_cast<int64_t>(phys) * p.blk_stride +
                          static_cast<int64_t>(tok - pg * p.bs) * p.slot_stride +
                          static_cast<int64_t>(kvh) * p.head_stride;
      if (lane < KS) s_off[grp][slot][lane] = ok ? off : -1;
      const uint64_t m = __ballot(ok);
      if (lane == 0) s_msk[grp][slot] = m;
    };
    // Staged chunks in flight. fp32 holds one tensor's at a time (its products are long enough
    // to cover a load): K's during the scores, then V's.
    PaChunk<T, KT> kst[LPT], vst_own[F32 ? 1 : LPT];
    auto& vst = [&]() -> auto& {
      if constexpr (F32) return kst;
      else return vst_own;
    }();
    // Chunk j of this thread: row chunk_row(j) of the step, dims NE * chunk_col(j) ..
    constexpr bool kRowsPerPass = GT % CPR == 0;
    auto chunk_row = [&](int j) {
      if constexpr (kRowsPerPass) return gtid / CPR + (GT / CPR) * j;
      else return (gtid + GT * j) / CPR;
    };
    auto chunk_col = [&](int j) {
      if constexpr (kRowsPerPass) return gtid % CPR;
      else return (gtid + GT * j) % CPR;
    };
    auto load_rows = [&](int slot, const KT* base, auto& st) {
#pragma unroll
      for (int j = 0; j < LPT; ++j) {
        const int d0 = NE * chunk_col(j);
        const int64_t off = s_off[grp][slot][chunk_row(j)];
        const bool ok = off >= 0 && d0 < D;
        if constexpr (VEC) {
          // No branch: a chunk without a row reads the cache's first one and is dropped.
          st[j].template load<true>(base + (ok ? off + d0 : 0), NE);
          if (!ok) st[j].clear();
        } else {
          st[j].clear();
          if (ok) st[j].template load<false>(base + off + d0, D - d0);
        }
      }
    };
    auto store_rows = [&](T* buf, int stride, const auto& st) {
#pragma unroll
      for (int j = 0; j < LPT; ++j)
        *reinterpret_cast<uint4*>(buf + chunk_row(j) * stride + NE * chunk_col(j)) =
            st[j].as_query_type();
    };

    const int tr_tok = lane >> 2 & 3;                          // transposed V reads: see
    const int tr_dim = 16 * (lane >> 4 & 1) + 4 * (lane & 3);  // the copying kernel
    // Weights of the step whose scores were last taken, as the B operands of P V (fp32: the
    // score registers' own; 16-bit: the two operands of chunk c of 32-key tile tl).
    float pf[F32 ? 16 : 1];
    uint4 ph[F32 ? 1 : NT][2], pl[F32 ? 1 : NT][2];
    // Scores and weights of the group's step s; between() runs once the scores are taken.
    // False: no row of the wave sees a key of the step.
    auto weigh = [&](int s, int slot, int buf, auto&& between) {
      const int t_base = s * KS;
      if (s >= end || t_base >= any_hi || t_base + KS <= any_lo) {
        between();
        return false;
      }
      T* const kb = kbuf(buf);
      const uint64_t msk_v = s_msk[grp][slot];
      const uint32_t mlo = __builtin_amdgcn_readfirstlane(static_cast<uint32_t>(msk_v));
      const uint32_t mhi = __builtin_amdgcn_readfirstlane(static_cast<uint32_t>(msk_v >> 32));
      const bool all = t_base >= wave_lo && t_base + KS <= wave_hi && mlo == 0xffffffffu &&
                       (KS == 32 || mhi == 0xffffffffu);
      mf_f32x16 sv[NT];
#pragma unroll
      for (int tl = 0; tl < NT; ++tl) {
        // Two chains in fp32: a wave's next product does not wait for its last one.
        mf_f32x16 st = zero16(), st1 = zero16();
        auto k_operand = [&](int j) {
          return *reinterpret_cast<const uint4*>(kb + (32 * tl + cc) * RSK + NE * (2 * j + hh));
        };
        uint4 ka_next = k_operand(0);
#pragma unroll
        for (int j = 0; j < JD; ++j) {
          const uint4 ka = ka_next;
          if (j + 1 < JD) ka_next = k_operand(j + 1);
          if constexpr (F32) {
            const uint32_t a[4] = {ka.x, ka.y, ka.z, ka.w};
            const uint32_t q[4] = {qb[j].x, qb[j].y, qb[j].z, qb[j].w};
#pragma unroll
            for (int e = 0; e < 4; e += 2) {
              st = __builtin_amdgcn_mfma_f32_32x32x2f32(__uint_as_float(a[e]), __uint_as_float(q[e]),
                                                        st, 0, 0, 0);
              st1 = __builtin_amdgcn_mfma_f32_32x32x2f32(__uint_as_float(a[e + 1]),
                                                         __uint_as_float(q[e + 1]), st1, 0, 0, 0);
            }
          } else {
            st = Mfma32<T>::mac(ka, qb[j], st);
          }
        }
        if constexpr (F32) st += st1;
        if (!all) {
          const uint32_t mk = (tl == 0 ? mlo : mhi) >> (4 * hh);
#pragma unroll
          for (int v = 0; v < 16; ++v) {
            const int k = (v & 3) + 8 * (v >> 2);
            const int tok = t_base + 32 * tl + 4 * hh + k;
            st[v] = tok >= lo_n && tok < hi_n && (mk >> k & 1u) ? st[v] : masked;
          }
        }
        sv[tl] = st;
      }
      between();
      // Online softmax as in the copying kernel: the weights with the current reference max
      // m, which moves only when a lane's weights sum past 2^8 or no key was seen yet.
      auto move_max = [&](float mt) {
        mt = halves_max(mt);
        const float m_new = fmaxf(m_run, mt);
        const float alpha = m_new != -INFINITY ? __builtin_amdgcn_exp2f(m_run - m_new) : 1.0f;
        l_run *= alpha;
        m_run = m_new;
        if (__any(alpha != 1.0f)) {
#pragma unroll
          for (int i = 0; i < ND; ++i) acc[i] *= alpha;
        }
      };
      auto lane_max = [&] {
        float mt = -INFINITY;
#pragma unroll
        for (int tl = 0; tl < NT; ++tl)
#pragma unroll
          for (int v = 0; v < 16; ++v) mt = fmaxf(mt, sv[tl][v] * p.scale_log2);
        return mt;
      };
      float pr[NT][16];
      float psum;
      auto weights = [&]() {
        const float m_use = m_run != -INFINITY ? m_run : 0.0f;
        float s0 = 0.0f, s1 = 0.0f;
#pragma unroll
        for (int tl = 0; tl < NT; ++tl)
#pragma unroll
          for (int v = 0; v < 16; v += 2) {
            pr[tl][v] = __builtin_amdgcn_exp2f(fmaf(sv[tl][v], p.scale_log2, -m_use));
            pr[tl][v + 1] = __builtin_amdgcn_exp2f(fmaf(sv[tl][v + 1], p.scale_log2, -m_use));
            s0 += pr[tl][v];
            s1 += pr[tl][v + 1];
          }
        psum = s0 + s1;
      };
      weights();
      if (__builtin_expect(__any(!(psum <= kPfSumBound) || m_run == -INFINITY), 0)) {
        move_max(lane_max());
        weights();
      }
      l_run += psum;
      if constexpr (F32) {
#pragma unroll
        for (int v = 0; v < 16; ++v) pf[v] = pr[0][v];
      } else {
#pragma unroll
        for (int tl = 0; tl < NT; ++tl)
#pragma unroll
          for (int c2 = 0; c2 < 2; ++c2) {
            uint32_t hi[4], lo[4];
#pragma unroll
            for (int k = 0; k < 4; ++k) {
              const float x = pr[tl][8 * c2 + 2 * k], y = pr[tl][8 * c2 + 2 * k + 1];
              hi[k] = pa_pack2_down<T>(x, y);
              float a, c;
              pa_unpack2<T>(hi[k], a, c);
              lo[k] = Pack2<T>::pack(fmaf(x - a, kLoScale, x * (kLoScale * 0x1p-24f)),
                                     fmaf(y - c, kLoScale, y * (kLoScale * 0x1p-24f)));
            }
            ph[tl][c2] = make_uint4(hi[0], hi[1], hi[2], hi[3]);
            pl[tl][c2] = make_uint4(lo[0], lo[1], lo[2], lo[3]);
          }
      }
      return true;
    };
    // O^T += V^T P^T with those weights, V in LDS buffer buf.
    auto add_values = [&](int buf) {
      T* const vb = vbuf(buf);
      if constexpr (F32) {
        // A step's 32 keys are summed on their own and then added to the running output: a
        // chain of 16 products and one add a step, where one chain over the whole context
        // would round every pair of keys against the output so far.
        const float* vr = reinterpret_cast<const float*>(vb) + 4 * hh * RSV + cc;
        constexpr int NC = ND % 2 == 0 ? 2 : 1;  // dim tiles summed side by side
#pragma unroll
        for (int i = 0; i < ND; i += NC) {
          mf_f32x16 o[NC];
#pragma unroll
          for (int c = 0; c < NC; ++c) o[c] = zero16();
#pragma unroll
          for (int v = 0; v < 16; ++v) {
#pragma unroll
            for (int c = 0; c < NC; ++c)
              o[c] = __builtin_amdgcn_mfma_f32_32x32x2f32(
                  vr[((v & 3) + 8 * (v >> 2)) * RSV + 32 * (i + c)], pf[v], o[c], 0, 0, 0);
          }
#pragma unroll
          for (int c = 0; c < NC; ++c) acc[i + c] += o[c];
        }
      } else {
        auto v_operand = [&](int tl, int c2, int i) {
          uint16_t* lo = reinterpret_cast<uint16_t*>(vb) +
                         (32 * tl + 16 * c2 + 4 * hh + tr_tok) * RSV + 32 * i + tr_dim;
          const uint2 x = __builtin_bit_cast(uint2, __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_s4*)lo));
          const uint2 y = __builtin_bit_cast(
              uint2, __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_s4*)(lo + 8 * RSV)));
          return make_uint4(x.x, x.y, y.x, y.y);
        };
        if constexpr (kLoScale == 1.0f) {
#pragma unroll
          for (int tl = 0; tl < NT; ++tl)
#pragma unroll
            for (int c2 = 0; c2 < 2; ++c2)
#pragma unroll
              for (int i = 0; i < ND; ++i) {
                const uint4 va = v_operand(tl, c2, i);
                acc[i] = Mfma32<T>::mac(va, ph[tl][c2], acc[i]);
                acc[i] = Mfma32<T>::mac(va, pl[tl][c2], acc[i]);
              }
        } else {  // the rests' products on their own, unscaled into the sum
#pragma unroll
          for (int i = 0; i < ND; ++i) {
            mf_f32x16 o = zero16();
#pragma unroll
            for (int tl = 0; tl < NT; ++tl)
#pragma unroll
              for (int c2 = 0; c2 < 2; ++c2) {
                const uint4 va = v_operand(tl, c2, i);
                acc[i] = Mfma32<T>::mac(va, ph[tl][c2], acc[i]);
                o = Mfma32<T>::mac(va, pl[tl][c2], o);
              }
#pragma unroll
            for (int v = 0; v < 16; ++v) acc[i][v] = fmaf(o[v], 1.0f / kLoScale, acc[i][v]);
          }
        }
      }
    };

    if (n_it > 0) {
      if (w == 0) {
        const int page0 = page_id(s_first), page1 = page_id(s_first + NG);
        put_offsets(s_first, 0, page0);
        put_offsets(s_first + NG, 1, page1);
      }
      __syncthreads();
      load_rows(0, kbase, kst);
      store_rows(kbuf(0), RSK, kst);
      load_rows(0, vbase, vst);
      store_rows(vbuf(0), RSV, vst);
      __syncthreads();
      int slot = 0;  // i % 3
      for (int i = 0; i < n_it; ++i) {
        const int s = s_first + NG * i;
        const int slot1 = slot == 2 ? 0 : slot + 1;
        const int slot2 = slot1 == 2 ? 0 : slot1 + 1;
        const int cur = i & 1;  // the other buffer's readers are past the last barrier
        const bool more = s + NG < end;
        if (more) {
          load_rows(slot1, kbase, kst);
          if constexpr (!F32) load_rows(slot1, vbase, vst);
        }
        int page = -1;
        if (w == 0) page = page_id(s + 2 * NG);
        const bool have = weigh(s, slot, cur, [&] {
          if constexpr (F32) {
            if (more) {
              store_rows(kbuf(cur ^ 1), RSK, kst);
              load_rows(slot1, vbase, vst);
            }
          }
        });
        if (have) add_values(cur);
        if (more) {
          if constexpr (!F32) store_rows(kbuf(cur ^ 1), RSK, kst);
          store_rows(vbuf(cur ^ 1), RSV, vst);
        }
        if (w == 0) put_offsets(s + 2 * NG, slot2, page);
        __syncthreads();
        slot = slot1;
      }
    }

    // Combine the key groups (same rows, same lane layout) through LDS, normalise, store.
    float a0 = 1.0f, a1 = 0.0f, M = m_run, l = l_run;
    float4* const s_acc = reinterpret_cast<float4*>(s_mem);
    float2* const s_ml = reinterpret_cast<float2*>(s_mem + kPfWaves * kWave * ND * 64);
    if constexpr (NG == 2) {
      if (grp == 1) {
#pragma unroll
        for (int i = 0; i < ND; ++i)
#pragma unroll
          for (int q = 0; q < 4; ++q)
            s_acc[((w * ND + i) * 4 + q) * kWave + lane] =
                make_float4(acc[i][4 * q], acc[i][4 * q + 1], acc[i][4 * q + 2], acc[i][4 * q + 3]);
        s_ml[w * kWave + lane] = make_float2(m_run, l_run);
      }
      __syncthreads();
      if (grp == 0) {
        const float2 o = s_ml[w * kWave + lane];
        M = fmaxf(m_run, o.x);
        a0 = M == -INFINITY ? 0.0f : __builtin_amdgcn_exp2f(m_run - M);
        a1 = M == -INFINITY ? 0.0f : __builtin_amdgcn_exp2f(o.x - M);
        l = l_run * a0 + o.y * a1;
      }
    }
    if (grp == 0) {
      l = halves_sum(l);
      auto merged = [&](int i, int q) {
        float4 x = make_float4(acc[i][4 * q], acc[i][4 * q + 1], acc[i][4 * q + 2], acc[i][4 * q + 3]);
        if constexpr (NG == 2) {
          const float4 o = s_acc[((w * ND + i) * 4 + q) * kWave + lane];
          x = make_float4(x.x * a0 + o.x * a1, x.y * a0 + o.y * a1, x.z * a0 + o.z * a1,
                          x.w * a0 + o.w * a1);
        }
        return x;
      };
      if (!full) {  // a share of a split task: its unnormalised partial
        if (row_ok) {
          const int64_t rs = (2 * share.share + (seg == 0 ? 0 : 1)) * kPfRows + (w * WROWS + cc);
          if (hh == 0) *reinterpret_cast<float2*>(p.sk_ml + rs * 2) = make_float2(M, l);
          float* const pa = p.sk_acc + rs * DP + 4 * hh;
#pragma unroll
          for (int i = 0; i < ND; ++i)
#pragma unroll
            for (int q = 0; q < 4; ++q) *reinterpret_cast<float4*>(pa + 32 * i + 8 * q) = merged(i, q);
        }
      } else if (row_ok) {
        const float inv = l > 0.0f ? 1.0f / l : 0.0f;
        T* op = static_cast<T*>(p.out) + out_row() * D;
#pragma unroll
        for (int i = 0; i < ND; ++i)
#pragma unroll
          for (int q = 0; q < 4; ++q) {
            const float4 o = merged(i, q);
            const int d = 32 * i + 8 * q + 4 * hh;
            pa_store4<T, VEC>(op + d, d, D, o.x * inv, o.y * inv, o.z * inv, o.w * inv);
          }
      }
    }
    __syncthreads();  // this task's LDS reads are done before the next task's writes
  }
}

// Fold of the tasks split between shares (prefill_sk_fold_kernel, for rows of any head
// size held DP floats apart): TPR threads a row, 4 dims a thread.
template <typename T, int DP, bool VEC>
__global__ __launch_bounds__(kPfFoldThreads) void prefill_any_fold_kernel(const PrefillParams p) {
  constexpr int TPR = next_pow2(DP / 4);
  constexpr int FR = kPfFoldThreads / TPR;
  constexpr int PER_TASK = kPfRows / FR;
  const unsigned task = blockIdx.x / PER_TASK;
  if (task >= static_cast<unsigned>(p.ntasks)) return;
  const int pv = p.sk_pre[task], p1 = p.sk_pre[task + 1], total = p.sk_pre[p.ntasks];
  const int p0 = pv + p.sk_pre[p.ntasks + 1];
  if (p1 <= p0 || total <= 0) return;
  const int G = pf_sk_shares(p.sk_groups, total);
  const int l_lo = pf_sk_owner(p0, total, G), l_hi = pf_sk_owner(p1 - 1, total, G);
  if (l_lo == l_hi) return;  // one share's: written whole
  const PfTask t = pf_task<kPfRows>(p, task);
  const int j = static_cast<int>(threadIdx.x) % TPR;
  const int r = static_cast<int>(blockIdx.x % PER_TASK) * FR + static_cast<int>(threadIdx.x) / TPR;
  if (r >= t.rows_here) return;  // (the row's TPR threads leave together)
  float M = -INFINITY, L = 0.0f;
  for (int l = l_lo + j; l <= l_hi; l += TPR) {
    const int64_t rs = static_cast<int64_t>(pf_sk_partial_slot(l, pv, total, G)) * kPfRows + r;
    const float2 ml = *reinterpret_cast<const float2*>(p.sk_ml + rs * 2);
    if (ml.x == -INFINITY) continue;
    const float Mn = fmaxf(M, ml.x);
    L = L * __builtin_amdgcn_exp2f(M - Mn) + ml.y * __builtin_amdgcn_exp2f(ml.x - Mn);
    M = Mn;
  }
#pragma unroll
  for (int o = 1; o < TPR; o <<= 1) {
    const float Mo = __shfl_xor(M, o, kWave);
    const float Lo = __shfl_xor(L, o, kWave);
    const float Mn = fmaxf(M, Mo);
    if (Mn != -INFINITY) {
      L = L * __builtin_amdgcn_exp2f(M - Mn) + Lo * __builtin_amdgcn_exp2f(Mo - Mn);
      M = Mn;
    }
  }
  if (4 * j >= DP) return;
  float4 a = make_float4(0.0f, 0.0f, 0.0f, 0.0f);
#pragma unroll 4
  for (int l = l_lo; l <= l_hi; ++l) {
    const int64_t rs = static_cast<int64_t>(pf_sk_partial_slot(l, pv, total, G)) * kPfRows + r;
    const float m = p.sk_ml[rs * 2];
    const float4 v = *reinterpret_cast<const float4*>(p.sk_acc + rs * DP + 4 * j);
    const float w = m == -INFINITY ? 0.0f : __builtin_amdgcn_exp2f(m - M);
    a.x = fmaf(v.x, w, a.x);
    a.y = fmaf(v.y, w, a.y);
    a.z = fmaf(v.z, w, a.z);
    a.w = fmaf(v.w, w, a.w);
  }
  const float inv = L > 0.0f ? 1.0f / L : 0.0f;
  const int row = t.row0 + r;
  const int i = row / p.G;
  const int64_t orow = (static_cast<int64_t>(t.b) * p.q_len + i) * p.H + t.kvh * p.G + (row - i * p.G);
  pa_store4<T, VEC>(static_cast<T*>(p.out) + orow * p.head_dim + 4 * j, 4 * j, p.head_dim, a.x * inv,
                    a.y * inv, a.z * inv, a.w * inv);
}

template <typename T, typename KT, int DP, bool VEC>
hipError_t launch_prefill_any_vec(const PrefillParams& p, hipStream_t stream) {
  const dim3 grid(static_cast<unsigned>(p.sk_groups > 0 ? p.sk_groups : kXcds * p.xcd_per));
  hipLaunchKernelGGL((prefill_any_kernel<T, KT, DP, VEC>), grid, dim3(pa_groups(DP) * kPfGroupThreads), 0,
                     stream, p);
  if (p.sk_groups > 0) {
    const hipError_t e = hipGetLastError();
    if (e != hipSuccess) return e;
    constexpr int per_task = kPfRows / (kPfFoldThreads / next_pow2(DP / 4));
    hipLaunchKernelGGL((prefill_any_fold_kernel<T, DP, VEC>), dim3(static_cast<unsigned>(p.ntasks * per_task)),
                       dim3(kPfFoldThreads), 0, stream, p);
  }
  return hipGetLastError();
}

template <typename T, typename KT, int DP>
hipError_t launch_prefill_any_one(const PrefillParams& p, hipStream_t stream) {
  return p.vec ? launch_prefill_any_vec<T, KT, DP, true>(p, stream)
               : launch_prefill_any_vec<T, KT, DP, false>(p, stream);
}

// Defined in prefill_any_<query type>_<cache type>.hip, a file a pair.
template <typename T, typename KT>
hipError_t launch_prefill_any(const PrefillParams& p, hipStream_t stream);

#define MSATTN_DECLARE_PA(T)                                                          \
  template <> hipError_t launch_prefill_any<T, float>(const PrefillParams&, hipStream_t);    \
  template <> hipError_t launch_prefill_any<T, _Float16>(const PrefillParams&, hipStream_t); \
  template <> hipError_t launch_prefill_any<T, bf16_t>(const PrefillParams&, hipStream_t);   \
  template <> hipError_t launch_prefill_any<T, fp8_t>(const PrefillParams&, hipStream_t);
MSATTN_DECLARE_PA(float)
MSATTN_DECLARE_PA(_Float16)
MSATTN_DECLARE_PA(bf16_t)
#undef MSATTN_DECLARE_PA

#define MSATTN_DEFINE_PA(T, KT)                                                       \
  template <>                                                                         \
  hipError_t launch_prefill_any<T, KT>(const PrefillParams& p, hipStream_t stream) {  \
    switch (pa_capacity(p.head_dim)) {                                                \
      case 32: return launch_prefill_any_one<T, KT, 32>(p, stream);                   \
      case 64: return launch_prefill_any_one<T, KT, 64>(p, stream);                   \
      case 96: return launch_prefill_any_one<T, KT, 96>(p, stream);                   \
      case 128: return launch_prefill_any_one<T, KT, 128>(p, stream);                 \
      case 192: return launch_prefill_any_one<T, KT, 192>(p, stream);                 \
      default: return launch_prefill_any_one<T, KT, 256>(p, stream);                  \
    }                                                                                 \
  }

}  // namespace msattn
